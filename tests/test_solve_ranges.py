"""The superposition solve on both sides of the range in which its divisions
run without range scaling (the covariance's mean magnitude between 1e-18 and
1e18): chains of ordinary size, of 1e-11 and of 1e-14 A, and rotated copies of
them.  The rotation must be the copy's within 1e-4 (single-precision
coordinates and sums over 120 residues), every residue aligned."""
import numpy as np
import pytest

from gtalign_alpha_amd import synth
from gtalign_alpha_amd.batch import GtaBatch
from gtalign_alpha_amd.capi import default_options
from gtalign_alpha_amd.chunk import Chunk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("factor", [1.0, 1e-11, 1e-14])
def test_solve_ranges(factor):
    rng = np.random.default_rng(5)
    x = synth.chain(77, 120).astype(np.float64)
    x -= x.mean(0)
    q, _ = np.linalg.qr(rng.normal(size=(3, 3)))
    rot = q * np.sign(np.linalg.det(q))
    a, b = (x * factor).astype(np.float32), (x @ rot.T * factor).astype(np.float32)
    qc, rc = Chunk.from_structures([a], ["A" * 120]), Chunk.from_structures([b], ["A" * 120])
    with GtaBatch(0, default_options(), max_qrys=1, max_qry_poss=120, max_refs=1, max_ref_poss=120) as bt:
        bt.TransferQueryPMDataToDevice(qc)
        bt.TransferCPMDataToDevice(rc)
        g = bt.ProcessBlock()
    assert g.alndata[0, 0, 4] == 120 and g.alndata[0, 0, 9] > 0.999
    assert np.abs(g.tfms[0, 0, :9].reshape(3, 3) - rot).max() < 1e-4

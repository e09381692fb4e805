"""Default DP forms of a chunk whose longest fills exceed the device's share:
the strips of those pairs go to workers ahead of the one-wave pairs of the same
launch, or, in the batched form, are taken by its persistent waves before the
queue.  Equal to one wave per pair bit for bit, on every replay."""
import numpy as np
import pytest

from gtalign_alpha_amd import synth
from gtalign_alpha_amd.batch import GtaBatch
from gtalign_alpha_amd.capi import default_options
from gtalign_alpha_amd.chunk import Chunk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batched", [0, 1], ids=["plain", "batched"])
@pytest.mark.parametrize("ss", [0, 1], ids=["", "search-by-ss"])
def test_default_grid_pairs(batched, ss):
    rng = np.random.default_rng(3)
    q = synth.chain(1, 385)                      # 7 groups of rows, one row in the last
    # the longest references hold noisy copies of the query, so that they continue
    tail = [np.concatenate([synth.chain(2 + i, n), synth.rigid_copy(rng, q, 0.8)]) for i, n in enumerate([1615, 1516])]
    refs = sorted(tail + [synth.chain(10 + i, int(n)) for i, n in enumerate(rng.integers(20, 120, 620))],
                  key=len, reverse=True)
    qc, rc = (Chunk.from_structures(xs, [synth.residues(rng, len(x)) for x in xs]) for xs in ([q], refs))
    kw = dict(max_qrys=1, max_qry_poss=qc.nposs, max_refs=rc.nstrs, max_ref_poss=rc.nposs)
    out, grid = [], []
    for forced in (True, False):
        with GtaBatch(0, default_options(batched=batched, addsearchbyss=ss), **kw) as b:
            if forced:
                b.set_dp_buckets(2**60, 2)       # one wave per pair
            b.TransferQueryPMDataToDevice(qc)
            b.TransferCPMDataToDevice(rc)
            out.append([b.ProcessBlock() for _ in range(3)])
            grid.append(b.dp_forms()[0]["grid"])
    assert grid == [0, 2]
    want = out[0][0]
    assert (want.alndata[0, :2] > 0).any()
    for g in out[1]:
        assert np.array_equal(g.alndata, want.alndata)
        assert np.array_equal(g.tfms, want.tfms)
        assert np.array_equal(g.alns, want.alns)

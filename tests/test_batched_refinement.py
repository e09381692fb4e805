"""Batched refinement where the persistent workgroups of 4 and 2 waves take
several pairs each and many refinements end at once because the last fill left
the alignment unchanged: every replay equals the plain form, in which a
workgroup refines one pair, bit for bit."""
import numpy as np
import pytest

from gtalign_alpha_amd import synth
from gtalign_alpha_amd.batch import GtaBatch
from gtalign_alpha_amd.capi import PREC_FP32, PREC_MIXED, default_options
from gtalign_alpha_amd.chunk import Chunk

pytestmark = pytest.mark.gpu


def family_set(nq, nr):
    """nq seed chains and nr noisy rigid copies of them, 30-90 residues."""
    rng = np.random.default_rng(5)
    seeds = [synth.chain(100 + i, int(rng.integers(30, 90))) for i in range(nq)]
    copies = [synth.rigid_copy(rng, seeds[i % nq], 0.2 + 0.4 * (i % 7)) for i in range(nr)]
    return [Chunk.from_structures(xs, [synth.residues(rng, len(x)) for x in xs])
            for xs in (sorted(seeds, key=len, reverse=True), sorted(copies, key=len, reverse=True))]


# up to 64 pairs per CU: 4 waves, 1,024 persistent workgroups; above: 2 waves, 2,048
@pytest.mark.parametrize("prec", [PREC_FP32, PREC_MIXED], ids=["fp32", "mixed"])
@pytest.mark.parametrize("nr", [1000, 2500], ids=["4-waves", "2-waves"])
def test_batched_refinement_of_unchanged_alignments(nr, prec):
    q, r = family_set(8, nr)
    kw = dict(max_qrys=q.nstrs, max_qry_poss=q.nposs, max_refs=r.nstrs, max_ref_poss=r.nposs)
    got = []
    for batched in (0, 1):
        with GtaBatch(0, default_options(precision=prec, batched=batched, prescore=0.0), **kw) as b:
            b.TransferQueryPMDataToDevice(q)
            b.TransferCPMDataToDevice(r)
            got.append([b.ProcessBlock() for _ in range(4 if batched else 1)])
    want = got[0][0]
    for g in got[1]:
        assert np.array_equal(g.alndata, want.alndata)
        assert np.array_equal(g.tfms, want.tfms)
        assert np.array_equal(g.alns, want.alns)

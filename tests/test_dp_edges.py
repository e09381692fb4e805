"""DP fill and walk at the edges of the strip sweep: rows at every remainder
of the strips of 64-256 rows (1-4 rows a lane), columns around the 16-step
blocks, the 64-column loads and the 128-entry ring, walks that leave their
window of 64 rows and 64 columns (references far longer or shorter than the
query), and undefined coordinates first and last."""
import numpy as np
import pytest

from gtalign_alpha_amd import synth
from gtalign_alpha_amd.batch import GtaBatch
from gtalign_alpha_amd.capi import default_options
from gtalign_alpha_amd.chunk import Chunk
from oracle import oracle

pytestmark = pytest.mark.gpu

QLENS = [1, 3, 63, 64, 65, 127, 128, 129, 191, 193, 255, 256, 257, 320, 385, 449, 513]
RLENS = [1, 2, 15, 16, 17, 33, 48, 49, 63, 64, 65, 79, 81, 127, 128, 129, 255, 256, 257, 700]


def chunk(rng, lens):
    xs = [synth.chain(int(rng.integers(1, 2**40)), L) for L in sorted(lens, reverse=True)]
    return Chunk.from_structures(xs, [synth.residues(rng, len(x)) for x in xs])


def check(q, r, tf, got, gap0, gapopen):
    for i in range(q.nstrs):
        for j in range(r.nstrs):
            d02 = float(oracle.d0(int(q.len[i]), int(r.len[j]))["d0"]) ** 2
            _, want = oracle.dp(q.coords(i), r.coords(j), tf[i, j], d02, gapopen, gap0)
            assert np.array_equal(got[i, j], want), (int(q.len[i]), int(r.len[j]))


@pytest.mark.parametrize("undefined", [False, True], ids=["defined", "undefined"])
@pytest.mark.parametrize("gap0,gapopen", [(True, 0.0), (False, -0.6)], ids=["gap0", "gap-0.6"])
@pytest.mark.parametrize("form", ["one-wave", "W-waves", "grid"])
def test_dp_edges(form, gap0, gapopen, undefined):
    rng = np.random.default_rng(11)
    q, r = chunk(rng, QLENS), chunk(rng, RLENS)
    if undefined:
        for c, v in ((q, 1.0e5), (r, -1.0e5)):
            for i in range(0, c.nstrs, 2):
                c.x[int(c.dst[i])] = v
                c.x[int(c.dst[i]) + int(c.len[i]) - 1] = v
    tf = np.zeros((q.nstrs, r.nstrs, 12), np.float32)
    tf[..., :9] = np.eye(3).reshape(-1)
    tf[..., 9:] = rng.normal(scale=2.0, size=tf[..., 9:].shape)
    with GtaBatch(0, default_options(), max_qrys=q.nstrs, max_qry_poss=q.nposs, max_refs=r.nstrs,
                  max_ref_poss=r.nposs) as b:
        # the W-wave and device-wide forms take pairs of >= 2 strips and >= 256 columns
        b.set_dp_buckets(2**60 if form == "one-wave" else 0, 2)
        b.set_dp_grid(1 if form == "grid" else 2)
        b.TransferQueryPMDataToDevice(q)
        b.TransferCPMDataToDevice(r)
        got = b.dp_under(tf, gap0, gapopen)
        forms, _ = b.dp_forms()
    n = {"one-wave": forms["one_wave"], "grid": forms["grid"]}.get(form, forms["w4"] + forms["w8"] + forms["w16"])
    assert n > 0
    check(q, r, tf, got, gap0, gapopen)

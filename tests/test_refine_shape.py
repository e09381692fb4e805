"""The workgroups of the refinement launches (host rule, no device), and the
batched form with more pairs than a persistent grid has workgroups."""
import numpy as np
import pytest

from gtalign_alpha_amd import synth
from gtalign_alpha_amd.batch import GtaBatch, lib
from gtalign_alpha_amd.capi import PREC_FP32, PREC_MIXED, REF_LOG, default_options
from gtalign_alpha_amd.chunk import Chunk

NCU = 256
DPREFINE, LOG = 0, 7


def shape(prec, mode, pairs=1000, maxaln=4000, fits1=1, batched=0):
    out = np.zeros(5, np.int32)
    assert lib().gta_test_refine_shape(prec, mode, NCU, pairs, maxaln, fits1, batched, out.ctypes.data) == 0
    return out.tolist()


@pytest.mark.parametrize("prec", [PREC_FP32, PREC_MIXED])
@pytest.mark.parametrize("mode", range(8))
@pytest.mark.parametrize("pairs", [1, 1000, 100000, 1000000])
def test_persistent_grid_fills_the_device(prec, mode, pairs):
    """16 waves per CU whatever the workgroup size, and in the FP32 forms LDS
    (2 KB a wave and the staged alignment) for all of them."""
    waves, wgs, cap, _, _ = shape(prec, mode, pairs)
    assert waves * wgs == 16 * NCU
    assert mode != LOG or waves == 2            # its steps run in one slot group
    if prec == PREC_FP32 or mode == DPREFINE:
        assert wgs // NCU * (2048 * waves + 24 * cap) <= 160 * 1024
    assert shape(prec, mode, pairs, maxaln=100)[2] == 100


@pytest.mark.parametrize("maxaln,pairs,waves", [
    (47, 256, 1), (47, 64000, 1), (90, 4000, 4), (90, 16000, 2), (90, 64000, 1), (150, 16000, 2), (200, 8000, 4),
    (200, 16000, 2), (200, 64000, 1), (300, 15000, 4), (300, 80000, 1), (1000, 16384, 4), (1000, 16385, 2),
    (1000, 100000, 2), (1000, 800000, 1), (65535, 1, 4), (65535, 262144, 2), (65535, 262145, 1)])
def test_dprefine_waves_follow_length_and_number(maxaln, pairs, waves):
    """Chunks of short chains take small workgroups, however few their pairs."""
    assert shape(PREC_FP32, DPREFINE, pairs, maxaln)[0] == waves
    if waves == 1:                              # never where many alignments exceed its LDS
        assert shape(PREC_FP32, DPREFINE, pairs, maxaln, fits1=0)[0] == (1 if maxaln <= 47 else 2)
    small = maxaln <= 47 and pairs <= 64 * NCU  # a persistent grid of one-wave workgroups only for many pairs
    assert shape(PREC_FP32, DPREFINE, pairs, maxaln, batched=1)[0] == (4 if small else waves)


@pytest.mark.parametrize("prec,maxaln,live,waves", [
    (PREC_FP32, 100, 0, 8), (PREC_FP32, 100, 512, 8), (PREC_FP32, 100, 513, 4), (PREC_FP32, 500, 2560, 8),
    (PREC_FP32, 500, 2561, 4), (PREC_MIXED, 100, 256, 8), (PREC_MIXED, 100, 257, 4), (PREC_MIXED, 211, 900, 4),
    (PREC_MIXED, 650, 1280, 8), (PREC_MIXED, 650, 1281, 4)])
def test_final_waves_follow_the_pairs_left(prec, maxaln, live, waves):
    """Not one size for every chunk: 900 frames of an ensemble fill the CUs
    with workgroups of half the size."""
    for mode in (1, 2, 3, 4):
        assert shape(prec, mode, live, maxaln)[0] == waves
    for mode in (5, 6):                         # FULLA: 768 slots a pair
        assert shape(prec, mode, live, maxaln)[0] == 8


@pytest.mark.gpu
@pytest.mark.parametrize("prec", [PREC_FP32, PREC_MIXED], ids=["fp32", "mixed"])
def test_final_stage_with_both_workgroups(prec):
    """700 copies of a chain (4-wave workgroups in the plain form, 8-wave ones
    in the batched form) against the same copies in two chunks of 350 and, in
    four, of 175."""
    rng = np.random.default_rng(9)
    x = synth.chain(41, 97)
    rs = [synth.rigid_copy(rng, x, 0.2 + 0.3 * (i % 8)) for i in range(700)]
    q, r = Chunk.from_structures([x], ["A" * 97]), Chunk.from_structures(rs, ["A" * 97] * 700)
    want = batched_equals_plain(q, r, precision=prec)
    live = int((want.alndata[..., 4] > 0).sum())
    assert shape(prec, 2, live, 97)[0] == 4 and shape(prec, 2, 175, 97)[0] == 8
    for n in (350, 175):
        for k in range(0, 700, n):
            part = r.subset(range(k, k + n))
            with GtaBatch(0, default_options(precision=prec), max_qrys=1, max_qry_poss=97, max_refs=n,
                          max_ref_poss=part.nposs) as b:
                b.TransferQueryPMDataToDevice(q)
                b.TransferCPMDataToDevice(part)
                g = b.ProcessBlock()
            assert np.array_equal(g.alndata, want.alndata[:, k:k + n])
            assert np.array_equal(g.tfms, want.tfms[:, k:k + n])


@pytest.mark.parametrize("mode", range(8))
@pytest.mark.parametrize("pairs", [1, 1000, 100000, 1000000])
def test_split_workgroups_leave_room_for_16_waves(mode, pairs):
    """The LDS of a split pair's workgroups follows from their own waves."""
    _, _, _, waves, cap = shape(PREC_FP32, mode, pairs)
    assert waves <= 2 and 16 // waves * (2048 * waves + 24 * cap) <= 160 * 1024


@pytest.mark.gpu
@pytest.mark.parametrize("prec", [PREC_FP32, PREC_MIXED], ids=["fp32", "mixed"])
def test_batched_log_search(prec):
    """2,500 copies of one chain: every pair reaches the log search, which has
    8 workgroups per CU."""
    rng = np.random.default_rng(6)
    x = synth.chain(31, 44)
    rs = [synth.rigid_copy(rng, x, 0.1 + 0.1 * (i % 9)) for i in range(2500)]
    q, r = Chunk.from_structures([x], ["A" * 44]), Chunk.from_structures(rs, ["A" * 44] * 2500)
    want = batched_equals_plain(q, r, refinement=REF_LOG, precision=prec)
    assert (want.alndata[..., 4] > 0).sum() > 8 * NCU


@pytest.mark.gpu
@pytest.mark.parametrize("nr,hi,waves", [(1000, 170, 4), (2500, 170, 2), (2500, 60, 1)])
def test_batched_dprefine_of_unchanged_alignments(nr, hi, waves):
    """Persistent workgroups of each size that take several pairs, many of
    whose refinements end at once because their alignment did not change."""
    rng = np.random.default_rng(8)
    seeds = [synth.chain(300 + i, int(rng.integers(30, hi + 1))) for i in range(7)] + [synth.chain(299, hi)]
    rs = [synth.rigid_copy(rng, seeds[i % 8], 0.2 + 0.4 * (i % 7)) for i in range(nr)]
    q, r = (Chunk.from_structures(xs, [synth.residues(rng, len(x)) for x in xs]) for xs in (seeds, rs))
    assert shape(PREC_FP32, DPREFINE, 8 * nr, hi, batched=1)[0] == waves
    batched_equals_plain(q, r, prescore=0.0)


def batched_equals_plain(q, r, **kw):
    """The batched form's first call and two replays equal the plain form's bits."""
    got = []
    for batched in (0, 1):
        with GtaBatch(0, default_options(batched=batched, **kw), max_qrys=q.nstrs, max_qry_poss=q.nposs,
                      max_refs=r.nstrs, max_ref_poss=r.nposs) as b:
            b.TransferQueryPMDataToDevice(q)
            b.TransferCPMDataToDevice(r)
            got.append([b.ProcessBlock() for _ in range(3 if batched else 1)])
    want = got[0][0]
    for g in got[1]:
        assert np.array_equal(g.alndata, want.alndata)
        assert np.array_equal(g.tfms, want.tfms)
        assert np.array_equal(g.alns, want.alns)
    return want

"""gta_process_into with buffers that a caller keeps from call to call: they
hold other bytes, or the results of another chunk, on entry, and the sections
are those of gta_process byte for byte -- copied whole (below 1 MiB, or most
pairs aligned) or as the packed rows of the aligned pairs."""
import ctypes as C

import numpy as np
import pytest

from gtalign_alpha_amd import synth
from gtalign_alpha_amd.batch import BlockResults, GtaBatch, lib
from gtalign_alpha_amd.capi import (GTA_ALN_NFIELDS, GTA_TFM_NFIELDS, Results, alignment_section_size,
                                    default_options)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["packed", "dense", "small"])
def test_reused_buffers(kind):
    qc, rc, _ = synth.config(1, scale=0.006)                 # 16 x 300
    q, nr = qc.subset([2, 9]), 30 if kind == "small" else 300
    first = rc.subset(range(nr))
    if kind == "dense":                                      # copies of one query: every pair of it aligns
        first = q.subset([0] * nr)
    other = q.subset([0, 1])
    other.x[:], other.y[:], other.z[:] = q.x[::-1], q.y[::-1], q.z[::-1]
    size = alignment_section_size(2, q.nposs, nr, first.nposs)
    assert (size > 1 << 20) == (kind != "small")
    alndata = np.full((2, nr, GTA_ALN_NFIELDS), -7, np.float32)
    tfms = np.full((2, nr, GTA_TFM_NFIELDS), -7, np.float32)
    alns = np.full(size + 64, 0xA5, np.uint8)                # longer than the section: the rest stays
    with GtaBatch(0, default_options(), max_qrys=2, max_qry_poss=q.nposs, max_refs=nr, max_ref_poss=first.nposs) as b:
        for qq in (q, other, q):
            b.TransferQueryPMDataToDevice(qq)
            b.TransferCPMDataToDevice(first)
            res = Results()
            assert lib().gta_process(b._h, C.byref(res)) == 0
            want = BlockResults(res)
            assert lib().gta_process_into(b._h, 2 * nr, alndata.ctypes.data, tfms.ctypes.data, alns.ctypes.data,
                                          alns.size, C.byref(res)) == 0
            assert np.array_equal(alns[:size], want.alns)
            assert np.array_equal(alndata, want.alndata) and np.array_equal(tfms, want.tfms)
            assert (alns[size:] == 0xA5).all()
        # none of the small set's pairs reaches the score threshold: a section of zeros
        assert want.alns.any() == (kind != "small")

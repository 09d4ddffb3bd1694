"""Batches large enough that their binning is enqueued before the host looks at
the reads: every short length with a few long reads, against the oracle, and a
read longer than the longest bin."""
import numpy as np
import pytest

import myers_amd as M
import oracle_lib as O

pytestmark = pytest.mark.gpu

SIZE = 2_000_000


def test_lengths_and_too_long_reads():
    print("[gpu-case] large scan", flush=True)
    ref = M.synth_reference(81, SIZE, 0.002)
    short = M.synth_batch(M.make_spec(1, 60_003, log_uniform=(1, 260), err_range=(0.0, 0.1), candidates=9,
                                      distance=0.1), ref, SIZE)
    long = M.synth_batch(M.make_spec(2, 2_500, log_uniform=(900, 1_300), err_range=(0.0, 0.1), candidates=2,
                                     distance=0.1), ref, SIZE)
    qi, ca = long["qinfo"].copy(), long["cands"].copy()
    qi[:, 0] += np.uint32(len(short["peq"]))
    ca["query"] += np.uint32(len(short["qinfo"]))
    peq = np.concatenate([short["peq"], long["peq"]])
    qinfo = np.concatenate([short["qinfo"], qi])
    cands = np.concatenate([short["cands"], ca])
    assert len(cands) >= 2048 * 256 and len(qinfo) % 4 != 0
    with M.Myers(ref, SIZE, avg_query=200, cands_per_query=9, buffer_bytes=512 << 20) as m:
        for mode in (M.WINDOW_ALIGNED, M.WINDOW_EXACT):
            got = m.verify(peq, qinfo, cands, 0.1, flags=mode)
            np.testing.assert_array_equal(got, O.myers_batch(ref, SIZE, peq, qinfo, cands, 0.1, mode))
        # a read of more words than the last bin: its candidates are skipped, the call says so
        wrong = qinfo.copy()
        wrong[7, 1] = 24_577
        with pytest.raises(Exception):
            m.verify(peq, wrong, cands, 0.1)
        got = m.verify(peq, qinfo, cands, 0.1)
        np.testing.assert_array_equal(got, O.myers_batch(ref, SIZE, peq, qinfo, cands, 0.1, M.WINDOW_ALIGNED))

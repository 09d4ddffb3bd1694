"""Read sizes near 2^32 (whose word count wraps to 0) in batches of every kernel:
their candidates are skipped, the others are as without them."""
import numpy as np
import pytest

import myers_amd as M
import oracle_lib as O

pytestmark = pytest.mark.gpu

SIZE = 1_000_000
WILD = [0xFFFFFFFF, 0xFFFFFFE1]


@pytest.mark.parametrize("length,reads,times", [(2000, 300, 80), (1000, 300, 250), (2000, 20, 1), (150, 20, 1)])
def test_candidates_are_skipped(length, reads, times):
    ref = M.synth_reference(93, SIZE, 0.001)
    b = M.synth_batch(M.make_spec(length, reads, length=length, err_range=(0.0, 0.1), candidates=4, distance=0.1), ref,
                      SIZE)
    want = O.myers_batch(ref, SIZE, b["peq"], b["qinfo"], b["cands"], 0.1, M.WINDOW_ALIGNED)
    qinfo = b["qinfo"].copy()
    for k, size in enumerate(WILD):
        qinfo[3 + 5 * k, 1] = size
        want[b["cands"]["query"] == 3 + 5 * k] = [0, 0xFFFFFFFF]
    with M.Myers(ref, SIZE, avg_query=length, cands_per_query=4, buffer_bytes=256 << 20) as m:
        for threshold in (-1.0, 0.2):
            print(f"[gpu-case] wild sizes length={length} times={times} threshold={threshold}", flush=True)
            m.set_threshold(threshold)
            got = m.verify(b["peq"], qinfo, np.tile(b["cands"], times), 0.1, flags=M.ENGINE_PERSISTENT)
            exp = want
            if threshold >= 0:
                exp = O.apply_threshold(b["qinfo"], b["cands"], want, threshold)
                exp[want[:, 1] == 0xFFFFFFFF] = [0, 0xFFFFFFFF]
            np.testing.assert_array_equal(got.reshape(times, -1, 2), np.broadcast_to(exp, (times,) + exp.shape))

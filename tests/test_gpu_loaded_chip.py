"""A batch beside others of the same library: while several buffers have a batch in
flight, mid-sized batches of long reads run split into fewer, larger parts, which
spend less of the chip per cell, and the count of those comes back to zero."""
import numpy as np
import pytest

import myers_amd as M
import oracle_lib as O
from launch_info import HANDOVERS, launch_info

pytestmark = pytest.mark.gpu

SIZE = 1_000_000


def test_split_launch_beside_others():
    ref = M.synth_reference(101, SIZE)
    b = M.synth_batch(M.make_spec(9, 50, log_uniform=(2000, 20000), err_range=(0.0, 0.12), candidates=4, distance=0.1),
                      ref, SIZE)
    want = O.myers_batch(ref, SIZE, b["peq"], b["qinfo"], b["cands"], 0.1, M.WINDOW_ALIGNED)
    with M.Myers(ref, SIZE, num_buffers=3, avg_query=8000, cands_per_query=40, buffer_bytes=64 << 20) as m:
        def send(i, times):
            m.send(b["peq"], b["qinfo"], np.tile(b["cands"], times), 0.1, i=i)

        def receive(i, times):
            got = m.receive(i, times * len(want))
            np.testing.assert_array_equal(got.reshape(times, -1, 2), np.broadcast_to(want, (times,) + want.shape))

        def words(i):
            info = launch_info(m, i)
            assert info.ran & HANDOVERS
            return info.split_words

        print("[gpu-case] split beside others", flush=True)
        for _ in range(3):
            send(2, 12)                               # alone: 2400 candidates
            receive(2, 12)
            alone = words(2)
            send(0, 12)
            send(1, 12)                               # one other
            assert words(0) == words(1) == alone
            send(2, 12)                               # two others
            assert words(2) > alone
            for i in (0, 1, 2):
                receive(i, 12)
        # a received buffer, a second receive and a synchronize do not count twice
        m.receive(0, 0)
        M.synchronize(m, 0)
        send(0, 1)
        receive(0, 1)
        send(1, 12)
        send(2, 12)
        assert words(2) == alone
        receive(1, 12)
        receive(2, 12)

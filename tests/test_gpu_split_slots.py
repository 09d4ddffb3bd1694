"""The split launch's hand-over slots used many times over: more boundaries between
parts than twice the slots, with skipped candidates between live ones, launch
after launch on one buffer and in replayed graphs, against the oracle."""
import numpy as np
import pytest

import myers_amd as M
import oracle_lib as O
from launch_info import HANDOVERS, launch_info

pytestmark = pytest.mark.gpu

SIZE = 1_000_000


# long windows (a large distance) take long slots, so there are few
@pytest.mark.parametrize("length,distance,times", [(24500, 3.0, 40), (20000, 4.0, 40), (12000, 6.0, 96)])
def test_slots_are_used_again(length, distance, times):
    ref = M.synth_reference(102, SIZE, 0.001)
    b = M.synth_batch(M.make_spec(length, 8, length=length, err_range=(0.0, 0.15), candidates=1, distance=0.1), ref, SIZE)
    b["cands"]["position"] %= np.uint64(SIZE - int(length * (1 + 2 * distance)) - 16)
    b["cands"]["position"][3] = SIZE - 1                 # skipped
    want = O.myers_batch(ref, SIZE, b["peq"], b["qinfo"], b["cands"], distance, M.WINDOW_ALIGNED)
    exact = O.myers_batch(ref, SIZE, b["peq"], b["qinfo"], b["cands"], distance, M.WINDOW_EXACT)
    assert list(want[3]) == [0, 0xFFFFFFFF] and (want[[0, 1, 2, 4, 5, 6, 7], 1] < length).all()
    cands = np.tile(b["cands"], times)
    with M.Myers(ref, SIZE, avg_query=length, cands_per_query=40, buffer_bytes=64 << 20) as m:
        for k in range(4):
            flags, expect = ((0, want), (M.USE_GRAPH, want), (M.ENGINE_PERSISTENT | M.WINDOW_EXACT, exact), (M.USE_GRAPH, want))[k]
            print(f"[gpu-case] split slots length={length} distance={distance} launch={k}", flush=True)
            got = m.verify(b["peq"], b["qinfo"], cands, distance, flags=flags)
            np.testing.assert_array_equal(got.reshape(times, -1, 2), np.broadcast_to(expect, (times,) + expect.shape))
            info = launch_info(m)
            assert info.ran & HANDOVERS
            parts = -(-((length + 31) // 32) // (64 * info.split_words))
            assert len(cands) * (parts - 1) > 2 * info.split_slots, (parts, info.split_slots)

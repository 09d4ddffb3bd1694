"""The sliced kernel of longer reads over bins of many lengths, against the oracle:
batches made larger until the launch takes that kernel."""
import numpy as np
import pytest

import myers_amd as M
import oracle_lib as O
from launch_info import WIDE_SLICE, launch_info

pytestmark = pytest.mark.gpu

SIZE = 1_000_000


@pytest.mark.parametrize("lo,hi,reads,times", [(1025, 2048, 60, 60), (1900, 3400, 45, 40), (3000, 7000, 45, 20),
                                               (6000, 8300, 45, 16), (8193, 24576, 36, 24), (12000, 13000, 36, 24)])
def test_ragged_lengths(lo, hi, reads, times):
    ref = M.synth_reference(103, SIZE, 0.0005)
    b = M.synth_batch(M.make_spec(lo, reads, log_uniform=(lo, hi), err_range=(0.0, 0.12), candidates=3, distance=0.1), ref,
                      SIZE)
    b["cands"]["position"][5::40] = SIZE - 1
    with M.Myers(ref, SIZE, avg_query=4000, cands_per_query=60, buffer_bytes=512 << 20) as m:
        for mode, threshold in ((M.WINDOW_ALIGNED, -1.0), (M.WINDOW_EXACT, 0.08)):
            want = O.myers_batch(ref, SIZE, b["peq"], b["qinfo"], b["cands"], 0.1, mode)
            if threshold >= 0:
                want = O.apply_threshold(b["qinfo"], b["cands"], want, threshold)
            m.set_threshold(threshold)
            ran = 0
            for n in (times, 4 * times, 16 * times):
                print(f"[gpu-case] wide slice {lo}..{hi} x {n} threshold={threshold}", flush=True)
                got = m.verify(b["peq"], b["qinfo"], np.tile(b["cands"], n), 0.1, flags=mode)
                np.testing.assert_array_equal(got.reshape(n, -1, 2), np.broadcast_to(want, (n,) + want.shape))
                ran = launch_info(m).ran
                if ran & WIDE_SLICE:
                    break
            assert ran & WIDE_SLICE

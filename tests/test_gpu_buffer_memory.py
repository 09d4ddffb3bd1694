"""Device memory of the buffers: creating them takes what bufferBytes says and a
small workspace each, and the launches that need more room find it, in the
buffer's own arrays or on first use, or run another way."""
import numpy as np
import pytest
import torch

import myers_amd as M
import oracle_lib as O
from launch_info import FIRST_ROWS, HANDOVERS, launch_info

pytestmark = pytest.mark.gpu

SIZE = 1_000_000
MIB = 1 << 20


def taken(ref, buffers):
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    with M.Myers(ref, SIZE, num_buffers=buffers, avg_query=150, cands_per_query=11, buffer_bytes=2 * MIB):
        return before - torch.cuda.mem_get_info()[0]


def test_creation():
    ref = M.synth_reference(95, SIZE)
    print("[gpu-case] buffer memory", flush=True)
    taken(ref, 1)                                    # (what the runtime keeps after the first)
    per_buffer = (taken(ref, 65) - taken(ref, 1)) / 64
    # 1.1 MiB of ranges, queue heads and block counts beside the budget; six arrays,
    # each of whole pages of up to 2 MiB
    assert per_buffer < (2 + 1.1 + 6 * 2) * MIB, per_buffer / MIB


@pytest.mark.parametrize("fill,entries,first_rows", [(1.0, 0, False), (0.9, 0, False), (0.9, 40_000, True),
                                                     (0.75, 0, True)])
def test_list_of_the_second_launch(fill, entries, first_rows):
    """Threshold mode over a batch that fills the buffer: the first rows run where
    the candidates or the Peq entries leave room for the list."""
    ref = M.synth_reference(96, SIZE)
    reads = 66_000
    b = M.synth_batch(M.make_spec(7, reads, choices=[1000, 900], err_range=(0.0, 0.2), candidates=5, distance=0.1), ref,
                      SIZE)
    nc, ne = len(b["cands"]), len(b["peq"])
    full = O.myers_batch(ref, SIZE, b["peq"], b["qinfo"], b["cands"], 0.1, M.WINDOW_ALIGNED)
    want = O.apply_threshold(b["qinfo"], b["cands"], full, 0.1)
    # the capacities: avg_query's entries per read, and bytes for nc / fill candidates
    per_cand = (8 * 80 + 8) / 5 + 28
    with M.Myers(ref, SIZE, avg_query=1000, cands_per_query=5, buffer_bytes=int(nc / fill * per_cand) + 200) as m:
        cap_e, _, cap_c = m.capacity()
        peq = np.zeros((cap_e - entries, 20), np.uint32)            # spare entries at the end
        peq[:ne] = b["peq"]
        print(f"[gpu-case] list fill={nc / cap_c:.3f} spare entries={cap_e - len(peq)}", flush=True)
        m.set_threshold(0.1)
        for _ in range(2):
            np.testing.assert_array_equal(m.verify(peq, b["qinfo"], b["cands"], 0.1), want)
            assert bool(launch_info(m).ran & FIRST_ROWS) == first_rows
        # a batch on the device leaves the buffer's arrays free
        dp, dq, dc = M.DeviceArray(b["peq"]), M.DeviceArray(b["qinfo"]), M.DeviceArray(b["cands"])
        dr = M.DeviceArray.empty((nc, 2), np.uint32)
        M.verify_device(m, dp, ne, dq, reads, dc, nc, 0.1, dr, h_qinfo=b["qinfo"])
        M.synchronize(m)
        np.testing.assert_array_equal(dr.get(), want)
        assert launch_info(m).ran & FIRST_ROWS
        for a in (dp, dq, dc, dr):
            a.free()


@pytest.mark.parametrize("flags", [0, M.USE_GRAPH])
def test_first_split_launch(flags):
    ref = M.synth_reference(97, SIZE)
    b = M.synth_batch(M.make_spec(8, 12, log_uniform=(3000, 15000), err_range=(0.0, 0.1), candidates=4, distance=0.1),
                      ref, SIZE)
    want = O.myers_batch(ref, SIZE, b["peq"], b["qinfo"], b["cands"], 0.1, M.WINDOW_ALIGNED)
    with M.Myers(ref, SIZE, num_buffers=2, avg_query=4000, cands_per_query=4, buffer_bytes=16 * MIB) as m:
        print(f"[gpu-case] first split launch flags={flags}", flush=True)
        for i in (0, 1, 0, 1):
            np.testing.assert_array_equal(m.verify(b["peq"], b["qinfo"], b["cands"], 0.1, flags=flags, i=i), want)
            assert launch_info(m, i).ran & HANDOVERS

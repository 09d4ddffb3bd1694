"""myersVerifyDeviceNoAlloc shares one static workspace among all calls, so it
never runs candidates whose parts wait for each other through memory that later
calls find as these leave it."""
import numpy as np
import pytest

import myers_amd as M
import oracle_lib as O
from launch_info import HANDOVERS, SPLIT, launch_info
from test_zz_no_alloc import run

pytestmark = pytest.mark.gpu

SIZE = 1_000_000


@pytest.mark.parametrize("engine", [M.ENGINE_AUTO, M.ENGINE_PERSISTENT])
@pytest.mark.parametrize("lengths", [[20000], [1000, 9000], [150], [300, 900]])
def test_no_handovers(lengths, engine):
    ref = M.synth_reference(94, SIZE)
    b = M.synth_batch(M.make_spec(lengths[0], 20, choices=lengths, err_range=(0.0, 0.1), candidates=4, distance=0.1), ref,
                      SIZE)
    want = O.myers_batch(ref, SIZE, b["peq"], b["qinfo"], b["cands"], 0.1, M.WINDOW_ALIGNED)
    L = M.lib()
    with M.Myers(ref, SIZE, avg_query=4000, cands_per_query=4, buffer_bytes=64 << 20) as m:
        print(f"[gpu-case] no-alloc split lengths={lengths} engine={engine}", flush=True)
        np.testing.assert_array_equal(run(m, L.myersVerifyDevice, b, engine), want)
        own = launch_info(m)
        assert own.ran & SPLIT
        assert bool(own.ran & HANDOVERS) == (max(lengths) > 2048)
        np.testing.assert_array_equal(run(m, L.myersVerifyDeviceNoAlloc, b, engine), want)
        assert not launch_info(m).ran & HANDOVERS

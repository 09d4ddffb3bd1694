"""Thresholds whose product with the read length is beyond 32 bits (up to
infinity) keep every verified candidate, in every kernel of threshold mode."""
import numpy as np
import pytest

import myers_amd as M
import oracle_lib as O

pytestmark = pytest.mark.gpu

SIZE = 1_000_000


@pytest.mark.parametrize("reads,lengths", [(140_000, [100, 150, 200]), (140_000, [600, 1000]), (500, [100, 250, 900]),
                                           (60, [1500, 5000])])
def test_every_candidate_is_reported(reads, lengths):
    ref = M.synth_reference(91, SIZE)
    b = M.synth_batch(M.make_spec(reads + lengths[0], reads, choices=lengths, err_range=(0.0, 0.3), candidates=4,
                                  distance=0.1), ref, SIZE)
    want = O.myers_batch(ref, SIZE, b["peq"], b["qinfo"], b["cands"], 0.1, M.WINDOW_ALIGNED)
    with M.Myers(ref, SIZE, avg_query=2000, cands_per_query=4, buffer_bytes=512 << 20) as m:
        for engine in (M.ENGINE_AUTO, M.ENGINE_PLAIN, M.ENGINE_PERSISTENT, M.ENGINE_BINNED):
            for e in (1.0e6, 2.5e7, 1.0e9, float("inf")):
                print(f"[gpu-case] huge threshold reads={reads} lengths={lengths} engine={engine} e={e}", flush=True)
                m.set_threshold(e)
                got = m.verify(b["peq"], b["qinfo"], b["cands"], 0.1, flags=engine)
                np.testing.assert_array_equal(got, want, err_msg=f"engine={engine} e={e}")


def test_resident_server():
    ref = M.synth_reference(92, SIZE)
    b = M.synth_batch(M.make_spec(5, 60, choices=[100, 400, 1000, 3000], err_range=(0.0, 0.3), candidates=4,
                                  distance=0.1), ref, SIZE)
    want = O.myers_batch(ref, SIZE, b["peq"], b["qinfo"], b["cands"], 0.1, M.WINDOW_ALIGNED)
    with M.Myers(ref, SIZE, avg_query=1000, cands_per_query=4, buffer_bytes=64 << 20) as m:
        m.set_threshold(1.0e9)
        print("[gpu-case] huge threshold resident server", flush=True)
        with M.Server(m, distance=0.1, flags=M.SERVE_RESIDENT) as sv:
            req, keep = M.Server.request(b["peq"], b["qinfo"], b["cands"])
            sv.wait(sv.submit(req))
            np.testing.assert_array_equal(keep[3], want)

"""Reads in small batches, their rows split over waves, against the oracle:
reads of one part and of the most parts, lengths at the parts' borders, more
hand-overs than slots, repeated launches and replayed graphs on one buffer, and
skipped candidates between live ones."""
import numpy as np
import pytest

import myers_amd as M
import oracle_lib as O

pytestmark = pytest.mark.gpu

SIZE = 2_000_000
LENGTHS = [97, 128, 150, 224, 225, 256, 257, 700, 1023, 1024, 1025, 2047, 2048, 2049, 4096, 4097, 6145, 8192, 8193, 16385, 20000, 24575, 24576]


@pytest.fixture(scope="module")
def library():
    ref = M.synth_reference(79, SIZE, 0.002)
    with M.Myers(ref, SIZE, avg_query=3000, cands_per_query=10, buffer_bytes=256 << 20) as m:
        yield ref, m


def check(ref, m, b, mode, flags=0, times=1, threshold=-1.0):
    want = O.myers_batch(ref, SIZE, b["peq"], b["qinfo"], b["cands"], 0.1, mode)
    if threshold >= 0:
        want = O.apply_threshold(b["qinfo"], b["cands"], want, threshold)
    m.set_threshold(threshold)
    got = m.verify(b["peq"], b["qinfo"], np.tile(b["cands"], times), 0.1, flags=mode | flags)
    m.set_threshold(-1.0)
    np.testing.assert_array_equal(got.reshape(times, -1, 2), np.broadcast_to(want, (times,) + want.shape))


@pytest.mark.parametrize("length", LENGTHS)
def test_parts(library, length):
    ref, m = library
    print(f"[gpu-case] split length={length}", flush=True)
    for reads, cands, mode in ((1, 1, M.WINDOW_ALIGNED), (7, 3, M.WINDOW_EXACT), (40, 4, M.WINDOW_ALIGNED)):
        b = M.synth_batch(M.make_spec(length + reads, reads, length=length, err_range=(0.0, 0.2), candidates=cands,
                                      distance=0.1), ref, SIZE)
        check(ref, m, b, mode)
        check(ref, m, b, mode, M.ENGINE_PERSISTENT, threshold=0.12)


@pytest.mark.parametrize("reads,times", [(12, 1), (60, 1), (30, 6)])
def test_ragged_lengths(library, reads, times):
    ref, m = library
    print(f"[gpu-case] split ragged reads={reads} times={times}", flush=True)
    b = M.synth_batch(M.make_spec(reads, reads, log_uniform=(300, 24576), err_range=(0.0, 0.15), candidates=3,
                                  distance=0.1), ref, SIZE)
    for _ in range(3):
        check(ref, m, b, M.WINDOW_EXACT, times=times)


def test_more_handovers_than_slots(library):
    # 400 candidates of 6 or 12 parts: over 2,000 boundaries, under 1,700 slots
    ref, m = library
    print("[gpu-case] split slots", flush=True)
    b = M.synth_batch(M.make_spec(3, 20, length=24500, err_range=(0.0, 0.15), candidates=1, distance=0.1), ref, SIZE)
    b["cands"]["position"][5:8] = SIZE - 1              # skipped ones between
    for _ in range(2):
        check(ref, m, b, M.WINDOW_ALIGNED, times=20)


def test_skipped_and_wild_peq(library):
    ref, m = library
    print("[gpu-case] split skipped", flush=True)
    b = M.synth_batch(M.make_spec(6, 12, length=5000, err_range=(0.0, 0.1), candidates=4, distance=0.1), ref, SIZE)
    b["cands"]["position"][::3] = SIZE - 5000 - np.arange(16) * 70
    b["cands"]["position"][1:6] = [0, 1, 7, 8, 33]
    peq = b["peq"].reshape(-1, 5, 4).copy()
    peq[3::7, :, 1] |= 0x10
    peq[5::9, :, 2] = 0
    b["peq"] = np.ascontiguousarray(peq.reshape(-1, 20))
    check(ref, m, b, M.WINDOW_EXACT)
    check(ref, m, b, M.WINDOW_ALIGNED)
    b["cands"]["position"][:] = SIZE - 1
    check(ref, m, b, M.WINDOW_ALIGNED)


def test_replayed_graph(library):
    ref, m = library
    print("[gpu-case] split graph", flush=True)
    b = M.synth_batch(M.make_spec(8, 20, log_uniform=(1100, 15000), err_range=(0.0, 0.1), candidates=4, distance=0.1),
                      ref, SIZE)
    want = O.myers_batch(ref, SIZE, b["peq"], b["qinfo"], b["cands"], 0.1, M.WINDOW_ALIGNED)
    dp, dq, dc = M.DeviceArray(b["peq"]), M.DeviceArray(b["qinfo"]), M.DeviceArray(b["cands"])
    nq, nc, ne = len(b["qinfo"]), len(b["cands"]), len(b["peq"])
    dr = M.DeviceArray.empty((nc, 2), np.uint32)
    for rep in range(4):
        clear = np.zeros((nc, 2), np.uint32)
        M.check(M.lib().myersMemcpyHtoD(dr.ptr, M._ptr(clear), clear.nbytes), "clear")
        M.verify_device(m, dp, ne, dq, nq, dc, nc, 0.1, dr, flags=M.USE_GRAPH, h_qinfo=b["qinfo"])
        M.synchronize(m)
        np.testing.assert_array_equal(dr.get(), want)
        check(ref, m, b, M.WINDOW_EXACT)                # eager work on the same buffer between the replays

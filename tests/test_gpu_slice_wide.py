"""The candidate-sliced kernel of reads of over 1024 bases against the oracle:
the least and the most rows per lane of each team of waves, bins of mixed
lengths, N in reads and windows, chunks without a live candidate, and Peq words
that are not one code per base.  The kernel takes batches that fill the chip, so
a few dozen candidates are verified many times over."""
import numpy as np
import pytest

import myers_amd as M
import oracle_lib as O

pytestmark = pytest.mark.gpu

SIZE = 2_000_000
# 1 wave: 17-32 rows; 2: 17-26; 3: 18-26; 4: 20-32; 12: 11-32
LENGTHS = [1025, 1088, 1089, 1536, 2048, 2049, 3328, 3329, 4992, 4993, 6656, 6657, 8192, 8193, 8449, 12289, 19968, 19969,
           24576]


@pytest.fixture(scope="module")
def library():
    ref = M.synth_reference(78, SIZE, 0.0005)
    with M.Myers(ref, SIZE, avg_query=3000, cands_per_query=40, buffer_bytes=512 << 20) as m:
        yield ref, m


def check(ref, m, b, mode, flags=0, threshold=-1.0):
    want = O.myers_batch(ref, SIZE, b["peq"], b["qinfo"], b["cands"], 0.1, mode)
    # twice the bit-vector kernels' time for one chunk's longest
    size = int(b["qinfo"][:, 1].max())
    times = 1 + int(2 * 120e12 * (1.25 * size + 1200) * 1e-6 / (1.25 * float(size) ** 2) / len(b["cands"]))
    if threshold >= 0:
        want = O.apply_threshold(b["qinfo"], b["cands"], want, threshold)
    m.set_threshold(threshold)
    got = m.verify(b["peq"], b["qinfo"], np.tile(b["cands"], times), 0.1, flags=mode | flags)
    m.set_threshold(-1.0)
    np.testing.assert_array_equal(got.reshape(times, -1, 2), np.broadcast_to(want, (times,) + want.shape))


@pytest.mark.parametrize("length", LENGTHS)
def test_rows(library, length):
    ref, m = library
    print(f"[gpu-case] wide slice length={length}", flush=True)
    for cands, mode in ((1, M.WINDOW_EXACT), (5, M.WINDOW_ALIGNED)):
        b = M.synth_batch(M.make_spec(length, 36 // cands, length=length, err_range=(0.0, 0.2), candidates=cands,
                                      distance=0.1), ref, SIZE)
        check(ref, m, b, mode, M.ENGINE_PERSISTENT if cands == 1 else 0)


@pytest.mark.parametrize("lo,hi", [(1025, 2048), (3000, 7000), (8193, 24576), (900, 1200)])
def test_ragged_lengths(library, lo, hi):
    ref, m = library
    print(f"[gpu-case] wide slice {lo}..{hi}", flush=True)
    b = M.synth_batch(M.make_spec(lo, 45, log_uniform=(lo, hi), err_range=(0.0, 0.12), candidates=3, distance=0.1), ref,
                      SIZE)
    check(ref, m, b, M.WINDOW_ALIGNED)
    check(ref, m, b, M.WINDOW_EXACT, threshold=0.08)


@pytest.mark.parametrize("length", [1500, 5000, 7000, 9000])
def test_peq_without_one_code_per_base(library, length):
    # a base that matches two codes and one that matches none, in some reads
    ref, m = library
    print(f"[gpu-case] wide slice odd Peq length={length}", flush=True)
    b = M.synth_batch(M.make_spec(length, 12, length=length, err_range=(0.0, 0.1), candidates=3, distance=0.1), ref, SIZE)
    peq = b["peq"].reshape(-1, 5, 4).copy()
    entries = (length + 127) // 128
    peq[2 * entries, :, 1] |= 0x10
    peq[7 * entries + entries - 1, :, 0] = 0
    b["peq"] = np.ascontiguousarray(peq.reshape(-1, 20))
    check(ref, m, b, M.WINDOW_EXACT)


def test_skipped_candidates(library):
    ref, m = library
    print("[gpu-case] wide slice skipped", flush=True)
    b = M.synth_batch(M.make_spec(5, 40, length=2000, err_range=(0.0, 0.1), candidates=1, distance=0.1), ref, SIZE)
    at = np.array([SIZE - 1, SIZE - 2000, SIZE - 2201, SIZE - 2200, SIZE - 2300, 0, 7, 31, 32, 33], dtype=np.uint64)
    b["cands"]["position"][:20:2] = at
    check(ref, m, b, M.WINDOW_ALIGNED)
    check(ref, m, b, M.WINDOW_EXACT)
    b["cands"]["position"][:] = SIZE - 1
    check(ref, m, b, M.WINDOW_EXACT)


def test_chunks_of_two_lengths(library):
    """Chunks at the border of two lengths: rows missing to a lane up to 2, up to
    8, and more than the sliced form takes (a bin table of the caller's)."""
    ref, m = library
    default = m.bin_table()
    table = default.copy()
    table[33:65] = m.variant_index(8, 8)
    m.set_bin_table(table)
    try:
        for lengths in ([1990, 2040], [1600, 2000], [1030, 2040], [1030, 1300, 1400, 1700, 2048]):
            print(f"[gpu-case] wide slice lengths={lengths}", flush=True)
            b = M.synth_batch(M.make_spec(lengths[0], 37, choices=lengths, err_range=(0.0, 0.1), candidates=1,
                                          distance=0.1), ref, SIZE)
            check(ref, m, b, M.WINDOW_ALIGNED)
    finally:
        m.set_bin_table(default)

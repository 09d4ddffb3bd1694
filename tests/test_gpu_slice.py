"""The candidate-sliced kernel of reads of up to 1024 bases against the oracle:
the rows per lane of each form from the least to the most, reads whose rows do
not fill the lanes, chunks of one read and of many, N in reads and windows,
Peq words that are not one code per base, and chunks without a live candidate."""
import numpy as np
import pytest

import myers_amd as M
import oracle_lib as O

pytestmark = pytest.mark.gpu

SIZE = 2_000_000
# one length: up to 7 words small batches run the bit-vector kernel, from
# 524,288 candidates on the chunks are of 128 candidates (16 lanes per group)
SMALL = [225, 256, 257, 400, 513, 767, 832, 833, 865, 992, 993, 1000, 1023, 1024]
LARGE = [1, 16, 17, 31, 32, 33, 48, 49, 100, 225, 368, 369, 384, 385]


@pytest.fixture(scope="module")
def library():
    ref = M.synth_reference(77, SIZE, 0.03)
    with M.Myers(ref, SIZE, avg_query=300, cands_per_query=6, buffer_bytes=512 << 20) as m:
        yield ref, m


def check(ref, m, b, mode, flags=0, threshold=-1.0):
    m.set_threshold(threshold)
    got = m.verify(b["peq"], b["qinfo"], b["cands"], 0.1, flags=mode | flags)
    m.set_threshold(-1.0)
    want = O.myers_batch(ref, SIZE, b["peq"], b["qinfo"], b["cands"], 0.1, mode)
    if threshold >= 0:
        want = O.apply_threshold(b["qinfo"], b["cands"], want, threshold)
    np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("length", SMALL)
def test_rows_of_small_batches(library, length):
    ref, m = library
    mode = M.WINDOW_EXACT if length % 2 else M.WINDOW_ALIGNED
    print(f"[gpu-case] slice length={length}", flush=True)
    for cands in (1, 11):
        b = M.synth_batch(M.make_spec(length, 300, length=length, err_range=(0.0, 0.2), candidates=cands,
                                      distance=0.1), ref, SIZE)
        check(ref, m, b, mode)
        check(ref, m, b, mode, threshold=0.15)


@pytest.mark.parametrize("length", LARGE)
def test_rows_of_large_batches(library, length):
    ref, m = library
    mode = M.WINDOW_EXACT if length % 2 else M.WINDOW_ALIGNED
    print(f"[gpu-case] slice large length={length}", flush=True)
    b = M.synth_batch(M.make_spec(length, 110_000, length=length, err_range=(0.0, 0.2), poisson=6, cap=40,
                                  distance=0.1), ref, SIZE)
    assert len(b["cands"]) > 524_288
    check(ref, m, b, mode)


@pytest.mark.parametrize("engine", [M.ENGINE_PLAIN, M.ENGINE_PERSISTENT, M.ENGINE_BINNED])
def test_ragged_lengths_every_engine(library, engine):
    """Every length class at once; the large batch also groups reads with N."""
    ref, m = library
    for reads, lengths in ((3_000, (1, 1024)), (60_000, (300, 1024))):
        print(f"[gpu-case] slice ragged reads={reads} engine={engine}", flush=True)
        b = M.synth_batch(M.make_spec(reads, reads, log_uniform=lengths, err_range=(0.0, 0.2), poisson=6, cap=40,
                                      distance=0.1), ref, SIZE)
        check(ref, m, b, M.WINDOW_ALIGNED, engine)


def test_peq_without_one_code_per_base(library):
    """Rows of no code, of two codes and of N: such chunks run the bit-vector
    kernel, the others of the batch do not."""
    ref, m = library
    for length in (40, 300, 1000):
        print(f"[gpu-case] slice wild peq length={length}", flush=True)
        b = M.synth_batch(M.make_spec(length, 400, length=length, err_range=(0.0, 0.1), candidates=5, distance=0.1),
                          ref, SIZE)
        peq = b["peq"].reshape(-1, 5, 4).copy()
        entries = (length + 127) // 128
        rng = np.random.default_rng(length)
        for read in rng.choice(400, size=12, replace=False):
            for p in rng.choice(length, size=5, replace=False):
                e, w, bit = int(b["qinfo"][read, 0]) + p // 128, p % 128 // 32, np.uint32(1 << (p % 32))
                kind = rng.integers(3)
                peq[e, :, w] &= ~bit
                for c in ([], rng.choice(4, size=2, replace=False), [4])[kind]:
                    peq[e, c, w] |= bit
        assert entries * 400 == len(peq)
        b["peq"] = np.ascontiguousarray(peq.reshape(-1, 20))
        check(ref, m, b, M.WINDOW_ALIGNED, M.ENGINE_PERSISTENT)


def test_one_bin_of_mixed_lengths(library):
    """A bin table that sends every short read to one variant: its chunks mix
    word counts, which the sliced form does not take."""
    ref, m = library
    default = m.bin_table()
    b = M.synth_batch(M.make_spec(5, 500, log_uniform=(1, 1024), err_range=(0.0, 0.1), candidates=7, distance=0.1),
                      ref, SIZE)
    table = default.copy()
    table[:33] = m.variant_index(1, 32)
    m.set_bin_table(table)
    try:
        check(ref, m, b, M.WINDOW_EXACT)
        check(ref, m, b, M.WINDOW_ALIGNED, M.ENGINE_PERSISTENT)
    finally:
        m.set_bin_table(default)


def test_skipped_candidates_and_the_reference_end(library):
    """Chunks with only skipped candidates, with some, and windows up to the
    reference's last base."""
    ref, m = library
    for length in (64, 250, 1000):
        b = M.synth_batch(M.make_spec(length + 1, 60, length=length, err_range=(0.0, 0.1), candidates=8,
                                      distance=0.1), ref, SIZE)
        n = int(np.float32(length) * (np.float32(1.0) + np.float32(2.0) * np.float32(0.1)))
        pos = b["cands"]["position"]
        pos[:192] = SIZE + np.arange(192)               # three chunks of skipped candidates
        pos[200:440:3] = SIZE - n                       # skipped: not more than the window left
        pos[201:440:3] = SIZE - n - 1 - np.arange(80) % 9
        print(f"[gpu-case] slice skipped length={length}", flush=True)
        for mode in (M.WINDOW_ALIGNED, M.WINDOW_EXACT):
            check(ref, m, b, mode)
            check(ref, m, b, mode, M.ENGINE_PERSISTENT)

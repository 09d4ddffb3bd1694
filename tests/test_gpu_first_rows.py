"""Threshold mode over large batches, where the first rows of a read rule its
candidate out, against the oracle: every word count, thresholds from few rows to
all rows, batches of mostly unrelated candidates and of none, skipped candidates,
and a bin of mixed lengths."""
import numpy as np
import pytest

import myers_amd as M
import oracle_lib as O

pytestmark = pytest.mark.gpu

SIZE = 2_000_000


@pytest.fixture(scope="module")
def library():
    ref = M.synth_reference(80, SIZE, 0.003)
    with M.Myers(ref, SIZE, avg_query=500, cands_per_query=8, buffer_bytes=512 << 20) as m:
        yield ref, m


def check(ref, m, spec, thresholds, mode=M.WINDOW_ALIGNED, change=None):
    b = M.synth_batch(spec, ref, SIZE)
    if change:
        change(b)
    assert len(b["cands"]) >= 300_000
    full = O.myers_batch(ref, SIZE, b["peq"], b["qinfo"], b["cands"], 0.1, mode)
    for e in thresholds:
        m.set_threshold(e)
        got = m.verify(b["peq"], b["qinfo"], b["cands"], 0.1, flags=mode)
        m.set_threshold(-1.0)
        np.testing.assert_array_equal(got, O.apply_threshold(b["qinfo"], b["cands"], full, e), err_msg=f"e={e}")


@pytest.mark.parametrize("lengths", [(120, 256), (257, 640), (641, 1024)])
def test_thresholds(library, lengths):
    ref, m = library
    print(f"[gpu-case] first rows {lengths}", flush=True)
    check(ref, m, M.make_spec(lengths[0], 40_000, log_uniform=lengths, err_range=(0.0, 0.3), poisson=8, cap=40,
                              distance=0.1), [0.0, 0.03, 0.1, 0.2, 0.31, 0.5])


@pytest.mark.parametrize("length", [250, 500, 1000])
def test_every_candidate_kept(library, length):
    # one candidate per read, at its place: nothing is ruled out
    ref, m = library
    print(f"[gpu-case] first rows kept {length}", flush=True)
    check(ref, m, M.make_spec(length, 330_000, length=length, err_range=(0.0, 0.1), candidates=1, distance=0.1), [0.2],
          M.WINDOW_EXACT)


def test_skipped_candidates(library):
    ref, m = library
    print("[gpu-case] first rows skipped", flush=True)

    def change(b):
        b["cands"]["position"][::5] = SIZE + 3
        b["cands"]["position"][1:200_000:7] = SIZE - 500
        b["cands"]["position"][130_000:140_000] = SIZE
    check(ref, m, M.make_spec(9, 80_000, log_uniform=(300, 420), err_range=(0.0, 0.1), candidates=4, distance=0.1),
          [0.1, 0.25], change=change)


def test_one_bin_of_mixed_lengths(library):
    # reads with fewer rows than the bin's first rows
    ref, m = library
    print("[gpu-case] first rows mixed bin", flush=True)
    default = m.bin_table()
    table = default.copy()
    table[:33] = m.variant_index(1, 32)
    m.set_bin_table(table)
    try:
        check(ref, m, M.make_spec(4, 41_000, choices=[100, 120, 1000], err_range=(0.0, 0.1), candidates=8,
                                  distance=0.1), [0.2])
    finally:
        m.set_bin_table(default)

"""Threshold mode over mid-sized batches: the cut-off kernel of a bin's launch at
the edges of its widths, and the first rows where they pay, against the oracle."""
import numpy as np
import pytest

import myers_amd as M
import oracle_lib as O
from launch_info import CUT, FIRST_ROWS, launch_info

pytestmark = pytest.mark.gpu

SIZE = 1_000_000


@pytest.fixture(scope="module")
def library():
    ref = M.synth_reference(99, SIZE, 0.002)
    with M.Myers(ref, SIZE, avg_query=1000, cands_per_query=5, buffer_bytes=256 << 20) as m:
        yield ref, m
        m.set_threshold(-1.0)


def check(ref, m, b, times, flags, e, mode=M.WINDOW_ALIGNED):
    full = O.myers_batch(ref, SIZE, b["peq"], b["qinfo"], b["cands"], 0.1, mode)
    want = O.apply_threshold(b["qinfo"], b["cands"], full, e)
    m.set_threshold(e)
    got = m.verify(b["peq"], b["qinfo"], np.tile(b["cands"], times), 0.1, flags=flags | mode)
    m.set_threshold(-1.0)
    np.testing.assert_array_equal(got.reshape(times, -1, 2), np.broadcast_to(want, (times,) + want.shape))
    return launch_info(m).ran


@pytest.mark.parametrize("length", [513, 544, 577, 608, 609, 704, 705, 800, 801, 897, 928, 929, 1000, 1024])
def test_cut_off_widths(library, length):
    ref, m = library
    b = M.synth_batch(M.make_spec(length, 60, length=length, err_range=(0.0, 0.2), candidates=5, distance=0.1), ref, SIZE)
    b["cands"]["position"][3::50] = SIZE - 4
    for e, mode in ((0.0, M.WINDOW_EXACT), (0.03, M.WINDOW_ALIGNED), (0.1, M.WINDOW_EXACT)):
        print(f"[gpu-case] cut-off length={length} e={e}", flush=True)
        assert check(ref, m, b, 280, M.ENGINE_PLAIN, e, mode) & CUT
    assert not check(ref, m, b, 280, M.ENGINE_PLAIN, 0.11) & CUT


@pytest.mark.parametrize("lengths", [[600, 1000], [530, 700, 1024]])
def test_cut_off_bins(library, lengths):
    ref, m = library
    print(f"[gpu-case] cut-off bins {lengths}", flush=True)
    b = M.synth_batch(M.make_spec(len(lengths), 120, choices=lengths, err_range=(0.0, 0.15), candidates=5, distance=0.1),
                      ref, SIZE)
    assert check(ref, m, b, 450, M.ENGINE_PLAIN, 0.05) & CUT


@pytest.mark.parametrize("length,times,first", [(1000, 170, False), (1000, 320, True), (600, 260, False), (600, 800, True)])
def test_first_rows_of_one_length(library, length, times, first):
    ref, m = library
    print(f"[gpu-case] first rows of one length {length} x {times}", flush=True)
    b = M.synth_batch(M.make_spec(length, 100, length=length, err_range=(0.0, 0.1), candidates=5, distance=0.1), ref, SIZE)
    for flags in (0, M.USE_GRAPH):
        assert bool(check(ref, m, b, times, flags, 0.05) & FIRST_ROWS) == first

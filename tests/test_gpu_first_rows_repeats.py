"""Threshold mode over large batches whose reads start in short tandem repeats,
against the oracle.  In a repeat the score of a read's first rows goes up and
down by one from column to column near zero, where a bound that takes eight
columns' falls without their rises would be less than zero."""
import numpy as np
import pytest

import myers_amd as M
import oracle_lib as O

pytestmark = pytest.mark.gpu

SIZE = 1_000_000


def repeats(seed, unit):
    """A random reference in which a repeat of `unit` bases and 40-300 bases long
    starts every 500 bases or so."""
    rng = np.random.default_rng(seed)
    codes = rng.integers(0, 4, SIZE).astype(np.uint8)
    at = 0
    while at < SIZE - 1000:
        length = int(rng.integers(40, 301))
        codes[at:at + length] = np.resize(rng.permutation(4)[:unit], length)
        at += length + int(rng.integers(150, 350))
    return O.pack_reference(codes)


@pytest.mark.parametrize("unit", [2, 3, 4])
@pytest.mark.parametrize("length", [600, 1000])
def test_reads_that_start_in_a_repeat(unit, length):
    ref = repeats(unit, unit)
    # a few shorter reads: a batch of several bins is binned, which the first rows need
    b = M.synth_batch(M.make_spec(length + unit, 76_000, choices=[length] * 7 + [length // 2], err_range=(0.0, 0.02),
                                  candidates=4, distance=0.1), ref, SIZE)
    assert len(b["cands"]) >= 300_000
    full = O.myers_batch(ref, SIZE, b["peq"], b["qinfo"], b["cands"], 0.1, M.WINDOW_ALIGNED)
    with M.Myers(ref, SIZE, avg_query=length, cands_per_query=4, buffer_bytes=256 << 20) as m:
        for e in (0.0, 0.01, 0.03, 0.1):
            print(f"[gpu-case] first rows in repeats unit={unit} length={length} e={e}", flush=True)
            want = O.apply_threshold(b["qinfo"], b["cands"], full, e)
            assert (want[:, 0] != 0xFFFFFFFF).sum() > (30_000 if e > 0.02 else 1_000)
            m.set_threshold(e)
            got = m.verify(b["peq"], b["qinfo"], b["cands"], 0.1)
            np.testing.assert_array_equal(got, want, err_msg=f"e={e}")

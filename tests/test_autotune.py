"""The autotuner's choice of variants to time (no GPU)."""
import os
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(os.path.dirname(HERE), "myers-gpu_amd", "python"))
import autotune  # noqa: E402

VARIANTS = [{"lanes": 1, "words": w} for w in range(1, 33)] + [{"lanes": lanes, "words": w} for lanes in (2, 4, 8, 64)
                                                                for w in (8, 12)]


@pytest.mark.parametrize("words", range(1, 33))
def test_a_short_row_holds_no_padding(words):
    timed = [VARIANTS[i] for i in autotune.candidates_for(VARIANTS, words)]
    assert [v["words"] for v in timed if v["lanes"] == 1] == [words]
    assert all(words <= v["lanes"] * v["words"] <= max(2 * words, words + 4) for v in timed)


def test_long_rows_are_timed_with_every_cover():
    timed = [VARIANTS[i] for i in autotune.candidates_for(VARIANTS, 48)]
    assert [(v["lanes"], v["words"]) for v in timed] == [(4, 12), (8, 8), (8, 12)]

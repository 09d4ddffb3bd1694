"""Bins of the engines: the persistent engine has a bin per word count whatever
rows a caller's table gives short reads, the engines with a launch per bin keep
its rows, and a bin of several word counts runs in every width, against the
oracle."""
import numpy as np
import pytest

import myers_amd as M
import oracle_lib as O

pytestmark = pytest.mark.gpu

SIZE = 1_000_000


@pytest.fixture(scope="module")
def library():
    ref = M.synth_reference(98, SIZE, 0.002)
    with M.Myers(ref, SIZE, avg_query=400, cands_per_query=5, buffer_bytes=256 << 20) as m:
        yield ref, m


def batch(ref, seed, reads, lo, hi):
    b = M.synth_batch(M.make_spec(seed, reads, log_uniform=(lo, hi), err_range=(0.0, 0.15), candidates=5, distance=0.1),
                      ref, SIZE)
    words = np.unique((b["qinfo"][:, 1] + 31) // 32)
    return b, words, O.myers_batch(ref, SIZE, b["peq"], b["qinfo"], b["cands"], 0.1, M.WINDOW_ALIGNED)


@pytest.mark.parametrize("flags", [0, M.USE_GRAPH])
@pytest.mark.parametrize("reads", [300, 20_000, 120_000])
def test_bins_of_each_engine(library, reads, flags):
    ref, m = library
    b, words, want = batch(ref, reads, reads, 300, 900)
    default = m.bin_table()
    coarse = default.copy()
    coarse[1:17], coarse[17:33] = m.variant_index(1, 16), m.variant_index(1, 32)
    try:
        for name, table in (("default", default), ("two rows", coarse)):
            m.set_bin_table(table)
            np.testing.assert_array_equal(m.bin_table(), table)
            for engine in (M.ENGINE_AUTO, M.ENGINE_PERSISTENT, M.ENGINE_PLAIN, M.ENGINE_BINNED):
                print(f"[gpu-case] bins reads={reads} table={name} engine={engine} flags={flags}", flush=True)
                np.testing.assert_array_equal(m.verify(b["peq"], b["qinfo"], b["cands"], 0.1, flags=engine | flags), want)
                if flags:
                    continue
                per_bin = engine in (M.ENGINE_PLAIN, M.ENGINE_BINNED)
                assert m.stats().variantsUsed == (len(np.unique(table[words])) if per_bin else len(words))
    finally:
        m.set_bin_table(default)


def test_default_table_has_few_short_bins(library):
    # a launch per bin: their number is what the plain engine's time goes with
    _, m = library
    assert len(np.unique(m.bin_table()[1:33])) <= 13


@pytest.mark.parametrize("width", list(range(1, 33)))
def test_bins_of_several_word_counts(library, width):
    ref, m = library
    b, _, want = batch(ref, width, 700, 20, 32 * width)
    default = m.bin_table()
    table = default.copy()
    table[:width + 1] = m.variant_index(1, width)
    m.set_bin_table(table)
    try:
        for engine in (M.ENGINE_PLAIN, M.ENGINE_BINNED):
            print(f"[gpu-case] one bin width={width} engine={engine}", flush=True)
            np.testing.assert_array_equal(m.verify(b["peq"], b["qinfo"], b["cands"], 0.1, flags=engine), want)
    finally:
        m.set_bin_table(default)

"""Batches of one short length through the buffer API, whose launch reads and
writes the host arrays itself, against the oracle: one buffer refilled again and
again with other reads, lengths and sizes, between batches that are copied."""
import numpy as np
import pytest

import myers_amd as M
import oracle_lib as O

pytestmark = pytest.mark.gpu

SIZE = 2_000_000


def test_refilled_buffers():
    ref = M.synth_reference(83, SIZE, 0.002)
    with M.Myers(ref, SIZE, avg_query=300, cands_per_query=8, buffer_bytes=128 << 20) as m:
        for k, (length, reads) in enumerate([(150, 1), (150, 1), (31, 300), (32, 300), (1024, 40), (1000, 3_000),
                                             (1025, 5), (100, 20_000), (100, 19_999), (224, 700), (225, 700), (7, 1)]):
            print(f"[gpu-case] host arrays length={length} reads={reads}", flush=True)
            b = M.synth_batch(M.make_spec(500 + k, reads, length=length, err_range=(0.0, 0.2), candidates=7,
                                          distance=0.1), ref, SIZE)
            b["cands"]["position"][::5] = SIZE - 1          # skipped ones write their results too
            for mode in (M.WINDOW_ALIGNED, M.WINDOW_EXACT):
                got = m.verify(b["peq"], b["qinfo"], b["cands"], 0.1, flags=mode)
                np.testing.assert_array_equal(got, O.myers_batch(ref, SIZE, b["peq"], b["qinfo"], b["cands"], 0.1, mode))

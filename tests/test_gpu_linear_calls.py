"""Linear calls on one PackedB8 handle, whose stream and buffers are kept
between calls: growing and shrinking row counts, padded rows after full
ones, several threads, against the CPU oracle."""
import concurrent.futures as cf

import numpy as np
import pytest

from helpers import f32_bits_equal, mismatch_report
from indecis_amd import linalg
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,n", [(768, 96), (70, 33)])
def test_linear_calls_one_handle(k, n):
    rng = np.random.default_rng(k)
    q, s = linalg.pack_b8(rng.standard_normal((n, k), dtype=np.float32))
    cs = q.astype(np.int32).sum(axis=1).astype(np.int32)
    bias = rng.standard_normal(n).astype(np.float32)
    b = linalg.PackedB8(q, s)
    calls = []
    for rows in (64, 1, 17, 200, 3, 15, 16, 33):
        x = rng.standard_normal((rows, k), dtype=np.float32)
        x[:, rng.choice(k, 3, replace=False)] *= 40
        for out in (True, False):
            calls.append((x, out, orc.linear8(x, q, s, cs, bias, out, 6.0)))
    for x, out, want in calls:
        got = linalg.linear8(x, b, bias, out, 6.0)
        assert f32_bits_equal(got, want), (x.shape, out, mismatch_report(got, want))
    with cf.ThreadPoolExecutor(6) as ex:
        for (x, out, want), got in zip(calls, ex.map(lambda t: linalg.linear8(t[0], b, bias, t[1], 6.0), calls)):
            assert f32_bits_equal(got, want), (x.shape, out, mismatch_report(got, want))
    b.close()

"""Linear calls on PackedB8 handles, whose streams and buffers are kept
between calls and shared by a device's handles: growing and shrinking row
counts, padded rows after full ones, several threads, against the CPU
oracle; what is kept, and that it is given back."""
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


def test_linear_workspaces_bounded():
    """Twelve handles (layers of a tower) called with 4,096 rows of 3,072 and
    outlier channels, about 115 MB of buffers a call: no more than 256 MiB
    stays with all of them together, an allocation that fails gives it back,
    and so does closing the last handle; calls of other shapes between give
    the oracle's bits."""
    import ctypes as C

    import torch

    from indecis_amd import _lib
    from indecis_amd.modernbert import Config, Model
    k, n, rows = 3072, 96, 4096
    rng = np.random.default_rng(7)
    q, s = linalg.pack_b8(rng.standard_normal((n, k), dtype=np.float32))
    q2, s2 = linalg.pack_b8(rng.standard_normal((33, 70), dtype=np.float32))
    cs2 = q2.astype(np.int32).sum(axis=1).astype(np.int32)
    layers, other = [linalg.PackedB8(q, s) for _ in range(12)], linalg.PackedB8(q2, s2)
    x, y = rng.standard_normal((rows, k), dtype=np.float32), rng.standard_normal((17, 70), dtype=np.float32)
    x[:, 5] *= 40
    want = orc.linear8(y, q2, s2, cs2, None, True, 6.0)

    def free():
        torch.cuda.synchronize()
        return torch.cuda.mem_get_info()[0]

    before, first = free(), None
    for b in layers:
        got = linalg.linear8(x, b, None, True, 6.0)
        first = got if first is None else first
        assert f32_bits_equal(got, first)
        assert f32_bits_equal(linalg.linear8(y, other, None, True, 6.0), want)
    assert before - free() <= (256 + 32) << 20
    huge = Model(None, cfg=Config(hidden=256, layers=1, heads=4, intermediate=512, vocab=700_000_000))
    tiny = np.zeros(16, np.float32)  # never read: the allocation fails first
    with pytest.raises(_lib.IxhError, match="out of memory|hip:"):
        _lib.check(_lib.lib().ixh_model_set_embeddings_f32(huge._h, tiny.ctypes.data_as(C.c_void_p)))
    huge.close()
    assert before - free() <= 32 << 20
    assert f32_bits_equal(linalg.linear8(x, layers[0], None, True, 6.0), first)
    for b in layers + [other]:
        b.close()
    assert before - free() <= 32 << 20


def test_linear_most_rows():
    """More row blocks of 16 than a grid's y dimension has (65,535), the last
    rows holding the massive values that make a channel an outlier."""
    k, n, rows = 16, 8, 65535 * 16 + 21
    rng = np.random.default_rng(11)
    q, s = linalg.pack_b8(rng.standard_normal((n, k), dtype=np.float32))
    cs = q.astype(np.int32).sum(axis=1).astype(np.int32)
    x = rng.standard_normal((rows, k), dtype=np.float32)
    x[-1, 3], x[-20, 7] = 500, -400
    b = linalg.PackedB8(q, s)
    got, want = linalg.linear8(x, b, None, True, 6.0), orc.linear8(x, q, s, cs, None, True, 6.0)
    assert f32_bits_equal(got, want), mismatch_report(got, want)
    b.close()

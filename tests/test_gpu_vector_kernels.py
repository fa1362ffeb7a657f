"""The standalone vector kernels at the edges of their splits: argmax at every alignment, remainders and special
values; RMSNorm at lengths off the multiples of 4 and past 4096, in place; the activation prep into a buffer of any
alignment."""
import ctypes as C

import numpy as np
import pytest

from weights import BF16, F32, MXFP4, Q4_0, Q8_0, rel_err

pytestmark = pytest.mark.gpu


def argmax_at(dev, x, off):
    """l3m_k_argmax of x placed off floats past a 16-byte boundary."""
    p, o = dev.put(np.concatenate([np.full(off, np.inf, np.float32), x])), dev.alloc(4)
    assert dev.lib.l3m_k_argmax(p + 4 * off, len(x), o, None) == 0
    return int(dev.get(o, 1, np.int32)[0])


@pytest.mark.parametrize("off", [0, 1, 2, 3])
@pytest.mark.parametrize("n", [1, 2, 3, 5, 63, 255, 256, 259, 1000, 1027, 4093, 4096, 4097, 4099, 24576, 24579, 50257, 131075])
def test_argmax_edges(dev, n, off):
    rng = np.random.default_rng(n + off)
    x = rng.standard_normal(n).astype(np.float32)
    assert argmax_at(dev, x, off) == int(np.argmax(x))
    for i in {0, n // 2, n - 1}:                               # one larger value at either end
        y = x.copy()
        y[i] = 50
        assert argmax_at(dev, y, off) == i
    y = np.full(n, -np.inf, np.float32)                        # all at the lowest: the first; NaN never wins
    assert argmax_at(dev, y, off) == 0
    y[0] = np.nan
    if n > 1:
        assert argmax_at(dev, y, off) == 1
        y[n // 2:] = 3.0
        assert argmax_at(dev, y, off) == max(n // 2, 1) - (n // 2 == 0)
    assert argmax_at(dev, np.full(n, np.nan, np.float32), off) == 0
    dev.free_all()


@pytest.mark.parametrize("n", [1, 3, 5, 255, 257, 1022, 4096, 4097, 16352])
def test_rmsnorm_edges(dev, n):
    rng = np.random.default_rng(n)
    x, w = rng.standard_normal(n).astype(np.float32), (1 + 0.1 * rng.standard_normal(n)).astype(np.float32)
    x64 = x.astype(np.float64)
    want = x64 / np.sqrt((x64 * x64).mean() + 1e-5) * w
    assert rel_err(dev.rmsnorm(x, w, 1e-5), want) < 1e-6       # a few roundings of 2^-24 and the sum's
    p = dev.put(np.concatenate([x, np.full(4, 7, np.float32)]))
    assert dev.lib.l3m_k_rmsnorm(p, p, dev.put(w), n, 1e-5, None) == 0     # in place, nothing past the end written
    got = dev.get(p, n + 4, np.float32)
    assert rel_err(got[:n], want) < 1e-6 and np.all(got[n:] == 7)
    dev.free_all()


@pytest.mark.parametrize("dtype", [F32, BF16, Q8_0, Q4_0, MXFP4])
@pytest.mark.parametrize("k", [2, 34, 1024, 1056, 4096])
def test_prep_any_alignment(dev, dtype, k):
    """The prepared bytes do not depend on where x and the output lie, and nothing is written past their end."""
    if dtype in (Q8_0, Q4_0, MXFP4):
        k = max(k // 32 * 32, 32)
    x = np.random.default_rng(k).standard_normal(k).astype(np.float32)
    want = dev.prep(dtype, x)
    n = len(want)
    src, dst = dev.put(np.concatenate([np.zeros(1, np.float32), x])), dev.put(np.full(n + 32, 0xA5, np.uint8))
    for off in (1, 2, 4, 8):
        assert dev.lib.l3m_k_prep(dtype, src + 4, k, dst + off, None) == 0
        got = dev.get(dst, n + 32, np.uint8)
        assert np.array_equal(got[off:off + n], want) and np.all(got[off + n:] == 0xA5)
        assert dev.lib.l3m_dev_upload(dst, np.full(n + 32, 0xA5, np.uint8).ctypes.data_as(C.c_void_p), n + 32) == 0
    dev.free_all()

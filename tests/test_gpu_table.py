"""The kernel table (l3m_kernels_hip) without the reference's library: host tiles repacked on the device equal the
host's l3m_lt_pack_ltiles byte for byte, and gemv and attend on host buffers meet the oracle."""
import ctypes as C

import numpy as np
import pytest

import l3m_amd as A
from weights import BF16, F32, MXFP4, Q4_0, Q8_0, rel_err, rows

pytestmark = pytest.mark.gpu
NAMES = {F32: "f32", BF16: "bf16", Q8_0: "q8_0", Q4_0: "q4_0", MXFP4: "mxfp4"}
TOL = {F32: 1e-3, BF16: 1e-3, Q8_0: 1e-3, Q4_0: 5e-3, MXFP4: 5e-3}   # test_gpu_kernels.py's bars
SCALE = {F32: 0, BF16: 0, Q8_0: 2, Q4_0: 2, MXFP4: 1}
BLOCK = {Q8_0: 32, Q4_0: 16, MXFP4: 16}


def make_tiles(dtype, w, n, k):
    """File rows as the reference's tiles (kernels.h:1-11)."""
    t = n // 16
    if dtype == F32:
        return np.ascontiguousarray(w.view(np.uint32).reshape(t, 16, k).transpose(0, 2, 1)).view(np.uint8).reshape(-1)
    if dtype == BF16:
        return np.ascontiguousarray(w.view(np.uint16).reshape(t, 16, k // 2, 2).transpose(0, 2, 1, 3)).view(np.uint8).reshape(-1)
    b = w.reshape(t, 16, k // 32, -1).transpose(0, 2, 1, 3)
    s, q = b[..., :SCALE[dtype]].reshape(t, k // 32, -1), b[..., SCALE[dtype]:]
    if dtype == Q8_0:
        q = (q ^ 0x80).reshape(t, k // 32, 16, 8, 4).transpose(0, 1, 3, 2, 4)
    else:
        c = np.concatenate([q & 15, q >> 4], 3).reshape(t, k // 32, 16, 4, 2, 4)
        q = (c[..., 0, :] | c[..., 1, :] << 4).transpose(0, 1, 3, 2, 4)
    return np.ascontiguousarray(np.concatenate([s, q.reshape(t, k // 32, -1)], 2)).reshape(-1)


@pytest.mark.parametrize("dtype", list(NAMES), ids=NAMES.get)
@pytest.mark.parametrize("ntiles,k", [(1, 32), (3, 288), (5, 2), (2, 18), (7, 1376), (128, 4096)])
def test_device_repack_equals_host(dev, dtype, ntiles, k):
    if dtype >= Q8_0 and k % 32:
        pytest.skip("quantized rows are whole blocks")
    lib = dev.lib
    lib.l3m_k_ltiles.argtypes = [C.c_int, C.c_int, C.c_int, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p]
    n = 16 * ntiles
    raw = np.random.default_rng(k + dtype).integers(0, 256, ntiles * (k * 64 if dtype == F32 else k * 32 if dtype == BF16 else
                                                    k // 32 * 16 * (BLOCK[dtype] + SCALE[dtype])), dtype=np.uint8)
    qs, ss = lib.l3m_lt_quant_size(dtype, n, k), lib.l3m_lt_scale_size(dtype, n, k)
    q, s = np.zeros(qs, np.uint8), np.zeros(max(ss, 1), np.uint8)
    lib.l3m_lt_pack_ltiles(dtype, ntiles, k, raw.ctypes.data, q.ctypes.data, s.ctypes.data)
    dr, dq, ds = dev.put(np.concatenate([raw, np.full(64, 0xA5, np.uint8)])), dev.alloc(qs), dev.alloc(max(ss, 16))
    assert lib.l3m_k_ltiles(dtype, ntiles, k, dr, dq, ds, None) == 0
    assert np.array_equal(dev.get(dq, qs, np.uint8), q)
    assert not ss or np.array_equal(dev.get(ds, ss, np.uint8), s[:ss])
    dev.free_all()


class Vec(C.Structure):                                # l3m_vec
    _fields_ = [(f, C.c_void_p) for f in ("f32", "bf16", "q8", "scale", "sum")]


class Table(C.Structure):                              # l3m_kernels
    _fields_ = [("name", C.c_char_p), ("gemv", C.CFUNCTYPE(None, C.c_void_p, C.c_void_p, C.c_int, C.c_int, C.c_void_p) * 5),
                ("attend", C.CFUNCTYPE(None, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p, C.c_int, C.c_int, C.c_int))]


@pytest.mark.parametrize("dtype", list(NAMES), ids=NAMES.get)
def test_table_gemv(oracle, dtype):
    """Sizes up, down and up again through the same staging buffers."""
    table = Table.in_dll(A.lib(), "l3m_kernels_hip")
    for k, ntiles in [(288, 3), (4096, 128), (32, 1), (1376, 5)]:
        n = 16 * ntiles
        w, x = rows(dtype, n, k, seed=k + dtype), np.random.default_rng(k).standard_normal(k).astype(np.float32)
        p = oracle.prepare(dtype, x)
        keep = {"f32": x, **p}
        v, y = Vec(**{f: a.ctypes.data for f, a in keep.items()}), np.full(n, np.nan, np.float32)
        tiles = make_tiles(dtype, w, n, k)
        table.gemv[dtype](y.ctypes.data, tiles.ctypes.data, ntiles, k, C.addressof(v))
        assert rel_err(y, oracle.gemv(dtype, w, n, k, x)) < TOL[dtype]


@pytest.mark.parametrize("hd,pos,stride", [(64, 100, 128), (48, 0, 48), (128, 511, 128), (64, 4000, 64)])
def test_table_attend(oracle, hd, pos, stride):
    table = Table.in_dll(A.lib(), "l3m_kernels_hip")
    rng = np.random.default_rng(9 + hd + pos)
    q, out = rng.standard_normal(hd).astype(np.float32), np.zeros(hd, np.float32)
    k, v = ((rng.integers(0, 1 << 16, (pos + 1) * stride, dtype=np.uint16) & 0xBFFF).astype(np.uint16) for _ in range(2))
    table.attend(out.ctypes.data, q.ctypes.data, k.ctypes.data, v.ctypes.data, pos, hd, stride)
    assert np.abs(out - oracle.attend(q, k, v, pos, hd, stride)).max() <= 1e-5

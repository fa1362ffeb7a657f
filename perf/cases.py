"""The work a program has this framework do, as cases that can be timed and compared.

Kinds of case:
  generate  Model.generate on a loaded model: `prompt` tokens, `new` greedy tokens after them; the logits of
            the last position (and the tokens, when there are any). A prompt with new = 0 is the time to the
            first logits.
  matvec    the activation prep and the matrix-vector product on device buffers (l3m_k_prep, l3m_k_gemv).
  mlp       an FFN block out of the single kernels: RMSNorm, prep, gate and up rows, SiLU, prep, down rows.
  head      a model's end out of the single kernels: RMSNorm, prep, the vocabulary's rows, argmax.
  attend    one query head over a K/V cache on device buffers (l3m_k_attend).
  table     the kernel table's matrix-vector product on host buffers (l3m_kernels_hip), as the reference's
            dispatcher calls it.
"""
import ctypes
import math
import struct
import tempfile
from pathlib import Path

import torch                              # before the library: both then use one HIP runtime
import numpy as np

import l3m_amd as A

# ------------------------------------------------------------------------------------------- cases


def _model(name, cfg, dtype, prompt, new, ctx=None):
    c = A.CONFIGS[cfg]
    return {"name": name, "kind": "generate", "arch": "llama", "dim": c.dim, "layers": c.n_layers, "heads": c.n_heads, "kv": c.n_kv_heads,
            "ffn": c.ffn_dim, "vocab": c.vocab, "ctx": ctx or c.ctx, "dtype": dtype, "prompt": prompt, "new": new}


def listed():
    return [
        # the benchmark's smallest model, one short completion: the launch and hand-over latency of decode
        _model("decode 15M bf16", "stories15M", "bf16", 1, 60),
        # the headline benchmark: greedy tokens from BOS until the context of 128 is full
        _model("decode 110M q4_0", "stories110M", "q4_0", 1, 126),
        # a long conversation: a prompt of 600 tokens, then tokens far into a context of 1024
        _model("long context 42M q8_0", "stories42M", "q8_0", 600, 64, ctx=1024),
        # the benchmark's chat prompt: 64 tokens to the first logits of the deepest model
        _model("prompt 64 135M q8_0", "smollm2", "q8_0", 64, 0),
        # a document as the prompt: nearly all of a context of 512
        _model("prompt 480 135M mxfp4", "smollm2", "mxfp4", 480, 0, ctx=512),
        # the same in the dtype whose activations are not quantized
        _model("prompt 200 15M bf16", "stories15M", "bf16", 200, 0),
        # the smallest matrix of the microbench: one call is launches and latency
        {"name": "matvec 768x288 bf16", "kind": "matvec", "rows": 768, "k": 288, "dtype": "bf16"},
        # its largest: the weight stream
        {"name": "matvec 14336x4096 q4_0", "kind": "matvec", "rows": 14336, "k": 4096, "dtype": "q4_0"},
        # an FFN block of a program that composes the kernels itself
        {"name": "mlp 768x2048 q8_0", "kind": "mlp", "dim": 768, "ffn": 2048, "dtype": "q8_0"},
        # the largest vocabulary of the configurations, with the greedy pick
        {"name": "head 49152x576 q8_0", "kind": "head", "dim": 576, "vocab": 49152, "dtype": "q8_0"},
        # one head at the end of a long cache
        {"name": "attend 4001 hd 128", "kind": "attend", "pos": 4000, "hd": 128, "stride": 128},
        # the drop-in table: the matrix comes from host memory on every call
        {"name": "table 2048x768 q8_0", "kind": "table", "rows": 2048, "k": 768, "dtype": "q8_0"},
    ]


def _log(rng, lo, hi, step=1):
    """A whole multiple of step from lo to hi, spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi + step)))
    return max(lo, min(hi, int(v) // step * step))


def draw(rng):
    kind = rng.choice(["decode", "prompt", "prompt", "matvec", "mlp", "head", "attend", "table"])
    dt = rng.choice(["bf16", "q8_0", "q4_0", "mxfp4"])
    if kind in ("decode", "prompt"):
        hd = rng.choice([32, 48, 64, 64])
        heads = rng.choice([4, 6, 8, 12] if hd == 48 else [4, 6, 8, 9, 12])
        arch = "gpt2" if kind == "decode" and dt != "mxfp4" and rng.random() < 0.2 else "llama"
        kv = heads if arch == "gpt2" else rng.choice([h for h in range(1, heads + 1) if heads % h == 0 and 4 * h >= heads])
        ctx = rng.choice([128, 256, 300, 512, 1024])
        case = {"kind": "generate", "arch": arch, "dim": heads * hd, "layers": rng.randint(2, 10), "heads": heads, "kv": kv,
                "ffn": _log(rng, 256, 2048, 32), "vocab": _log(rng, 1000, 49152), "ctx": ctx, "dtype": dt}
        if kind == "prompt":
            return {**case, "prompt": _log(rng, 8, ctx - 2), "new": 0}
        one = work({**case, "prompt": 1, "new": 0})["bytes"]
        return {**case, "prompt": 1, "new": min(_log(rng, 8, 100), int(6e9 / one) - 1)}
    if kind == "matvec":
        return {"kind": "matvec", "rows": _log(rng, 64, 14336), "k": _log(rng, 64, 4096, 32), "dtype": dt}
    if kind == "mlp":
        return {"kind": "mlp", "dim": _log(rng, 256, 1024, 32), "ffn": _log(rng, 512, 4096, 32), "dtype": dt}
    if kind == "head":
        return {"kind": "head", "dim": _log(rng, 256, 1024, 32), "vocab": _log(rng, 4096, 49152), "dtype": dt}
    if kind == "attend":
        hd = 8 * rng.randint(4, 16)
        return {"kind": "attend", "pos": _log(rng, 1, 8001) - 1, "hd": hd, "stride": hd * rng.choice([1, 1, 2, 3])}
    return {"kind": "table", "rows": 16 * _log(rng, 8, 256), "k": _log(rng, 128, 2048, 32), "dtype": dt}


# ------------------------------------------------------------------------------------------ inputs
# Weight blocks as the microbench specifies them: bf16 N(0, 0.02); q8_0 codes uniform with an f16 scale
# |N(0, 0.02)| / 127; q4_0 codes uniform, scale N(0, 0.02) / 8; mxfp4 codes uniform, exponents 119..123.

E2M1 = np.array([0, 0.5, 1, 1.5, 2, 3, 4, 6, 0, -0.5, -1, -1.5, -2, -3, -4, -6])


def _gen(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed((seed * 1000003 + salt) % (1 << 62))
    return g


def _host(t):
    return t.cpu().numpy()


def _bf16_bits(t):
    return _host(t.to(torch.bfloat16).view(torch.int16)).view(np.uint16)


def _rows(dtype, n, k, seed, salt):
    """File rows (uint8 [n, row bytes]) of an n x k matrix."""
    g = _gen(seed, salt)
    if dtype == "bf16":
        return _bf16_bits(torch.randn((n, k), generator=g, device="cuda") * 0.02).view(np.uint8).reshape(n, -1)
    nb = k // 32
    if dtype == "mxfp4":
        d = torch.randint(119, 124, (n, nb, 1), generator=g, device="cuda", dtype=torch.uint8)
    else:
        s = torch.randn((n, nb, 1), generator=g, device="cuda") * 0.02
        d = (s.abs() / 127 if dtype == "q8_0" else s / 8).to(torch.float16).view(torch.uint8)
    if dtype == "q8_0":
        q = torch.randint(-127, 128, (n, nb, 32), generator=g, device="cuda", dtype=torch.int8).view(torch.uint8)
    else:
        q = torch.randint(0, 256, (n, nb, 16), generator=g, device="cuda", dtype=torch.uint8)
    return _host(torch.cat([d, q], 2)).reshape(n, -1)


def _values(dtype, raw, k):
    """File rows in float64."""
    n = len(raw)
    if dtype == "f32":
        return torch.from_numpy(np.ascontiguousarray(raw).view(np.float32).reshape(n, k).copy()).cuda().double()
    if dtype == "bf16":
        return torch.from_numpy(np.ascontiguousarray(raw).view(np.int16).reshape(n, k).copy()).cuda().view(torch.bfloat16).double()
    b = torch.from_numpy(np.ascontiguousarray(raw).reshape(n, k // 32, -1).copy()).cuda()
    if dtype == "mxfp4":
        d, q = torch.exp2(b[..., :1].double() - 127), b[..., 1:]
    else:
        d, q = b[..., :2].contiguous().view(torch.float16).double(), b[..., 2:].contiguous()
    if dtype == "q8_0":
        v = q.view(torch.int8).double()
    else:
        c = torch.cat([q & 15, q >> 4], 2).long()
        v = c.double() - 8 if dtype == "q4_0" else torch.from_numpy(E2M1).cuda()[c]
    return (v * d).reshape(n, k)


def _matrix(dtype, raw, k):
    """A device matrix in the library's layout, as a program lays its weights out once."""
    dev = A.Device()
    return dev, dev.matrix(A.DTYPES[dtype], raw, k)


class _Owned:
    """Device buffers of a state, freed with it."""

    def __init__(self):
        self.devs = []

    def matrix(self, dtype, raw, k):
        dev, m = _matrix(dtype, raw, k)
        self.devs.append(dev)
        return m

    def __del__(self):
        for d in self.devs:
            d.free_all()


def _vec(n, seed, salt, mean=0.0, std=1.0):
    return mean + std * torch.randn(n, generator=_gen(seed, salt), device="cuda")


def _act(dtype, k):
    return torch.zeros(A.lib().l3m_act_bytes(A.DTYPES[dtype], k), dtype=torch.uint8, device="cuda")


def _model_file(case, seed, folder):
    c = A.Config("case", case["dim"], case["layers"], case["heads"], case["kv"], case["ffn"], case["vocab"], case["ctx"], case["dtype"])
    return A.write_model(Path(folder) / "m.l3m", c, seed=seed + 1, std=0.005, norm_jitter=0.1, arch=case["arch"])


def _ids(case, seed):
    return [0] if case["prompt"] == 1 else A.prompt(seed + 1, case["vocab"], case["prompt"])


class _Vec(ctypes.Structure):             # l3m_vec (include/l3m_hip.h)
    _fields_ = [(n, ctypes.c_void_p) for n in ("f32", "bf16", "q8", "scale", "sum")]


class _Table(ctypes.Structure):           # l3m_kernels
    _fields_ = [("name", ctypes.c_char_p), ("gemv", ctypes.CFUNCTYPE(None, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_void_p) * 5),
                ("attend", ctypes.c_void_p)]


def _prepared(x):
    """l3m_vec_prepare of float32 x: per 32 values q = rint(x * 127 / amax), the scale amax / 127, the sum of q."""
    b = x.reshape(-1, 32).astype(np.float32)
    am = np.abs(b).max(1, keepdims=True)
    inv = np.where(am > 0, np.float32(127) / np.where(am > 0, am, np.float32(1)), np.float32(0)).astype(np.float32)
    q = np.rint(b * inv)
    return q.astype(np.int8).reshape(-1), (am / np.float32(127)).reshape(-1), q.sum(1).astype(np.int32)


def _tiles(dtype, raw, n, k):
    """The reference's host tiles of 16 rows: bf16 [k/2][16][2]; else per 32 inputs the 16 scales, then q8 bytes
    (value + 128) at (i / 4 * 16 + row) * 4 + i % 4, or nibbles (8g + j low, 8g + 4 + j high) at (g * 16 + row) * 4 + j."""
    t = n // 16
    if dtype == "bf16":
        return np.ascontiguousarray(raw.view(np.uint16).reshape(t, 16, k // 2, 2).transpose(0, 2, 1, 3)).view(np.uint8).reshape(-1)
    b = raw.reshape(t, 16, k // 32, -1).transpose(0, 2, 1, 3)
    w = 1 if dtype == "mxfp4" else 2
    s, q = b[..., :w].reshape(t, k // 32, -1), b[..., w:]
    if dtype == "q8_0":
        q = (q ^ 0x80).reshape(t, k // 32, 16, 8, 4).transpose(0, 1, 3, 2, 4)
    else:
        c = np.concatenate([q & 15, q >> 4], 3).reshape(t, k // 32, 16, 4, 2, 4)
        q = (c[..., 0, :] | c[..., 1, :] << 4).transpose(0, 1, 3, 2, 4)
    return np.ascontiguousarray(np.concatenate([s, q.reshape(t, k // 32, -1)], 2)).reshape(-1)


def prepare(case, seed):
    kind, lib = case["kind"], A.lib()
    if kind == "generate":
        with tempfile.TemporaryDirectory() as d:
            return {"kind": kind, "model": A.Model(_model_file(case, seed, d), ctx=case["ctx"]), "ids": _ids(case, seed), "new": case["new"]}
    s = {"kind": kind, "lib": lib, "own": _Owned(), "dtype": A.DTYPES.get(case.get("dtype"))}
    if kind == "matvec":
        n, k, dt = case["rows"], case["k"], case["dtype"]
        s.update(k=k, w=s["own"].matrix(dt, _rows(dt, n, k, seed, 1), k), x=_vec(k, seed, 2), act=_act(dt, k), y=torch.empty(n, device="cuda"))
    elif kind == "mlp":
        d, f, dt = case["dim"], case["ffn"], case["dtype"]
        s.update(d=d, f=f, wg=s["own"].matrix(dt, _rows(dt, f, d, seed, 1), d), wu=s["own"].matrix(dt, _rows(dt, f, d, seed, 2), d),
                 wd=s["own"].matrix(dt, _rows(dt, d, f, seed, 3), f), x=_vec(d, seed, 4), nw=_vec(d, seed, 5, 1.0, 0.1),
                 h=torch.empty(d, device="cuda"), g=torch.empty(f, device="cuda"), u=torch.empty(f, device="cuda"),
                 a=_act(dt, d), b=_act(dt, f), y=torch.empty(d, device="cuda"))
    elif kind == "head":
        d, v, dt = case["dim"], case["vocab"], case["dtype"]
        s.update(d=d, v=v, w=s["own"].matrix(dt, _rows(dt, v, d, seed, 1), d), x=_vec(d, seed, 2), nw=_vec(d, seed, 3, 1.0, 0.1),
                 h=torch.empty(d, device="cuda"), a=_act(dt, d), y=torch.empty(v, device="cuda"), tok=torch.zeros(1, dtype=torch.int32, device="cuda"))
    elif kind == "attend":
        n, hd, st = case["pos"] + 1, case["hd"], case["stride"]
        s.update(pos=case["pos"], hd=hd, stride=st, q=_vec(hd, seed, 1), kc=_vec(n * st, seed, 2).to(torch.bfloat16), vc=_vec(n * st, seed, 3).to(torch.bfloat16),
                 y=torch.empty(hd, device="cuda"))
    else:
        n, k, dt = case["rows"], case["k"], case["dtype"]
        x = _host(_vec(k, seed, 2))
        keep = {"f32": x, "bf16": _bf16_bits(torch.from_numpy(x)), **dict(zip(("q8", "scale", "sum"), _prepared(x)))}
        s.update(k=k, ntiles=n // 16, tiles=_tiles(dt, _rows(dt, n, k, seed, 1), n, k), keep=keep, y=np.zeros(n, np.float32),
                 v=_Vec(**{f: a.ctypes.data for f, a in keep.items()}), table=_Table.in_dll(lib, "l3m_kernels_hip"))
    return s


# --------------------------------------------------------------------------------------------- run

def _ok(rc):
    if rc:
        raise RuntimeError((A.lib().l3m_dev_error() or b"?").decode())


def run(s):
    kind = s["kind"]
    if kind == "generate":
        toks = s["model"].generate(s["ids"], s["new"])
        out = {"logits": s["model"].logits}
        if s["new"]:
            out["tokens"] = np.array(toks, np.int32)
        return out
    lib, dt = s["lib"], s["dtype"]
    ref = ctypes.byref
    p = {n: t.data_ptr() for n, t in s.items() if isinstance(t, torch.Tensor)}
    if kind == "matvec":
        _ok(lib.l3m_k_prep(dt, p["x"], s["k"], p["act"], None))
        _ok(lib.l3m_k_gemv(ref(s["w"]), p["act"], s["k"], p["y"], None))
        return s["y"]
    if kind == "mlp":
        _ok(lib.l3m_k_rmsnorm(p["h"], p["x"], p["nw"], s["d"], 1e-5, None))
        _ok(lib.l3m_k_prep(dt, p["h"], s["d"], p["a"], None))
        _ok(lib.l3m_k_gemv(ref(s["wg"]), p["a"], s["d"], p["g"], None))
        _ok(lib.l3m_k_gemv(ref(s["wu"]), p["a"], s["d"], p["u"], None))
        _ok(lib.l3m_k_silu_mul(p["u"], p["g"], s["f"], None))
        _ok(lib.l3m_k_prep(dt, p["u"], s["f"], p["b"], None))
        _ok(lib.l3m_k_gemv(ref(s["wd"]), p["b"], s["f"], p["y"], None))
        return s["y"]
    if kind == "head":
        _ok(lib.l3m_k_rmsnorm(p["h"], p["x"], p["nw"], s["d"], 1e-5, None))
        _ok(lib.l3m_k_prep(dt, p["h"], s["d"], p["a"], None))
        _ok(lib.l3m_k_gemv(ref(s["w"]), p["a"], s["d"], p["y"], None))
        _ok(lib.l3m_k_argmax(p["y"], s["v"], p["tok"], None))
        return {"logits": s["y"], "token": s["tok"]}
    if kind == "attend":
        _ok(lib.l3m_k_attend(p["y"], p["q"], p["kc"], p["vc"], s["pos"], s["hd"], s["stride"], None))
        return s["y"]
    s["table"].gemv[dt](s["y"].ctypes.data, s["tiles"].ctypes.data, s["ntiles"], s["k"], ctypes.addressof(s["v"]))
    return s["y"]


# -------------------------------------------------------------------------------------------- work

def _wbytes(dtype, n):
    return n * {"f32": 4.0, "bf16": 2.0, "q8_0": 34 / 32, "q4_0": 18 / 32, "mxfp4": 17 / 32}[dtype]


def work(case):
    kind, dt = case["kind"], case.get("dtype")
    if kind == "generate":
        d, L, hd = case["dim"], case["layers"], case["dim"] // case["heads"]
        body = L * (2 * d * d + 2 * d * hd * case["kv"] + (2 if case["arch"] == "gpt2" else 3) * d * case["ffn"])
        P, new, head = case["prompt"], case["new"], d * case["vocab"]
        row = L * case["kv"] * hd * 2 * 2                     # K and V of one position, bf16
        passes = 1 + new                                      # the prompt in one, then a pass a token
        seen = sum(range(P, P + new + 1))
        return {"bytes": passes * (_wbytes(dt, body) + _wbytes(dt, head)) + row * (P + new + seen) + 4 * case["vocab"],
                "flops": 2.0 * body * (P + new) + 2.0 * head * passes + 4.0 * L * d * sum(range(1, P + new + 1))}
    if kind in ("matvec", "table"):
        n = case["rows"] * case["k"]
        return {"bytes": _wbytes(dt, n) + 4 * (case["rows"] + case["k"]), "flops": 2.0 * n}
    if kind == "mlp":
        n = 3 * case["dim"] * case["ffn"]
        return {"bytes": _wbytes(dt, n) + 12 * case["dim"], "flops": 2.0 * n}
    if kind == "head":
        n = case["dim"] * case["vocab"]
        return {"bytes": _wbytes(dt, n) + 8 * case["dim"] + 4 * case["vocab"], "flops": 2.0 * n}
    return {"bytes": 4.0 * (case["pos"] + 1) * case["hd"] + 8 * case["hd"], "flops": 4.0 * (case["pos"] + 1) * case["hd"]}


def tolerance(case):
    kind = case["kind"]
    if kind == "generate":
        # int8 activations (q8_0, q4_0, mxfp4 bodies): one rounding more or less in a layer flips rint decisions
        # in all that follow. The batched prefill against token by token, 2 to 30 layers: rel up to 0.0097, max
        # up to 0.039. bf16 rounds its activations to 8 bits (0.0029 from the 64-bit logits).
        return {"rel": 0.01, "max": 0.1} if case["dtype"] == "bf16" else {"rel": 0.03, "max": 0.15}
    if kind in ("mlp", "head"):
        return {"rel": 2e-3, "max": 0.05}                     # a flipped rint of the normalized activation
    return {"rel": 1e-5, "max": 1e-4}                         # 32-bit sums of exact products


# ------------------------------------------------------------------------------------------- exact

def _read(path):
    """name -> (dtype, rows, cols, bytes) of a .l3m file's tensors."""
    raw = np.fromfile(path, np.uint8)
    n, toc = struct.unpack_from("<I", raw, 64)[0], struct.unpack_from("<Q", raw, 72)[0]
    out = {}
    for e in range(toc, toc + 120 * n, 120):
        name = bytes(raw[e:e + 64]).split(b"\0")[0].decode()
        dt, nd = struct.unpack_from("<2I", raw, e + 64)
        shape = struct.unpack_from("<4Q", raw, e + 72)[:nd]
        off, size = struct.unpack_from("<2Q", raw, e + 104)
        out[name] = (A.DTYPE_NAMES[dt], shape if nd == 2 else (1, shape[0]), raw[off:off + size])
    return out


def _norm(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5) * w


def _exact_prompt(case, seed):
    """The logits after the prompt with every value in 64 bits (activations and K/V rows unrounded)."""
    with tempfile.TemporaryDirectory() as d:
        t = _read(_model_file(case, seed, d))

    def mat(name):
        dt, (r, c), raw = t[name]
        return _values(dt, raw.reshape(r, -1), c)

    P, H, KV, hd = case["prompt"], case["heads"], case["kv"], case["dim"] // case["heads"]
    ids = torch.tensor(_ids(case, seed), device="cuda")
    x = mat("embed")[ids]
    i = torch.arange(hd // 2, device="cuda", dtype=torch.float64)
    ang = torch.arange(P, device="cuda", dtype=torch.float64)[:, None] * 10000.0 ** (-2 * i / hd)
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]

    def rope(v):
        a, b = v[..., 0::2], v[..., 1::2]
        return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).flatten(-2)

    mask = torch.ones(P, P, device="cuda", dtype=torch.bool).tril()
    for layer in range(case["layers"]):
        def m(name):
            return mat(f"blk.{layer}.{name}")
        h = _norm(x, m("attn_norm"))
        q, k, v = rope((h @ m("wq").T).view(P, H, hd)), rope((h @ m("wk").T).view(P, KV, hd)), (h @ m("wv").T).view(P, KV, hd)
        o = []
        for j in range(H):
            sc = (q[:, j] @ k[:, j * KV // H].T / math.sqrt(hd)).masked_fill(~mask, -math.inf)
            o.append(torch.softmax(sc, -1) @ v[:, j * KV // H])
        x = x + torch.cat(o, 1) @ m("wo").T
        h = _norm(x, m("ffn_norm"))
        x = x + (torch.nn.functional.silu(h @ m("w_gate").T) * (h @ m("w_up").T)) @ m("w_down").T
    return (_norm(x[-1:], mat("norm")) @ mat("embed").T)[0]


def exact(case, seed):
    kind, dt = case["kind"], case.get("dtype")
    if kind == "generate":
        # greedy tokens are a chain of choices: no 64-bit value of the logits at its end
        if case["new"] or case["arch"] != "llama":
            return None
        return {"logits": _exact_prompt(case, seed)}
    if kind in ("matvec", "table"):
        # the product of the weights with the prepared activation, whose rounding the formats define
        x = _vec(case["k"], seed, 2)
        if dt == "bf16":
            a = x.to(torch.bfloat16).double()
        else:
            q, sc, _ = _prepared(_host(x))
            a = torch.from_numpy(q.reshape(-1, 32).astype(np.float64) * sc[:, None].astype(np.float64)).cuda().reshape(-1)
        return _values(dt, _rows(dt, case["rows"], case["k"], seed, 1), case["k"]) @ a
    if kind == "mlp":
        d, f = case["dim"], case["ffn"]
        h = _norm(_vec(d, seed, 4).double(), _vec(d, seed, 5, 1.0, 0.1).double())
        g, u = (_values(dt, _rows(dt, f, d, seed, i), d) @ h for i in (1, 2))
        return _values(dt, _rows(dt, d, f, seed, 3), f) @ (torch.nn.functional.silu(g) * u)
    if kind == "head":
        d = case["dim"]
        h = _norm(_vec(d, seed, 2).double(), _vec(d, seed, 3, 1.0, 0.1).double())
        return {"logits": _values(dt, _rows(dt, case["vocab"], d, seed, 1), d) @ h, "token": None}
    n, hd, st = case["pos"] + 1, case["hd"], case["stride"]
    q = _vec(hd, seed, 1).double()
    k, v = (_vec(n * st, seed, i).to(torch.bfloat16).double().view(n, st)[:, :hd] for i in (2, 3))
    return torch.softmax(k @ q / math.sqrt(hd), 0) @ v

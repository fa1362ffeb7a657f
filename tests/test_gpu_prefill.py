"""Batched prompt prefill on the GPU (int8 GEMMs on the matrix cores), through the l3m.h API.

A prompt of at least L3M_PREFILL_MIN (8) tokens runs its positions before the last in one batched pass
that fills the K/V cache; decoding then starts at the last prompt token. The logits after the prompt
must meet the engine bar of test_gpu_engine.py against the oracle (the reference's token-by-token order)
and against the GPU's own token-by-token path (L3M_PREFILL=0): equal argmax, KL < 0.01 nats, max-abs
within 2% of max|logit| (the int8 activation noise floor of the quantized paths). Prompts of 8 (the
threshold: 7 positions, less than one 16-token tile), 9 and 17 (a tile boundary), 40 and 100 tokens cover one to seven
16-token tiles of the GEMM and the attention (hd 64, 32 and 48 on the matrix cores, 32-position chunks), and 65
ends exactly at a tile's and a chunk's boundary; whole 32-blocks per head prepare the attention output inside the
attention kernel, hd 48 in one of its own. q4_0 and
mxfp4 bodies run the same int8 GEMM on q8_0 copies of their matrices with the same values (an mxfp4 block's
scale 2^(e-128) is an f16 and its doubled e2m1 codes are int8).
"""
import numpy as np
import pytest

import l3m_amd as A
from weights import read_tensors, to_bf16

pytestmark = pytest.mark.gpu
GQA = A.Config("pf_gqa", dim=192, n_layers=3, n_heads=6, n_kv_heads=2, ffn_dim=512, vocab=512, ctx=128, dtype="q8_0")
MHA = A.Config("pf_mha", dim=256, n_layers=2, n_heads=4, n_kv_heads=4, ffn_dim=640, vocab=512, ctx=128, dtype="q4_0")
MX = A.Config("pf_mx", dim=192, n_layers=2, n_heads=6, n_kv_heads=3, ffn_dim=512, vocab=512, ctx=128, dtype="mxfp4")
# hd 48: the attention output's blocks span heads, so it is prepared by a kernel of its own
HD48 = A.Config("pf_hd48", dim=192, n_layers=3, n_heads=4, n_kv_heads=2, ffn_dim=512, vocab=512, ctx=128, dtype="q8_0")


def kl(lr, lf):
    lr, lf = np.float64(lr), np.float64(lf)
    pr = np.exp(lr - lr.max()); pr /= pr.sum()
    lpr = lr - lr.max() - np.log(np.exp(lr - lr.max()).sum())
    lpf = lf - lf.max() - np.log(np.exp(lf - lf.max()).sum())
    return float((pr * (lpr - lpf)).sum())


def bf16(u):
    return (np.asarray(u, np.uint32) << 16).view(np.float32).astype(np.float64)


def ulps(a, b):
    """Distance in bf16 units in the last place (values of one sign; a sign change counts through zero)."""
    def key(u):
        u = np.asarray(u, np.int64)
        return np.where(u & 0x8000, -(u & 0x7FFF), u)
    return np.abs(key(a) - key(b))


def close(a, b):
    return int(np.argmax(a)) == int(np.argmax(b)) and kl(b, a) < 0.01 and np.abs(a - b).max() <= 0.02 * np.abs(b).max()


@pytest.mark.parametrize("n_prompt", [8, 9, 17, 40, 65, 100])
@pytest.mark.parametrize("cfg", [GQA, MHA, MX, HD48], ids=["q8_0-gqa", "q4_0-mha", "mxfp4-gqa", "q8_0-hd48"])
def test_prefill_logits(models, oracle, monkeypatch, cfg, n_prompt):
    print(f"case {cfg.name} prompt {n_prompt}", flush=True)
    path = models.get(cfg, cfg.dtype, seed=9, std=0.05, norm_jitter=0.1)
    ids = A.prompt(9, cfg.vocab, n_prompt)
    fast = A.Model(path)
    fast.generate(ids, 0)
    assert fast.prefilled == n_prompt - 1
    lf = fast.logits
    monkeypatch.setenv("L3M_PREFILL", "0")
    step = A.Model(path)
    step.generate(ids, 0)
    assert step.prefilled == 0
    ls = step.logits
    om = oracle.load(path)
    om.generate(ids, 0)
    lo = om.logits()
    assert close(lf, lo), (kl(lo, lf), np.abs(lf - lo).max() / np.abs(lo).max())
    assert close(lf, ls)
    # the K/V rows the prefill wrote, against the oracle's (the reference's token-by-token order) and the
    # GPU's own token-by-token rows
    hd, P = cfg.dim // cfg.n_heads, n_prompt - 1
    worst = {}
    for layer in range(cfg.n_layers):
        for kvh in range(cfg.n_kv_heads):
            kp, vp = fast.kv_rows(layer, kvh, 0, P, hd)
            ks, vs = step.kv_rows(layer, kvh, 0, P, hd)
            ko, vo = om.kv_rows(layer, kvh, 0, P, hd)
            for name, got_, tok_, ora in (("k", kp, ks, ko), ("v", vp, vs, vo)):
                g, t, o = bf16(got_), bf16(tok_), bf16(ora)
                scale = np.abs(o).max()
                assert np.abs(g - o).max() <= 0.02 * scale, (layer, kvh, name)
                assert np.abs(g - t).max() <= 0.02 * scale, (layer, kvh, name)
                if layer == 0:                        # before activation rounding can cascade: nearly exact
                    assert np.abs(g - o).max() <= 0.005 * scale, (layer, kvh, name)
                    assert np.mean(ulps(got_, ora) <= 1) >= 0.99, (layer, kvh, name)
                worst[name] = max(worst.get(name, 0.0), float(np.abs(g - o).max() / scale))
    print(f"prefill K/V vs oracle, worst max-abs / max|x|: {worst}", flush=True)
    # the continuation decodes over the prefilled cache: at every one of its 8 steps the GPU's token is the
    # oracle's argmax given the same prefix (its top two at a near-tie)
    got = fast.generate(ids, 8)
    assert fast.prefilled == P
    om2 = oracle.load(path)
    seq = list(ids) + got
    for k in range(len(got)):
        pos = len(ids) - 1 + k
        if k == 0:
            for p in range(pos):
                om2.forward(seq[p], p, logits=False)
        lg = om2.forward(seq[pos], pos).astype(np.float64)
        order = np.argsort(-lg, kind="stable")
        lv = np.sort(lg)
        tie = (lv[-1] - lv[-2]) / np.abs(lv).max() < 0.005
        assert got[k] == order[0] or (tie and got[k] == order[1]), (k, got, order[:2])


def test_prefill_graph_replays_equal_loose_launches(models, monkeypatch):
    """A prompt length's second prompt is captured as a graph and replayed from then on (its first, and all with
    L3M_PREFILL_GRAPH=0, are launched kernel by kernel). Every call, with decoding and other lengths run in between
    and a longer prompt's rows left in the buffers, gives logits and K/V rows bit-identical to the loose launches of
    the same prompt."""
    cfg = GQA
    path = models.get(cfg, cfg.dtype, seed=9, std=0.05, norm_jitter=0.1)
    hd = cfg.dim // cfg.n_heads
    graph = A.Model(path)
    monkeypatch.setenv("L3M_PREFILL_GRAPH", "0")
    loose = A.Model(path)
    for i, n_prompt in enumerate([40, 100, 40, 57, 100, 40, 100, 57, 57, 40]):
        print(f"call {i}: prompt {n_prompt}", flush=True)
        ids = A.prompt(20 + i, cfg.vocab, n_prompt)
        got = graph.generate(ids, 3)
        want = loose.generate(ids, 3)
        assert graph.prefilled == loose.prefilled == n_prompt - 1
        assert got == want
        assert np.array_equal(graph.logits, loose.logits)
        for layer in range(cfg.n_layers):
            for kvh in range(cfg.n_kv_heads):
                kg, vg = graph.kv_rows(layer, kvh, 0, n_prompt - 1, hd)
                kl_, vl = loose.kv_rows(layer, kvh, 0, n_prompt - 1, hd)
                assert np.array_equal(kg, kl_) and np.array_equal(vg, vl), (i, layer, kvh)


LONG = A.Config("pf_long", dim=128, n_layers=2, n_heads=4, n_kv_heads=2, ffn_dim=256, vocab=512, ctx=256, dtype="q8_0")


def test_prefill_past_128_positions(models, oracle, monkeypatch):
    """A 200-token prompt at ctx 256: 199 prefilled positions, past the 128-slot logits ring and over seven of
    the attention's 32-position chunks. The logits after the prompt meet the engine bar against the oracle
    and the GPU's token-by-token path, and each of the 30 greedy tokens that follow is the oracle's argmax
    given the same prefix (its second at a near-tie)."""
    path = models.get(LONG, "q8_0", seed=3, std=0.08, norm_jitter=0.2)
    ids = A.prompt(7, LONG.vocab, 200)
    om = oracle.load(path, ctx=256)
    om.generate(ids, 0)
    lo = om.logits()
    with A.Model(path, ctx=256) as m:
        m.generate(ids, 0)
        assert m.prefilled == 199
        lf = m.logits
        got = m.generate(ids, 30)
    om2, seq = oracle.load(path, ctx=256), list(ids) + got
    for p in range(len(ids) - 1):
        om2.forward(seq[p], p, logits=False)
    for k in range(len(got)):
        pos = len(ids) - 1 + k
        lg = om2.forward(seq[pos], pos).astype(np.float64)
        order, lv = np.argsort(-lg, kind="stable"), np.sort(lg)
        tie = (lv[-1] - lv[-2]) / np.abs(lv).max() < 0.005
        assert got[k] == order[0] or (tie and got[k] == order[1]), (k, got[k], order[:2])
    monkeypatch.setenv("L3M_PREFILL", "0")
    with A.Model(path, ctx=256) as m:
        m.generate(ids, 0)
        assert m.prefilled == 0
        ls = m.logits
    assert close(lf, lo), (kl(lo, lf), np.abs(lf - lo).max() / np.abs(lo).max())
    assert close(lf, ls)


def test_prefill_graph_cache_replaces_the_oldest(models, monkeypatch):
    """More prompt lengths than the eight a model keeps graphs of: eleven lengths, three prompts each (launched one by
    one, captured, replayed), then the first three so again (each replaced since) and the last (still kept). Every
    call's tokens and logits equal the loose launches' bit for bit."""
    path = models.get(GQA, GQA.dtype, seed=9, std=0.05, norm_jitter=0.1)
    graph = A.Model(path)
    monkeypatch.setenv("L3M_PREFILL_GRAPH", "0")
    loose = A.Model(path)
    lengths = list(range(10, 32, 2))
    for i, n_prompt in enumerate([n for n in lengths + lengths[:3] for _ in range(3)] + lengths[-1:]):
        ids = A.prompt(40 + n_prompt + i, GQA.vocab, n_prompt)
        got, want = graph.generate(ids, 2), loose.generate(ids, 2)
        assert graph.prefilled == loose.prefilled == n_prompt - 1
        assert got == want, (i, n_prompt)
        assert np.array_equal(graph.logits, loose.logits), (i, n_prompt)
    graph.close(); loose.close()


@pytest.mark.parametrize("n_prompt", [8, 17, 34, 130])
@pytest.mark.parametrize("hd", [16, 24, 80, 96, 112, 128])
@pytest.mark.parametrize("dtype", ["q8_0", "bf16"])
def test_prefill_attention_head_dims(models, oracle, dtype, hd, n_prompt):
    """The prompt's attention at head dims off the other tests': multiples of 16 up to 128 on the matrix cores
    (16-token tiles, 32-position chunks dealt to four wavefronts: 7, 16, 33 and 129 positions), 24 in the form
    with a wavefront per token and head; grouped KV heads. Logits and the second layer's K/V rows (which the
    first layer's attention enters) meet the bars of test_prefill_logits against the oracle."""
    heads = 4
    cfg = A.Config(f"pf_attn{hd}", dim=heads * hd, n_layers=2, n_heads=heads, n_kv_heads=2, ffn_dim=256, vocab=512, ctx=160, dtype=dtype)
    path = models.get(cfg, dtype, seed=11, std=0.05, norm_jitter=0.1)
    ids = A.prompt(12, cfg.vocab, n_prompt)
    om = oracle.load(path, ctx=160)
    om.generate(ids, 0)
    with A.Model(path, ctx=160) as m:
        m.generate(ids, 0)
        assert m.prefilled == n_prompt - 1
        assert close(m.logits, om.logits())
        for kvh in range(2):
            for got, want in zip(m.kv_rows(1, kvh, 0, n_prompt - 1), om.kv_rows(1, kvh, 0, n_prompt - 1, hd)):
                g, w = bf16(got), bf16(want)
                assert np.abs(g - w).max() <= 0.02 * np.abs(w).max(), kvh


# 33 tiles of 32 output rows in Wo and Wdown, 99 in q/k/v, 65 blocks of ffn: odd counts at every split of the GEMM
WIDE = A.Config("pf_wide", dim=1056, n_layers=2, n_heads=11, n_kv_heads=11, ffn_dim=2080, vocab=512, ctx=1024, dtype="q8_0")


@pytest.mark.parametrize("n_prompt", [34, 162, 500, 1000])
@pytest.mark.parametrize("dtype", ["q8_0", "bf16"])
def test_prefill_gemm_splits(models, monkeypatch, dtype, n_prompt):
    """The GEMM's three splits: 32 x 16 tiles over up to 8 wavefronts (Wo and Wdown at 33 positions), 32 x 32 tiles
    over 4 (q/k/v and gate/up at 33, all at 161, Wo and Wdown at 499), a wavefront a tile (q/k/v and gate/up at
    499, all at 999), with ragged last token tiles. Against the GPU's token-by-token path: the logits' bar of
    test_prefill_logits, the K/V rows within 2% of the largest, the first layer's (one matrix, before activation
    rounding can cascade) within 0.5%."""
    path = models.get(WIDE, dtype, seed=13, std=0.03, norm_jitter=0.1)
    ids = A.prompt(14, WIDE.vocab, n_prompt)
    out = []
    for prefill in ("1", "0"):
        monkeypatch.setenv("L3M_PREFILL", prefill)
        with A.Model(path, ctx=1024) as m:
            m.generate(ids, 0)
            assert m.prefilled == (n_prompt - 1 if prefill == "1" else 0)
            out.append((m.logits, [[m.kv_rows(layer, kvh, 0, n_prompt - 1) for kvh in (0, 5, 10)] for layer in (0, 1)]))
    (lf, kf), (ls, ks) = out
    assert close(lf, ls), (kl(ls, lf), np.abs(lf - ls).max() / np.abs(ls).max())
    for layer, bar in ((0, 0.005), (1, 0.02)):
        for got, want in zip(kf[layer], ks[layer]):
            for g, w in zip(got, want):
                g, w = bf16(g), bf16(w)
                assert np.abs(g - w).max() <= bar * np.abs(w).max(), (layer, np.abs(g - w).max() / np.abs(w).max())


@pytest.mark.parametrize("n_prompt", [8, 9, 17, 65, 100])
@pytest.mark.parametrize("cfg", [GQA, HD48], ids=["gqa", "hd48"])
def test_prefill_bf16(models, oracle, monkeypatch, cfg, n_prompt):
    """A bf16 body's prompt in one batched pass (bf16 products on the matrix cores): the logits' bars of
    test_prefill_logits against the oracle and the token-by-token path, both layers' K/V rows within 1% of the
    oracle's largest (an activation rounded to bf16, 2^-9 of its value, the other way after a sum in another
    order)."""
    path = models.get(cfg, "bf16", seed=9, std=0.05, norm_jitter=0.1)
    ids, hd, P = A.prompt(9, cfg.vocab, n_prompt), cfg.dim // cfg.n_heads, n_prompt - 1
    om = oracle.load(path)
    om.generate(ids, 0)
    with A.Model(path) as m:
        m.generate(ids, 0)
        assert m.prefilled == P
        lf, kv = m.logits, [m.kv_rows(layer, kvh, 0, P) for layer in range(cfg.n_layers) for kvh in range(cfg.n_kv_heads)]
    monkeypatch.setenv("L3M_PREFILL", "0")
    with A.Model(path) as m:
        m.generate(ids, 0)
        assert m.prefilled == 0
        ls = m.logits
    # KL and max-abs bars alone: two logits vectors within d of each other can differ in argmax where the top two
    # lie within 2 d (65 tokens of the hd 48 model: the token-by-token path and the oracle do)
    for ref in (om.logits(), ls):
        assert kl(ref, lf) < 0.01 and np.abs(lf - ref).max() <= 0.02 * np.abs(ref).max()
    want = [om.kv_rows(layer, kvh, 0, P, hd) for layer in range(cfg.n_layers) for kvh in range(cfg.n_kv_heads)]
    for g, w in zip(kv, want):
        for a, b in zip(g, w):
            assert np.abs(bf16(a) - bf16(b)).max() <= 0.01 * np.abs(bf16(b)).max()


def patch(path, out, edit):
    """A copy of the .l3m file at path with its tensors changed by edit(name -> writable uint8 view, 2-D for matrices)."""
    raw = np.fromfile(path, np.uint8)
    tensors, _ = read_tensors(path)
    toc = int(raw[72:80].view(np.uint64)[0])
    views = {}
    for i, (name, (_, _, data)) in enumerate(tensors.items()):
        off, size = (int(v) for v in raw[toc + 120 * i + 104:toc + 120 * i + 120].view(np.uint64))
        views[name] = raw[off:off + size].reshape(data.shape)
    edit(views)
    raw.tofile(out)
    return out


class Codes:
    """Element writes into a matrix of file rows: q8_0 codes (and block scales), or bf16 values."""

    def __init__(self, dtype, rows):
        self.q8, self.n = dtype == "q8_0", len(rows)
        self.r = rows.reshape(self.n, -1, 34) if self.q8 else rows.view(np.uint16)

    def put(self, row, col, code, scale=None, alone=False):
        """Column col = code (q8_0) or code * scale (bf16; scale 1 / 127); alone: the rest of its 32-block zero."""
        if self.q8:
            b = self.r[row, col // 32]
            if alone:
                b[..., 2:] = 0
            b[..., 2 + col % 32] = np.int8(code).view(np.uint8)
            if scale is not None:
                b[..., :2] = np.array([scale], np.float16).view(np.uint8)
        else:
            if alone:
                self.r[row, col // 32 * 32:col // 32 * 32 + 32] = 0
            self.r[row, col] = to_bf16([code * (1 / 127 if scale is None else scale)])[0]


@pytest.mark.parametrize("kind", ["nan_v", "inf_k"])
@pytest.mark.parametrize("hd", [32, 48, 64])
@pytest.mark.parametrize("dtype", ["q8_0", "bf16"])
def test_prefill_values_that_are_not_finite(models, oracle, tmp_path, dtype, hd, kind):
    """A prompt token X (position 5 of 20) whose K or V row in layer 0 is not finite, in one kv head; every other row
    is. nan_v: its V row holds NaN in every other dim (a sum of +inf and -inf), which the tokens before it never attend, so their second
    layer's rows are the oracle's; int8 bodies drop a NaN in the next rounding, so there the later tokens' are too.
    inf_k: its K row ends in infinities against which every q is negative: p is 0 exactly, and every row is the
    oracle's. Bar: 2% of the largest, as test_prefill_logits."""
    cfg = A.Config(f"pf_odd{hd}", dim=4 * hd, n_layers=2, n_heads=4, n_kv_heads=2, ffn_dim=256, vocab=128, ctx=64, dtype=dtype)
    base = models.get(cfg, dtype, seed=21, std=0.05, norm_jitter=0.1)
    P, at, X = 20, 5, 7
    ids = [X if i == at else 10 + i for i in range(P + 1)]
    a, b, const = 0, 32, 64                           # input columns: X alone is not 0 in a and b; no token is in const

    def edit(t):
        embed = Codes(dtype, t["embed"])
        for col in (a, b):
            embed.put(slice(None), col, 0)
            embed.put(X, col, 100)
        t["blk.0.attn_norm"].view(np.float32)[[a, b]] = 1e36
        wq, wk, wv = (Codes(dtype, t[f"blk.0.{n}"]) for n in ("wq", "wk", "wv"))
        for col in (a, b):
            for w in (wq, wk, wv):
                w.put(slice(None), col, 0)
        if kind == "nan_v":
            for col, code in ((a, 127), (b, -127)):
                wv.put(slice(0, hd, 2), col, code, 6e4, alone=True)
        else:
            embed.put(slice(None), const, 100)
            # the last RoPE pair hardly turns: +inf in row hd - 2 of kv head 0 from X makes both of its pair, and that
            # pair's q rows are negative for every token in the head's two query heads
            wk.put(slice(hd - 2, hd - 1), a, 127, 6e4, alone=True)
            for h in (0, 1):
                rows = slice((h + 1) * hd - 2, (h + 1) * hd)
                if dtype == "q8_0":
                    wq.r[rows, :, 2:] = 0
                else:
                    wq.r[rows] = 0
                wq.put(rows, const, -127)

    path = patch(base, tmp_path / "odd.l3m", edit)
    om = oracle.load(path)
    om.generate(ids, 0)
    with A.Model(path) as m:
        m.generate(ids, 0)
        assert m.prefilled == P
        for kvh in range(2):
            first = [bf16(w) for w in om.kv_rows(0, kvh, 0, P, hd)]
            bad = first[1] if kind == "nan_v" else first[0]
            assert (kvh == 0) == (not np.isfinite(bad[at]).all()) and np.isfinite(np.delete(bad, at, 0)).all()
            for name, got, want in zip("kv", m.kv_rows(1, kvh, 0, P), om.kv_rows(1, kvh, 0, P, hd)):
                g, w = bf16(got), bf16(want)
                if kind == "nan_v" and dtype == "bf16":
                    g, w = g[:at], w[:at]
                assert np.isfinite(w).all() and np.isfinite(g).all(), (name, kvh)
                assert np.abs(g - w).max() <= 0.02 * np.abs(w).max(), (name, kvh, np.abs(g - w).max() / np.abs(w).max())

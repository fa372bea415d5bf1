"""F32 weights: the prompt's products on the fp32 matrix cores and the decode
step's matvecs against float64 on the GPU's own inputs, at the edges of their
tiles and row segments.

Bound per output: kernel_check's for float32 sums, 1e-6 of sum |w||x| plus
two ulps of the result.  Of an output's K terms a wave adds K / 4 in a chain,
so K / 4 roundings of at most 2^-24 of the partial sum, which walk like their
square root: at K = 2080 about 23 x 6e-8 = 1.4e-6 of a partial sum that is
itself near sum |w||x| / K^0.5, far below the bound.
"""
import numpy as np
import pytest

import kernel_check as kc
from emberllm_amd import _native, configs, emberllm

pytestmark = pytest.mark.gpu


def model(name, dim, hidden, heads, kv, hd, bias, vocab=320):
    cfg = dict(configs.TINY["t_f32"], dim=dim, hidden_dim=hidden, n_heads=heads, n_kv_heads=kv, head_dim=hd,
               qkv_bias=bias, max_seq_len=1024, vocab_size=vocab)
    return configs.model_path("f32w_" + name, cfg)


def check(rep, name, W, x, out, pre=None, bias=None):
    y, mag = np.empty((len(x), W.rows)), np.empty((len(x), W.rows))
    x = x.astype(np.float64)
    r0 = 0
    for r0, w in W.chunks():
        y[:, r0:r0 + len(w)] = x @ w.T
        mag[:, r0:r0 + len(w)] = np.abs(x) @ np.abs(w).T
    if bias is not None:
        y += bias
    if pre is not None:
        y += pre
    rep.add(name, out, y, kc.SUM_TOL * mag + 2 * kc.F32_ULP * np.abs(y) + 1e-30)


# K of 3 blocks (a wave without any), 25 (uneven quarters) and 65; outputs and
# tokens that end inside a tile; the last two reach the 64 x 64 tiles
SHAPES = [("t", 96, 192, 2, 1, 48, 0), ("u", 800, 1056, 16, 8, 64, 1), ("v", 2080, 608, 2, 1, 64, 0)]


@pytest.mark.parametrize("shape,n", [(s, n) for s in SHAPES for n in (2, 31, 33, 70)] + [(SHAPES[1], 1000), (SHAPES[2], 1000)],
                         ids=lambda v: v[0] if isinstance(v, tuple) else str(v))
def test_prefill_products(shape, n):
    path = model(*shape)
    mf = kc.ModelFile(path)
    eng = emberllm.Engine(path, ctx=1024)
    ids = np.random.default_rng(n).integers(0, mf.V, n)
    got = []
    for layer in (0, 1):
        eng.debug_capture_prefill(layer, 0)
        eng.prefill(ids)
        got.append([np.asarray(eng.debug_read_prefill(s)[0]) for s in range(6)])
    eng.debug_capture_prefill(-1, 0)
    eng.close()
    xin, qkv, o, xmid, h13, xout = got[0]
    rep = kc.Report(f"{shape[0]} n {n}")
    bias = np.concatenate([mf.vec(f"layers.0.{w}_bias") for w in ("wq", "wk", "wv")]) if shape[6] else None
    check(rep, "qkv", mf.mat(mf.layer(0, "qkv")), kc.rmsnorm_f32(xin, mf.vec("layers.0.attn_norm"), mf.eps), qkv, bias=bias)
    check(rep, "wo", mf.mat(mf.layer(0, "wo")), o, xmid, pre=xin)
    check(rep, "w1|w3", mf.mat(mf.layer(0, "w13")), kc.rmsnorm_f32(xmid, mf.vec("layers.0.ffn_norm"), mf.eps), h13)
    check(rep, "w2", mf.mat(mf.layer(0, "w2")), kc.swiglu_f32(h13, mf.hid), xout, pre=xmid)
    print(rep, flush=True)
    assert rep.ok, str(rep)
    # the second run's layer 0 had its SwiGLU in the w1|w3 product, the first
    # run's as a kernel of its own: the same sums, the same function
    np.testing.assert_array_equal(got[1][0], xout)


# a pass that fills its context, whose last tile ends behind the last row of
# every buffer: the same logits as in a larger context
@pytest.mark.parametrize("shape,n", [(SHAPES[0], 33), (SHAPES[1], 70), (SHAPES[2], 1001)], ids=lambda v: v[0] if isinstance(v, tuple) else str(v))
def test_a_pass_that_fills_its_context(shape, n):
    path = model(*shape)
    ids = np.random.default_rng(n).integers(0, 320, n)
    out = []
    for ctx in (n, 1024):
        eng = emberllm.Engine(path, ctx=ctx)
        out.append(eng.prefill(ids))
        eng.close()
    assert np.isfinite(out[0]).all()
    np.testing.assert_array_equal(out[0], out[1])


# a row of 24 chunks (part of a wave), of 200, of 520 (two segments of 8 x 64
# chunks, the second short, with the looped activation prologue) and the
# widths of each segment size; the vocabulary's rows four to a wave
DECODE = SHAPES + [("w", 512, 768, 8, 4, 64, 0), ("x", 1024, 2048, 2, 1, 64, 1)]


@pytest.mark.parametrize("shape", DECODE, ids=lambda v: v[0])
def test_decode_products(shape):
    path = model(*shape, vocab=4101)
    mf = kc.ModelFile(path)
    eng = emberllm.Engine(path, ctx=1024)
    eng.prefill(np.arange(5))
    rep = kc.Report(shape[0])
    for step, layer in enumerate((0, 1)):
        eng.debug_capture(layer)
        logits = eng.forward(40 + step, 5 + step)
        xin, qkv, o, xmid, h, xout = (eng.debug_read(s)[None] for s in range(6))
        p = f"layers.{layer}."
        bias = np.concatenate([mf.vec(p + w + "_bias") for w in ("wq", "wk", "wv")]) if shape[6] else None
        check(rep, f"L{layer} qkv", mf.mat(mf.layer(layer, "qkv")), kc.rmsnorm_f32(xin, mf.vec(p + "attn_norm"), mf.eps), qkv, bias=bias)
        check(rep, f"L{layer} wo", mf.mat(mf.layer(layer, "wo")), o, xmid, pre=xin)
        x = kc.rmsnorm_f32(xmid, mf.vec(p + "ffn_norm"), mf.eps).astype(np.float64)
        w = np.concatenate([c for _, c in mf.mat(mf.layer(layer, "w13")).chunks()])
        g, u = (x @ w.T)[:, :mf.hid], (x @ w.T)[:, mf.hid:]
        mg, mu = (np.abs(x) @ np.abs(w).T)[:, :mf.hid], (np.abs(x) @ np.abs(w).T)[:, mf.hid:]
        sg = 1.0 / (1.0 + np.exp(-g))
        bound = kc.SUM_TOL * (np.abs(sg * (1.0 + g * (1.0 - sg)) * u) * mg + np.abs(g * sg) * mu) + 8 * kc.F32_ULP * np.abs(g * sg * u) + 1e-30
        rep.add(f"L{layer} swiglu", h, g * sg * u, bound)
        check(rep, f"L{layer} w2", mf.mat(mf.layer(layer, "w2")), h, xout, pre=xmid)
    check(rep, "head", mf.mat(mf.head_names()), kc.rmsnorm_f32(xout, mf.vec("final_norm"), mf.eps), logits[None])
    eng.debug_capture(-1)
    eng.close()
    print(rep, flush=True)
    assert rep.ok, str(rep)


# the attention on the product's raw rows: a fresh pass of one and of four
# row tiles, one behind a history, with interleaved and neox RoPE
@pytest.mark.parametrize("kv16", [False, True])
@pytest.mark.parametrize("hd,n,start", [(64, 5, 0), (64, 128, 0), (64, 33, 300), (128, 70, 0), (128, 3, 61)])
def test_attention_on_raw_rows(hd, n, start, kv16):
    cfg = dict(configs.TINY["t_f32"], dim=256, hidden_dim=1056, n_heads=4, n_kv_heads=2, head_dim=hd, max_seq_len=1024,
               qk_norm=int(hd == 128), rope_style=_native.ROPE_NEOX if hd == 128 else _native.ROPE_INTERLEAVED)
    path = configs.model_path(f"f32w_raw{hd}", cfg)
    mf = kc.ModelFile(path)
    ids = np.random.default_rng(n).integers(0, mf.V, start + n)
    eng = emberllm.Engine(path, ctx=1024, kv_fp16=kv16)
    if start:
        eng.prefill(ids[:start])
    eng.debug_capture_prefill(1, 0)
    eng.prefill(ids[start:], start=start)
    qkv, o = (np.asarray(eng.debug_read_prefill(s)[0], dtype=np.float32) for s in (1, 2))
    k, v = (kc.cache_rows(eng.kv_read(w, 1, start + n), mf, kv16) for w in (0, 1))
    eng.debug_capture_prefill(-1, 0)
    eng.close()
    rep = kc.Report(f"raw rows, hd {hd}, n {n} at {start} kv16={kv16}")
    pos = start + np.arange(n)
    kc.check_kv_rows(rep, "kv store", mf, 1, qkv, pos, k, v, kv16)
    kc.check_attention(rep, "attention", mf, 1, qkv, pos, k, v, o)
    print(rep, flush=True)
    assert rep.ok, str(rep)

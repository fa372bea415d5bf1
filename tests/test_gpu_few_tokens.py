"""Passes of few tokens: their products (gemm_few.hip), and their attention
behind a history (k_pf_few_attn, k_pf_few_merge), against float64 on the GPU's
own inputs at the edges of their tiles (kernel_check's bounds).

The products' sums: K is split over up to 16 waves of at most 16 blocks each,
so a sum is a chain of at most 16 fmas and one of at most 15 additions, within
the depth kernel_check's 1e-6 of sum |terms| is stated for."""
import numpy as np
import pytest

import kernel_check as kc
from emberllm_amd import _native, configs, emberllm

pytestmark = pytest.mark.gpu

Q8, Q4 = _native.DT_Q8_0, _native.DT_Q4_0


def model(name, dim, hidden, heads, kv, hd, dtype, **kw):
    cfg = dict(configs.TINY["t_qwen3"], dim=dim, hidden_dim=hidden, n_heads=heads, n_kv_heads=kv, head_dim=hd, dtype=dtype,
               max_seq_len=2048, vocab_size=640, tied=1, qk_norm=kw.get("norm", 0), qkv_bias=kw.get("bias", 0),
               rope_style=kw.get("rope", _native.ROPE_NEOX))
    return configs.model_path("few_" + name, cfg)


# K of 3, 8, 9, 18, 28 and 32 blocks in the normalized products, of 4 to 257
# in wo and w2; 1, 2, 3 and 7 query heads per kv head
SHAPES = {
    "a": ("a", 96, 1056, 2, 2, 64, Q8, dict(rope=_native.ROPE_INTERLEAVED)),
    "b": ("b", 576, 1536, 9, 3, 64, Q4, dict(bias=1)),
    "c": ("c", 896, 5120, 14, 2, 64, Q8, dict(bias=1, norm=1)),
    "d": ("d", 1024, 3072, 16, 8, 128, Q8, dict(norm=1)),
    "e": ("e", 1024, 1024, 4, 2, 128, Q4, dict(norm=1)),
    # raw rows with a bias and interleaved RoPE; w2 of the most inputs, four
    # chunks per wave, and of one block more, which the staged kernels take
    "f": ("f", 256, 8192, 4, 2, 128, Q8, dict(bias=1, rope=_native.ROPE_INTERLEAVED)),
    "g": ("g", 288, 8192, 3, 1, 128, Q4, dict(bias=1, norm=1, rope=_native.ROPE_INTERLEAVED)),
    "h": ("h", 256, 8224, 4, 2, 64, Q8, dict()),
}


def run(shape, n, kv16, start):
    *s, kw = SHAPES[shape]
    path = model(*s, **kw)
    mf = kc.ModelFile(path)
    ids = np.random.default_rng(n + start).integers(0, mf.V, start + n)
    eng = emberllm.Engine(path, ctx=max(start + n, 512), kv_fp16=kv16)
    if start:
        eng.prefill(ids[:start])
    rep = kc.Report(f"{shape} n {n} at {start} kv16={kv16}")
    for layer in (0, 1):
        eng.debug_capture_prefill(layer, 0)
        eng.prefill(ids[start:], start=start)
        slots = [np.asarray(eng.debug_read_prefill(k)[0]) for k in range(6)]
        k, v = (kc.cache_rows(eng.kv_read(w, layer, start + n), mf, kv16) for w in (0, 1))
        kc.check_prefill_layer(rep, mf, layer, slots, start, k, v, kv16)
    eng.debug_capture_prefill(-1, 0)
    eng.close()
    print(rep, flush=True)
    assert rep.ok, str(rep)


@pytest.mark.parametrize("n", [1, 15, 17, 128])
@pytest.mark.parametrize("shape", list(SHAPES))
def test_products(shape, n):
    run(shape, n, False, 0)


# two token tiles per workgroup in w1|w3 alone and in wo and w2, the last one
# with a single token
@pytest.mark.parametrize("shape,n", [("b", 81), ("d", 49), ("d", 97), ("b", 241)])
def test_two_token_tiles(shape, n):
    run(shape, n, True, 0)


# a history inside the first tile, on a tile's edge, off it, of many key
# ranges; rows that fill 64-row tiles to the last and past it, up to the four
# the kernel takes and one more, which it does not
@pytest.mark.parametrize("shape,n,start,kv16", [("a", 1, 1, False), ("a", 64, 640, True), ("b", 22, 129, False), ("b", 85, 1500, True),
                                                ("c", 36, 63, True), ("c", 37, 640, False), ("d", 23, 517, True), ("d", 128, 1900, False),
                                                ("d", 2, 126, False), ("d", 16, 250, True), ("d", 1, 63, False), ("d", 9, 64, True),
                                                ("e", 33, 65, True), ("e", 9, 2000, False), ("f", 16, 250, True),
                                                ("g", 7, 63, False)])
def test_attention_behind_a_history(shape, n, start, kv16):
    run(shape, n, kv16, start)

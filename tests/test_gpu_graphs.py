"""Captured graphs of decode steps and prefill passes against plain launches."""
import numpy as np
import pytest

from emberllm_amd import _native, configs, emberllm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["t_qwen3", "t_f32"])
def test_a_graph_that_cannot_be_had(monkeypatch, name):
    """A step or pass whose graph cannot be instantiated has run all the same:
    it returns its logits, and so do the next ones, without graphs."""
    path = configs.model_path(name)
    V = configs.ALL[name]["vocab_size"]
    plain = emberllm.Engine(path)
    plain.set_graph(False)
    monkeypatch.setenv("EHIP_GRAPH_TEST_FAIL", "1")
    eng = emberllm.Engine(path)
    rng = np.random.default_rng(3)
    for round_ in range(3):
        ids = rng.integers(0, V, 7)
        np.testing.assert_array_equal(eng.prefill(ids), plain.prefill(ids))
        for pos in range(7, 11):
            tok = int(rng.integers(0, V))
            np.testing.assert_array_equal(eng.forward(tok, pos), plain.forward(tok, pos))
        if round_ == 1:
            eng.set_graph(True)   # tries once more
    eng.close()
    plain.close()


Q8, Q4, F32 = _native.DT_Q8_0, _native.DT_Q4_0, _native.DT_F32


def wide(name, **kw):
    """Two layers whose passes take the few-token products (inputs of at least 1,024 in one of them)."""
    cfg = dict(configs.TINY["t_qwen3"], dim=256, hidden_dim=1056, n_heads=4, n_kv_heads=2, head_dim=64, qk_norm=0, tied=1,
               vocab_size=640, max_seq_len=1024)
    cfg.update(kw)
    return configs.model_path("graphs_" + name, cfg)


MODELS = {
    "q8_64": dict(dtype=Q8),
    "q8_128": dict(dtype=Q8, head_dim=128, qk_norm=1),     # raw rows up to 16 tokens
    "q4_128": dict(dtype=Q4, head_dim=128, qk_norm=1),
    "f32_64": dict(dtype=F32, rope_style=_native.ROPE_INTERLEAVED),   # raw rows
    "f32_128": dict(dtype=F32, head_dim=128, qk_norm=1),
    "narrow": dict(dtype=Q8, hidden_dim=512),              # exact-order attention
}
# (first position, tokens): one and several row tiles, behind a history of a
# few key tiles and of many (with the merge), longer than the few-token
# products; more than the eight graphs a state keeps, the first one again at
# the end
PASSES = [(0, 5), (0, 33), (0, 128), (0, 300), (0, 700), (63, 2), (64, 64), (300, 23), (640, 9), (700, 40), (0, 5)]


@pytest.mark.parametrize("kv16", [False, True])
@pytest.mark.parametrize("name", list(MODELS))
def test_every_pass_of_a_shape(name, kv16):
    """A prefill pass shape is launched, launched and captured, then replayed:
    each time, with other tokens, it gives the logits and the cache of plain
    launches, also after its graph had to make room for others."""
    path = wide(name, **MODELS[name])
    eng, plain = (emberllm.Engine(path, ctx=768, kv_fp16=kv16) for _ in range(2))
    plain.set_graph(False)
    rng = np.random.default_rng(len(name))
    for start, n in PASSES:
        for call in range(4):
            ids = rng.integers(0, 640, n)
            got, want = eng.prefill(ids, start=start), plain.prefill(ids, start=start)
            assert np.isfinite(want).all()
            np.testing.assert_array_equal(got, want, err_msg=f"{n} tokens at {start}, call {call}")
            tok = int(rng.integers(0, 640))   # a decode step between the passes
            np.testing.assert_array_equal(eng.forward(tok, start + n), plain.forward(tok, start + n))
        for layer in (0, 1):
            for which in (0, 1):
                a, b = (e.kv_read(which, layer, start + n + 1) for e in (eng, plain))
                np.testing.assert_array_equal(a, b)
    eng.close()
    plain.close()

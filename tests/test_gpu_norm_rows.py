"""The RMSNorm of a prompt's rows has one order of summation: the rows behind
layer 0's attn_norm (normalized with the embedding, k_quant_rows) and behind
its ffn_norm (k_norm_rows) agree bit for bit where their inputs do.

The model makes the two visible: wo is zero, so both norms see the embedded
rows; wq and w1 are identities, so their products are the normalized rows (a
sum of one term and zeros has no rounding)."""
import shutil

import numpy as np
import pytest

import kernel_check as kc
from emberllm_amd import configs, emberllm

pytestmark = pytest.mark.gpu


# one and two 16-byte pieces per thread, the last one short
@pytest.mark.parametrize("dim,kv", [(128, 2), (960, 15), (1024, 8), (1088, 17), (2048, 8)])
def test_one_order_of_summation(tmp_path, dim, kv):
    cfg = dict(configs.TINY["t_f32"], dim=dim, hidden_dim=dim, n_heads=dim // 64, n_kv_heads=kv, head_dim=64, vocab_size=320)
    path = str(tmp_path / "norms.ember")
    shutil.copy(configs.model_path(f"norms{dim}", cfg), path)
    mf = kc.ModelFile(path)
    raw = np.memmap(path, dtype=np.uint8, mode="r+")

    def put(name, value):
        off, n = int(mf.t[name].offset), int(mf.t[name].nbytes)
        raw[off:off + n].view("<f4")[:] = np.asarray(value, dtype=np.float32).ravel()

    norm = np.random.default_rng(dim).uniform(0.5, 1.5, dim)
    put("layers.0.attn_norm", norm)
    put("layers.0.ffn_norm", norm)
    put("layers.0.wq", np.eye(dim))
    put("layers.0.w1", np.eye(dim))
    put("layers.0.wo", np.zeros((dim, dim)))
    raw.flush()
    eng = emberllm.Engine(path, ctx=64)
    eng.debug_capture_prefill(0, 0)
    eng.prefill(np.arange(64) * 5 % 320)
    xin, qkv, _, xmid, h13, _ = (np.asarray(eng.debug_read_prefill(s)[0]) for s in range(6))
    eng.close()
    np.testing.assert_array_equal(xin, xmid)
    np.testing.assert_array_equal(qkv[:, :dim], h13[:, :dim])
    want = kc.rmsnorm_f32(xin, norm.astype(np.float32), mf.eps)
    np.testing.assert_allclose(h13[:, :dim], want, rtol=1e-5)

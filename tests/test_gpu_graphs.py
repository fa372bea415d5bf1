"""Captured graphs of decode steps and prefill passes against plain launches."""
import numpy as np
import pytest

from emberllm_amd import configs, emberllm

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

"""Prompt passes of fp32 files whose hidden_dim is not a multiple of 64: the copy's rows of w2 are filled up with zeros.

The product kernels of the copy and the fused ones multiply the same bf16 values in the same order, and a zero weight adds nothing:
logits and cache are equal bit for bit, at every length and after the buffers have grown."""
import numpy as np
import pytest

from test_gpu_model import _model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,hidden", [(64, 8), (64, 56), (128, 72), (192, 1376), (64, 4200)])
def test_hidden_between_steps(pkg, dim, hidden):
    from llama2_jl_amd import synth
    lm = _model(pkg, "PLAN_F32", dim=dim, hidden_dim=hidden, n_layers=2, n_heads=dim // 32, n_kv_heads=dim // 32, vocab_size=128, seq_len=330,
                rope_freq_base=10000.0, rope_is_neox=False)
    dev = lm.device()
    for n in (1, 17, 64, 65, 130, 321):
        prompt = synth.seeded_prompt(n, n, 128)
        got = []
        for copy in (True, False):
            dev.set_prefill_copy(copy)
            dev.reset()
            logits, nxt = dev.prefill(prompt, 0)
            assert not dev.prefill_library
            got.append((logits.copy(), nxt, *[a.copy() for a in dev.kv_read(1, 0, n)]))
        assert got[0][1] == got[1][1]
        for a, b in zip(got[0], got[1]):
            assert np.array_equal(a, b), n

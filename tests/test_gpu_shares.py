"""Dense products of a bf16 prompt whose positions go in equal shares of 64 to 320: each size of a share, shares of unequal size, a last one with a single
position; Llama's w1 | w3 (the same sums as from the quantized blocks, bit for bit) and the layered models' gated and plain feed-forwards."""
import numpy as np
import pytest

import layered_cases as lc
from test_gpu_tiles import SAME, TOL, _model

pytestmark = pytest.mark.gpu

# (positions, rows): one share of 1 .. 5 units; 3 + 3, 4 + 4 + 3, 2 + 1, ... by what fits the compute units
SIZES = [(60, 28672), (120, 28672), (190, 28672), (250, 28672), (320, 28672), (321, 28672), (700, 28672), (129, 28672), (385, 9216), (1025, 9216), (129, 512), (577, 2560)]


@pytest.mark.parametrize("n,rows", SIZES)
def test_llama(pkg, n, rows):
    from llama2_jl_amd import synth
    cfg = pkg.ModelConfig(dim=256, hidden_dim=rows // 2, n_layers=1, n_heads=4, n_kv_heads=2, vocab_size=320, seq_len=n, rope_freq_base=10000.0, rope_is_neox=False)
    lm = synth.synthetic_model(cfg, synth.PLAN_Q4_K_S, seed=5)
    tok = lc.tokens(n, 320, 2)
    got = []
    for copy in (True, False):
        lm._device = None
        dev = lm.device()
        dev.set_prefill_library(False)
        dev.set_prefill_copy(copy)
        got.append(dev.prefill_logits(tok, np.arange(n)))
        dev.close()
    assert np.isfinite(got[0]).all() and np.array_equal(got[0], got[1])


@pytest.mark.parametrize("kind", ["gated", "plain"])
@pytest.mark.parametrize("n,rows", [(n, r) for n, r in SIZES if n >= 128])
def test_layered(pkg, kind, n, rows):
    lm, ref = _model(pkg, kind, rows - 6, n)
    tok = lc.tokens(n, 50, 2)
    want, got = ref.run(tok), {}
    for images in (True, False):
        lm._device = None
        dev = lm.device()
        dev.set_prefill_copy(images)
        got[images] = dev.prefill_logits(tok, np.arange(n))
        assert dev.chosen("tile_images") == (1 if images else 0)
        dev.close()
    for lo in range(0, n, 64):
        assert lc.error(got[True][lo:lo + 64], want[lo:lo + 64]) <= TOL, lo
        assert lc.error(got[True][lo:lo + 64], got[False][lo:lo + 64]) <= SAME, lo

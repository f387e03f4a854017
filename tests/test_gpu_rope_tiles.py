"""The launch between projections and attention of a Llama prompt (rotation, cache rows, attention tiles): a prompt in pieces.

A piece's first tile of 32 keys may hold earlier positions (from the fp32 cache) and new ones (from the projections).  Rotation,
cache rows and the tiles' bf16 values of a position don't depend on where the pieces begin, and neither do an fp32 file's other steps
(own product kernels: one order of sums for every position): caches and logits equal those of one piece, bit for bit."""
import numpy as np
import pytest

from test_gpu_model import _model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size,neox", [(32, False), (64, True), (96, True), (128, False)])
def test_prompt_in_pieces(pkg, size, neox):
    from llama2_jl_amd import synth
    lm = _model(pkg, "PLAN_F32", dim=4 * size, hidden_dim=256, n_layers=2, n_heads=4, n_kv_heads=2, vocab_size=128, seq_len=150,
                rope_freq_base=10000.0, rope_is_neox=neox)
    dev = lm.device()
    dev.set_prefill_library(False)
    tok = synth.seeded_prompt(size, 150, 128)
    want = None
    for cuts in ((0, 150), (0, 1, 33, 64, 150), (0, 31, 32, 95, 129, 150), (0, 45, 46, 149, 150)):
        dev.reset()
        for a, b in zip(cuts, cuts[1:]):
            logits, nxt = dev.prefill(tok[a:b], a)
        got = [logits.copy(), np.int32(nxt)] + [x.copy() for l in range(2) for x in dev.kv_read(l, 0, 150)]
        want = want or got
        for a, b in zip(want, got):
            assert np.array_equal(a, b), cuts

"""bf16 products of 17 to 200 positions (and fewer, of many inputs): tiles of 32 and 64 rows x 32 and 64 positions, workgroups that share a tile's inputs,
experts' rows a tile at a time, inputs that do not go round four wavefronts, row counts that are no multiple of anything.  Against the restatement, and every
call again: the same bits, whoever was through last."""
import numpy as np
import pytest

import layered_cases as lc
from oracle import layered_np as ref

pytestmark = pytest.mark.gpu

TOL = 3e-2  # bf16 activations against 64 bits, as for the other prompts


def _check(pkg, c, sizes, seed):
    t = lc.settle_routers(c, ref.random_tensors(c, seed), seed)
    tok = lc.tokens(max(sizes), c["vocab"], 4)
    want = ref.Sequence(c, t).run(tok)
    dev = lc.language_model(pkg, c, t, precision="bfloat16").device()
    dev.set_prefill_library(False)
    for n in sizes:
        at = np.arange(max(0, n - 70), n)
        got = dev.prefill_logits(tok[:n], at)
        assert lc.error(got, want[at]) <= TOL, n
        assert np.array_equal(got, dev.prefill_logits(tok[:n], at)), n
    dev.close()


# inputs of the down product: 65, 64 and 130 steps of 64, shared by 4, 4 and 8 workgroups a tile; of 1300 rows by 2 from 129 positions on
@pytest.mark.parametrize("width,ff,sizes", [(334, 4150, (3, 16, 17, 32, 33, 64, 65, 130)), (66, 8310, (9, 40, 96)), (1300, 4096, (24, 60, 129, 190))])
def test_shared_inputs(pkg, width, ff, sizes):
    c = lc.config([lc.attention(heads=2, kv_heads=1, dim=32, vdim=32, rot=32, mlp=lc.dense(ff))], width=width, vocab=120)
    _check(pkg, c, sizes, 61)


# logits of up to 70 positions: 32 x 32, 64 x 32 and 64 x 64 of 8210 rows, 32 x 64 of 4120; 5 and 6 steps of inputs
@pytest.mark.parametrize("vocab,width", [(8210, 334), (4120, 300), (16390, 257)])
def test_many_rows(pkg, vocab, width):
    c = lc.config([lc.attention(heads=2, kv_heads=1, dim=16, vdim=16, rot=16, mlp=lc.dense(515))], width=width, vocab=vocab)
    _check(pkg, c, (5, 8, 17, 32, 33, 64, 65, 70), 62)


# few inputs, 2, 3, 4 and 6 steps: the other kernel's tiles of 16 x 32 and 32 x 64, k_gemm's from 65 positions on of many rows, the ring's where it has one round
@pytest.mark.parametrize("width,vocab", [(66, 8210), (130, 16400), (200, 4120), (250, 16390), (330, 12300)])
def test_few_inputs(pkg, width, vocab):
    c = lc.config([lc.attention(heads=2, kv_heads=1, dim=16, vdim=16, rot=16, mlp=lc.dense(515))], width=width, vocab=vocab)
    _check(pkg, c, (17, 33, 64, 65), 65)


# (experts, chosen, rows of the up product): few rows, up to 8 positions an expert on average and more; many rows; an expert with more than 64
@pytest.mark.parametrize("experts,top,rows", [(8, 2, 70), (8, 4, 2100), (3, 1, 520)])
def test_experts(pkg, experts, top, rows):
    c = lc.config([lc.attention(heads=2, kv_heads=1, dim=16, vdim=16, rot=16, mlp=lc.moe(experts, top, rows))], width=330, vocab=60)
    _check(pkg, c, (6, 17, 33, 70, 110, 127), 63)


# w1 | w3 in tiles of 32 x 32, 32 x 64, 64 x 32 and 64 x 64; eighths of 7, 9 and 21 steps of inputs, of which one is empty or some are longer; of 2, 3 and 6
# steps, and up to 16 positions of 2048 rows, straight to registers, in tiles of 32 x 32 and 64 x 64
@pytest.mark.parametrize("dim,hidden,lengths", [(128, 2048, (33, 65, 128, 130)), (192, 8192, (1, 8, 17, 40, 64)), (1344, 4160, (24, 64, 70, 128)),
                                                (384, 1088, (64, 300)), (448, 4096, (33, 65, 128)), (576, 1024, (1, 16, 17))])
def test_llama(pkg, dim, hidden, lengths):
    """Against the products that sum their inputs in one part: one more rounding to bf16 the other way for the odd element, as for other prompts with
    and without the library's products"""
    from llama2_jl_amd import synth
    cfg = pkg.ModelConfig(dim=dim, hidden_dim=hidden, n_layers=2, n_heads=dim // 32, n_kv_heads=1, vocab_size=256, seq_len=max(lengths), rope_freq_base=10000.0,
                          rope_is_neox=False)
    dev = synth.synthetic_model(cfg, synth.PLAN_F32, seed=3).device()
    for n in lengths:
        prompt, got = synth.seeded_prompt(n, n, 256), []
        for library in (True, False, True):
            dev.set_prefill_library(library)
            dev.reset()
            got.append(dev.prefill_logits(prompt, np.arange(n)))
            assert dev.prefill_library == library
        assert np.array_equal(got[0], got[2]), n
        assert np.linalg.norm(got[0] - got[1]) <= 1.5e-2 * np.linalg.norm(got[1]), n
    dev.close()


# prompts that have tile images: both, one and none of the experts' products from the plain rows; an expert's last block with a single row
@pytest.mark.parametrize("experts,top,rows,sizes", [(8, 2, 300, (130, 257, 500, 516)), (5, 1, 4100, (129, 400)), (70, 2, 260, (140,))])
def test_experts_with_images(pkg, experts, top, rows, sizes):
    c = lc.config([lc.attention(heads=2, kv_heads=1, dim=16, vdim=16, rot=16, mlp=lc.moe(experts, top, rows))], width=330, vocab=60)
    t = lc.settle_routers(c, ref.random_tensors(c, 64), 64)
    tok = lc.tokens(max(sizes), c["vocab"], 4)
    want = ref.Sequence(c, t).run(tok)
    for images in (True, False):
        dev = lc.language_model(pkg, c, t, seq_len=520, precision="bfloat16").device()
        dev.set_prefill_copy(images)
        for n in sizes:
            got = dev.prefill_logits(tok[:n], np.arange(n))
            assert dev.chosen("tile_images") == (2 if images else 0)
            for lo in range(0, n, 64):
                assert lc.error(got[lo:lo + 64], want[lo:min(lo + 64, n)]) <= TOL, (n, lo)
        dev.close()

"""The experts' products of a bf16 prompt from tile images, in blocks of 64 to 320 positions: one of every size, an expert's positions in several blocks of
unequal size, experts without positions, last blocks with one row more than a smaller one would hold.  Against the restatement and against the product
kernels without images."""
import numpy as np
import pytest

import layered_cases as lc
import lezepel_cases as zc
from oracle import layered_np, lezepel_np

pytestmark = pytest.mark.gpu

TOL = 3e-2   # bf16 activations against 64 bits, as for the other prompts
SAME = 4e-3  # the same operands and fp32 sums in another order, so that a result may be the next bf16 number (2^-8 of it)


# (positions, experts, chosen, rows of an expert's up product): many rows of few inputs want an expert's positions in as few blocks as there can be,
# few rows of many inputs in blocks of 64
@pytest.mark.parametrize("kind", ["gated", "plain"])
@pytest.mark.parametrize("n,experts,top,rows", [(130, 8, 2, 4096), (400, 8, 2, 4096), (700, 8, 2, 4096), (1000, 8, 2, 4096), (1210, 8, 2, 4096),
                                                (1500, 8, 2, 4096), (1300, 2, 1, 640), (321, 1, 1, 2048), (129, 70, 1, 200), (500, 3, 3, 200)])
def test_blocks(pkg, kind, n, experts, top, rows):
    if kind == "gated":
        c = zc.config([zc.layer(heads=2, dim=12, rot_dim=4, vdim=16, kv_rank=20, q_rank=24, mlp=zc.moe(experts, top, rows // 2))], width=200, vocab=50, scale=1.0)
        t = zc.settle_routers(c, lezepel_np.random_tensors(c, 8), 8)
        lm, ref = zc.language_model(pkg, c, t, n, "bfloat16"), lezepel_np.Sequence(c, t)
    else:
        c = lc.config([lc.attention(heads=2, kv_heads=1, dim=16, vdim=16, rot=8, mlp=lc.moe(experts, top, rows))], width=200, vocab=50)
        t = lc.settle_routers(c, layered_np.random_tensors(c, 8), 8)
        lm, ref = lc.language_model(pkg, c, t, n, "bfloat16"), layered_np.Sequence(c, t)
    tok = lc.tokens(n, 50, 2)
    want = ref.run(tok)
    got = {}
    for images in (True, False):
        lm._device = None
        dev = lm.device()
        dev.set_prefill_copy(images)
        got[images] = dev.prefill_logits(tok, np.arange(n))
        assert dev.chosen("tile_images") == (2 if images else 0)  # (up and down)
        dev.close()
    for lo in range(0, n, 64):  # (every part by itself: a block left out is not to hide in the mean)
        assert lc.error(got[True][lo:lo + 64], want[lo:lo + 64]) <= TOL, lo
        assert lc.error(got[True][lo:lo + 64], got[False][lo:lo + 64]) <= SAME, lo


# (positions, experts, chosen, rows of an expert's up product): the same few experts take every position, so that blocks of whole tiles are chosen where the
# experts' mean asks for blocks of 128, with a thread an expert in one wavefront or in two
@pytest.mark.parametrize("n,experts,top,rows", [(700, 24, 3, 4096), (700, 65, 8, 2048)])
def test_few_experts_take_all(pkg, n, experts, top, rows):
    c = zc.config([zc.layer(heads=2, dim=12, rot_dim=4, vdim=16, kv_rank=20, q_rank=24, mlp=zc.moe(experts, top, rows // 2))], width=200, vocab=50, scale=1.0)
    t = zc.settle_routers(c, lezepel_np.random_tensors(c, 8), 8)
    bias = t["l0.mlp.router.b"]
    bias[:] = np.where(np.arange(experts) % (experts // top) == 1, 60.0, 0.0)
    bias[np.flatnonzero(bias)[top:]] = 0.0
    bias[bias > 0] += np.arange(top)
    t["l0.mlp.router.b"] = lezepel_np.bf16(bias)
    tok = lc.tokens(n, 50, 2)
    want = lezepel_np.Sequence(c, t).run(tok)
    got = {}
    lm = zc.language_model(pkg, c, t, n, "bfloat16")
    for images in (True, False):
        lm._device = None
        dev = lm.device()
        dev.set_prefill_copy(images)
        got[images] = dev.prefill_logits(tok, np.arange(n))
        assert dev.chosen("tile_images") == (2 if images else 0)
        dev.close()
    for lo in range(0, n, 64):
        assert lc.error(got[True][lo:lo + 64], want[lo:lo + 64]) <= TOL, lo
        assert lc.error(got[True][lo:lo + 64], got[False][lo:lo + 64]) <= SAME, lo

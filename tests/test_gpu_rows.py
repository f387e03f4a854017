"""Decode steps where their products' prologues change form: the choice of experts by every wavefront for itself (up to 40) or by the workgroup, sigmoid and
softmax; the head norm whose factors are requested ahead (four partial sums a head, up to 4096 elements) or formed one by one.  Against the fp64
restatements."""
import numpy as np
import pytest

import layered_cases as lc
import lezepel_cases as zc
from oracle import layered_np, lezepel_np

pytestmark = pytest.mark.gpu

TOL = 2e-5  # decode steps are fp32 sums of at most a few thousand terms, relative to the largest logit; as for the other decode steps


def _steps(dev, ref, c, t, n=5):
    tok = lc.tokens(n, c["vocab"])
    s = ref.Sequence(c, t)
    want = np.array([s.step(int(a)) for a in tok])
    got = np.array([dev.forward(int(a), i)[0] for i, a in enumerate(tok)])
    dev.close()
    assert lc.error(got, want) <= TOL


@pytest.mark.parametrize("design", ["sigmoid", "softmax"])
@pytest.mark.parametrize("experts,top", [(1, 1), (7, 7), (8, 3), (39, 5), (40, 40), (41, 5), (63, 5), (64, 64), (65, 5), (65, 64)])
def test_choice_of_experts(pkg, design, experts, top):
    if design == "sigmoid":
        c = lc.config([lc.attention(mlp=lc.moe(experts, top, 17)), lc.attention(mlp=lc.moe(experts, top, 40))], width=136)
        t = lc.settle_routers(c, layered_np.random_tensors(c, 3), 3)
        _steps(lc.language_model(pkg, c, t).device(), layered_np, c, t)
    else:
        c = zc.config([zc.layer(mlp=zc.moe(experts, top, 17)), zc.layer(mlp=zc.moe(experts, top, 40))], width=136, vocab=50, scale=1.0)
        t = zc.settle_routers(c, lezepel_np.random_tensors(c, 3), 3)
        _steps(zc.language_model(pkg, c, t).device(), lezepel_np, c, t)


@pytest.mark.parametrize("heads,vdim", [(3, 128), (32, 128), (33, 128), (5, 100), (5, 97), (4, 96), (4, 132), (41, 100)])
def test_head_norm(pkg, heads, vdim):
    c = lc.config([lc.delta(heads=heads, kv_heads=1, dim=20, vdim=vdim, conv=2, ranks=(8, 8))])
    t = layered_np.random_tensors(c, 4)
    _steps(lc.language_model(pkg, c, t).device(), layered_np, c, t)


@pytest.mark.parametrize("design,tiny", [
    ("vudelix", "embed"),         # the norm in front of a layer's first product
    ("vudelix", "l0.mix.q"),      # a query's norm
    ("vudelix", "l0.side.proj"),  # a pending update's norm
    ("lezepel", "embed"),
    ("lezepel", "l0.mix.dq"),     # norms inside latent attention
    ("lezepel", "l0.mix.dkv"),
])
def test_norms_of_vectors_whose_squares_are_denormal(pkg, design, tiny):
    """norm_eps 0 and vectors of 2^-66: their mean squares are fp32 numbers below 2^-126, of 17 bits, each rounded by 2^-18 at most, so that the root of
    their mean is off by far less than the tolerance.  (Not of a delta rule's heads, whose outputs differ by more than that range.)"""
    if design == "vudelix":
        c = lc.config([lc.attention()], eps=0.0, side=40 if "side" in tiny else 0)
        cases, ref = lc, layered_np
    else:
        c = zc.config([zc.layer()], eps=0.0, scale=1.0)
        cases, ref = zc, lezepel_np
    t = {k: np.array(v) for k, v in ref.random_tensors(c, 6).items()}
    t[tiny] = t[tiny] * 2.0 ** -66
    if tiny == "l0.mix.dkv":  # (only the compressed keys and values: the rotated part's scale is in the scores)
        rank = t["l0.mix.dkv.norm"].size
        t[tiny][rank:] *= 2.0 ** 66
    _steps(cases.language_model(pkg, c, t).device(), ref, c, t)

"""fp32 products of a prompt with infinities and NaN, in every form of the tiles (32 and 64 positions, one and two groups of wavefronts, blocks of an expert's
rows): what they meet comes out as plain sums give it, and everything else as it does without them."""
import numpy as np
import pytest

import layered_cases as lc
from oracle import layered_np as ref

pytestmark = pytest.mark.gpu

TOL = 2e-5  # fp32 runs of layered models

# (width: inputs, vocabulary: rows, positions): tiles of 32 positions, of 64 with two groups, with one
PLAIN = [(100, 5500, 100), (1000, 8200, 64), (100, 9001, 129)]


def run(pkg, c, t, tok):
    dev = lc.language_model(pkg, c, t, seq_len=len(tok), precision="float32").device()
    dev.keep_residuals()
    got = dev.prefill_logits(tok, np.arange(len(tok)), 0)
    res = dev.residuals(0, len(tok))
    dev.close()
    return got, res


def oracle(c, t, tok):
    s, logits, res = ref.Sequence(c, t), [], []
    with np.errstate(all="ignore"):
        for a in tok:
            logits.append(s.step(int(a)))
            res.append(s.residuals[0])
    return np.array(logits), np.array(res)


def same_kind(got, want):
    return np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.where(np.isinf(got), np.sign(got), 0), np.where(np.isinf(want), np.sign(want), 0))


def model(width, vocab, seed, **more):
    # (one key a query: positions do not see each other)
    c = lc.config([lc.attention(heads=2, kv_heads=1, dim=16, vdim=16, size=1, rot=16, **more)], width=width, vocab=vocab)
    return c, {k: ref.bf16(np.array(v)) for k, v in ref.random_tensors(c, seed).items()}


@pytest.mark.parametrize("width,vocab,n", PLAIN)
def test_infinite_weights_of_the_logits(pkg, width, vocab, n):
    c, t = model(width, vocab, 6)
    tok = lc.tokens(n, vocab)
    clean, _ = run(pkg, c, t, tok)
    t["head"] = t["head"].copy()
    t["head"][[0, 77, vocab - 1], [width - 1, 3, 0]] = [np.inf, -np.inf, np.inf]
    got, _ = run(pkg, c, t, tok)
    want, _ = oracle(c, t, tok)
    assert same_kind(got, want) and np.isinf(got).sum() == 3 * n
    rest = np.isfinite(want)
    assert np.array_equal(got[rest], clean[rest])


@pytest.mark.parametrize("value", [np.inf, np.nan])
@pytest.mark.parametrize("width,vocab,n", PLAIN)
def test_tokens_that_are_not_finite(pkg, width, vocab, n, value):
    c, t = model(width, vocab, 7)
    tok = lc.tokens(n, vocab)
    tok[n // 2] = tok[n - 1]  # (the last position of a tile and one in the middle)
    clean, _ = run(pkg, c, t, tok)
    t["embed"] = t["embed"].copy()
    t["embed"][tok[n - 1], width // 3] = value
    got, _ = run(pkg, c, t, tok)
    bad = tok == tok[n - 1]
    # (attention takes 16 queries at a time, and a masked value that is NaN times zero is one)
    block = np.isin(np.arange(n) // 16, np.nonzero(bad)[0] // 16)
    assert np.isnan(got[bad]).all() and np.array_equal(got[~block], clean[~block])


# (experts, chosen, elements, width, positions): both products of an expert in two groups; the first in one; the second in one
@pytest.mark.parametrize("matrix", ["up", "down"])
@pytest.mark.parametrize("experts,top,ff,width,n", [(4, 2, 1030, 1100, 130), (4, 2, 1030, 300, 130), (4, 2, 400, 1100, 130)])
def test_infinite_weights_of_an_expert(pkg, experts, top, ff, width, n, matrix):
    c, t = model(width, 50, 8, mlp=lc.moe(experts, top, ff))
    t = lc.settle_routers(c, t, 8)
    tok = lc.tokens(n, 50)
    clean, clean_res = run(pkg, c, t, tok)
    # (the second product has an infinite activation where the first has an infinite weight; rows of zeros there give NaN)
    name = "l0.mlp.e2." + matrix
    t[name] = t[name].copy()
    t[name][7 if matrix == "up" else width - 1, 11] = np.inf
    got, res = run(pkg, c, t, tok)
    want, want_res = oracle(c, t, tok)
    assert same_kind(res, want_res) and np.isinf(res).any() and np.isfinite(res).all(1).any()
    rest = np.isfinite(want_res).all(1)
    assert lc.error(res[rest], want_res[rest]) <= TOL and lc.error(got[rest], want[rest]) <= TOL
    if matrix == "down":  # (a single element of each position is not finite)
        rest = np.isfinite(want_res)
        assert np.array_equal(res[rest], clean_res[rest])

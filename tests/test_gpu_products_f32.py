"""fp32 products of a prompt on the bf16 matrix cores (activations in three exact parts): odd numbers of positions, rows and inputs, one and two groups of
wavefronts a tile, blocks of an expert's rows, and infinite weights, against the oracle."""
import numpy as np
import pytest

import layered_cases as lc
from oracle import layered_np as ref

pytestmark = pytest.mark.gpu

# fp32 sums of up to 1000 products, relative to the rms of the logits: as the other fp32 runs of layered models
TOL = 2e-5


def check(pkg, c, t, n):
    tok = lc.tokens(n, c["vocab"])
    s = ref.Sequence(c, t)
    want = np.array([s.step(int(a)) for a in tok])
    dev = lc.language_model(pkg, c, t, seq_len=n, precision="float32").device()
    got = dev.prefill_logits(tok, np.arange(n), 0)
    dev.close()
    return got, want


# (width: inputs of the logits, vocabulary, positions): more results each than small products have.  60 inputs are one step, 449 eight, 577 ten, 1000
# sixteen, a group's share being half of them; tiles of 32 and 64 positions, the last with one, two groups and (9001) one
@pytest.mark.parametrize("width,vocab,n", [(60, 2731, 97), (60, 12345, 65), (449, 4099, 65), (577, 2049, 129), (1000, 8200, 64), (1000, 4110, 161), (520, 9001, 129)])
def test_logits(pkg, width, vocab, n):
    c = lc.config([lc.attention(heads=2, kv_heads=1, dim=16, vdim=16, size=8, rot=16)], width=width, vocab=vocab)
    t = {k: ref.bf16(np.array(v)) for k, v in ref.random_tensors(c, 3).items()}
    got, want = check(pkg, c, t, n)
    assert lc.error(got, want) <= TOL


# one and two steps of inputs (60, 64, 100, 128) with every epilogue that a prompt's products of them have: results, activations, gates and decays; more tiles than CUs, edges
@pytest.mark.parametrize("width,ff,ranks,n", [(60, 2050, (64, 100), 130), (64, 16500, (1, 128), 97), (100, 2049, (128, 65), 161), (128, 9001, (100, 60), 64)])
def test_few_inputs(pkg, width, ff, ranks, n):
    c = lc.config([lc.delta(heads=24, kv_heads=4, dim=100, vdim=90, conv=4, ranks=ranks, mlp=lc.dense(ff))], width=width, vocab=2500)
    t = {k: ref.bf16(np.array(v)) for k, v in ref.random_tensors(c, 12).items()}
    got, want = check(pkg, c, t, n)
    assert lc.error(got, want) <= TOL


# (experts, chosen, elements, width, positions): about 60, 65, 150 and 80 positions an expert
@pytest.mark.parametrize("experts,top,ff,width,n", [(9, 3, 530, 72, 181), (4, 2, 1030, 600, 130), (3, 3, 333, 515, 150), (5, 2, 1100, 110, 200)])
def test_experts(pkg, experts, top, ff, width, n):
    c = lc.config([lc.attention(heads=2, kv_heads=1, dim=16, vdim=16, size=8, rot=16, mlp=lc.moe(experts, top, ff))], width=width, vocab=50)
    t = {k: ref.bf16(np.array(v)) for k, v in ref.random_tensors(c, 4).items()}
    t = lc.settle_routers(c, t, 4)
    got, want = check(pkg, c, t, n)
    assert lc.error(got, want) <= TOL


def test_infinite_weights(pkg):
    c = lc.config([lc.attention(heads=2, kv_heads=1, dim=16, vdim=16, size=8, rot=16)], width=100, vocab=5500)
    t = {k: ref.bf16(np.array(v)) for k, v in ref.random_tensors(c, 5).items()}
    got, want = check(pkg, c, t, 100)
    assert lc.error(got, want) <= TOL
    head = [k for k in t if t[k].shape == (5500, 100)]
    assert head
    # a row of the logits' matrix alone: the model's tokens are smaller numbers than it
    tok = lc.tokens(100, c["vocab"])
    row = next(r for r in range(5499, 0, -1) if r not in tok)
    for k in head:
        t[k] = t[k].copy()
        t[k][row, 37] = np.inf
    inf, _ = check(pkg, c, t, 100)
    assert np.isinf(inf[:, row]).all() and (inf[:, row] > 0).any() and (inf[:, row] < 0).any()
    rest = np.arange(5500) != row
    assert np.array_equal(inf[:, rest], got[:, rest])

"""Decode steps in which latent attention and a gated feed-forward share launches: against the fp64 restatement, at the borders of what
the shared launches take (rank, head and rotated sizes), of the runs of keys (32 a workgroup, four runs that each request their
value rows, 16 runs, longer runs behind) and where a model is just beyond them and goes one launch after the other."""
import numpy as np
import pytest

import layered_cases as lc
import lezepel_cases as zc
from oracle import lezepel_np as ref

pytestmark = pytest.mark.gpu

TOL = 2e-5  # decode steps are fp32 sums of at most a few thousand terms, relative to the largest logit; as for the other decode steps


def _case(mlp, width=72, **kw):
    return zc.config([zc.layer(mlp=m, **kw) for m in mlp], width=width, vocab=50, scale=1.0)


SHAPES = {
    "largest": _case([zc.moe(5, 2, 40), zc.dense(100)], heads=2, dim=128, rot_dim=64, vdim=128, kv_rank=512, q_rank=96, scale=0.07),
    "rank_beyond": _case([zc.moe(5, 2, 40)], heads=2, dim=24, rot_dim=8, vdim=20, kv_rank=516, q_rank=40),
    "odd_query": _case([zc.dense(50)], heads=3, dim=9, rot_dim=2, vdim=11, kv_rank=30, q_rank=20),
    "seventeen_heads": _case([zc.dense(70), zc.moe(9, 4, 24)], heads=17, dim=20, rot_dim=6, vdim=13, kv_rank=100, q_rank=36),
    "one_head": _case([zc.moe(3, 3, 5)], heads=1, dim=2, rot_dim=2, vdim=1, kv_rank=1, q_rank=3),
    "wide": _case([zc.dense(2100), zc.moe(6, 2, 2050)], width=2112, heads=4, dim=40, rot_dim=16, vdim=24, kv_rank=260, q_rank=130),
}


@pytest.mark.parametrize("shape", sorted(SHAPES))
def test_borders(pkg, shape):
    c = SHAPES[shape]
    t = zc.settle_routers(c, ref.random_tensors(c, 5), 5)
    n = 40 if shape == "wide" else 530
    tok = lc.tokens(n, c["vocab"])
    s, want = ref.Sequence(c, t), []
    for a in tok:
        want.append(s.step(int(a)))
    want = np.array(want)
    dev = zc.language_model(pkg, c, t, seq_len=n).device()
    assert dev.chosen("shared_steps") == (0 if shape in ("rank_beyond", "odd_query") else len(c["layers"]))
    borders = (0, 30, 62, 126, 158, 510)
    for b in borders:
        if b >= n:
            continue
        if b:
            dev.prefill_logits(tok[:b], [], 0)
        got = np.array([dev.forward(int(tok[p]), p)[0] for p in range(b, min(b + 6, n))])
        assert lc.error(got, want[b:b + len(got)]) <= TOL, (shape, b)
    # replays of the recorded step, host work between them: the counts of the runs are back at zero every time
    dev.reset()
    for p in range(n if n < 100 else 140):
        got = dev.forward(int(tok[p]), p)[0]
        assert lc.error(got, want[p]) <= TOL, (shape, p)
    dev.close()


def test_padding_behind_the_heads(pkg):
    """A narrow layer behind which a wide one leaves its values in the same buffer, at positions where a head has several runs of keys: what the wide one
    left from a sequence of numbers that are none must not reach the next sequence's output product."""
    c = _case([zc.dense(70)], heads=3, dim=20, rot_dim=6, vdim=13, kv_rank=100, q_rank=36)
    wide = _case([zc.dense(70)], heads=5, dim=20, rot_dim=6, vdim=40, kv_rank=100, q_rank=36)
    c["layers"] += wide["layers"]
    t = {k: np.array(v) for k, v in ref.random_tensors(c, 5).items()}
    t["embed"][7, 3] = np.inf
    n = 160
    tok = lc.tokens(n, c["vocab"])
    tok[tok == 7] = 8
    s, want = ref.Sequence(c, t), []
    for a in tok:
        want.append(s.step(int(a)))
    dev = zc.language_model(pkg, c, t, seq_len=n).device()
    assert dev.chosen("shared_steps") == 2
    for at in (40, 70, 100, 130, 150):
        dev.reset()
        with np.errstate(invalid="ignore"):
            assert not np.isfinite(dev.forward(7, 0)[0]).all()
        dev.reset()
        dev.prefill_logits(tok[:at], [], 0)
        got = np.array([dev.forward(int(tok[p]), p)[0] for p in range(at, at + 4)])
        assert lc.error(got, want[at:at + 4]) <= TOL, at
    dev.close()

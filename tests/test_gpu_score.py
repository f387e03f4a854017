"""Logits of several wanted positions (l2h_prefill_logits): one pass over the classifier's weights for up to 8 of them.

A position asked for alone runs the decode step's classifier on the same hidden state: the same q8_K inputs and the same exact terms
(integers, or fp32 products in fp64), summed in fp64 in another order.  Two such sums of T terms differ by at most T * 2^-53 of the
sum of magnitudes, far below half a unit of the fp32 that they are rounded to except where they lie that close to a rounding
boundary: at most one unit in the last place, of a few logits."""
import numpy as np
import pytest

from test_gpu_model import _model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("plan,dim,vocab", [
    ("PLAN_Q4_K_S", 256, 333),    # q6_K: one block a row, the last 16 rows in part
    ("PLAN_Q4_K", 768, 777),      # q4_K: three blocks, the last 8 rows in part
    ("Q5_K", 512, 33001),         # q5_K: more rows than one round of the workgroups takes
    ("PLAN_Q4_K_S", 7424, 300),   # four images fit into 64 KiB, eight don't
    ("PLAN_F32", 96, 301),        # fp32: 24 pieces for 16 lanes, the last 4 rows in part
    ("PLAN_F32", 2304, 260),      # fp32, four images
    ("PLAN_F32", 4160, 64),       # too long for four: one position at a time
])
def test_wanted_positions(pkg, plan, dim, vocab):
    from llama2_jl_amd import synth
    heads = dim // 64 if dim % 64 == 0 else dim // 32
    plan = dict(synth.PLAN_Q4_K, output=synth.TYPE_Q5_K) if plan == "Q5_K" else plan
    lm = _model(pkg, plan, dim=dim, hidden_dim=256, n_layers=1, vocab_size=vocab, seq_len=64, rope_freq_base=10000.0, rope_is_neox=False, n_heads=heads,
                n_kv_heads=heads)
    dev = lm.device()
    tok = synth.seeded_prompt(3, 40, vocab)
    alone = np.stack([dev.prefill_logits(tok, [i])[0] for i in range(40)])
    for want in ([0, 39], [1, 2, 3], [4, 9, 20, 31], [0, 7, 8, 9, 39], np.arange(3, 11), np.arange(9), np.arange(1, 40, 3), np.arange(40)):
        got = dev.prefill_logits(tok, want)
        ulp = np.spacing(np.abs(alone[want]))
        assert np.all(np.abs(got - alone[want]) <= ulp), want
        assert np.mean(got != alone[want]) <= 1e-3, want
        assert np.array_equal(dev.state("logits"), got[-1])  # the last of them is the model's state


def test_more_wanted_positions_than_the_workspace_has_rows(pkg):
    """The logits' workspace is 64 MiB, 130 rows of a vocabulary of 128 256: positions on both sides of its border, in one call of 140."""
    from llama2_jl_amd import synth
    vocab, n = 128256, 150
    lm = _model(pkg, synth.PLAN_Q4_K_S, dim=256, hidden_dim=256, n_layers=1, vocab_size=vocab, seq_len=160, rope_freq_base=10000.0, rope_is_neox=False,
                n_heads=4, n_kv_heads=4)
    dev = lm.device()
    tok = synth.seeded_prompt(5, n, vocab)
    want = np.arange(7, 147)
    got = dev.prefill_logits(tok, want)
    assert np.array_equal(dev.state("logits"), got[-1])
    for i in (0, 1, 121, 127, 128, 129, 130, 131, 137, 138, 139):
        alone = dev.prefill_logits(tok, [want[i]])[0]
        assert np.all(np.abs(got[i] - alone) <= np.spacing(np.abs(alone))), i
        assert np.mean(got[i] != alone) <= 1e-3, i

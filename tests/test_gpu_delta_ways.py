"""The delta rule's prompt pass in chunks of 16 (delta_plan.h), for many heads and for wide values, and in chunks of 32 with wide values from 512 tokens on: from an
empty state and going on from one; in several passes over the chunks; and up to 47 tokens one by one."""
import numpy as np
import pytest

import layered_cases as lc
from oracle import layered_np as ref

pytestmark = pytest.mark.gpu

TOL = {"float32": 2e-5, "bfloat16": 3e-2}  # as the other runs of layered models: fp32 rounding, bf16 activations


# (heads, key heads, dim, vdim, lengths one after the other); 768 heads have eight chunks a pass: 256 tokens
@pytest.mark.parametrize("precision", sorted(TOL))
@pytest.mark.parametrize("heads,kv_heads,dim,vdim,cuts", [(64, 2, 100, 100, (47, 48, 49, 80)), (4, 2, 48, 130, (63, 64, 511, 512, 600)), (100, 1, 65, 129, (48, 61)),
                                                          (768, 1, 8, 8, (48, 256, 257, 545)), (3, 3, 128, 128, (46, 47, 48, 49))])
def test_chunks(pkg, heads, kv_heads, dim, vdim, cuts, precision):
    c = lc.config([lc.delta(heads=heads, kv_heads=kv_heads, dim=dim, vdim=vdim, conv=4, ranks=(8, 12))], width=72, vocab=60)
    t = {k: ref.bf16(np.array(v)) for k, v in ref.random_tensors(c, 4).items()}
    tok = lc.tokens(sum(cuts) + 1, c["vocab"])
    s = ref.Sequence(c, t)
    want = np.array([s.step(int(a)) for a in tok])
    dev = lc.language_model(pkg, c, t, seq_len=len(tok), precision=precision).device()
    at = 0
    for n in cuts:
        for first in sorted({0, at}):
            dev.reset()
            if first:
                dev.prefill(tok[:first])
            got = dev.prefill_logits(tok[first:first + n], np.arange(n), first)
            assert lc.error(got, want[first:first + n]) <= TOL[precision], (n, first)
        at += n
        assert lc.error(dev.forward(int(tok[at]), at)[0], want[at]) <= TOL[precision], at
    dev.close()

"""The delta rule's prompt pass from an empty state and going on from one, heads at the edges of what a wavefront takes.  From 48 tokens on lengths around
chunks (of 32; of 16 where a head has more than 128 value elements) and three of them, the operands under way; below that it goes token by token."""
import numpy as np
import pytest

import layered_cases as lc
from oracle import layered_np as ref

pytestmark = pytest.mark.gpu

TOL = {"float32": 2e-5, "bfloat16": 3e-2}  # as the other runs of layered models: fp32 rounding, bf16 activations


@pytest.mark.parametrize("precision", sorted(TOL))
@pytest.mark.parametrize("dim,vdim", [(64, 16), (65, 17), (128, 128), (192, 145), (256, 256)])
def test_borders(pkg, dim, vdim, precision):
    c = lc.config([lc.delta(heads=2, kv_heads=1, dim=dim, vdim=vdim, conv=4, ranks=(8, 12))], width=72, vocab=60)
    t = {k: ref.bf16(np.array(v)) for k, v in ref.random_tensors(c, 4).items()}
    tok = lc.tokens(292, c["vocab"])
    s = ref.Sequence(c, t)
    want = np.array([s.step(int(a)) for a in tok])
    dev = lc.language_model(pkg, c, t, seq_len=len(tok), precision=precision).device()
    for n in (24, 31, 32, 33, 48, 49, 95, 96, 97, 129):
        for at in (0, n):
            got = dev.prefill_logits(tok[at:at + n], np.arange(n), at)
            assert lc.error(got, want[at:at + n]) <= TOL[precision], (n, at)
        assert lc.error(dev.forward(int(tok[2 * n]), 2 * n)[0], want[2 * n]) <= TOL[precision], n
    dev.close()

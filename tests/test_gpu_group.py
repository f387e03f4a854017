"""The grouping of a prompt's tokens by expert: more choices than a thread keeps (8 x 1024), more experts than a wavefront's threads, experts without tokens."""
import numpy as np
import pytest

import layered_cases as lc
from oracle import layered_np as ref

pytestmark = pytest.mark.gpu

TOL = 2e-5  # fp32 runs of layered models


@pytest.mark.parametrize("experts,top,ff,width,n", [(9, 6, 24, 64, 1500), (300, 2, 8, 320, 90), (7, 7, 20, 64, 3), (5, 1, 20, 64, 1100)])
def test_choices(pkg, experts, top, ff, width, n):
    c = lc.config([lc.attention(heads=2, kv_heads=1, dim=8, vdim=8, rot=4, size=5, mlp=lc.moe(experts, top, ff))], width=width, vocab=30)
    t = lc.settle_routers(c, ref.random_tensors(c, 8), 8)
    tok = lc.tokens(n, c["vocab"])
    s = ref.Sequence(c, t)
    want = np.array([s.step(int(a)) for a in tok])
    dev = lc.language_model(pkg, c, t, seq_len=n, precision="float32").device()
    assert lc.error(dev.prefill_logits(tok, np.arange(n)), want) <= TOL
    dev.close()

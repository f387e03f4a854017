"""The dense product of a long prompt where its tiles of 256 x 256 are a little more than whole rounds of the compute units, the rest going as
halves of 128 positions: against the fp64 restatement, where the rest is smallest and largest and just beyond, and where halves are partly or
wholly past the last position."""
import numpy as np
import pytest

import layered_cases as lc
import lezepel_cases as zc
from oracle import lezepel_np as ref

pytestmark = pytest.mark.gpu

TOL = 3e-2  # bf16 activations, as for the other prompts


# (positions, row groups of 256): items = groups x blocks of 256 positions; a gated layer has two rows for every one of its ff outputs
@pytest.mark.parametrize("n,groups", [(264, 129), (400, 192), (400, 193), (512, 130), (520, 86)])
def test_rest_as_halves(pkg, n, groups):
    c = zc.config([zc.layer(heads=2, dim=12, rot_dim=4, vdim=16, kv_rank=20, q_rank=24, mlp=zc.dense(128 * groups - 3))], width=48, vocab=50, scale=1.0)
    t = ref.random_tensors(c, 8)
    tok = lc.tokens(n, 50, 2)
    want = ref.Sequence(c, t).run(tok)
    dev = zc.language_model(pkg, c, t, seq_len=n).device()
    got = dev.prefill_logits(tok, np.arange(n))
    for lo in range(0, n, 64):  # (every part by itself: a block left out is not to hide in the mean)
        assert lc.error(got[lo:lo + 64], want[lo:lo + 64]) <= TOL, (n, groups, lo)
    dev.close()

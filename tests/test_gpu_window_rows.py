"""fp32 window attention of a prompt at the borders of its kernel's forms (heads of up to 64, 128 and 256 elements, sizes that are no multiple of four), of a
block of queries (16) and of the tiles of keys that its wavefronts take in turn."""
import numpy as np
import pytest

import layered_cases as lc
from oracle import layered_np as ref

pytestmark = pytest.mark.gpu

# fp32 sums of up to 256 products and 150 keys, relative to the rms of the logits: as the other fp32 runs of layered models
TOL = 2e-5

# (key elements, value elements, window)
SHAPES = [(3, 1, 1), (5, 64, 16), (64, 7, 17), (65, 30, 150), (40, 128, 33), (128, 128, 129), (130, 66, 48), (256, 254, 90)]


@pytest.mark.parametrize("dim,vdim,size", SHAPES)
def test_borders(pkg, dim, vdim, size):
    c = lc.config([lc.attention(heads=4, kv_heads=2, dim=dim, vdim=vdim, size=size, rot=2 * min(dim // 2, 8), scale=dim ** -0.5)], width=60, vocab=50)
    t = ref.random_tensors(c, 9)
    t = {k: ref.bf16(np.array(v)) for k, v in t.items()}
    tok = lc.tokens(150, c["vocab"])
    s = ref.Sequence(c, t)
    want = np.array([s.step(int(a)) for a in tok])
    dev = lc.language_model(pkg, c, t, seq_len=150, precision="float32").device()
    for cuts in ([150], [15, 16, 17, 102], [2, 63, 85]):
        at = 0
        for n in cuts:
            got = dev.prefill_logits(tok[at:at + n], np.arange(n), at)
            assert lc.error(got, want[at:at + n]) <= TOL, (cuts, at)
            at += n
    dev.close()

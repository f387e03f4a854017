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


# (heads, key/value heads, key elements, value elements, window, positions): one wavefront a block (many blocks) with one tile of keys and with several, and two, four and
# eight of them, for heads of up to 64, 128 and 256 elements; and activations that are rounded to bf16
FORMS = [(32, 4, 16, 12, 1, 530), (32, 4, 16, 12, 40, 530), (17, 1, 100, 66, 20, 1000), (9, 3, 256, 129, 40, 1000), (9, 3, 132, 200, 1, 1000), (2, 2, 64, 60, 20, 200),
         (2, 1, 128, 100, 50, 200), (2, 1, 36, 33, 150, 200), (1, 1, 200, 180, 60, 200), (8, 8, 20, 16, 200, 1030), (2, 2, 126, 128, 170, 200)]


@pytest.mark.parametrize("heads,kv_heads,dim,vdim,size,n", FORMS)
def test_wavefronts(pkg, heads, kv_heads, dim, vdim, size, n):
    c = lc.config([lc.attention(heads=heads, kv_heads=kv_heads, dim=dim, vdim=vdim, size=size, rot=2 * min(dim // 2, 8), scale=dim ** -0.5)], width=60, vocab=50)
    t = {k: ref.bf16(np.array(v)) for k, v in ref.random_tensors(c, 10).items()}
    tok = lc.tokens(n, c["vocab"])
    s = ref.Sequence(c, t)
    want = np.array([s.step(int(a)) for a in tok])
    dev = lc.language_model(pkg, c, t, seq_len=n, precision="float32").device()
    assert lc.error(dev.prefill_logits(tok, np.arange(n), 0), want) <= TOL
    at = n - n // 3
    dev.reset()
    dev.prefill(tok[:at])
    assert lc.error(dev.prefill_logits(tok[at:], np.arange(n - at), at), want[at:]) <= TOL
    dev.close()


@pytest.mark.parametrize("dim,vdim", [(133, 21), (136, 72), (256, 256)])
def test_bf16_outputs(pkg, dim, vdim):
    """(heads that the bf16 attention has no tile for)"""
    c = lc.config([lc.attention(heads=3, kv_heads=1, dim=dim, vdim=vdim, size=70, rot=16, scale=dim ** -0.5)], width=60, vocab=50)
    t = {k: ref.bf16(np.array(v)) for k, v in ref.random_tensors(c, 11).items()}
    tok = lc.tokens(150, c["vocab"])
    s = ref.Sequence(c, t)
    want = np.array([s.step(int(a)) for a in tok])
    dev = lc.language_model(pkg, c, t, seq_len=150, precision="bfloat16").device()
    assert lc.error(dev.prefill_logits(tok, np.arange(150), 0), want) <= 3e-2  # as the other bf16 runs
    dev.close()

"""The dense product of a long bf16 prompt in tiles of 256 x 256: where they are a little more than whole rounds of the compute units, the rest
going as halves of 128 positions (the rest smallest, largest and just beyond; halves partly or wholly past the last position), and where no
tile is cut and their number is no multiple of the eight XCDs.  Gated feed-forwards (Lezepel) and plain ones (Vudelix)."""
import numpy as np
import pytest

import layered_cases as lc
import lezepel_cases as zc
from oracle import layered_np, lezepel_np

pytestmark = pytest.mark.gpu

TOL = 3e-2   # bf16 activations against 64 bits, as for the other prompts
SAME = 4e-3  # against the product kernel that has no tile images: the same operands and fp32 sums in another order, so that a result may be the next bf16
             # number (2^-8 of it)


def _model(pkg, kind, rows, seq_len):
    if kind == "gated":  # two rows for every one of the layer's outputs
        c = zc.config([zc.layer(heads=2, dim=12, rot_dim=4, vdim=16, kv_rank=20, q_rank=24, mlp=zc.dense(rows // 2))], width=48, vocab=50, scale=1.0)
        t = lezepel_np.random_tensors(c, 8)
        return zc.language_model(pkg, c, t, seq_len, "bfloat16"), lezepel_np.Sequence(c, t)
    c = lc.config([lc.attention(heads=2, kv_heads=1, dim=16, vdim=16, rot=8, mlp=lc.dense(rows))], width=48, vocab=50)
    t = layered_np.random_tensors(c, 8)
    return lc.language_model(pkg, c, t, seq_len, "bfloat16"), layered_np.Sequence(c, t)


# (positions, row groups of 256): tiles = groups x blocks of 256 positions; a layer has at most 36 864 outputs
GATED = [(264, 129), (400, 192), (400, 193), (512, 130), (520, 86), (400, 215), (400, 226), (1030, 86)]
PLAIN = [(264, 129), (700, 128), (700, 129), (512, 130), (520, 86), (900, 113), (1030, 86)]


@pytest.mark.parametrize("kind,n,groups", [("gated", *s) for s in GATED] + [("plain", *s) for s in PLAIN])
def test_rest_as_halves_and_none(pkg, kind, n, groups):
    lm, ref = _model(pkg, kind, 256 * groups - 6, n + 40)
    tok, other = lc.tokens(n, 50, 2), lc.tokens(n + 40, 50, 3)
    want = ref.run(tok)
    got = {}
    for images in (True, False):
        lm._device = None
        dev = lm.device()
        dev.set_prefill_copy(images)
        dev.prefill_logits(other, [0])  # (what a tile that nobody computes would leave in place)
        assert dev.chosen("tile_images") == (1 if images else 0)
        dev.reset()
        got[images] = dev.prefill_logits(tok, np.arange(n))
        dev.close()
    for lo in range(0, n, 64):  # (every part by itself: a block left out is not to hide in the mean)
        assert lc.error(got[True][lo:lo + 64], want[lo:lo + 64]) <= TOL, lo
        assert lc.error(got[True][lo:lo + 64], got[False][lo:lo + 64]) <= SAME, lo

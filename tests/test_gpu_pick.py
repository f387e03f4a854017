"""The greedy token of a layered model's decode steps, which the classifier's workgroups leave a key each of and the next step (or the end of the
call) picks: the first index of the largest logit, with rows that tie inside a workgroup, across workgroups, across its wavefronts (more than 64 rows a workgroup:
the largest vocabulary) and at the ends."""
import numpy as np
import pytest

import layered_cases as lc
from oracle import layered_np as ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("side", (0, 5))
@pytest.mark.parametrize("vocab", (1, 3, 65, 520, 41003))
def test_first_of_the_largest(pkg, vocab, side):
    c = lc.config([lc.attention(heads=2, kv_heads=1, dim=8, vdim=8, rot=4), lc.attention(heads=2, kv_heads=1, dim=8, vdim=8, rot=4)], width=40, vocab=vocab,
                  side=side)
    t = {k: np.array(v) for k, v in ref.random_tensors(c, 3).items()}
    # every row of the classifier occurs at several places: the largest logit does, whichever row it is
    head = t["head"]
    n = min(vocab, 37)
    for at in range(n, vocab, n):
        head[at:at + n] = head[:min(n, vocab - at)]
    head[-n:] = head[:n][::-1]
    t["head"] = ref.bf16(head)
    dev = lc.language_model(pkg, c, t, seq_len=64).device()
    prompt = lc.tokens(3, vocab)
    want, p = [], list(prompt)
    for i in range(12):  # one step a call
        logits, got = dev.forward(int(p[i]), i)
        first = int(np.argmax(logits))
        assert got == first
        if i >= len(prompt) - 1:
            want.append(first)
            p.append(first)
    for k in (10, 1, 2):  # several steps a call, the prompt's among them
        dev.reset()
        ids = np.asarray(dev.generate_greedy(list(prompt), k))
        assert list(ids) == want[:k]
    ids = dev.generate_greedy([want[1]], 3, pos0=4)  # (goes on where the call of two steps ended)
    assert list(ids) == want[2:5]
    dev.close()

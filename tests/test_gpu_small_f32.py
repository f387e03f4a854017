"""Decoding of small fp32 models by the single-launch kernel against the per-phase path, bit for bit.  Both form exact products and
fp64 sums that are rounded once, so that another order of a sum shows only where it lies within 1e-15 of the middle between two
floats."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _pair(pkg, seed, dim, hidden, layers, heads, kv, vocab, neox):
    from llama2_jl_amd import synth
    from llama2_jl_amd.inference import DeviceModel
    cfg = pkg.ModelConfig(dim=dim, hidden_dim=hidden, n_layers=layers, n_heads=heads, n_kv_heads=kv, vocab_size=vocab, seq_len=320,
                          rope_freq_base=10000.0, rope_is_neox=neox)
    lm = synth.synthetic_model(cfg, synth.PLAN_F32, seed=seed)
    fast, slow = DeviceModel(cfg, lm.weights, path=3), DeviceModel(cfg, lm.weights, path=1)
    assert fast.path == 3 and slow.path == 1
    return fast, slow


def _same(fast, slow, prompt, n_new):
    fast.reset()
    slow.reset()
    (a, la), (b, lb) = (d.generate_greedy(prompt, n_new, want_logits=True) for d in (fast, slow))
    assert np.asarray(a).tolist() == np.asarray(b).tolist()
    assert np.array_equal(la.view(np.uint32), lb.view(np.uint32))
    for name in ("x", "xb", "q", "hb"):
        assert np.array_equal(fast.state(name).view(np.uint32), slow.state(name).view(np.uint32)), name


# the smallest of each kernel: (hidden, whether the kernel for small models takes it)
@pytest.mark.parametrize("hidden,small", [(4, 0), (56, 1), (120, 1)])
@pytest.mark.parametrize("n_new", [2, 7, 19])
def test_keys_of_the_steps_before_in_one_launch(pkg, n_new, hidden, small):
    """A layer so small that nothing sweeps the vector cache between a step's read of a line of keys and the next step's"""
    from llama2_jl_amd import synth
    fast, slow = _pair(pkg, 31, 256, hidden, 2, 8, 8, 300, False)
    assert fast.steps_per_launch == 8 and fast.chosen("small_kernel") == small
    _same(fast, slow, synth.seeded_prompt(70, 2, 300), n_new)
    fast.close()
    slow.close()


SHAPES = [
    # (small, dim, hidden, layers, heads, kv heads, vocabulary, neox): hidden sizes around the slices of 512 that w2's rows are cut into, the shortest and the
    # longest of each head size that the kernel for small models takes (small = 1) and some just beyond, where the general fp32 kernel runs; row counts
    # that leave workgroups, wavefronts and the last pair of the classifier without rows
    (0, 256, 4, 2, 8, 8, 1, False),
    (1, 256, 512, 2, 4, 2, 255, True),
    (1, 256, 516, 1, 8, 1, 4097, False),
    (1, 256, 56, 2, 8, 8, 33, True),
    (1, 256, 1920, 2, 8, 2, 1000, False),
    (1, 256, 1984, 2, 4, 4, 1000, True),
    (0, 256, 1988, 2, 4, 4, 1000, True),
    (1, 512, 1376, 2, 8, 8, 32000, False),
    (1, 512, 2052, 2, 16, 4, 3, True),
    (1, 512, 48, 2, 16, 16, 500, False),
    (1, 512, 3840, 1, 16, 4, 1000, True),
    (1, 512, 3968, 1, 8, 2, 1000, False),
    (1, 512, 60, 2, 4, 4, 500, True),
    (1, 512, 252, 2, 4, 1, 1, False),
    (1, 512, 4032, 2, 4, 4, 1000, False),
    (0, 512, 4096, 2, 4, 4, 1000, False),
]


@pytest.mark.parametrize("shape", range(len(SHAPES)))
def test_rows_slices_and_heads(pkg, shape):
    from llama2_jl_amd import synth
    small, *sizes = SHAPES[shape]
    fast, slow = _pair(pkg, 40 + shape, *sizes)
    assert fast.chosen("small_kernel") == small and slow.chosen("small_kernel") == 0
    for rep, n_new in enumerate((19, 290)):  # the second run crosses into the attention of long caches
        _same(fast, slow, synth.seeded_prompt(70 + rep, 2 + 5 * rep, sizes[5]), n_new)
    fast.close()
    slow.close()


def test_gives_up_and_recovers(pkg):
    """a wait bound of zero, set from the host: every wavefront leaves at the next barrier, and the model decodes as before afterwards"""
    from llama2_jl_amd import synth
    cfg = pkg.ModelConfig(dim=512, hidden_dim=1376, n_layers=2, n_heads=8, n_kv_heads=8, vocab_size=500, seq_len=64, rope_freq_base=10000.0)
    dev = synth.synthetic_model(cfg, synth.PLAN_F32, seed=5).device(path=3)
    prompt = synth.seeded_prompt(11, 6, 500)
    want = np.asarray(dev.generate_greedy(prompt, 12)).tolist()
    dev.set_wait_limit(0)
    dev.reset()
    with pytest.raises(pkg.L2HError):
        dev.generate_greedy(prompt, 12)
    dev.set_wait_limit(1 << 20)
    for _ in range(2):
        dev.reset()
        assert np.asarray(dev.generate_greedy(prompt, 12)).tolist() == want
    dev.close()

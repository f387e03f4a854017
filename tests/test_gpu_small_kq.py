"""Decoding of small k-quant models by the single-launch kernel against the per-phase path, bit for bit: the same integers and exact
products, fp64 sums rounded once, so that another order of a sum shows only where it lies within 1e-15 of the middle between two floats."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

Q4, Q5, Q6 = 12, 13, 14


def _pair(pkg, seed, plan, dim, hidden, layers, heads, kv, vocab, neox):
    from llama2_jl_amd import synth
    from llama2_jl_amd.inference import DeviceModel
    cfg = pkg.ModelConfig(dim=dim, hidden_dim=hidden, n_layers=layers, n_heads=heads, n_kv_heads=kv, vocab_size=vocab, seq_len=320,
                          rope_freq_base=10000.0, rope_is_neox=neox)
    lm = synth.synthetic_model(cfg, plan, seed=seed)
    fast, slow = DeviceModel(cfg, lm.weights), DeviceModel(cfg, lm.weights, path=1)
    assert fast.path == 3 and slow.path == 1 and fast.steps_per_launch == 8 and fast.chosen("small_kernel") == 1
    return fast, slow


def _same(fast, slow, prompt, n_new):
    fast.reset()
    slow.reset()
    (a, la), (b, lb) = (d.generate_greedy(prompt, n_new, want_logits=True) for d in (fast, slow))
    assert np.asarray(a).tolist() == np.asarray(b).tolist()
    assert np.array_equal(la.view(np.uint32), lb.view(np.uint32))
    for name in ("x", "xb", "q", "hb"):
        assert np.array_equal(fast.state(name).view(np.uint32), slow.state(name).view(np.uint32)), name


SHAPES = [
    # (plan, dim, hidden, layers, heads, kv heads, vocabulary, neox): one and two slices of w2's rows and those that leave places in them
    # empty, vocabularies that end inside a piece, both head sizes, shared and own key/value heads
    ("PLAN_Q4_K_S", 512, 1024, 4, 8, 2, 2048, False),
    ("PLAN_Q5_K_M", 512, 256, 3, 8, 8, 1, True),
    ("PLAN_Q4_K_S", 512, 768, 2, 16, 4, 515, True),
    ("PLAN_Q5_K_M", 512, 2304, 2, 16, 1, 4097, False),
    ("PLAN_Q4_K_S", 512, 3840, 1, 8, 8, 32000, False),
    ("PLAN_Q4_K_S", 1024, 2816, 2, 16, 4, 1000, False),
    ("PLAN_Q5_K_M", 1024, 3840, 2, 16, 16, 32003, True),
    ("PLAN_Q5_K_M", 1024, 256, 2, 32, 8, 300, False),
    # the longest with heads of 32
    ("PLAN_Q4_K_S", 512, 3584, 2, 16, 4, 300, False),
    ("PLAN_Q5_K_M", 1024, 3584, 2, 32, 32, 300, True),
]


@pytest.mark.parametrize("shape", range(len(SHAPES)))
def test_rows_slices_and_heads(pkg, shape):
    from llama2_jl_amd import synth
    plan, *sizes = SHAPES[shape]
    fast, slow = _pair(pkg, 40 + shape, getattr(synth, plan), *sizes)
    for rep, n_new in enumerate((19, 290)):  # the second run crosses into the attention of long caches
        _same(fast, slow, synth.seeded_prompt(70 + rep, 2 + 5 * rep, sizes[5]), n_new)
    fast.close()
    slow.close()


def test_asked_for_by_number_it_is_refused_as_before(pkg):
    from llama2_jl_amd import synth
    cfg = pkg.ModelConfig(dim=512, hidden_dim=1024, n_layers=1, n_heads=8, n_kv_heads=2, vocab_size=500, seq_len=64, rope_freq_base=10000.0)
    with pytest.raises(pkg.L2HError):
        synth.synthetic_model(cfg, synth.PLAN_Q4_K_S, seed=5).device(path=3)


@pytest.mark.parametrize("dim,hidden,heads", [(512, 3840, 16), (1024, 3840, 32), (512, 4096, 8), (1024, 1024, 8), (256, 512, 8)])
def test_just_beyond_it_runs_on_path_1(pkg, dim, hidden, heads):
    from llama2_jl_amd import synth
    cfg = pkg.ModelConfig(dim=dim, hidden_dim=hidden, n_layers=1, n_heads=heads, n_kv_heads=heads, vocab_size=300, seq_len=64, rope_freq_base=10000.0)
    dev = synth.synthetic_model(cfg, synth.PLAN_Q4_K_S, seed=5).device()
    assert dev.path == 1 and dev.chosen("small_kernel") == 0 and dev.path_reason
    dev.close()


@pytest.mark.parametrize("n_new", [2, 7, 19])
def test_keys_of_the_steps_before_in_one_launch(pkg, n_new):
    """as for the fp32 kernel: a layer whose rows sweep little of the vector cache between a step's read of a line of keys and the next step's"""
    from llama2_jl_amd import synth
    fast, slow = _pair(pkg, 31, synth.PLAN_Q4_K_S, 512, 256, 2, 16, 16, 300, False)
    _same(fast, slow, synth.seeded_prompt(70, 2, 300), n_new)
    fast.close()
    slow.close()


def test_gives_up_and_recovers(pkg):
    """a wait bound of zero, set from the host: every wavefront leaves at the next barrier; a model whose path was not asked for goes on on path 1"""
    from llama2_jl_amd import synth
    cfg = pkg.ModelConfig(dim=512, hidden_dim=1024, n_layers=2, n_heads=8, n_kv_heads=2, vocab_size=500, seq_len=64, rope_freq_base=10000.0)
    dev = synth.synthetic_model(cfg, synth.PLAN_Q4_K_S, seed=5).device()
    prompt = synth.seeded_prompt(11, 6, 500)
    want = np.asarray(dev.generate_greedy(prompt, 12)).tolist()
    dev.set_wait_limit(0)
    dev.reset()
    with pytest.raises(pkg.L2HError):
        dev.generate_greedy(prompt, 12)
    for _ in range(2):
        dev.reset()
        assert np.asarray(dev.generate_greedy(prompt, 12)).tolist() == want
    dev.close()


def test_memory_of_the_cache_follows_the_path(pkg):
    """uncached for several steps a launch; a model that leaves the kernel takes its cache's rows along, one that never ran it has an ordinary cache"""
    from llama2_jl_amd import synth
    fast, slow = _pair(pkg, 9, synth.PLAN_Q4_K_S, 512, 1024, 2, 8, 2, 500, False)
    assert fast.chosen("uncached_cache") == 1 and slow.chosen("uncached_cache") == 0
    prompt = synth.seeded_prompt(11, 6, 500)
    for d in (fast, slow):
        ids = np.asarray(d.generate_greedy(prompt, 40))
    fast.set_wait_limit(0)
    with pytest.raises(pkg.L2HError):
        fast.forward(int(ids[-1]), 45)
    assert fast.chosen("uncached_cache") == 0
    for l in range(2):
        for a, b in zip(fast.kv_read(l, 0, 45), slow.kv_read(l, 0, 45)):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    (a, la), (b, lb) = (d.generate_greedy([int(ids[-1])], 30, pos0=45, want_logits=True) for d in (fast, slow))
    assert a.tolist() == b.tolist() and np.array_equal(la.view(np.uint32), lb.view(np.uint32))
    fast.close()
    slow.close()
    # heads of 80, each with keys of its own: path 1
    cfg = pkg.ModelConfig(dim=1280, hidden_dim=1024, n_layers=1, n_heads=16, n_kv_heads=16, vocab_size=500, seq_len=64, rope_freq_base=10000.0)
    dev = synth.synthetic_model(cfg, synth.PLAN_Q4_K_S, seed=5).device()
    assert dev.path == 1 and dev.chosen("uncached_cache") == 0
    dev.close()


def test_a_call_that_cannot_run_here_runs_on_path_1(pkg, monkeypatch):
    """the library's own bound, forced to zero from the host: the call that finds it met gives path 1's results, from the rows that the cache held"""
    from llama2_jl_amd import _lib, synth
    monkeypatch.setenv("L2H_FLOW_SPINS", "0")
    fast, slow = _pair(pkg, 13, synth.PLAN_Q4_K_S, 512, 1024, 2, 8, 2, 500, False)
    tok = synth.seeded_prompt(3, 37, 500)
    got = []
    for d in (fast, slow):
        d.prefill(tok)
        ids, logits = d.generate_greedy(tok[:5], 20, pos0=37, want_logits=True)
        got.append((ids.tolist(), logits.tobytes(), d.forward(int(ids[-1]), 61)[0].tobytes()))
    assert got[0] == got[1]
    assert _lib.lib().l2h_model_path(fast.handle) == 1 and "one kernel per phase" in _lib.lib().l2h_model_path_reason(fast.handle).decode()
    fast.close()
    slow.close()

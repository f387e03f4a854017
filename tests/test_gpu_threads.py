"""Two host threads, each with a context and a model of its own, decode on one device at the same time: every call gives what it gives alone.  The kernels
of launch paths 2 and 3 read a model's arguments from the device's constant memory and need all of their workgroups resident."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MODELS = {
    # (plan, dim, hidden, layers, heads, kv heads, vocabulary, path asked for, path taken)
    "small_kq": ("PLAN_Q4_K_S", 512, 1024, 4, 8, 2, 2048, 0, 3),
    "small_kq_1024": ("PLAN_Q5_K_M", 1024, 2816, 2, 16, 4, 1000, 0, 3),
    "small_f32": ("PLAN_F32", 512, 1376, 2, 8, 8, 500, 0, 3),
    "pieces": ("PLAN_Q4_K", 2048, 2048, 2, 16, 4, 512, 0, 3),
    "persistent": ("PLAN_Q4_K_S", 512, 1024, 2, 8, 2, 320, 2, 2),
    "per_phase": ("PLAN_Q4_K_S", 256, 512, 2, 4, 2, 320, 0, 1),
}


def _device(pkg, name, seed):
    from llama2_jl_amd import _lib, synth
    from llama2_jl_amd.inference import DeviceModel
    plan, dim, hidden, layers, heads, kv, vocab, asked, path = MODELS[name]
    cfg = pkg.ModelConfig(dim=dim, hidden_dim=hidden, n_layers=layers, n_heads=heads, n_kv_heads=kv, vocab_size=vocab, seq_len=96,
                          rope_freq_base=10000.0)
    dev = DeviceModel(cfg, synth.synthetic_model(cfg, getattr(synth, plan), seed=seed).weights, ctx=_lib.Context(), path=asked)
    assert dev.path == path
    return dev


def _calls(dev, n, results):
    """n calls of three kinds, each from a fresh cache"""
    from llama2_jl_amd import synth
    vocab = dev.config.vocab_size
    for i in range(n):
        prompt = synth.seeded_prompt(100 + i, 2 + i % 7, vocab)
        dev.reset()
        ids, logits = dev.generate_greedy(prompt, 3 + 5 * (i % 5), want_logits=True)
        results.append((np.asarray(ids).tolist(), logits.tobytes()))
        tok, pos = int(ids[-1]), prompt.size - 1 + len(ids)
        for _ in range(3):
            logits, tok = dev.forward(tok, pos)
            pos += 1
            results.append((tok, logits.tobytes()))


@pytest.mark.parametrize("pair", [("small_kq", "small_kq_1024"), ("small_kq", "small_kq"), ("small_kq", "pieces"), ("small_f32", "small_kq"),
                                  ("persistent", "small_kq"), ("per_phase", "pieces")])
def test_each_gives_what_it_gives_alone(pkg, pair):
    n = 40
    devs = [_device(pkg, name, 5 + k) for k, name in enumerate(pair)]
    alone, together, errors = [[], []], [[], []], []
    for d, r in zip(devs, alone):
        _calls(d, n, r)

    def body(d, r):
        try:
            _calls(d, n, r)
        except Exception as e:  # (reported by the main thread)
            errors.append(e)

    threads = [threading.Thread(target=body, args=a) for a in zip(devs, together)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    assert together == alone
    for d, name in zip(devs, pair):
        from llama2_jl_amd import _lib
        assert _lib.lib().l2h_model_path(d.handle) == MODELS[name][8]
        ctx = d.ctx
        d.close()
        ctx.close()

"""Draws (l2h_sample) whose target lies between the running sums of two threads, or of two runs of logits, as they are rounded: every target has an element that
reaches it.  A classifier of rows c_i h / |h|^2 gives the model's final hidden state h the logits c_i, to fp32 rounding."""
import numpy as np
import pytest

from test_gpu_model import CASES, _model

pytestmark = pytest.mark.gpu


def _device(pkg, logits):
    plan, kw = CASES["f32"]
    lm = _model(pkg, plan, **dict(kw, vocab_size=len(logits), n_layers=1))
    dim = lm.config.dim
    rows = np.zeros((len(logits), dim), np.float32)
    rows[:dim] = np.eye(dim)
    lm.weights.output_weight = rows
    dev = lm.device()
    h = dev.forward(2, 0)[0][:dim].astype(np.float64)
    dev.close()
    lm.weights.output_weight = np.outer(logits, h / (h @ h)).astype(np.float32)
    dev = lm.device()
    got = dev.forward(2, 0)[0]
    assert np.allclose(got, logits, rtol=1e-5, atol=1e-5)
    return dev


# e^-37.82 is 3.76e-17: four of them come to 1.5e-16 beside a 1, where a last bit is 2.2e-16
@pytest.mark.parametrize("vocab,likely", [(300, 4), (4096, 4), (4097, 4), (5200, 4),  # in the run of the four; up to 4096 logits there is one
                                          (5200, 1024), (5200, 5199)])                # in another run, the last one among them
def test_targets_between_two_sums(pkg, vocab, likely):
    logits = np.full(vocab, -200.0)
    logits[:4] = -37.82
    logits[likely] = 0.0
    dev = _device(pkg, logits)
    four = 4 * np.exp(-37.82)
    for u, want in [(0.0, 0), (1e-17, 0), (1e-16, 2), (1.4e-16, 3), (1.6e-16, likely), (2e-16, likely), (2.2e-16, likely), (3e-16, likely), (0.5, likely),
                    (float(np.nextafter(np.float32(1), np.float32(0))), likely)]:
        assert abs(u - four) > 5e-18
        assert dev.sample_token(1.0, u) == want, u
    # (targets on both sides of the four's sum)
    for u in np.linspace(1.45e-16, 1.55e-16, 41):
        assert dev.sample_token(1.0, float(u)) in (3, likely), u
    dev.close()

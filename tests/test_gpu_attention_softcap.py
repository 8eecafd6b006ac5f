"""The soft cap of the logits, cap tanh(s / cap), on both sides of where its form changes (|s| = 0.8 cap), far beyond it and at infinity.

Bound: fp32 logits off by at most 4 units in the last place of the logit (the quotient, the polynomial or the exponential form and the
product), the probabilities by that, the sum over the keys and the exponential: 4 * 2^-24 * cap + 1e-6 relative, against float64."""
import math

import pytest
import torch

from _util import kernels_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cap", [0.5, 2.0, 30.0, 1000.0])
@pytest.mark.parametrize("D", [32, 64, 128, 256])
@pytest.mark.parametrize("spread", [0.05, 1.0, 20.0])
def test_capped_logits(D, cap, spread):
    from aidotnet.tensors_amd import Mi355Backend, Mi355Engine
    eng = Mi355Engine(Mi355Backend())
    gen = torch.Generator(device="cuda").manual_seed(D)
    q = torch.randn(2, 2, 45, D, device="cuda", generator=gen)
    k = torch.randn(2, 2, 83, D, device="cuda", generator=gen)
    v = torch.randn(2, 2, 83, D, device="cuda", generator=gen)
    scale = spread * cap / math.sqrt(D)                    # logits of a standard deviation of `spread` caps
    if not scale < 2.0 ** 20:
        pytest.skip("scale")
    o, w = eng.ScaledDotProductAttention(q, k, v, None, scale, softcap=cap)
    s = (q.double() @ k.double().transpose(-1, -2)) * scale
    p = torch.softmax(cap * torch.tanh(s / cap), -1)
    # a logit is a sum of D products, each rounded in fp32 as is every partial sum: off by some 2^-24 of sum |q k|, which is sqrt(D) times the
    # logit where the terms cancel, of which 1 / cosh^2 passes the cap; the cap itself adds its four units
    size = (q.double().abs() @ k.double().abs().transpose(-1, -2)) * scale
    slope = torch.cosh(torch.clamp(s / cap, -300, 300)).pow(-2)
    logit_err = (slope * size).amax(-1, keepdim=True) * 4 * 2.0 ** -24 + 4 * 2.0 ** -24 * cap
    bound = 2 * torch.expm1(logit_err) + 2e-6
    assert bool(((w.double() - p).abs() <= bound * p + 1e-30).all()), float(((w.double() - p).abs() / p).max())
    want = p @ v.double()
    assert bool(((o.double() - want).abs() <= bound * (p @ v.double().abs()) + 1e-30).all())


def test_infinite_and_nan_logits():
    from aidotnet.tensors_amd import Mi355Backend, Mi355Engine
    eng = Mi355Engine(Mi355Backend())
    q = torch.ones(1, 1, 3, 64, device="cuda"); k = torch.zeros(1, 1, 40, 64, device="cuda"); v = torch.ones(1, 1, 40, 64, device="cuda")
    k[0, 0, 7] = 3e38; k[0, 0, 9] = -3e38                  # logits of +inf and -inf: +-cap
    _, w = eng.ScaledDotProductAttention(q, k, v, None, 1.0, softcap=5.0)
    s = torch.zeros(40, dtype=torch.float64); s[7], s[9] = 5.0, -5.0
    assert torch.allclose(w[0, 0].cpu().double(), torch.softmax(s, 0).expand(3, 40), rtol=2e-6, atol=0)
    q[0, 0, 1, 0] = float("nan")
    o, w = eng.ScaledDotProductAttention(q, k, v, None, 1.0, softcap=5.0)
    assert bool(o[0, 0, 1].isnan().all()) and not bool(o[0, 0, 0].isnan().any()) and not bool(o[0, 0, 2].isnan().any())

"""Attention with a scale of zero (every visible key weighs the same) and below it: causal, padded and ragged key sequences, all types and widths.

Bounds: 4e-6 of the norm for fp32 sums, 1e-2 for 16-bit probabilities and values."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

KIND = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


@pytest.fixture(scope="module")
def eng():
    from aidotnet.tensors_amd import Mi355Engine
    return Mi355Engine()


def reference(q, k, v, scale, hidden):
    s = (torch.matmul(q.double(), k.double().transpose(2, 3).contiguous()) * scale).masked_fill(hidden, -math.inf)
    return torch.matmul(torch.softmax(s, -1), v.double()), torch.logsumexp(s, -1), torch.softmax(s, -1)


def inputs(D, Sq, Sk, kind="f32"):
    gen = torch.Generator(device="cuda").manual_seed(Sk + D)
    return [torch.randn(2, 2, n, D, device="cuda", generator=gen).to(KIND[kind]) for n in (Sq, Sk, Sk)]


@pytest.mark.parametrize("scale", [0.0, -0.125])
@pytest.mark.parametrize("Sq,Sk", [(70, 70), (33, 300)])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("D", [32, 64, 128, 256])
@pytest.mark.parametrize("kind", list(KIND))
def test_causal_and_ragged(eng, kind, D, causal, Sq, Sk, scale):
    q, k, v = inputs(D, Sq, Sk, kind)
    hidden = causal & (torch.arange(Sk, device="cuda")[None, :] > torch.arange(Sq, device="cuda")[:, None])
    want, lse, _ = reference(q, k, v, scale, hidden)
    o, l = eng.FlashAttention(q, k, v, scale, causal)
    tol = 4e-6 if kind == "f32" else 1e-2
    assert float((o.double() - want).norm() / want.norm()) <= tol
    assert float((l.double() - lse).abs().max()) <= (1e-5 if kind == "f32" else 1e-3)


@pytest.mark.parametrize("scale", [0.0, -0.125])
@pytest.mark.parametrize("D", [32, 64, 128, 256])
def test_padded_and_probabilities(eng, D, scale):
    q, k, v = inputs(D, 70, 131)
    keep = (torch.arange(131, device="cuda")[None, :] < torch.tensor([[60], [127]], device="cuda"))[:, None, None, :]
    want, _, p = reference(q, k, v, scale, ~keep)
    o, w = eng.ScaledDotProductAttention(q, k, v, keep, scale)
    assert float((o.double() - want).norm() / want.norm()) <= 4e-6 and float((w.double() - p).norm() / p.norm()) <= 4e-6

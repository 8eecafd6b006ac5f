"""Rounding of 16-bit attention behind a block table and under a key mask at head dimension 128: the direct-to-LDS kernel, split by key
ranges or not, is no further from float64 than the recurrence over 64-key tiles whose probabilities are rounded to the storage type
against the row's running maximum (the largest one of a row is then exactly 1) and whose sums are exact.

Bound: both errors are norms over some 10^5 outputs of independent roundings of the same width, so their ratio is known to about 1 %; a
reference that lags behind the row maximum raises it by 5 to 13 % on these shapes (the largest probability is rounded like the others)."""
import math

import pytest
import torch

from _util import TORCH16

pytestmark = pytest.mark.gpu


def exact_and_rounded(q, k, v, hidden, dtype):
    """q [H, Sq, D], k, v [H, Sk, D] in float64; hidden [Sq, Sk] or [1, Sk].  The attention in float64, and the recurrence above."""
    s = (torch.matmul(q, k.transpose(1, 2).contiguous()) / math.sqrt(q.shape[-1])).masked_fill(hidden, float("-inf"))
    m = torch.full(s.shape[:2] + (1,), float("-inf"), dtype=s.dtype, device=s.device)
    l, o = torch.zeros_like(m), torch.zeros(s.shape[:2] + (v.shape[-1],), dtype=s.dtype, device=s.device)
    for k0 in range(0, s.shape[-1], 64):
        x = s[..., k0:k0 + 64]
        m_new = torch.maximum(m, x.amax(-1, keepdim=True))
        ref = torch.where(torch.isinf(m_new), torch.zeros_like(m_new), m_new)
        p, w = torch.exp(x - ref), torch.exp(m - ref)
        l = l * w + p.sum(-1, keepdim=True)
        o = o * w + torch.matmul(p.to(dtype).double(), v[:, k0:k0 + 64])
        m = m_new
    return torch.matmul(torch.softmax(s, -1), v), o / l


@pytest.fixture(scope="module")
def be():
    from aidotnet.tensors_amd import Mi355Backend
    return Mi355Backend()


@pytest.mark.parametrize("kind", ["f16", "bf16"])
@pytest.mark.parametrize("heads,kv,block,nq,start", [(12, 12, 32, 182, 0), (32, 16, 64, 88, 66), (16, 4, 16, 60, 722), (8, 2, 16, 200, 3000)])
def test_paged_prefill(be, kind, heads, kv, block, nq, start):
    gen = torch.Generator(device="cuda").manual_seed(nq + start)
    keys, d = start + nq, 128
    blocks = (keys + block - 1) // block
    randn = lambda *s: torch.randn(*s, device="cuda", generator=gen).to(TORCH16[kind])
    q, kp, vp = randn(nq, heads, d), randn(blocks, block, kv, d), randn(blocks, block, kv, d)
    table = torch.randperm(blocks, device="cuda", generator=gen).to(torch.int32)
    W = be.WrapTensor
    got = be.PagedAttentionHalf(kind, W(q), W(kp), W(vp), W(table), heads, kv, d, block, nq, start, 1 / math.sqrt(d)).tensor.double().view(nq, heads, d)
    flat = lambda p: p[table.long()].reshape(-1, kv, d)[:keys].double().permute(1, 0, 2).repeat_interleave(heads // kv, 0).contiguous()
    i, j = torch.arange(nq, device="cuda")[:, None], torch.arange(keys, device="cuda")[None, :]
    want, rounded = exact_and_rounded(q.double().permute(1, 0, 2).contiguous(), flat(kp), flat(vp), j > i + start, TORCH16[kind])
    assert float((got.permute(1, 0, 2) - want).norm()) <= 1.02 * float((rounded - want).norm())


@pytest.mark.parametrize("kind", ["f16", "bf16"])
@pytest.mark.parametrize("H,Sq,Sk", [(16, 149, 149), (8, 130, 600), (8, 40, 2100)])
def test_key_mask(be, kind, H, Sq, Sk):
    from aidotnet.tensors_amd import AttnDesc
    gen = torch.Generator(device="cuda").manual_seed(Sq + Sk)
    d = 128
    randn = lambda *s: torch.randn(*s, device="cuda", generator=gen).to(TORCH16[kind])
    q, k, v = randn(H, Sq, d), randn(H, Sk, d), randn(H, Sk, d)
    keep = torch.rand(Sk, device="cuda", generator=gen) < 0.8
    o = torch.empty(H, Sq, d, device="cuda")
    W = be.WrapTensor
    be._attn(kind, W(q), W(k), W(v), W(o), None, None, W(keep), None, AttnDesc(B=1, H=H, Hkv=H, Sq=Sq, Sk=Sk, D=d, scale=1 / math.sqrt(d), mask_mode=3))
    want, rounded = exact_and_rounded(q.double(), k.double(), v.double(), ~keep[None, :], TORCH16[kind])
    assert float((o.double() - want).norm()) <= 1.02 * float((rounded - want).norm())

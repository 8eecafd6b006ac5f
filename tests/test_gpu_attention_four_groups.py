"""fp32 attention over two 128-key tiles of head dimension 64 on a small grid: the fp32 pipe with four waves to a row's keys, on both sides of the
edges of its range.

Bound: fp32 products and sums: 4e-6 of the norm against float64, the log-sum-exp 1e-5."""
import math

import pytest
import torch

from _util import kernels_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("B,H,Sq,Sk,groups", [(1, 4, 65, 192, True), (1, 4, 256, 256, True), (2, 16, 225, 225, True), (1, 4, 64, 200, False), (1, 4, 200, 191, False),
                                              (1, 4, 200, 257, False), (4, 16, 256, 256, False)])
def test_four_groups(B, H, Sq, Sk, groups, causal):
    from aidotnet.tensors_amd import Mi355Backend, Mi355Engine
    eng = Mi355Engine(Mi355Backend())
    gen = torch.Generator(device="cuda").manual_seed(Sk)
    q, k, v = (torch.randn(B, H, n, 64, device="cuda", generator=gen) for n in (Sq, Sk, Sk))
    names = kernels_of(lambda: eng.FlashAttention(q, k, v, isCausal=causal))
    if not causal or Sq > 64:                              # (up to 64 visible keys stay on the fp32 pipe too)
        assert len(names) == 1 and names[0].startswith("attn_fwd_kernel" if groups else "attn_split_kernel"), names
    o, lse = eng.FlashAttention(q, k, v, isCausal=causal)
    s = (q.double() @ k.double().transpose(-1, -2).contiguous()) * 0.125
    if causal:
        s = s.masked_fill(torch.arange(Sk, device="cuda")[None, :] > torch.arange(Sq, device="cuda")[:, None], -math.inf)
    want = torch.softmax(s, -1) @ v.double()
    assert float((o.double() - want).norm() / want.norm()) <= 4e-6 and float((lse.double() - torch.logsumexp(s, -1)).abs().max()) <= 1e-5

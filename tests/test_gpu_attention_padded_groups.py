"""16-bit attention layers under a padding mask, head dimension 64: two key groups to a query tile up to 768 workgroups of 64 queries, on both sides of
the line, against float64.

Bounds: a layer is a chain of roundings to the storage type: projections, probabilities, attention rows and result, each 2^-9 (bf16) or 2^-12 (fp16) at most
and an independent 0.58 of that in the 2-norm, with the sums of the projections 5e-3 and 6.5e-4."""
import math

import pytest
import torch

from _util import TORCH16, kernels_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,bound", [("bf16", 5e-3), ("f16", 6.5e-4)])
@pytest.mark.parametrize("B,S,H,groups", [(8, 512, 12, 2), (2, 70, 4, 2), (6, 500, 16, 2), (13, 512, 8, 1), (5, 1000, 12, 1)])
def test_padded_layer(kind, bound, B, S, H, groups):
    from aidotnet.tensors_amd import Mi355Engine
    eng = Mi355Engine()
    dM = 64 * H
    gen = torch.Generator(device="cuda").manual_seed(S)
    x = torch.randn(B, S, dM, device="cuda", generator=gen).to(TORCH16[kind])
    w = [(torch.randn(dM, dM, device="cuda", generator=gen) / math.sqrt(dM)).to(TORCH16[kind]) for _ in range(4)]
    lengths = torch.randint((S + 1) // 2, S + 1, (B,), device="cuda", generator=gen)
    keep = (torch.arange(S, device="cuda")[None, :] < lengths[:, None])[:, None, None, :]
    call = lambda: eng.MultiHeadAttentionForward(x, *w, H, keep)
    names = [n for n in kernels_of(call) if n.startswith("attn_fwd_kernel")]
    assert len(names) == 1 and names[0].rstrip(">").endswith(", %d" % groups), names
    heads = lambda i: (x.double().view(B * S, dM) @ w[i].double()).view(B, S, H, 64).transpose(1, 2).contiguous()
    q, k, v = heads(0), heads(1), heads(2)
    s = (torch.matmul(q, k.transpose(2, 3).contiguous()) / 8).masked_fill(~keep, -math.inf)
    want = (torch.matmul(torch.softmax(s, -1), v).transpose(1, 2).reshape(B * S, dM) @ w[3].double()).view(B, S, dM)
    assert float((call().double() - want).norm() / want.norm()) <= bound

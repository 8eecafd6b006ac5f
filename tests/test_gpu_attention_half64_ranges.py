"""16-bit attention at head dimension 64 with few query tiles over many keys: ranges of the keys and a merge, with dense and paged K and V.

Bound: probabilities rounded to the operand type, 2^-9 (bf16) and 2^-12 (fp16) of each against a row's sum: 7e-3 and 8e-4 of the norm against
float64 on the same rounded inputs, as in one range; the log-sum-exp 1e-5."""
import math

import pytest
import torch

from _util import TORCH16, kernels_of

pytestmark = pytest.mark.gpu
LIMIT = {"f16": 8e-4, "bf16": 7e-3}


def reference(q, k, v, scale, first=None):
    g = q.shape[1] // k.shape[1]
    k, v = k.repeat_interleave(g, 1).double(), v.repeat_interleave(g, 1).double()
    s = (q.double() @ k.transpose(-1, -2).contiguous()) * scale
    if first is not None:
        s = s.masked_fill(torch.arange(k.shape[2], device="cuda")[None, :] > torch.arange(q.shape[2], device="cuda")[:, None] + first, -math.inf)
    return torch.softmax(s, -1) @ v, torch.logsumexp(s, -1)


@pytest.mark.parametrize("kind", ["f16", "bf16"])
@pytest.mark.parametrize("causal", [False, True])
# (the shortest keys that are cut and one more, ranges that end short, one row and several tiles, 256 workgroups and fewer)
@pytest.mark.parametrize("B,H,Hkv,Sq,Sk", [(1, 2, 2, 1, 1152), (1, 8, 2, 65, 1153), (2, 3, 3, 31, 3000), (1, 1, 1, 200, 8200), (1, 16, 16, 189, 3984), (1, 8, 8, 1000, 1700)])
def test_dense(B, H, Hkv, Sq, Sk, causal, kind):
    from aidotnet.tensors_amd import Mi355Backend, Mi355Engine
    eng = Mi355Engine(Mi355Backend()); be = eng.backend; W = be.WrapTensor
    gen = torch.Generator(device="cuda").manual_seed(Sk)
    q, k, v = (torch.randn(B, h, n, 64, device="cuda", generator=gen).to(TORCH16[kind]) for h, n in ((H, Sq), (Hkv, Sk), (Hkv, Sk)))
    call = lambda: eng.FlashAttention(q, k, v, 0.125, causal, queryOffset=Sk - Sq if causal else 0)
    assert [n.split("<")[0] for n in kernels_of(call)] == ["attn_fwd_kernel", "attn_split_merge_kernel"]
    o, lse = call()
    want, true = reference(q, k, v, 0.125, Sk - Sq if causal else None)
    assert float((o.double() - want).norm() / want.norm()) <= LIMIT[kind] and float((lse.double() - true).abs().max()) <= 1e-5
    raw = torch.full((B * H * Sq * 64 + 64,), -7.0, device="cuda", dtype=q.dtype)
    be.FlashAttentionHalf(kind, W(q), W(k), W(v), W(raw), None, B, H, Sq, Sk, 64, 0.125, causal, Sk - Sq if causal else 0, Hkv, True)
    assert float((raw[:-64].view(B, H, Sq, 64).double() - want).norm() / want.norm()) <= 1.5 * LIMIT[kind] and bool((raw[-64:] == -7.0).all())


@pytest.mark.parametrize("kind", ["f16", "bf16"])
@pytest.mark.parametrize("block", [16, 40, 64])
@pytest.mark.parametrize("H,Hkv,S,start", [(16, 16, 189, 3795), (12, 6, 614, 2524), (4, 1, 8, 16000)])
def test_paged(H, Hkv, S, start, block, kind):
    from aidotnet.tensors_amd import Mi355Backend
    be = Mi355Backend(); W = be.WrapTensor
    gen = torch.Generator(device="cuda").manual_seed(S)
    n = start + S
    blocks = (n + block - 1) // block
    table = torch.randperm(blocks + 3, device="cuda", generator=gen)[:blocks].int()
    kp, vp = (torch.randn(blocks + 3, block, Hkv, 64, device="cuda", generator=gen).to(TORCH16[kind]) for _ in range(2))
    q = torch.randn(S, H, 64, device="cuda", generator=gen).to(TORCH16[kind])
    call = lambda: be.PagedAttentionHalf(kind, W(q), W(kp), W(vp), W(table), H, Hkv, 64, block, S, start, 0.125)
    assert [x.split("<")[0] for x in kernels_of(call)] == ["attn_fwd_kernel", "attn_split_merge_kernel"]
    out = call().tensor.view(S, H, 64)
    k, v = (x[table.long()].reshape(-1, Hkv, 64)[:n].transpose(0, 1)[None] for x in (kp, vp))
    want, _ = reference(q.transpose(0, 1)[None], k, v, 0.125, start)
    assert float((out.double() - want[0].transpose(0, 1)).norm() / want.norm()) <= LIMIT[kind]


def test_not_a_number_stays():
    from aidotnet.tensors_amd import Mi355Backend, Mi355Engine
    eng = Mi355Engine(Mi355Backend())
    q, k, v = (torch.randn(1, 2, n, 64, device="cuda").bfloat16() for n in (40, 2000, 2000))
    q[0, 1, 5, 3] = math.nan
    o, _ = eng.FlashAttention(q, k, v)
    assert bool(o[0, 1, 5].isnan().all()) and bool(o[0, 0].isfinite().all()) and bool(o[0, 1, :5].isfinite().all()) and bool(o[0, 1, 6:].isfinite().all())

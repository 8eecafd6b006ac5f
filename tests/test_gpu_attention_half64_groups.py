"""16-bit attention at head dimension 64: how many waves share the keys of a query tile, and on which key tiles, on both sides of each line, with rows
that end inside a wave's block of 32 keys.

Bounds: probabilities rounded to the operand type against float64 on the same rounded inputs.  A rounding is 2^-9 (bf16) or 2^-12 (fp16) at most and
0.41 to 0.58 of that in the 2-norm; the largest of each group are exactly one, which takes off what fewer groups would add: 1.45e-3 and 1.85e-4 over the
rows measured here, one group 1.55e-3 and 2e-4; the log-sum-exp 1e-5."""
import math

import pytest
import torch

from _util import TORCH16, kernels_of

pytestmark = pytest.mark.gpu
LIMIT = {"f16": 1.85e-4, "bf16": 1.48e-3}


def reference(q, k, v, first):
    g = q.shape[1] // k.shape[1]
    s = torch.matmul(q.double(), k.double().repeat_interleave(g, 1).transpose(2, 3).contiguous()) / 8
    if first is not None:
        s = s.masked_fill(torch.arange(k.shape[2], device="cuda")[None, :] > torch.arange(q.shape[2], device="cuda")[:, None] + first, -math.inf)
    return torch.matmul(torch.softmax(s, -1), v.double().repeat_interleave(g, 1)), torch.logsumexp(s, -1)


def tile_and_groups(call):
    """(keys to a tile, key groups) of the attention kernel that `call` launches"""
    names = [n for n in kernels_of(call) if n.startswith("attn_fwd_kernel")]
    assert len(names) == 1, names
    args = names[0].split("<", 1)[1].rstrip("> ").split(", ")
    return int(args[3]), int(args[-1])


@pytest.mark.parametrize("kind", ["f16", "bf16"])
@pytest.mark.parametrize("B,H,Sq,Sk,causal,plan", [
    (1, 8, 300, 191, False, (64, 2)), (1, 8, 300, 192, False, (128, 4)), (2, 16, 256, 257, False, (128, 4)), (2, 16, 257, 257, False, (64, 2)),
    (2, 16, 257, 319, False, (64, 2)), (2, 16, 257, 321, False, (128, 4)), (1, 16, 1024, 385, False, (128, 4)), (1, 16, 1025, 385, False, (64, 2)),
    (2, 12, 449, 449, True, (128, 4)), (2, 12, 513, 513, True, (128, 2)), (4, 12, 512, 512, True, (128, 2)), (4, 32, 257, 257, True, (64, 2)),
    (4, 16, 450, 450, True, (128, 2)), (4, 16, 513, 513, True, (64, 2)), (2, 10, 1023, 1023, True, (128, 2)), (2, 10, 1024, 1024, True, (128, 4)), (2, 10, 1025, 1025, True, (128, 2)),
    (2, 16, 1152, 1200, True, (128, 2)), (2, 16, 1153, 1200, True, (64, 2))])
def test_dense(B, H, Sq, Sk, causal, plan, kind):
    from aidotnet.tensors_amd import Mi355Engine
    eng = Mi355Engine()
    gen = torch.Generator(device="cuda").manual_seed(Sk)
    q, k, v = (torch.randn(B, H, n, 64, device="cuda", generator=gen).to(TORCH16[kind]) for n in (Sq, Sk, Sk))
    call = lambda: eng.FlashAttention(q, k, v, 0.125, causal)
    assert tile_and_groups(call) == plan
    o, lse = call()
    want, true = reference(q, k, v, 0 if causal else None)
    assert float((o.double() - want).norm() / want.norm()) <= LIMIT[kind] and float((lse.double() - true).abs().max()) <= 1e-5


@pytest.mark.parametrize("kind", ["f16", "bf16"])
@pytest.mark.parametrize("H,Hkv,S,start,block,plan", [(16, 4, 130, 95, 32, (128, 4)), (16, 4, 130, 95, 16, (64, 2)), (16, 4, 130, 95, 48, (64, 2)), (32, 8, 500, 411, 96, (128, 2)),
                                                     (32, 8, 500, 411, 16, (64, 2)), (32, 8, 600, 511, 64, (128, 4)), (32, 8, 1100, 13, 64, (128, 2))])
def test_paged(H, Hkv, S, start, block, plan, kind):
    from aidotnet.tensors_amd import Mi355Backend
    be = Mi355Backend(); W = be.WrapTensor
    gen = torch.Generator(device="cuda").manual_seed(S)
    n = start + S
    blocks = (n + block - 1) // block
    table = torch.randperm(blocks + 3, device="cuda", generator=gen)[:blocks].int()
    kp, vp = (torch.randn(blocks + 3, block, Hkv, 64, device="cuda", generator=gen).to(TORCH16[kind]) for _ in range(2))
    q = torch.randn(S, H, 64, device="cuda", generator=gen).to(TORCH16[kind])
    call = lambda: be.PagedAttentionHalf(kind, W(q), W(kp), W(vp), W(table), H, Hkv, 64, block, S, start, 0.125)
    assert tile_and_groups(call) == plan
    out = call().tensor.view(S, H, 64)
    k, v = (x[table.long()].reshape(-1, Hkv, 64)[:n].transpose(0, 1)[None].contiguous() for x in (kp, vp))
    want, _ = reference(q.transpose(0, 1)[None].contiguous(), k, v, start)
    assert float((out.double() - want[0].transpose(0, 1)).norm() / want.norm()) <= LIMIT[kind]

"""Decode with four query heads per workgroup on both sides of 512 workgroups (the loads of one or of two iterations in flight), with lengths
that end inside an iteration, contiguous and behind a block table, against a float64 softmax; fp32 after the load, held at 1e-4."""
import math

import pytest
import torch

from _util import TORCH16

pytestmark = pytest.mark.gpu
DT = {"f32": torch.float32, **TORCH16}


# B, H, Hkv, D, keys, splits: B H / 4 x splits workgroups
@pytest.mark.parametrize("kind", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("B,H,Hkv,D,S,splits", [
    (8, 16, 2, 64, 4099, 16), (8, 16, 2, 64, 4330, 17), (5, 16, 2, 32, 6530, 26), (33, 64, 16, 64, 70, 1), (20, 8, 1, 256, 3701, 14), (45, 16, 4, 80, 777, 3)])
def test_contiguous(kind, B, H, Hkv, D, S, splits):
    from aidotnet.tensors_amd import Mi355Backend
    be = Mi355Backend()
    gen = torch.Generator(device="cuda").manual_seed(S)
    q, k, v = (torch.randn(*s, device="cuda", generator=gen).to(DT[kind]) for s in ((B, H, 1, D), (B, Hkv, S, D), (B, Hkv, S, D)))
    o = torch.empty(B, H, 1, D, device="cuda")
    be.DecodeAttention(kind, *(be.WrapTensor(t) for t in (q, k, v, o)), B, H, S, D, 1 / math.sqrt(D), numKVHeads=Hkv, splits=splits)
    g = H // Hkv
    for b in range(B):
        K, V = k[b].double(), v[b].double()
        p = torch.softmax(torch.matmul(q[b].double().reshape(Hkv, g, D), K.transpose(1, 2).contiguous()) / math.sqrt(D), -1)
        want = torch.matmul(p, V).reshape(H, 1, D)
        assert float(((o[b].double() - want).abs() / (1 + want.abs())).max()) <= 1e-4, b


@pytest.mark.parametrize("kind", ["f32", "bf16"])
@pytest.mark.parametrize("H,Hkv,D,block,S", [(64, 16, 64, 16, 9001), (64, 8, 64, 48, 12345)])
def test_block_table(kind, H, Hkv, D, block, S):
    from aidotnet.tensors_amd import Mi355Backend
    be = Mi355Backend()
    gen = torch.Generator(device="cuda").manual_seed(S)
    blocks = (S + block - 1) // block
    T = DT[kind]
    q, kp, vp = (torch.randn(*s, device="cuda", generator=gen).to(T) for s in ((1, H, D), (blocks + 3, block, Hkv, D), (blocks + 3, block, Hkv, D)))
    table = torch.randperm(blocks + 3, device="cuda", generator=gen)[:blocks].to(torch.int32)
    W = be.WrapTensor
    got = be._paged("decode", kind, W(q), W(kp), W(vp), W(table), H, Hkv, D, block, 1, S, 0, 1 / math.sqrt(D), 35, True).tensor.reshape(H, D)
    K, V = (t[table.long()].reshape(-1, Hkv, D)[:S].double().transpose(0, 1).contiguous() for t in (kp, vp))
    p = torch.softmax(torch.matmul(q[0].double().reshape(Hkv, H // Hkv, D), K.transpose(1, 2).contiguous()) / math.sqrt(D), -1)
    want = torch.matmul(p, V).reshape(H, D)
    assert float(((got.double() - want).abs() / (1 + want.abs())).max()) <= 1e-4

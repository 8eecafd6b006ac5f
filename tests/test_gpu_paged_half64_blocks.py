"""16-bit paged prefill at head dimension 64 in one range: every block size, also those of which a tile's loads see only half a group of 32 keys.

Bound: probabilities rounded to the operand type: 7e-3 (bf16) and 8e-4 (fp16) of the norm against float64 on the same rounded inputs."""
import pytest
import torch

from _util import TORCH16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["f16", "bf16"])
@pytest.mark.parametrize("block", [16, 24, 32, 48, 64, 80])
@pytest.mark.parametrize("H,Hkv,S,start", [(32, 8, 300, 200), (8, 8, 70, 30), (64, 8, 700, 0)])
def test_blocks(H, Hkv, S, start, block, kind):
    from aidotnet.tensors_amd import Mi355Backend
    be = Mi355Backend(); W = be.WrapTensor
    gen = torch.Generator(device="cuda").manual_seed(S)
    n = start + S
    blocks = (n + block - 1) // block
    table = torch.randperm(blocks + 3, device="cuda", generator=gen)[:blocks].int()
    kp, vp = (torch.randn(blocks + 3, block, Hkv, 64, device="cuda", generator=gen).to(TORCH16[kind]) for _ in range(2))
    q = torch.randn(S, H, 64, device="cuda", generator=gen).to(TORCH16[kind])
    out = be.PagedAttentionHalf(kind, W(q), W(kp), W(vp), W(table), H, Hkv, 64, block, S, start, 0.125).tensor.view(S, H, 64)
    k, v = (x[table.long()].reshape(-1, Hkv, 64)[:n].transpose(0, 1).repeat_interleave(H // Hkv, 0).double() for x in (kp, vp))
    s = (q.transpose(0, 1).double() @ k.transpose(-1, -2).contiguous()) * 0.125
    s = s.masked_fill(torch.arange(n, device="cuda")[None, :] > torch.arange(S, device="cuda")[:, None] + start, -float("inf"))
    want = (torch.softmax(s, -1) @ v).transpose(0, 1)
    assert float((out.double() - want).norm() / want.norm()) <= {"f16": 8e-4, "bf16": 7e-3}[kind]

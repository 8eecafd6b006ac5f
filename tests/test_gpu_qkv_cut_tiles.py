"""The three products of an attention layer in one launch, where their widths leave the last tile column partly filled: each product's
stores end at its own columns, which the next one's begin behind.  Named by the kernel that ran.

Bounds on |error| / |result| (2-norms) against float64 with the layer's own roundings to storage: bf16 rounds the result once and what is
left of three roundings before it, each at most 2^-9; fp32 sums as everywhere."""
import pytest
import torch

from _util import kernels_of

pytestmark = pytest.mark.gpu

CASES = [(8, 512, 5, torch.bfloat16, "gemm_dl16_kernel<bf16_t, bf16_t, 2, true, false, 4, true>"),
         (16, 512, 5, torch.bfloat16, "gemm_dl16_kernel<bf16_t, bf16_t, 2, true, false, 2, true>"),
         (8, 512, 13, torch.bfloat16, "gemm_dl16_kernel<bf16_t, bf16_t, 3, false, false, 4, true>"),
         (16, 512, 5, torch.float32, "gemm_split_kernel<128, 2, 3, 1>"), (8, 512, 13, torch.float32, "gemm_split_kernel<64, 2, 3, 1>"),
         (8, 512, 12, torch.float32, "gemm_split_kernel<64, 2, 3, 0>")]


@pytest.mark.parametrize("B,S,H,dt,kernel", CASES)
def test_attention_layer(B, S, H, dt, kernel):
    from aidotnet.tensors_amd import Mi355Engine
    eng = Mi355Engine()
    d, dM = 64, 64 * H
    gen = torch.Generator(device="cuda").manual_seed(B + H)
    x = torch.randn(B, S, dM, device="cuda", generator=gen).to(dt)
    w = [(torch.randn(dM, dM, device="cuda", generator=gen) / dM ** 0.5).to(dt) for _ in range(4)]
    out = []
    names = kernels_of(lambda: out.append(eng.MultiHeadAttentionForward(x, *w, H, None)))
    assert names[0] == kernel, names
    q, k, v = ((x.double() @ w[i].double()).to(dt).double().view(B, S, H, d).transpose(1, 2) for i in range(3))
    att = torch.softmax(q @ k.transpose(-1, -2).contiguous() / 8.0, -1) @ v
    want = att.to(dt).double().transpose(1, 2).reshape(B, S, dM) @ w[3].double()
    assert float((out[0].double() - want).norm() / want.norm()) <= (4e-6 if dt == torch.float32 else 3 * 2.0 ** -9)

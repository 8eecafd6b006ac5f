"""16-bit products of 9 to 15 columns over very many rows: from about 10^10 multiply-adds on, with K a multiple of 64, B and C go through
padded copies while A is read where it is and takes no workspace.

Bound: 16-bit operands, fp32 sums, one rounding of the result: 2^-9 relative (bf16) and 2^-11 (fp16) of each, held at 2^-8 and 2^-10 of the
norm; rows sampled over the whole range, float64."""
import pytest
import torch

from _util import TORCH16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["f16", "bf16"])
@pytest.mark.parametrize("M,N,K", [(100000, 13, 8192), (262147, 9, 4096), (140000, 15, 4096)])
def test_narrow_tall(M, N, K, kind):
    from aidotnet.tensors_amd import Mi355Backend
    be = Mi355Backend(); W = be.WrapTensor
    gen = torch.Generator(device="cuda").manual_seed(N)
    x = torch.empty(M, K, dtype=TORCH16[kind], device="cuda")
    for r in range(0, M, 16384):
        x[r:r + 16384] = torch.randn(min(16384, M - r), K, device="cuda", generator=gen).to(x.dtype)
    w = (torch.randn(K, N, device="cuda", generator=gen) / K ** 0.5).to(x.dtype)
    y = torch.empty(M, N, dtype=x.dtype, device="cuda")
    (be.Hgemm if kind == "f16" else be.Bf16Gemm)(W(x), W(w), W(y), M, N, K)
    assert be.WorkspaceBytes() < M * K // 4
    rows = torch.cat([torch.arange(300), torch.arange(M - 300, M), torch.randint(0, M, (1000,))]).cuda()
    want = x[rows].double() @ w.double()
    assert float((y[rows].double() - want).norm() / want.norm()) <= (2.0 ** -10 if kind == "f16" else 2.0 ** -8)

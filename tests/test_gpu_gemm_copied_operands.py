"""Which 16-bit products off the 16-byte grid go through padded copies (told by the workspace: at least B's copy, or the partial sums of
the K ranges alone) and their values on both sides of the line.

Bound: 16-bit operands, fp32 sums, one rounding of the result: 2^-9 relative (bf16) and 2^-11 (fp16) of each, held at 2^-8 and 2^-10 of the
norm; sampled rows, float64."""
import pytest
import torch

from _util import TORCH16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["f16", "bf16"])
@pytest.mark.parametrize("M,N,K,copied", [(1677, 3683, 3455, True), (3722, 1021, 7711, True), (4096, 4095, 4096, True),
                                          (372, 2901, 4904, False), (210, 1063, 6344, False), (700, 9001, 801, False), (2189, 571, 1347, False)])
def test_copied_or_in_place(M, N, K, copied, kind):
    from aidotnet.tensors_amd import Mi355Backend
    be = Mi355Backend(); W = be.WrapTensor
    gen = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn(M, K, device="cuda", generator=gen).to(TORCH16[kind])
    w = (torch.randn(K, N, device="cuda", generator=gen) / K ** 0.5).to(x.dtype)
    y = torch.empty(M, N, dtype=x.dtype, device="cuda")
    (be.Hgemm if kind == "f16" else be.Bf16Gemm)(W(x), W(w), W(y), M, N, K)
    assert (be.WorkspaceBytes() >= K * N * 2) == copied
    rows = torch.cat([torch.arange(70), torch.arange(M - 70, M), torch.randint(0, M, (200,))]).cuda()
    want = x[rows].double() @ w.double()
    assert float((y[rows].double() - want).norm() / want.norm()) <= (2.0 ** -10 if kind == "f16" else 2.0 ** -8)

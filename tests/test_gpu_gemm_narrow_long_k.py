"""16-bit products of fewer than 128 columns over a long K: K ranges of the 128 x 128 tile, summed by a pass of their own.

Bound: 16-bit operands, fp32 sums, one rounding of the result: 2^-9 relative (bf16) and 2^-11 (fp16) of each, held at 2^-8 and 2^-10 of the
norm, float64; without ranges 1e-5 of the norm for an fp32 result (fp32 sums of up to 8192 products)."""
import pytest
import torch

from _util import TORCH16, kernels_of

pytestmark = pytest.mark.gpu


# (the fewest and the most columns, a partial and several row tiles, the shortest K and one whose last range is shorter)
@pytest.mark.parametrize("kind", ["f16", "bf16"])
@pytest.mark.parametrize("M,N,K", [(1, 8, 2048), (4, 64, 3008), (129, 64, 1856), (300, 120, 8128), (1433, 64, 5120), (16384, 32, 2048)])
def test_narrow_long_k(M, N, K, kind):
    from aidotnet.tensors_amd import Mi355Backend
    be = Mi355Backend(); W = be.WrapTensor
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(M, K, device="cuda", generator=gen).to(TORCH16[kind])
    w = (torch.randn(K, N, device="cuda", generator=gen) / K ** 0.5).to(TORCH16[kind])
    want = x.double() @ w.double()
    raw = torch.full((M * N + 64,), -7.0, device="cuda", dtype=x.dtype)
    raw32 = torch.full((M * N + 64,), -7.0, device="cuda")
    fn, fn32 = (be.Hgemm, be.GemmFp16In32fOut) if kind == "f16" else (be.Bf16Gemm, be.GemmBf16In32fOut)
    names = kernels_of(lambda: fn(W(x), W(w), W(raw), M, N, K))
    if M * K < 2 ** 24:                                    # (few row tiles: ranges pay)
        assert len(names) == 2 and names[0].startswith("gemm_dl16_kernel"), names
    fn32(W(x), W(w), W(raw32), M, N, K)
    assert float((raw[:M * N].view(M, N).double() - want).norm() / want.norm()) <= (2.0 ** -10 if kind == "f16" else 2.0 ** -8)
    assert float((raw32[:M * N].view(M, N).double() - want).norm() / want.norm()) <= 1e-5
    assert bool((raw[M * N:] == -7.0).all()) and bool((raw32[M * N:] == -7.0).all())

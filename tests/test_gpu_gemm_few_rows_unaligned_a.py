"""Up to 16 rows of A off the 16-byte grid on an aligned B of at most 256 x 16384: the general kernel runs (the bits of its forced 64 x 64
tile), the sizes one past each line run elsewhere; both against float64.

Bound: 16-bit operands, fp32 sums, one rounding of the result: 2^-9 relative (bf16) and 2^-11 (fp16) of each, held at 2^-8 and 2^-10 of the
norm."""
import pytest
import torch

from _util import TORCH16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["f16", "bf16"])
@pytest.mark.parametrize("M,N,K,offset,general", [(2, 15424, 209, 0, True), (16, 16384, 255, 0, True), (1, 24, 101, 0, True), (9, 4096, 256, 1, True), (4, 1024, 65, 0, True),
                                                  (17, 4096, 255, 0, False), (2, 16392, 209, 0, False), (2, 4096, 257, 0, False)])
def test_few_rows(M, N, K, offset, general, kind):
    from aidotnet.tensors_amd import Mi355Backend
    be = Mi355Backend(); W = be.WrapTensor
    gen = torch.Generator(device="cuda").manual_seed(N + K)
    raw = torch.randn(M * K + offset, device="cuda", generator=gen).to(TORCH16[kind])
    x = raw[offset:].view(M, K)
    w = (torch.randn(K, N, device="cuda", generator=gen) / K ** 0.5).to(x.dtype)
    y, z = torch.empty(M, N, dtype=x.dtype, device="cuda"), torch.empty(M, N, dtype=x.dtype, device="cuda")
    call = be.Hgemm if kind == "f16" else be.Bf16Gemm
    call(W(x), W(w), W(y), M, N, K)
    be.SetGemmTile(64)
    call(W(x), W(w), W(z), M, N, K)
    if general:
        assert torch.equal(y, z)
    want = x.double() @ w.double()
    for got in (y, z):
        assert float((got.double() - want).norm() / want.norm()) <= (2.0 ** -10 if kind == "f16" else 2.0 ** -8)

"""Which kernels a 16-bit product runs, where its rules meet: the estimates behind them may be fitted anew, but not silently lose these sizes."""
import pytest
import torch

from _util import kernels_of

pytestmark = pytest.mark.gpu

RANGES = ["gemm_dl16_kernel<bf16_t, float, 2, true", "skinny_reduce_kernel"]       # K ranges of 128 x 128 tiles and their sum
TILE64 = ["gemm_dl_kernel<bf16_t, bf16_t, false, 64"]                              # 64 x 64 tiles without edge handling
CASES = [(2048, 512, 2048, RANGES), (1000, 1024, 2048, RANGES), (512, 1024, 1792, RANGES), (1024, 1024, 2048, RANGES),
         (512, 4672, 512, TILE64), (384, 6976, 768, TILE64), (640, 3648, 832, TILE64), (1152, 4032, 128, TILE64)]


@pytest.mark.parametrize("M,N,K,want", CASES)
def test_plan_and_product(M, N, K, want):
    from aidotnet.tensors_amd import Mi355Backend
    be = Mi355Backend(); W = be.WrapTensor
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    a, b = ((torch.randint(-8, 9, s, generator=gen, device="cuda") / 8).bfloat16() for s in ((M, K), (K, N)))
    c = torch.empty(M, N, device="cuda", dtype=torch.bfloat16)
    names = kernels_of(lambda: be.Bf16Gemm(W(a), W(b), W(c), M, N, K))
    assert len(names) == len(want) and all(n.startswith(w) for n, w in zip(names, want)), names
    # (every partial sum of these inputs is exact in fp32: one rounding)
    assert torch.equal(c, (a.double() @ b.double()).float().bfloat16())

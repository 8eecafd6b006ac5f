"""Which kernels a 16-bit product runs, where its rules meet: the estimates behind them may be fitted anew, but not silently lose these sizes."""
import pytest
import torch

from _util import kernels_of

pytestmark = pytest.mark.gpu

RANGES = ["gemm_dl16_kernel<bf16_t, float, 2, true, false, 4, false>", "skinny_reduce_kernel"]      # K ranges of 128 x 128 tiles and their sum
CUT_RANGES = ["gemm_dl16_kernel<bf16_t, float, 2, true, false, 4, true>", "skinny_reduce_kernel"]
TILE64 = ["gemm_dl_kernel<bf16_t, bf16_t, false, 64"]                              # 64 x 64 tiles without edge handling
EDGE64 = ["gemm_dl_kernel<bf16_t, bf16_t, true, 64"]
FEW = ["gemm_skinny_kernel<bf16_t, 7>", "skinny_reduce_kernel"]


def cut(tile):                                                                     # the 16 x 16 x 32 kernel with a partial last column
    return ["gemm_dl16_kernel<bf16_t, bf16_t, %s, true>" % tile]


CASES = [(2048, 512, 2048, RANGES), (1000, 1024, 2048, RANGES), (512, 1024, 1792, RANGES), (1024, 1024, 2048, RANGES),
         (512, 4672, 512, TILE64), (384, 6976, 768, TILE64), (640, 3648, 832, TILE64), (1152, 4032, 128, TILE64),
         # the sizes of test_gpu_gemm_ragged_columns.py
         (1000, 11008, 64, cut("3, false, false, 4")), (1000, 11000, 128, cut("3, false, false, 4")), (4000, 4088, 64, cut("2, true, false, 2")),
         (2040, 4088, 6208, cut("2, false, false, 4")), (2040, 4088, 128, cut("2, true, false, 2")), (2000, 2040, 64, cut("2, true, false, 4")),
         (300, 64, 192, EDGE64), (129, 136, 1088, EDGE64), (200, 1032, 2624, CUT_RANGES), (64, 4104, 4160, CUT_RANGES),
         (1000, 8192, 8256, ["gemm_dl16_kernel<bf16_t, bf16_t, 2, false, false, 4, false>"]), (33, 1000, 2112, EDGE64),
         (1, 136, 2560, FEW), (32, 248, 2624, FEW), (32, 1000, 4160, FEW), (32, 4104, 1536, FEW), (5, 8200, 8192, FEW),
         (7, 11000, 1600, ["gemm_skinny_kernel<bf16_t, 3>", "skinny_reduce_kernel"]), (17, 50264, 128, cut("2, true, false, 2")),
         (1000, 8192, 10560, ["gemm_dl16_kernel<bf16_t, float, 4, false, true, 4, false>", "skinny_reduce_kernel"]),
         (1000, 12296, 768, cut("4, false, false, 4")), (2000, 6152, 768, cut("4, false, false, 4")), (8192, 13000, 1024, cut("4, false, true, 4"))]


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

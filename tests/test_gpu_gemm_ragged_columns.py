"""16-bit products of aligned rows whose columns do not fill whole tiles: every tile width of the 16 x 16 x 32 kernel with a partial last
column, K ranges of uneven length, the few-row stream past the last slab of 128 columns.

Dyadic inputs make every product and partial sum exact in fp32, so results must equal the float64 product rounded once; bias and activation
are held to fp32 arithmetic plus that rounding (2^-8 of bf16, relative)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# 256 x 192 / 256 x 128 / 128 x 128 on both rings with a partial last column; K ranges of 128 x 128 tiles; few rows (one, two slabs, two workgroups
# per CU); 256 x 256 in two K ranges of uneven length; 256 x 256 with a partial last column, twice, and with non-temporal stores
# (test_gpu_gemm_plans.py holds which kernel each of them runs)
SHAPES = [(1000, 11008, 64), (1000, 11000, 128), (4000, 4088, 64), (2040, 4088, 6208), (2040, 4088, 128), (2000, 2040, 64), (300, 64, 192),
          (129, 136, 1088), (128, 136, 1088), (200, 1032, 2624), (64, 4104, 4160), (1000, 8192, 8256), (33, 1000, 2112),
          (1, 136, 2560), (32, 248, 2624), (32, 1000, 4160), (32, 4104, 1536), (7, 11000, 1600), (17, 50264, 128), (5, 8200, 8192),
          (1000, 8192, 10560), (1000, 12296, 768), (2000, 6152, 768), (8192, 13000, 1024)]


def operands(M, N, K, dt):
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    a = torch.randint(-8, 9, (M, K), generator=gen, device="cuda").to(dt) / 8
    b = torch.randint(-8, 9, (K, N), generator=gen, device="cuda").to(dt) / 8
    return a, b, a.double() @ b.double()


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_exact_products(M, N, K, dt):
    from aidotnet.tensors_amd import Mi355Backend
    be = Mi355Backend(); W = be.WrapTensor
    a, b, want = operands(M, N, K, dt)
    for out, call in ((dt, be.Hgemm if dt == torch.float16 else be.Bf16Gemm),
                      (torch.float32, be.GemmFp16In32fOut if dt == torch.float16 else be.GemmBf16In32fOut)):
        c = torch.full((M * N + 64,), -7.0, device="cuda", dtype=out)
        call(W(a), W(b), W(c), M, N, K)
        torch.cuda.synchronize()
        assert torch.equal(c[:M * N].view(M, N), want.float().to(out)) and bool((c[M * N:] == -7.0).all())


@pytest.mark.parametrize("act", ["None", "Swish"])
@pytest.mark.parametrize("M,N,K", [(1000, 11000, 128), (4000, 4088, 64), (2000, 2040, 64), (200, 1032, 2624), (32, 1000, 4160)])
def test_bias_and_activation(M, N, K, act):
    from aidotnet.tensors_amd import Mi355Engine
    a, b, z = operands(M, N, K, torch.bfloat16)
    bias = torch.randn(N, generator=torch.Generator().manual_seed(N)).cuda()
    y = Mi355Engine().FusedLinear(a, b, bias, act).double()
    z = z + bias.double()
    want = z if act == "None" else z * torch.sigmoid(z)
    assert torch.allclose(y, want, rtol=2.0 ** -8, atol=1e-5)

"""fp32 products on the bf16 matrix pipe (three bf16 values to an operand, two to an fp16 weight): mostly tiles of 64 rows by 128 columns in
K ranges, with K remainders, columns past the end, operands at any element (every instance by name: test_gpu_gemm_split_tiles.py).

Bound: every 32 of K add one fp32 rounding of the running sum, the sums inside them and what the split leaves out stay below ten more:
|error| <= (K / 32 + 10) 2^-24 sum |a| |b|."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(9, 2, 2049), (10, 3, 3001), (33, 127, 2046), (63, 129, 4127), (64, 130, 2080), (65, 255, 4097), (129, 257, 1057), (1025, 1155, 33),
          (1024, 1152, 512), (2000, 2001, 65), (2048, 2048, 96), (1537, 2176, 100), (4096, 3072, 64), (4095, 3072, 64), (300, 40001, 31)]


def operands(M, N, K, half, seed, lead=0):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    def place(t, dt):
        raw = torch.full((lead + t.numel(),), float("nan"), dtype=dt, device="cuda")
        raw[lead:] = t.reshape(-1)
        return raw[lead:].view(t.shape)
    a = torch.randn(M, K, device="cuda", generator=gen)
    b = torch.randn(K, N, device="cuda", generator=gen)
    return place(a, torch.float32), place(b, torch.float16 if half else torch.float32)


def call(a, b, bias=None, act=0, out=None):
    from aidotnet.tensors_amd import Mi355Backend
    be = Mi355Backend(); W = be.WrapTensor
    M, K = a.shape
    N = b.shape[1]
    c = torch.full((M, N), float("nan"), device="cuda") if out is None else out
    f = be.GemmFp16WeightB if b.dtype == torch.float16 else be.GemmBiasActivationInto
    f(W(a), W(b), W(bias) if bias is not None else None, W(c), M, N, K, act, 0.0)
    torch.cuda.synchronize()
    return c


def check(c, a, b, K, extra=0.0):
    want = a.double() @ b.double()
    bound = (K / 32 + 10) * 2.0 ** -24 * (a.double().abs() @ b.double().abs())
    assert bool(((c.double() - want).abs() <= bound + extra).all())


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("lead", [0, 1])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_products(M, N, K, lead, half):
    a, b = operands(M, N, K, half, M + N + K, lead)
    raw = torch.full((lead + M * N + 8,), -7.0, device="cuda")
    c = call(a, b, out=raw[lead:lead + M * N].view(M, N))
    check(c, a, b, K)
    assert bool((raw[:lead] == -7).all()) and bool((raw[lead + M * N:] == -7).all())


@pytest.mark.parametrize("M,N,K", [(65, 255, 4097), (2000, 2001, 65), (4096, 3072, 64)])
def test_bias_and_relu(M, N, K):
    a, b = operands(M, N, K, False, 5)
    bias = torch.linspace(-4, 4, N, device="cuda")
    c = call(a, b, bias, 1)
    want = torch.relu(a.double() @ b.double() + bias.double())
    bound = (K / 32 + 12) * 2.0 ** -24 * (a.double().abs() @ b.double().abs() + bias.double().abs())
    assert bool(((c.double() - want).abs() <= bound).all())


@pytest.mark.parametrize("M,N,K", [(1025, 1155, 513), (130, 140, 2049)])
def test_alpha_beta_and_batches(M, N, K):
    from aidotnet.tensors_amd import Mi355Backend
    be = Mi355Backend(); W = be.WrapTensor
    a, b = operands(3 * M, N, K, False, 6)
    b = torch.stack([b, b + 1, -b])
    c0 = torch.randn(3, M, N, device="cuda")
    for batch in (1, 3):
        c = c0[:batch].clone()
        (be.Gemm if batch == 1 else lambda *x: be.BatchedGemm(*x[:6], batch, *x[6:]))(W(a), W(b), W(c), M, N, K, 0.5, -2.0)
        torch.cuda.synchronize()
        for i in range(batch):
            ai = a[i * M:(i + 1) * M].double()
            want = 0.5 * ai @ b[i].double() - 2.0 * c0[i].double()
            bound = (K / 32 + 14) * 2.0 ** -24 * (ai.abs() @ b[i].double().abs() + 2.0 * c0[i].double().abs())
            assert bool(((c[i].double() - want).abs() <= bound).all())


# a tile whose operands a split does not hold is computed on the fp32 pipe
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("M,N,K", [(65, 255, 4097), (2000, 2001, 65), (4096, 3072, 64)])
def test_infinities_and_nan(M, N, K, half):
    a, b = operands(M, N, K, half, 7)
    b[K // 2, 1] = 0.0
    a[3, K // 2] = float("inf"); a[M - 1, K - 1] = float("-inf"); a[7, 0] = float("nan"); b[0, N - 1] = float("inf")
    a[9, 5] = 3.4e38
    c = call(a, b)
    want = a.double() @ b.double()
    want[want.abs() > 3.4028236e38] *= float("inf")
    assert torch.equal(torch.isnan(c), torch.isnan(want))
    assert torch.equal(torch.isinf(c) & (c > 0), torch.isinf(want) & (want > 0))
    ok = torch.isfinite(want)
    ok[9] = False                                                  # (one term a million times the rest's bound)
    bound = (K + 10) * 2.0 ** -24 * (a.double().abs() @ b.double().abs())       # the fp32 pipe rounds after every other product
    assert bool(((c.double() - want).abs()[ok] <= bound[ok]).all())


@pytest.mark.parametrize("scale_a,scale_b", [(2.0 ** -120, 2.0 ** 100), (2.0 ** -120, 1.0), (2.0 ** 100, 2.0 ** -118), (2.0 ** 60, 2.0 ** 60), (2.0 ** -60, 2.0 ** -60)])
@pytest.mark.parametrize("M,N,K", [(65, 255, 4097), (4096, 3072, 64)])
def test_extreme_magnitudes(M, N, K, scale_a, scale_b):
    a, b = operands(M, N, K, False, 8)
    a *= scale_a; b *= scale_b
    a[:, 1] = 0.0
    c = call(a, b)
    want = a.double() @ b.double()
    # (results below 2^-126 are whole multiples of 2^-149, and so is every partial sum)
    bound = (K + 10) * (2.0 ** -24 * (a.double().abs() @ b.double().abs()) + 2.0 ** -149)
    assert bool(((c.double() - want).abs() <= bound).all())


# one to three terms: exact products and a rounding per term, |error| <= K 2^-24 sum |a| |b|
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("K", [1, 2, 3])
def test_shortest_sums(K, half):
    a, b = operands(2047, 2049, K, half, 20 + K)
    c = call(a, b).double()
    assert bool(((c - a.double() @ b.double()).abs() <= K * 2.0 ** -24 * (a.double().abs() @ b.double().abs())).all())

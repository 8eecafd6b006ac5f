"""Every instance of the split kernel (fp32 products on the bf16 matrix pipe), named by the kernel that ran: products, infinities and NaN,
values a split cuts, and results that depend on their own row and column alone."""
import pytest
import torch

from _util import kernels_of
from test_gpu_gemm_split import check, operands

pytestmark = pytest.mark.gpu

# (M, N, K, fp16 weights, kernel): tile rows, columns to a thread, parts of a value of B, 0 whole tiles / 1 ragged M or N / 2 a remainder of K
INSTANCES = [(2816, 4416, 96, False, "128, 3, 3, 0"), (1280, 4992, 64, False, "128, 2, 3, 0"), (3583, 1727, 64, False, "128, 2, 3, 1"),
             (3583, 1727, 65, False, "128, 2, 3, 2"), (4096, 1536, 96, False, "64, 2, 3, 0"), (4095, 3072, 64, False, "64, 2, 3, 1"),
             (300, 40001, 33, False, "64, 2, 3, 2"), (1000, 1153, 2049, False, "128, 2, 3, 2"), (65, 255, 4097, False, "64, 2, 3, 2"),
             (1280, 4992, 64, True, "128, 2, 2, 0"), (3583, 1727, 64, True, "128, 2, 2, 1"), (3583, 1727, 65, True, "128, 2, 2, 2"),
             (2048, 2048, 96, True, "64, 2, 2, 0"), (4095, 3072, 64, True, "64, 2, 2, 1"), (1025, 1155, 33, True, "64, 2, 2, 2")]


def run(a, b, kernel):
    from aidotnet.tensors_amd import Mi355Backend
    be = Mi355Backend(); W = be.WrapTensor
    (M, K), N = a.shape, b.shape[1]
    raw = torch.full((M * N + 64,), -7.0, device="cuda")
    f = be.GemmFp16WeightB if b.dtype == torch.float16 else be.GemmBiasActivationInto
    names = kernels_of(lambda: f(W(a), W(b), None, W(raw), M, N, K, 0, 0.0))
    assert names[0] == "gemm_split_kernel<%s>" % kernel, names
    assert bool((raw[M * N:] == -7.0).all())
    return raw[:M * N].view(M, N)


@pytest.mark.parametrize("M,N,K,half,kernel", INSTANCES)
def test_products(M, N, K, half, kernel):
    a, b = operands(M, N, K, half, M + N + K)
    check(run(a, b, kernel), a, b, K)


# infinities, NaN, a value that rounds to an infinity, values that a split cuts, zeros: in four rows and two columns of tiles whose other
# results keep their bits
@pytest.mark.parametrize("M,N,K,half,kernel", INSTANCES)
def test_odd_values_and_their_neighbours(M, N, K, half, kernel):
    a, b = operands(M, N, K, half, 7)
    a[8] = 0.0
    b[:, 5] = 0.0
    plain = run(a, b, kernel).clone()
    a[3, K // 2] = float("inf"); a[M - 1, K - 1] = float("nan"); a[9, 5] = 3.4e38; a[12, :] *= 2.0 ** -118
    b[0, N - 1] = float("inf")
    c = run(a, b, kernel)
    want = a.double() @ b.double()
    want[want.abs() > 3.4028236e38] *= float("inf")
    assert torch.equal(torch.isnan(c), torch.isnan(want))
    assert torch.equal(c == float("inf"), want == float("inf")) and torch.equal(c == -float("inf"), want == -float("inf"))
    ok = torch.isfinite(want)
    bound = (K + 10) * (2.0 ** -24 * (a.double().abs() @ b.double().abs()) + 2.0 ** -149)      # the fp32 pipe rounds after every other product
    assert bool(((c.double() - want).abs()[ok] <= bound[ok]).all())
    rows = torch.ones(M, dtype=torch.bool, device="cuda")
    rows[[3, M - 1, 9, 12]] = False
    assert torch.equal(c[rows][:, :N - 1], plain[rows][:, :N - 1])


# around 2^-110, where the third part of a value ends among the bf16 subnormals, and below, beside ordinary and beside large values
SCALES = [(-105, 0), (-109, 29), (-112, 0), (-112, 100), (-120, 60), (-100, -20), (29, -109), (0, -125)]
SMALLEST = [i + s for i in INSTANCES if i[:3] in ((2816, 4416, 96), (3583, 1727, 65), (65, 255, 4097)) for s in SCALES if not i[3] or abs(s[1]) <= 10]


@pytest.mark.parametrize("M,N,K,half,kernel,scale_a,scale_b", SMALLEST)
def test_smallest_values(M, N, K, half, kernel, scale_a, scale_b):
    a, b = operands(M, N, K, half, 8)
    a *= 2.0 ** scale_a; b *= 2.0 ** scale_b
    a[:, 1] = 0.0
    a[5] = 0.0
    c = run(a, b, kernel)
    want = a.double() @ b.double()
    # (results below 2^-126 are whole multiples of 2^-149, and so is every partial sum)
    bound = (K + 10) * (2.0 ** -24 * (a.double().abs() @ b.double().abs()) + 2.0 ** -149)
    assert bool(((c.double() - want).abs() <= bound).all())


# probabilities of a wide softmax: most of a row below 2^-110, in ranges of K without its largest ones too
@pytest.mark.parametrize("M,N,K,kernel", [(2816, 4416, 96, "128, 3, 3, 0"), (1000, 1153, 2049, "128, 2, 3, 2"), (65, 255, 4097, "64, 2, 3, 2")])
def test_probabilities(M, N, K, kernel):
    a, b = operands(M, N, K, False, 9)
    a = torch.softmax(a * 60, -1).contiguous()
    b[:, 3] = 0.0
    b[:, 4] *= 2.0 ** -70
    c = run(a, b, kernel)
    check(c, a, b, K)
    assert bool((c[:, 3] == 0).all())


# what a product takes does not hang on the values in it: before, one NaN cost fifteen times the product and a zero row a fifth of it.
# (Generous: the medians of five; a NaN is 1.4 times the product here.)
def test_time_does_not_hang_on_values():
    from aidotnet.tensors_amd import Mi355Backend
    be = Mi355Backend(synchronous=False); W = be.WrapTensor
    M, N, K = 2048, 2048, 4096
    a, b = operands(M, N, K, False, 10)
    c = torch.empty(M, N, device="cuda")

    def time(x):
        times = []
        for _ in range(6):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            for _ in range(4):
                be.GemmBiasActivationInto(W(x), W(b), None, W(c), M, N, K, 0, 0.0)
            e1.record()
            torch.cuda.synchronize()
            times.append(e0.elapsed_time(e1))
        return sorted(times[1:])[2]
    base = time(a)
    one = a.clone(); one[M // 2, K // 2] = float("nan")
    assert time(one) < 3.0 * base

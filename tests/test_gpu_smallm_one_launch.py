"""Products of at most eight fp32 rows in one launch (K up to 1024, weights up to four million elements): each row count's instance, sizes
on and around the 64 columns of a workgroup and the 64 / 384 k-rows of a round, columns past a multiple of four, fp16 weights, alpha and
beta, bias and activation, a C with elements behind it, and the line to the two-launch form on either side.

Bound: fp32 sums of K products of N(0,1) times N(0,1/K) values, K 2^-24 < 7e-5 in the worst case, held at 2e-6 of the result's norm
(sums of random signs: sqrt(K) 2^-24)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(1, 64, 64), (2, 63, 65), (3, 65, 63), (4, 130, 384), (5, 129, 385), (8, 768, 768), (7, 501, 499), (1, 4096, 1024), (8, 4097, 1023),
          (8, 100, 1025), (2, 5000, 1), (6, 4099, 2)]


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_few_rows(M, N, K, half):
    from aidotnet.tensors_amd import Mi355Backend
    be = Mi355Backend(); W = be.WrapTensor
    gen = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=gen)
    w = torch.randn(K, N, generator=gen) / K ** 0.5
    if half:
        w = w.half()
    bias = torch.randn(N, generator=gen)
    out = torch.full((M * N + 5,), -7.0, device="cuda")
    for act, fn in ((0, lambda z: z), (1, lambda z: z.clamp(min=0)), (6, lambda z: z * torch.sigmoid(z))):
        call = be.GemmFp16WeightB if half else be.GemmBiasActivationInto
        call(W(x.cuda()), W(w.cuda()), W(bias.cuda()), W(out), M, N, K, act, 0.01)
        want = fn(x.double() @ w.double() + bias.double())
        got = out[:M * N].cpu().double().view(M, N)
        assert float((got - want).norm() / want.norm()) <= 2e-6
        assert bool((out[M * N:] == -7.0).all())
    if not half:
        c0 = torch.randn(M, N, generator=gen)
        c = c0.cuda()
        be.Gemm(W(x.cuda()), W(w.cuda()), W(c), M, N, K, 0.5, -2.0)
        want = 0.5 * (x.double() @ w.double()) - 2.0 * c0.double()
        assert float((c.cpu().double() - want).norm() / want.norm()) <= 2e-6
        # off the 16-byte grid: the same loads at element alignment, the same bits
        raw = torch.empty(K * N + 1, device="cuda"); raw[1:] = w.reshape(-1).cuda()
        c1, c2 = torch.empty(M, N, device="cuda"), torch.empty(M, N, device="cuda")
        be.Gemm(W(x.cuda()), W(w.cuda()), W(c1), M, N, K)
        be.Gemm(W(x.cuda()), W(raw[1:].view(K, N)), W(c2), M, N, K)
        assert torch.equal(c1, c2)

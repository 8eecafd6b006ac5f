"""C = alpha A B + beta C on the general kernel at sizes that are no multiple of its tiles: the old values of C are read at clamped
addresses, so the last row and column must still get their own, and nothing behind C is touched.

Bound: fp32 sums of K products, 2e-6 of the result's norm (random signs, sqrt(K) 2^-24 with K up to 333)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(33, 70, 50), (65, 63, 33), (129, 131, 77), (100, 65, 333), (9, 1, 7), (500, 333, 77)])
@pytest.mark.parametrize("tile", [0, 64, 128])
def test_beta(M, N, K, tile):
    from aidotnet.tensors_amd import Mi355Backend
    be = Mi355Backend(); W = be.WrapTensor
    be.SetGemmTile(tile)
    gen = torch.Generator(device="cuda").manual_seed(M * N)
    x, w, c0 = (torch.randn(*s, device="cuda", generator=gen) for s in ((M, K), (K, N), (M, N)))
    raw = torch.full((M * N + 7,), float("nan"), device="cuda")
    raw[:M * N] = c0.reshape(-1)
    be.Gemm(W(x), W(w), W(raw[:M * N]), M, N, K, 0.5, -2.0)
    want = 0.5 * (x.double() @ w.double()) - 2.0 * c0.double()
    assert float((raw[:M * N].view(M, N).double() - want).norm() / want.norm()) <= 2e-6
    assert bool(torch.isnan(raw[M * N:]).all())

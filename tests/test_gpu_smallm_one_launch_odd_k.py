"""One and two fp32 rows in one launch at inner dimensions whose rows of A do not end on 16 bytes: the waves' sums, stored 16 bytes at a
time, must start on the grid at any K (with A in front of them they started K or 2 K floats in).

Bound: as for the other row counts, 2e-6 of the result's norm (sums of random signs, sqrt(K) 2^-24)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("M,N,K", [(1, 4096, 1), (1, 5001, 2), (1, 300, 255), (1, 77, 385), (1, 2050, 1023), (2, 4100, 1), (2, 129, 1023)])
def test_rows_of_any_length(M, N, K, half):
    from aidotnet.tensors_amd import Mi355Backend
    be = Mi355Backend(); W = be.WrapTensor
    gen = torch.Generator().manual_seed(M + N + K)
    x, w, bias = torch.randn(M, K, generator=gen), torch.randn(K, N, generator=gen) / K ** 0.5, torch.randn(N, generator=gen)
    w = w.half() if half else w
    out = torch.empty(M, N, device="cuda")
    (be.GemmFp16WeightB if half else be.GemmBiasActivationInto)(W(x.cuda()), W(w.cuda()), W(bias.cuda()), W(out), M, N, K, 0, 0.0)
    want = x.double() @ w.double() + bias.double()
    assert float((out.cpu().double() - want).norm() / want.norm()) <= 2e-6

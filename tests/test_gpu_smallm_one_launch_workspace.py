"""Few fp32 rows on a weight of a few megabytes: the one-launch form holds no workspace, so it is also what a stream under capture runs
without a reservation."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("M,N,K", [(1, 4096, 1024), (8, 768, 768), (5, 501, 499), (8, 16384, 64)])
def test_no_workspace(M, N, K, half):
    from aidotnet.tensors_amd import Mi355Backend
    be = Mi355Backend(synchronous=False); W = be.WrapTensor
    gen = torch.Generator(device="cuda").manual_seed(N)
    x, w = torch.randn(M, K, device="cuda", generator=gen), torch.randn(K, N, device="cuda", generator=gen)
    w = w.half() if half else w
    y, z = torch.empty(M, N, device="cuda"), torch.empty(M, N, device="cuda")
    call = lambda out: (be.GemmFp16WeightB if half else be.GemmBiasActivationInto)(W(x), W(w), None, W(out), M, N, K, 0, 0.0)
    call(y)
    assert be.WorkspaceBytes() == 0
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call(z)
    for _ in range(3):
        z.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, z)                    # the same kernel: the same bits


@pytest.mark.parametrize("M,N,K,one", [(8, 16384, 1, True), (8, 16385, 1, False), (1, 16385, 127, False), (1, 16385, 128, True), (2, 32768, 128, True), (4, 262144, 16, False),
                                       (8, 1 << 22, 1, False)])
def test_wide_weights_of_few_rows(M, N, K, one):
    """More than 16384 columns (a workgroup of 64 on every CU) of fewer than 128 rows take the two-launch form, which holds its partials
    in the workspace.  Bound: 2e-6 of the result's norm, as for the other sizes."""
    from aidotnet.tensors_amd import Mi355Backend
    be = Mi355Backend(); W = be.WrapTensor
    gen = torch.Generator(device="cuda").manual_seed(K)
    x, w, y = torch.randn(M, K, device="cuda", generator=gen), torch.randn(K, N, device="cuda", generator=gen), torch.empty(M, N, device="cuda")
    be.Gemm(W(x), W(w), W(y), M, N, K)
    assert (be.WorkspaceBytes() == 0) == one
    want = x.double() @ w.double()
    assert float((y.double() - want).norm() / want.norm()) <= 2e-6

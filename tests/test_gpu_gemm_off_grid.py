"""16-bit products whose dimensions are multiples of 8 and whose operands lie off the 16-byte grid: the last K-tile from clamped addresses
(K around multiples of 64, columns and rows that do not fill their tiles), K ranges (few tiles over a long K), the fused epilogue, and
nothing read past either operand.  Against float64; fp32 sums of K products of N(0,1) values, at most 2 K 2^-24 of sum |a||b| (~0.64 K)."""
import pytest
import torch

from _util import TORCH16

pytestmark = pytest.mark.gpu

SHAPES = [(1, 16, 8), (3, 24, 56), (17, 136, 64), (20, 272, 248), (64, 128, 128), (65, 1000, 72), (100, 264, 504), (130, 2064, 1384), (300, 4096, 320), (3000, 2040, 264),
          (1, 664, 4216), (7, 144, 5072), (3, 3080, 960), (33, 128, 8192)]


@pytest.mark.parametrize("kind", ["f16", "bf16"])
@pytest.mark.parametrize("which", ["a", "b", "ab"])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_values(M, N, K, which, kind):
    from aidotnet.tensors_amd import Mi355Engine
    eng = Mi355Engine()
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    dt = TORCH16[kind]
    def operand(rows, cols, off):
        # the neighbours of an operand are NaN: a value read from them and used would show
        buf = torch.full((rows * cols + 64,), float("nan"), device="cuda", dtype=dt)
        at = 33 if off else 32
        view = buf[at:at + rows * cols].view(rows, cols)
        view.copy_(torch.randn(rows, cols, device="cuda", generator=gen))
        assert (view.data_ptr() % 16 != 0) == off
        return view
    a, b = operand(M, K, "a" in which), operand(K, N, "b" in which)
    got = eng.TensorMatMul(a, b, out_dtype=torch.float32).double()
    want = torch.matmul(a.double(), b.double())
    scale = torch.matmul(a.double().abs(), b.double().abs())
    assert bool(((got - want).abs() <= 2 * K * 2.0 ** -24 * scale + 1e-30).all())
    bias = torch.randn(N, device="cuda", generator=gen)
    act = eng.FusedLinear(a, b, bias, "ReLU", out_dtype=torch.float32).double()
    assert bool(((act - (want + bias.double()).clamp_min(0)).abs() <= 2 * K * 2.0 ** -24 * (scale + bias.double().abs()) + 1e-30).all())


def test_ranges_ask_for_their_workspace():
    """A product of few tiles over a long K has a workspace for its ranges whichever way its operands lie."""
    from aidotnet.tensors_amd import Mi355Backend, Mi355Engine
    eng = Mi355Engine(Mi355Backend())
    a = torch.randn(664 * 4216 + 8, device="cuda").to(torch.bfloat16)
    eng.TensorMatMul(a[1:4217].view(1, 4216), a[:4216 * 664].view(4216, 664))
    assert eng.backend.WorkspaceBytes() >= 2 * 664 * 4

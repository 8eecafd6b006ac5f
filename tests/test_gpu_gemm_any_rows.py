"""16-bit products whose rows start anywhere (N or K not a multiple of 8, operands off the 16-byte grid), read in place: 64- and 128-row
tiles and K ranges, sizes on and around the tile edges (64 / 128 rows, 128 columns, 64 of K), the last K-tile whole, one element long and
one short, infinities next to the padding, and outputs that start on an odd element.

Dyadic inputs make every product and partial sum exact in fp32, so results must equal the float64 product rounded once; bias and activation
are held to fp32 arithmetic plus that rounding (2^-8 of bf16, relative)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(1, 17, 1), (3, 129, 7), (64, 127, 63), (65, 257, 64), (63, 135, 65), (128, 128, 129), (129, 1001, 191), (64, 50257, 72),
          (300, 20001, 70), (257, 16385, 193), (1, 148, 481), (30, 301, 4097), (70, 1003, 2049), (200, 264, 1021), (5, 16, 300)]


def operands(M, N, K, dt, seed, la=0, lb=0):
    gen = torch.Generator().manual_seed(seed)
    a = torch.randint(-8, 9, (M, K), generator=gen).double() / 8
    b = torch.randint(-8, 9, (K, N), generator=gen).double() / 8
    def place(t, lead):
        raw = torch.full((lead + t.numel(),), float("nan"), dtype=dt, device="cuda")
        raw[lead:] = t.reshape(-1).to(dt).cuda()
        return raw[lead:].view(t.shape)
    return a, b, place(a, la), place(b, lb)


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("la,lb", [(0, 0), (1, 3)])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_exact_products(M, N, K, la, lb, dt):
    from aidotnet.tensors_amd import Mi355Backend
    be = Mi355Backend(); W = be.WrapTensor
    a, b, da, db = operands(M, N, K, dt, M + N + K, la, lb)
    want = a @ b
    for lead in (0, 1):
        c = torch.full((lead + M * N + 8,), -7.0, device="cuda", dtype=dt)
        (be.Hgemm if dt == torch.float16 else be.Bf16Gemm)(W(da), W(db), W(c[lead:]), M, N, K)
        torch.cuda.synchronize()
        assert torch.equal(c[lead:lead + M * N].cpu().view(M, N), want.float().to(dt))
        assert bool((c[:lead] == -7.0).all()) and bool((c[lead + M * N:] == -7.0).all())
    c32 = torch.full((M * N + 8,), -7.0, device="cuda")
    (be.GemmFp16In32fOut if dt == torch.float16 else be.GemmBf16In32fOut)(W(da), W(db), W(c32), M, N, K)
    torch.cuda.synchronize()
    assert torch.equal(c32[:M * N].cpu().view(M, N), want.float()) and bool((c32[M * N:] == -7.0).all())


@pytest.mark.parametrize("act", ["None", "ReLU", "Swish"])
@pytest.mark.parametrize("M,N,K", [(65, 131, 63), (1, 148, 481), (40, 301, 2049), (200, 30001, 66)])
def test_bias_and_activation(M, N, K, act):
    from aidotnet.tensors_amd import Mi355Engine
    eng = Mi355Engine()
    a, b, da, db = operands(M, N, K, torch.bfloat16, M * N)
    bias = torch.randn(N, generator=torch.Generator().manual_seed(N))
    y = eng.FusedLinear(da, db / 4, bias.cuda(), act).double().cpu()
    z = a @ b / 4 + bias.double()
    want = {"None": z, "ReLU": z.clamp(min=0), "Swish": z * torch.sigmoid(z)}[act]
    assert float(((y - want).abs() / (1e-6 + want.abs())).max()) <= 2.0 ** -8 + 1e-4 or torch.allclose(y, want, rtol=2.0 ** -8, atol=1e-5)


def test_infinities_stay_in_their_rows_and_columns():
    """The elements a tile loads beyond its operands (the next row, the next columns) must not leak into the result."""
    from aidotnet.tensors_amd import Mi355Engine
    eng = Mi355Engine()
    for M, N, K in ((66, 131, 67), (3, 141, 483)):
        a, b, da, db = operands(M, N, K, torch.bfloat16, K)
        da[1, 0] = float("inf"); db[K - 1, 0] = float("inf"); db[2, N - 1] = float("nan")
        y = eng.TensorMatMul(da, db, out_dtype=torch.float32).cpu()
        bad = ~torch.isfinite(y)
        a2, b2 = da.double().cpu(), db.double().cpu()
        assert torch.equal(bad, ~torch.isfinite(a2 @ b2))
        assert torch.equal(y[~bad].double(), (a2 @ b2)[~bad])

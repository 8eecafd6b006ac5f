"""Values of the fused activations over the whole range of their argument, through every kernel that applies them.  A is a shifted
identity, so the product is exactly the chosen values and only the epilogue is looked at.

Bound: relative error <= 4e-7 for the functions built on the logistic function where the result is above 1e-30 (the hardware exponential
and its argument's rounding, the sum with 1 and the quotient: at most 2.75 units of 2^-23, 3.3e-7, see the last test); GELU's inner
cubic adds 2 |2u| 2^-24 relative, below 3e-6 for |u| <= 22, beyond which the result is x or below 1e-19."""
import math

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

VALUES = np.array([0.0, -0.0, 1e-30, -1e-30, 1e-4, -1e-4, 0.3, -0.3, 1.0, -1.0, 2.5, -2.5, 6.0, -6.0, 10.0, -10.0, 25.0, -25.0, 60.0, -60.0,
                   86.9, -86.9, 88.0, -88.0, 120.0, -120.0, 1e4, -1e4, 1e20, -1e20], np.float32)


def reference(x, act):
    x = x.astype(np.float64)
    with np.errstate(over="ignore"):
        if act == 1: return np.maximum(x, 0)
        if act == 2: return x / (1 + np.exp(-2 * 0.7978845608 * (x + 0.044715 * x ** 3)))
        if act == 3: return 1 / (1 + np.exp(-x))
        if act == 4: return np.tanh(x)
        if act == 5: return np.where(x > 0, x, 0.125 * x)
        if act == 6: return x / (1 + np.exp(-x))
    return x


# (M, N, K): few rows, the 64 / 128 / 256-wide direct-to-LDS tiles with and without edges, the general kernel (rows off the 16-byte grid)
@pytest.mark.parametrize("M,N,K", [(4, 256, 64), (64, 64, 64), (130, 132, 32), (512, 4096, 32), (70, 33, 31), (24, 128, 64)])
@pytest.mark.parametrize("act", range(7))
def test_activation_values_fp32(M, N, K, act):
    from aidotnet.tensors_amd import Mi355Engine
    eng = Mi355Engine()
    x = VALUES[(np.arange(K)[:, None] * 7 + np.arange(N)[None, :]) % len(VALUES)]
    a = np.zeros((M, K), np.float32); a[np.arange(M), np.arange(M) % K] = 1.0
    got = eng.FusedLinear(torch.from_numpy(a).cuda(), torch.from_numpy(x).cuda(), None, act, 0.125).cpu().numpy().astype(np.float64)
    arg = x[np.arange(M) % K]
    want = reference(arg, act)
    assert np.array_equal(np.isfinite(got), np.isfinite(want))
    big = np.abs(want) > 1e-30
    rel = np.abs(got - want)[big] / np.abs(want)[big]
    u = np.abs(2 * 0.7978845608 * (arg.astype(np.float64) + 0.044715 * arg.astype(np.float64) ** 3))[big]
    assert np.all(rel <= 4e-7 + (np.minimum(u, 100) * 2.0 ** -23 if act == 2 else 0.0))
    assert np.all(np.abs(got[~big]) <= 2e-30)


@pytest.mark.parametrize("M,N,K", [(64, 256, 64), (512, 1024, 64), (100, 200, 64)])
@pytest.mark.parametrize("act", range(7))
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_activation_values_16bit(M, N, K, act, dtype):
    """The 16-bit result is the fp32 epilogue rounded once: half a unit of the type (2^-11 fp16, 2^-8 bf16 ... relative) and, in fp16,
    of the smallest subnormal."""
    from aidotnet.tensors_amd import Mi355Engine
    eng = Mi355Engine()
    vals = VALUES[np.abs(VALUES) <= 1e4]
    x = torch.from_numpy(vals[(np.arange(K)[:, None] * 7 + np.arange(N)[None, :]) % len(vals)]).cuda().to(dtype)
    a = torch.zeros(M, K, dtype=dtype, device="cuda"); a[torch.arange(M), torch.arange(M) % K] = 1.0
    got = eng.FusedLinear(a, x, None, act, 0.125).double().cpu().numpy()
    want = reference(x.float().cpu().numpy()[np.arange(M) % K], act)
    unit = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    assert np.all(np.abs(got - want) <= 1.01 * unit * np.abs(want) + 2.0 ** -25)


def test_nan_stays_nan():
    from aidotnet.tensors_amd import Mi355Engine
    eng = Mi355Engine()
    w = torch.full((64, 64), float("nan"), device="cuda")
    for act in range(7):
        assert bool(torch.isnan(eng.FusedLinear(torch.ones(64, 64, device="cuda"), w, None, act, 0.1)).all()), act


def test_errors_of_the_logistic_functions():
    """Over the whole range of their argument.  In units of 2^-23: the hardware exponential 1, its argument's rounding ln 2 / 4, the sum with
    1 compensated up to 2^24 and at most 1 where it begins to be (e^-x itself beyond), the quotient 1/2: 2.75.  Subnormal results (sigmoid
    below -87.3) within the smallest subnormal beside that.  GELU where the rounding of its argument 2 u (three halves, times 2 u and the
    logistic function of -2 u) does not lead."""
    from aidotnet.tensors_amd import Mi355Engine
    eng = Mi355Engine()
    gen = torch.Generator(device="cuda").manual_seed(3)
    one = torch.ones(1, 1, device="cuda")
    for act in (3, 6, 2):
        for lo, hi in ((-88.7, -87.3), (-87.3, -20.0), (-20.0, -2.0), (-2.0, 0.1), (-0.1, 2.0), (2.0, 20.0), (20.0, 120.0)):
            if act == 2 and lo < -2.0:
                continue
            x = lo + (hi - lo) * torch.rand(1, 1 << 16, device="cuda", generator=gen)
            got = eng.FusedLinear(one, x, None, act).double()
            z = x.double()
            u2 = 2 * 0.7978845608 * (z + 0.044715 * z ** 3) if act == 2 else z
            want = (1.0 if act == 3 else z) / (1 + torch.exp(-u2))
            bound = 2.75 * 2.0 ** -23 + (1.5 * 2.0 ** -23 * u2.abs() * torch.sigmoid(-u2) if act == 2 else 0.0)
            assert bool(((got - want).abs() <= bound * want.abs() + 2.0 ** -149).all()), (act, lo)

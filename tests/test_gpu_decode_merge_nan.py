"""A row of which a value or logit is not a number: the merge of key ranges answers as a single range does (zeros where the row sum is no
number, NaN nowhere else)."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["f32", "bf16"])
@pytest.mark.parametrize("D,splits", [(128, 2), (128, 16), (256, 4)])
def test_nan_key(D, splits, kind):
    from aidotnet.tensors_amd import Mi355Backend
    be = Mi355Backend()
    dtype = torch.float32 if kind == "f32" else torch.bfloat16
    gen = torch.Generator(device="cuda").manual_seed(D + splits)
    B, H, S = 2, 4, 4096
    q, k, v = (torch.randn(B, H, s, D, device="cuda", generator=gen).to(dtype) for s in (1, S, S))
    k[0, 1, 700] = float("nan")
    def run(n):
        o = torch.full((B, H, 1, D), 7.0, device="cuda")
        be.DecodeAttention(kind, *(be.WrapTensor(t) for t in (q, k, v, o)), B, H, S, D, 1 / math.sqrt(D), splits=n)
        return o
    one, many = run(1), run(splits)
    assert torch.equal(torch.isnan(one), torch.isnan(many)) and torch.equal(one[0, 1] == 0, many[0, 1] == 0)
    assert torch.allclose(one.nan_to_num(0.0), many.nan_to_num(0.0), rtol=1e-4, atol=1e-5)

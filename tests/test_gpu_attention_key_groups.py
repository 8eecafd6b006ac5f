"""One, two and four waves per query row's keys (launch_attn picks by the size of the grid): query counts on and around the 32-, 64- and
128-row workgroups, key counts around the 32-key share of a wave and the 64- / 128-key tiles, key groups that see no key at all (short
sequences, causal rows), and infinite inputs on either side of the merge.  Against a float64 softmax.

Bounds: fp32 logits and one exponential of a difference below 20, (D + 20) 2^-24 < 2e-5, held at 1e-4; 16-bit operands round P once,
2^-9 relative (bf16) of values that are averages of N(0,1) rows, held at 2e-2."""
import numpy as np
import pytest
import torch

from _util import mixed_err

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    from aidotnet.tensors_amd import Mi355Engine
    return Mi355Engine()


def reference(q, k, v, scale, causal):
    g = q.shape[1] // k.shape[1]
    s = (q @ np.repeat(k, g, 1).transpose(0, 1, 3, 2)) * scale
    Sq, Sk = s.shape[-2:]
    if causal:                                              # top-left: query i sees keys 0 .. i
        s[..., np.arange(Sk)[None, :] > np.arange(Sq)[:, None]] = -np.inf
    m = s.max(-1, keepdims=True)
    p = np.exp(s - m)
    l = p.sum(-1, keepdims=True)
    return (p / l) @ np.repeat(v, g, 1), (m + np.log(l))[..., 0]


# B, H, Hkv, Sq, Sk, D: two groups (short keys, or another head dimension), four (head dimension 64 from 192 keys on), one (large grids)
SHAPES = [(1, 2, 2, 1, 1, 64), (1, 2, 1, 31, 33, 64), (2, 2, 2, 65, 63, 64), (1, 3, 3, 64, 191, 64),
          (1, 2, 2, 32, 192, 64), (1, 2, 1, 33, 257, 64), (2, 2, 2, 129, 224, 64), (1, 1, 1, 300, 385, 64), (2, 4, 4, 260, 260, 64),
          (1, 2, 2, 65, 97, 128), (2, 2, 1, 130, 161, 128), (1, 2, 2, 40, 31, 128), (1, 2, 2, 100, 90, 80), (1, 2, 2, 70, 129, 32), (1, 1, 1, 33, 65, 20),
          (8, 64, 64, 65, 66, 64), (4, 64, 64, 129, 70, 64), (4, 64, 64, 65, 40, 128), (4, 64, 32, 65, 40, 80)]


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("kind", ["f32", "bf16"])
@pytest.mark.parametrize("B,H,Hkv,Sq,Sk,D", SHAPES)
def test_key_groups(eng, B, H, Hkv, Sq, Sk, D, kind, causal):
    gen = torch.Generator().manual_seed(Sq * 1000 + Sk + D)
    dt = torch.float32 if kind == "f32" else torch.bfloat16
    q, k, v = (torch.randn(B, h, s, D, generator=gen).to(dt) for h, s in ((H, Sq), (Hkv, Sk), (Hkv, Sk)))
    o, lse = eng.FlashAttention(q.cuda(), k.cuda(), v.cuda(), None, causal)
    want, want_lse = reference(*(t.double().numpy() for t in (q, k, v)), 1.0 / np.sqrt(D), causal)
    assert mixed_err(o.cpu().numpy(), want) <= (1e-4 if kind == "f32" else 2e-2)
    # (16-bit: at head dimension 128 the row sum is taken over the probabilities as rounded for the product, 2^-9 relative each)
    assert mixed_err(lse.cpu().numpy(), want_lse) <= (1e-4 if kind == "f32" else 2e-3)


@pytest.mark.parametrize("Sk", [64, 256])
def test_infinite_values_and_logits(eng, Sk):
    """An infinite value spoils its head-dim column alone; a logit of +inf makes its row NaN, one of -inf a weight of zero -- in whichever
    key group it lies."""
    gen = torch.Generator().manual_seed(Sk)
    q, k, v = (torch.randn(1, 2, 40, 64, generator=gen), torch.randn(1, 2, Sk, 64, generator=gen), torch.randn(1, 2, Sk, 64, generator=gen))
    for key in (3, 40, Sk - 20):
        vi = v.clone(); vi[0, 0, key, 5] = float("inf")
        o, _ = eng.FlashAttention(q.cuda(), k.cuda(), vi.cuda())
        assert torch.isinf(o[0, 0, :, 5]).all() and torch.isfinite(o[0, 0, :, :5]).all() and torch.isfinite(o[0, 1]).all()
        qp = q.clone(); qp[..., 0] = q[..., 0].abs() + 0.1
        ki = k.clone(); ki[0, 0, key, 0] = float("-inf")
        o, _ = eng.FlashAttention(qp.cuda(), ki.cuda(), v.cuda())
        want, _ = reference(qp.double().numpy(), ki.double().numpy(), v.double().numpy(), 0.125, False)
        assert mixed_err(o.cpu().numpy(), want) <= 1e-4
        ki[0, 0, key, 0] = float("inf")
        o, _ = eng.FlashAttention(qp.cuda(), ki.cuda(), v.cuda())
        assert torch.isnan(o[0, 0]).all() and torch.isfinite(o[0, 1]).all()

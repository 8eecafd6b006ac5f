"""Keep-masks of the keys alone ([B or 1, 1, 1, Sk]: padding), which the kernels follow as one row of bytes per batch: every kernel form
that takes one (direct-to-LDS at head dimensions 64 and 128, the general form, the probabilities), sequence lengths on and around the
64- and 32-key tiles, tiles that are whole, mixed, empty at the end and empty at the start, a batch without a visible key, and masks that
come as strided views or as numbers.  Against a float64 softmax.

Bounds: fp32 as for the probabilities (1e-4, derived there); 16-bit operands round P and O once each, 2^-9 relative (bf16) of values that
are averages of N(0,1) rows, held at 2e-2 absolute-or-relative."""
import numpy as np
import pytest
import torch

from _util import dev, mixed_err

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    from aidotnet.tensors_amd import Mi355Engine
    return Mi355Engine()


def keep_rows(rng, B, Sk, how):
    if how == "padded":                                     # right padding, one sequence of full length
        lengths = rng.integers(1, Sk + 1, B); lengths[0] = Sk
        return np.arange(Sk)[None, :] < lengths[:, None]
    if how == "left":                                       # left padding: the first tiles are empty
        return np.arange(Sk)[None, :] >= rng.integers(0, Sk, B)[:, None]
    keep = rng.random((B, Sk)) < 0.5                        # "holes", and a batch that sees nothing
    keep[B - 1] = False
    return keep


def reference(q, k, v, keep, scale, causal=False, softcap=0.0):
    g = q.shape[1] // k.shape[1]
    k, v = np.repeat(k, g, 1).astype(np.float64), np.repeat(v, g, 1).astype(np.float64)
    s = (q.astype(np.float64) @ k.transpose(0, 1, 3, 2)) * scale
    if softcap > 0:
        s = softcap * np.tanh(s / softcap)
    Sq, Sk = s.shape[-2:]
    hidden = np.broadcast_to(~keep[:, None, None, :], s.shape).copy()
    if causal:
        hidden |= np.arange(Sk)[None, :] > np.arange(Sq)[:, None] + Sk - Sq
    s[hidden] = -np.inf
    m = s.max(-1, keepdims=True); m[~np.isfinite(m)] = 0.0
    p = np.exp(s - m)
    l = p.sum(-1, keepdims=True)
    p = p / np.where(l > 0, l, 1.0)
    return p @ v, p


@pytest.mark.parametrize("how", ["padded", "left", "holes"])
@pytest.mark.parametrize("B,H,Hkv,Sq,Sk,D,causal,softcap", [
    (2, 2, 2, 64, 64, 64, False, 0.0), (3, 2, 1, 130, 193, 64, False, 0.0), (2, 2, 2, 300, 300, 64, True, 0.0), (2, 1, 1, 1, 63, 64, False, 0.0),
    (2, 2, 2, 96, 96, 128, False, 0.0), (2, 4, 2, 129, 161, 128, True, 0.0),
    (2, 2, 2, 70, 150, 32, False, 0.0), (2, 2, 2, 65, 65, 80, True, 0.0), (2, 2, 2, 100, 140, 64, False, 20.0)])
def test_sdpa_key_mask(eng, B, H, Hkv, Sq, Sk, D, causal, softcap, how):
    rng = np.random.default_rng(Sq * 1000 + Sk + D)
    q = rng.standard_normal((B, H, Sq, D)).astype(np.float32)
    k, v = (rng.standard_normal((B, Hkv, Sk, D)).astype(np.float32) for _ in range(2))
    keep = keep_rows(rng, B, Sk, how)
    want, pw = reference(q, k, v, keep, 1 / np.sqrt(D), causal, softcap)
    o, w = eng.ScaledDotProductAttention(dev(q), dev(k), dev(v), torch.from_numpy(keep).cuda()[:, None, None, :], softcap=softcap, isCausal=causal)
    assert mixed_err(w.cpu().numpy(), pw) <= 1e-4 and mixed_err(o.cpu().numpy(), want) <= 1e-4


@pytest.mark.parametrize("how", ["padded", "left", "holes"])
@pytest.mark.parametrize("kind", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("B,S,H,D", [(2, 64, 2, 64), (3, 200, 2, 64), (3, 129, 2, 128), (2, 512, 1, 128), (2, 70, 4, 32), (2, 1, 2, 64)])
def test_mha_key_mask_equals_the_materialised_mask(eng, B, S, H, D, kind, how):
    """The layer with the mask as [B,1,1,S] against the same layer with it written out per query."""
    dtype = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}[kind]
    gen = torch.Generator().manual_seed(S * 10 + D)
    dM = H * D
    x = torch.randn(B, S, dM, generator=gen).to(dtype).cuda()
    ws = [(torch.randn(dM, dM, generator=gen) / dM ** 0.5).to(dtype).cuda() for _ in range(4)]
    keep = torch.from_numpy(keep_rows(np.random.default_rng(S), B, S, how)).cuda()[:, None, None, :]
    got = eng.MultiHeadAttentionForward(x, *ws, H, keep)
    want = eng.MultiHeadAttentionForward(x, *ws, H, keep.expand(B, H, S, S).contiguous() if S > 1 else keep.expand(B, H, 1, 1).contiguous())
    assert mixed_err(got.float().cpu().numpy(), want.float().cpu().numpy()) <= (1e-4 if kind == "f32" else 2e-2)


def test_key_mask_forms(eng):
    """One row for all batches, a strided view, numbers instead of booleans: the same result; a short buffer is refused."""
    from aidotnet.tensors_amd.backend import ArgumentException
    rng = np.random.default_rng(5)
    B, H, S, D = 2, 2, 100, 64
    q, k, v = (dev(rng.standard_normal((B, H, S, D)).astype(np.float32)) for _ in range(3))
    row = torch.from_numpy(rng.random(S) < 0.6).cuda()
    run = lambda m: eng.ScaledDotProductAttention(q, k, v, m, returnWeights=False)[0]
    base = run(row.expand(B, H, S, S))
    wide = torch.zeros(2 * S, dtype=torch.bool, device="cuda"); wide[::2] = row
    for m in (row[None, None, None, :], row.expand(B, 1, 1, S), wide[::2][None, None, None, :], row.float()[None, None, None, :] * 3, row.int()[None, None, None, :]):
        assert mixed_err(run(m).cpu().numpy(), base.cpu().numpy()) <= 1e-5
    with pytest.raises(ArgumentException):
        be, W = eng.backend, eng.backend.WrapTensor
        be.ScaledDotProductAttention(W(q), W(k), W(v), W(torch.empty_like(q)), None, W(row), B, H, S, S, D, 0.125, False, keyMask=True)

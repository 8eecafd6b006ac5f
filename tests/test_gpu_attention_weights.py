"""The probabilities that ScaledDotProductAttention returns beside its output: tiles of 64 queries x 128 keys, so the sizes here lie
on and around those edges, with head dimensions of one, several and partial fragment steps (fp32: 8 elements; parts of 32), aligned
and unaligned rows, and each option of the operator.  Against a float64 softmax; rows must sum to one where a key is visible.

Bound: both sides form fp32 logits from up to D products of N(0,1) values and one exponential of a difference below 20 in magnitude,
(D + 20) 2^-24 < 2e-5 relative for D <= 256; held at 1e-4."""
import numpy as np
import pytest
import torch

from _util import dev, mixed_err

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    from aidotnet.tensors_amd import Mi355Engine
    return Mi355Engine()


# B, H, Hkv, Sq, Sk, D, causal, masked, softcap
CASES = [
    (1, 1, 1, 1, 1, 8, False, False, 0.0),
    (1, 2, 2, 64, 128, 32, False, False, 0.0),          # exactly one tile
    (2, 2, 1, 65, 129, 64, True, False, 0.0),           # one past the tile, grouped heads, bottom-right causal
    (1, 3, 3, 63, 127, 40, True, False, 0.0),           # one short; head dim of one whole and one partial 128-byte part
    (1, 2, 2, 200, 200, 128, True, False, 0.0),         # four parts: the two-stage ring is refilled
    (1, 1, 1, 130, 260, 256, False, False, 5.0),        # eight parts, soft-cap
    (2, 4, 4, 96, 300, 64, False, True, 0.0),           # mask
    (1, 2, 2, 70, 90, 20, True, True, 3.0),             # D not a multiple of the step: guarded loads; every option
    (1, 2, 2, 33, 65, 7, False, False, 0.0),            # rows off the 16-byte grid
    (1, 1, 1, 300, 140, 16, True, False, 0.0),          # Sq > Sk: the early rows see no key at all
]


@pytest.mark.parametrize("B,H,Hkv,Sq,Sk,D,causal,masked,softcap", CASES)
def test_returned_probabilities(eng, B, H, Hkv, Sq, Sk, D, causal, masked, softcap):
    rng = np.random.default_rng(Sq * 1000 + Sk + D)
    q = rng.standard_normal((B, H, Sq, D)).astype(np.float32)
    k = rng.standard_normal((B, Hkv, Sk, D)).astype(np.float32); v = rng.standard_normal((B, Hkv, Sk, D)).astype(np.float32)
    keep = (rng.random((B, 1, 1, Sk)) < 0.7) if masked else None
    scale = 1.0 / np.sqrt(D)
    o, w = eng.ScaledDotProductAttention(dev(q), dev(k), dev(v), torch.from_numpy(keep).cuda() if masked else None, scale, softcap, causal)
    w = w.cpu().numpy().astype(np.float64)

    g = H // Hkv
    s = np.einsum("bhid,bhjd->bhij", q.astype(np.float64), np.repeat(k, g, 1).astype(np.float64)) * scale
    if softcap > 0:
        s = softcap * np.tanh(s / softcap)
    hidden = np.zeros((B, H, Sq, Sk), bool)
    if causal:
        hidden |= np.arange(Sk)[None, :] > np.arange(Sq)[:, None] + Sk - Sq
    if masked:
        hidden |= ~np.broadcast_to(keep, hidden.shape)
    s[hidden] = -np.inf
    m = np.where(np.isfinite(s.max(-1, keepdims=True)), s.max(-1, keepdims=True), 0.0)
    p = np.exp(s - m)
    l = p.sum(-1, keepdims=True)
    want = np.where(l > 0, p / np.where(l > 0, l, 1.0), 0.0)

    assert np.all(w[hidden] == 0.0)
    assert mixed_err(w, want) <= 1e-4
    visible = l[..., 0] > 0
    assert np.max(np.abs(w.sum(-1)[visible] - 1.0), initial=0.0) <= 1e-4
    assert mixed_err(o.cpu().numpy(), want @ np.repeat(v, g, 1).astype(np.float64)) <= 1e-4

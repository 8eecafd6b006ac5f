"""fp32 attention of few query tiles over many keys: ranges of the keys as workgroups of their own and a merge.

Bound: fp32 logits, probabilities and sums, so 4e-6 of the norm against float64 as in one range; values near the ends of the fp32 range against
float64 at 1e-5 of each row's largest value."""
import math

import pytest
import torch

from _util import kernels_of

pytestmark = pytest.mark.gpu


def engine():
    from aidotnet.tensors_amd import Mi355Backend, Mi355Engine
    return Mi355Engine(Mi355Backend())


def reference(q, k, v, scale, causal_from=None, keep=None, softcap=0.0):
    g = q.shape[1] // k.shape[1]
    k, v = k.repeat_interleave(g, 1).double(), v.repeat_interleave(g, 1).double()
    s = (q.double() @ k.transpose(-1, -2).contiguous()) * scale
    if softcap > 0:
        s = softcap * torch.tanh(s / softcap)
    if keep is not None:
        s = s.masked_fill(~keep, -math.inf)
    if causal_from is not None:
        i = torch.arange(q.shape[2], device="cuda")[:, None] + causal_from
        s = s.masked_fill(torch.arange(k.shape[2], device="cuda")[None, :] > i, -math.inf)
    p = torch.softmax(s, -1).nan_to_num(0.0)
    return p @ v, p, torch.logsumexp(s, -1)


def rel(x, y):
    return float((x.double() - y).norm() / y.norm())


# (the shortest keys that are cut and one more, last ranges that are short or empty, one and several query tiles, widths that fill a tile row or not)
CASES = [(1, 4, 4, 40, 225, 128), (1, 4, 4, 40, 384, 128), (1, 8, 2, 130, 385, 128), (2, 3, 3, 31, 1000, 80), (1, 2, 1, 1, 2049, 128), (1, 8, 8, 64, 768, 64), (2, 4, 4, 65, 769, 64),
         (1, 6, 3, 100, 1111, 32), (1, 1, 1, 17, 8200, 24), (1, 4, 4, 500, 900, 128)]


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("B,H,Hkv,Sq,Sk,D", CASES)
def test_ranges(B, H, Hkv, Sq, Sk, D, causal):
    eng = engine()
    gen = torch.Generator(device="cuda").manual_seed(Sk + D)
    q, k, v = (torch.randn(B, h, n, D, device="cuda", generator=gen) for h, n in ((H, Sq), (Hkv, Sk), (Hkv, Sk)))
    scale = 1 / math.sqrt(D)
    call = lambda: eng.ScaledDotProductAttention(q, k, v, None, scale, isCausal=causal)
    names = kernels_of(call)
    assert [n.split("<")[0] for n in names] == ["attn_split_kernel", "attn_split_merge_kernel", "attn_weights_split_kernel"], names
    o, w = call()
    want, p, lse = reference(q, k, v, scale, Sk - Sq if causal else None)
    assert rel(o, want) <= 4e-6 and rel(w, p) <= 4e-6, (rel(o, want), rel(w, p))
    if Hkv == H and not causal:
        o2, l2 = eng.FlashAttention(q, k, v, scale)
        assert rel(o2, want) <= 4e-6 and float((l2.double() - lse).abs().max()) <= 1e-5


@pytest.mark.parametrize("D", [32, 64])
def test_options(D):
    """A key mask that hides whole ranges and, in one batch, every key; a mask plane; a soft cap."""
    eng = engine()
    gen = torch.Generator(device="cuda").manual_seed(D)
    q, k, v = (torch.randn(2, 4, n, D, device="cuda", generator=gen) for n in (70, 1030, 1030))
    scale = 1 / math.sqrt(D)
    keys = torch.ones(2, 1, 1, 1030, dtype=torch.bool, device="cuda")
    keys[0, ..., 200:900] = False
    keys[1] = False
    plane = torch.rand(1, 1, 70, 1030, device="cuda", generator=gen) < 0.5
    plane[..., 3, :] = False
    for mask, cap in ((keys, 0.0), (plane, 0.0), (None, 20.0), (keys, 20.0)):
        call = lambda: eng.ScaledDotProductAttention(q, k, v, mask, scale, softcap=cap)
        assert any(n.startswith("attn_split_merge_kernel") for n in kernels_of(call))
        o, w = call()
        want, p, _ = reference(q, k, v, scale, keep=mask, softcap=cap)
        assert rel(o, want) <= 4e-6 and rel(w, p) <= 4e-6
        hidden = p.sum(-1) == 0
        assert bool((o[hidden] == 0).all()) and bool((w[hidden] == 0).all())


@pytest.mark.parametrize("block", [16, 33])
@pytest.mark.parametrize("H,Hkv,D,S,start", [(16, 4, 128, 31, 882), (4, 4, 64, 127, 1027), (2, 1, 128, 8, 4000)])
def test_paged(H, Hkv, D, S, start, block):
    eng = engine(); be = eng.backend; W = be.WrapTensor
    gen = torch.Generator(device="cuda").manual_seed(S)
    n = start + S
    blocks = (n + block - 1) // block
    table = torch.randperm(blocks + 3, device="cuda", generator=gen)[:blocks].int()
    kp, vp = (torch.randn(blocks + 3, block, Hkv, D, device="cuda", generator=gen) for _ in range(2))
    q = torch.randn(S, H, D, device="cuda", generator=gen)
    names = kernels_of(lambda: be.PagedAttentionPrefillGqa(W(q), W(kp), W(vp), W(table), H, Hkv, D, block, S, start, 1 / math.sqrt(D)))
    assert [x.split("<")[0] for x in names] == ["attn_split_kernel", "attn_split_merge_kernel"], names
    out = be.PagedAttentionPrefillGqa(W(q), W(kp), W(vp), W(table), H, Hkv, D, block, S, start, 1 / math.sqrt(D)).tensor.view(S, H, D)
    k, v = (x[table.long()].reshape(-1, Hkv, D)[:n].transpose(0, 1)[None] for x in (kp, vp))
    want, _, _ = reference(q.transpose(0, 1)[None], k, v, 1 / math.sqrt(D), start)
    assert rel(out, want[0].transpose(0, 1)) <= 4e-6


@pytest.mark.parametrize("size", [1e-30, 1e30, 1.5e38])
def test_values_near_the_ends(size):
    """V far from one, in some ranges or in all: the partials keep within fp32 wherever the result does; NaN and infinities reach their rows alone."""
    eng = engine()
    gen = torch.Generator(device="cuda").manual_seed(7)
    q, k, v = (torch.randn(1, 2, n, 128, device="cuda", generator=gen) for n in (40, 1600, 1600))
    v = v.clamp(-2, 2)
    for part in (slice(0, 1600), slice(300, 500))[:1 if size > 1e38 else 2]:      # (two scales in a head, the larger one at the end: beyond the fp32 pipe's sums)
        u = v.clone()
        u[:, :, part] *= size
        o, _ = eng.FlashAttention(q, k, u)
        want, _, _ = reference(q, k, u, 128 ** -0.5)
        top = want.abs().amax(-1, keepdim=True)
        assert bool(o.isfinite().all()) and float(((o.double() - want).abs() / top).max()) <= 1e-5
    q[0, 1, 5, 3] = math.nan
    v[0, 0, 900, 7] = math.inf
    o, _ = eng.FlashAttention(q, k, v)
    assert bool(o[0, 1, 5].isnan().all()) and bool(o[0, 1, :5].isfinite().all()) and bool((o[0, 0, :, 7] == math.inf).all())
    o[0, 0, :, 7] = 0
    assert bool(o[0, 0].isfinite().all())

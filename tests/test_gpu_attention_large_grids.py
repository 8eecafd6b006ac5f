"""Attention on grids past the lines up to which several waves share a row's keys (launch_attn): the instances with one wave per row that
larger batches run -- key masks (64-key tiles, and in fp32 at head dimension 128 the 32-key tiles), mask planes, biases and soft-caps, and
block tables (fp32 at head dimension 128: eight keys per wave and tile) -- and block tables at head dimension 256; then key masks on
sequences whose keys are cut into ranges.  Against a float64 softmax.

Bounds: fp32 logits and one exponential, (D + 20) 2^-24 < 2e-5, held at 1e-4; 16-bit operands round P once, 2^-9 relative (bf16) of
averages of N(0,1) rows, held at 2e-2, and at head dimension 128 their row sums are of the rounded probabilities (LSE 2e-3)."""
import math

import pytest
import torch

from _util import TORCH16

pytestmark = pytest.mark.gpu
DT = {"f32": torch.float32, **TORCH16}


@pytest.fixture(scope="module")
def be():
    from aidotnet.tensors_amd import Mi355Backend
    return Mi355Backend()


def close(got, want, tol):
    return float(((got.double() - want).abs() / (1 + want.abs())).max()) <= tol


def reference(q, k, v, hidden, scale, softcap=0.0, bias=None):
    """q [B,H,Sq,D], k, v [B,H,Sk,D] float64, hidden broadcastable to [B,H,Sq,Sk]: (O, LSE); a row without keys is zeros / -inf."""
    s = torch.matmul(q, k.transpose(-1, -2).contiguous()) * scale
    if softcap > 0:
        s = softcap * torch.tanh(s / softcap)
    if bias is not None:
        s = s + bias.double()
    s = s.masked_fill(hidden, float("-inf"))
    lse = torch.logsumexp(s, -1)
    return torch.matmul(torch.exp(s - torch.where(torch.isinf(lse), torch.zeros_like(lse), lse)[..., None]), v), lse


def attn(be, kind, q, k, v, causal=False, softcap=0.0, mask=None, mask_mode=0, bias=None):
    from aidotnet.tensors_amd._lib import AttnDesc
    (B, H, Sq, D), (Hkv, Sk) = q.shape, k.shape[1:3]
    o, lse = torch.empty(B, H, Sq, D, device="cuda"), torch.empty(B, H, Sq, device="cuda")
    d = AttnDesc(B=B, H=H, Hkv=Hkv, Sq=Sq, Sk=Sk, D=D, scale=1 / math.sqrt(D), causal=int(causal), causal_query_offset=Sk - Sq,
                 softcap=softcap, mask_mode=mask_mode)
    W = lambda t: be.WrapTensor(t) if t is not None else None
    be._attn(kind, W(q), W(k), W(v), W(o), W(lse), W(bias), W(mask), None, d)
    return o, lse


def operands(kind, B, H, Sq, Sk, D):
    gen = torch.Generator(device="cuda").manual_seed(Sq * 1000 + Sk + D)
    return [torch.randn(B, H, s, D, device="cuda", generator=gen).to(DT[kind]) for s in (Sq, Sk, Sk)], gen


def key_rows(how, B, Sk, gen):
    at = torch.arange(Sk, device="cuda")[None, :]
    cut = torch.randint(1, Sk, (B, 1), device="cuda", generator=gen)
    keep = at < cut if how == "padded" else at >= cut if how == "left" else torch.rand(B, Sk, device="cuda", generator=gen) < 0.5
    if how == "padded": keep[0] = True
    if how == "holes": keep[B - 1] = False
    return keep


def causal_hidden(Sq, Sk, on):
    return torch.arange(Sk, device="cuda")[None, :] > torch.arange(Sq, device="cuda")[:, None] + (Sk - Sq if on else Sk)


@pytest.mark.parametrize("how", ["padded", "left", "holes"])
@pytest.mark.parametrize("kind,B,H,Sq,Sk,D,causal", [
    ("f32", 8, 64, 129, 130, 64, False), ("f32", 8, 64, 129, 129, 64, True), ("f16", 8, 64, 129, 130, 64, False), ("bf16", 8, 64, 190, 190, 64, True),
    ("f32", 4, 64, 129, 97, 128, False), ("f32", 4, 64, 129, 129, 128, True), ("f32", 8, 64, 129, 63, 64, False), ("f32", 4, 64, 129, 31, 128, False)])
def test_key_mask(be, kind, B, H, Sq, Sk, D, causal, how):
    (q, k, v), gen = operands(kind, B, H, Sq, Sk, D)
    keep = key_rows(how, B, Sk, gen)
    o, lse = attn(be, kind, q, k, v, causal, mask=keep, mask_mode=3)
    hidden = ~keep[:, None, None, :] | causal_hidden(Sq, Sk, causal)
    want, want_lse = reference(q.double(), k.double(), v.double(), hidden, 1 / math.sqrt(D))
    empty = torch.isinf(want_lse)
    assert close(o, want, 1e-4 if kind == "f32" else 2e-2)
    assert torch.equal(torch.isinf(lse), empty) and close(lse[~empty], want_lse[~empty], 1e-4)


@pytest.mark.parametrize("how", ["padded", "left", "holes"])
@pytest.mark.parametrize("kind", ["f16", "bf16"])
@pytest.mark.parametrize("B,H,Sq,Sk,causal", [(3, 2, 7, 1024, False), (2, 2, 130, 1500, False), (2, 2, 33, 1500, True), (3, 1, 70, 4100, False)])
def test_key_mask_with_key_ranges(be, kind, B, H, Sq, Sk, causal, how):
    """Head dimension 128: masks that empty the first or the last range, and a batch that sees nothing."""
    (q, k, v), gen = operands(kind, B, H, Sq, Sk, 128)
    keep = key_rows(how, B, Sk, gen)
    if how == "padded": keep[1] = torch.arange(Sk, device="cuda") < 70
    if how == "left": keep[1] = torch.arange(Sk, device="cuda") >= Sk - 70
    o, lse = attn(be, kind, q, k, v, causal, mask=keep, mask_mode=3)
    hidden = ~keep[:, None, None, :] | causal_hidden(Sq, Sk, causal)
    want, want_lse = reference(q.double(), k.double(), v.double(), hidden, 1 / math.sqrt(128))
    empty = torch.isinf(want_lse)
    assert close(o, want, 2e-2)
    assert torch.equal(torch.isinf(lse), empty) and close(lse[~empty], want_lse[~empty], 2e-3)


@pytest.mark.parametrize("what", ["plane", "full", "softcap", "bias"])
@pytest.mark.parametrize("kind,B,H,Sq,Sk,D,causal", [
    ("f32", 8, 64, 129, 130, 64, False), ("f32", 8, 64, 129, 129, 64, True), ("f32", 8, 64, 129, 70, 32, False), ("bf16", 8, 64, 129, 130, 64, False),
    ("f16", 4, 64, 190, 190, 128, True), ("bf16", 4, 64, 129, 100, 80, False)])
def test_masks_biases_and_softcaps(be, kind, B, H, Sq, Sk, D, causal, what):
    (q, k, v), gen = operands(kind, B, H, Sq, Sk, D)
    hidden = causal_hidden(Sq, Sk, causal)
    kw, softcap, bias = {}, 0.0, None
    if what in ("plane", "full"):
        keep = torch.rand(*((Sq, Sk) if what == "plane" else (B, H, Sq, Sk)), device="cuda", generator=gen) < 0.6
        keep[..., 0] = True
        kw = {"mask": keep.float(), "mask_mode": 1 if what == "plane" else 2}
        hidden = hidden | ~keep
    elif what == "softcap":
        softcap = kw["softcap"] = 4.0
    else:
        bias = kw["bias"] = torch.randn(1, H, Sq, Sk, device="cuda", generator=gen)
    o, lse = attn(be, kind, q, k, v, causal, **kw)
    want, want_lse = reference(q.double(), k.double(), v.double(), hidden, 1 / math.sqrt(D), softcap, bias)
    assert close(o, want, 1e-4 if kind == "f32" else 2e-2) and close(lse, want_lse, 1e-4)


# heads, kvHeads, D, block, queries, start
@pytest.mark.parametrize("kind,heads,kv,d,block,nq,start", [
    ("f32", 32, 8, 128, 16, 830, 1273), ("f32", 64, 64, 128, 48, 390, 5),            # 32-key tiles, past 64 of them; blocks that straddle them
    ("f32", 64, 8, 64, 16, 1030, 3101), ("f16", 64, 8, 64, 32, 1030, 3101), ("bf16", 64, 16, 64, 48, 1030, 70),
    ("f16", 4, 2, 256, 16, 130, 61), ("bf16", 4, 2, 256, 48, 70, 2100), ("f16", 2, 2, 256, 64, 33, 0), ("bf16", 4, 4, 256, 8, 40, 100)])
def test_block_tables(be, kind, heads, kv, d, block, nq, start):
    gen = torch.Generator(device="cuda").manual_seed(nq * 7919 + start)
    keys = start + nq
    blocks = (keys + block - 1) // block
    pool = blocks + 3
    randn = lambda *s: torch.randn(*s, device="cuda", generator=gen).to(DT[kind])
    q, kp, vp = randn(nq, heads, d), randn(pool, block, kv, d), randn(pool, block, kv, d)
    table = torch.randperm(pool, device="cuda", generator=gen)[:blocks].to(torch.int32)
    spare = torch.ones(pool, dtype=torch.bool, device="cuda"); spare[table.long()] = False
    kp[spare] = float("nan"); vp[spare] = float("nan")                        # blocks of other sequences must not be touched
    if keys % block:
        kp[table[-1].long(), keys % block:] = float("nan"); vp[table[-1].long(), keys % block:] = float("nan")
    W, scale = be.WrapTensor, 1 / math.sqrt(d)
    args = (W(q), W(kp), W(vp), W(table))
    out = (be.PagedAttentionPrefillGqa(*args, heads, kv, d, block, nq, start, scale) if kind == "f32"
           else be.PagedAttentionHalf(kind, *args, heads, kv, d, block, nq, start, scale))
    got = out.tensor.reshape(nq, heads, d)
    K, V = (t[table.long()].reshape(-1, kv, d)[:keys].double() for t in (kp, vp))
    hidden = torch.arange(keys, device="cuda")[None, :] > torch.arange(nq, device="cuda")[:, None] + start
    for h in range(heads):
        g = h // (heads // kv)
        want, _ = reference(q[:, h].double(), K[:, g].contiguous(), V[:, g].contiguous(), hidden, scale)
        assert close(got[:, h], want, 1e-4 if kind == "f32" else 2e-2), h


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("kind", ["f32", "bf16"])
@pytest.mark.parametrize("H,Sq,Sk,D", [(256, 33, 64, 64), (257, 33, 64, 64), (257, 129, 64, 64), (512, 64, 64, 64), (128, 129, 64, 64), (171, 129, 64, 64),
                                       (171, 129, 65, 64), (200, 140, 130, 32), (218, 219, 239, 64), (110, 500, 500, 64), (90, 62, 32, 128), (90, 62, 33, 128), (300, 62, 33, 128)])
def test_lines_of_short_sequences(be, kind, H, Sq, Sk, D, causal):
    """Both sides of the lines that the key groups of short sequences have, and head counts that 8 does not divide."""
    (q, k, v), _ = operands(kind, 1, H, Sq, Sk, D)
    o, lse = attn(be, kind, q, k, v, causal)
    hidden = causal_hidden(Sq, Sk, causal)
    want, want_lse = reference(q.double(), k.double(), v.double(), hidden, 1 / math.sqrt(D))
    empty = torch.isinf(want_lse)
    assert close(o, want, 1e-4 if kind == "f32" else 2e-2)
    assert torch.equal(torch.isinf(lse), empty) and close(lse[~empty], want_lse[~empty], 1e-4 if kind == "f32" else 2e-3)

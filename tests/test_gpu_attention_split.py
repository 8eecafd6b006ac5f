"""fp32 attention and its probabilities on the fp16 matrix pipe: edges of the query and key tiles, key groups, head dimensions, options, and the values
that two scaled fp16 numbers do not hold.

Bounds: 1.5e-6 in the 2-norm per (batch, head) and output, five times what such sums of up to 700 terms show; what is computed again comes from the fp32
pipe and meets the same bound."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    from aidotnet.tensors_amd import Mi355Engine
    return Mi355Engine()


def exact(q, k, v, scale, hidden, softcap=0.0, bias=None):
    q, k, v = q.double(), k.double(), v.double()
    groups = q.shape[1] // k.shape[1]
    k, v = k.repeat_interleave(groups, 1), v.repeat_interleave(groups, 1)
    s = torch.matmul(q, k.transpose(2, 3).contiguous()) * scale
    if softcap:
        s = softcap * torch.tanh(s / softcap)
    if bias is not None:
        s = s + bias.double()
    s = s.masked_fill(hidden, float("-inf"))
    w = torch.softmax(s, -1)
    return torch.matmul(w, v), torch.logsumexp(s, -1), w


def close(got, want):
    err = (got.double() - want).flatten(2).norm(dim=2) / want.flatten(2).norm(dim=2)
    return float(err.max()) <= 1.5e-6


def causal_mask(Sq, Sk, offset, device="cuda"):
    return torch.arange(Sk, device=device)[None, :] > torch.arange(Sq, device=device)[:, None] + offset


def randn(seed, *shapes):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn(*s, device="cuda", generator=gen) for s in shapes]


# (B, H, Hkv, Sq, Sk, D): one row, tile edges of 32 / 64 / 128 rows and keys, every workgroup form, D in whole chunks of eight and padded ones
SHAPES = [(1, 2, 2, 1, 65, 64), (1, 2, 1, 33, 127, 64), (1, 3, 3, 64, 129, 64), (2, 2, 2, 130, 192, 64), (1, 12, 12, 200, 449, 64), (8, 48, 48, 129, 131, 64),
          (1, 2, 2, 40, 3, 32), (1, 4, 2, 100, 500, 24), (1, 4, 4, 65, 64, 8), (13, 60, 30, 70, 95, 32),
          (1, 2, 2, 20, 31, 128), (1, 4, 2, 130, 225, 128), (1, 2, 2, 128, 230, 80), (5, 60, 60, 129, 97, 96)]


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("B,H,Hkv,Sq,Sk,D", SHAPES)
def test_shapes(eng, B, H, Hkv, Sq, Sk, D, causal):
    q, k, v = randn(Sq + 3 * Sk + D, (B, H, Sq, D), (B, Hkv, Sk, D), (B, Hkv, Sk, D))
    offset = Sk - Sq if causal and Sk > Sq else 0
    want, lse, w = exact(q, k, v, 1 / math.sqrt(D), causal_mask(Sq, Sk, offset) if causal else torch.zeros(Sq, Sk, dtype=torch.bool, device="cuda"))
    o, l = eng.FlashAttention(q, k, v, isCausal=causal, queryOffset=offset)
    assert close(o, want) and float((l.double() - lse).abs().max()) <= 4e-6
    if not causal or Sk >= Sq:
        o, p = eng.ScaledDotProductAttention(q, k, v, isCausal=causal)
        assert close(o, want) and close(p, w)


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("Sq,Sk", [(70, 70), (130, 200), (300, 300)])
@pytest.mark.parametrize("option", ["padding", "plane", "softcap", "bias"])
def test_options(eng, option, Sq, Sk, D):
    B, H = 2, 4
    q, k, v, bias = randn(Sk + D, (B, H, Sq, D), (B, H, Sk, D), (B, H, Sk, D), (B, H, Sq, Sk))
    hidden, mask, softcap = torch.zeros(B, 1, 1, Sk, dtype=torch.bool, device="cuda"), None, 0.0
    if option == "padding":
        hidden = (torch.arange(Sk, device="cuda")[None, :] >= torch.tensor([[Sk // 2], [max(Sk - 65, 1)]], device="cuda"))[:, None, None, :]
        mask = ~hidden
    elif option == "plane":
        hidden = bias > 0.5
        hidden[..., 0] = False
        mask = ~hidden
    elif option == "softcap":
        softcap = 2.0
    if option == "bias":
        want, lse, w = exact(q, k, v, 1 / math.sqrt(D), hidden, bias=bias)
        o, l = eng.FlashAttention(q, k, v, attentionBias=bias)
        assert close(o, want) and float((l.double() - lse).abs().max()) <= 4e-6
    else:
        want, lse, w = exact(q, k, v, 1 / math.sqrt(D), hidden, softcap)
        o, p = eng.ScaledDotProductAttention(q, k, v, mask, softcap=softcap)
        assert close(o, want) and close(p, w)


@pytest.mark.parametrize("Sq,Sk,D", [(40, 200, 64), (130, 300, 128)])
@pytest.mark.parametrize("case", ["k later", "v later", "k hidden", "k zeros of q", "v column", "v tiny column", "v zero column", "first tile zero", "scaled",
                                  "large logits"])
def test_values_beyond_the_scale(eng, case, Sq, Sk, D):
    q, k, v = randn(Sk, (1, 2, Sq, D), (1, 2, Sk, D), (1, 2, Sk, D))
    causal, offset = False, 0
    if case == "k later":                 # a later tile far beyond the first one's scale: its logits rule
        k[:, :, 150:] *= 1e4
    elif case == "v later":
        v[:, :, 150:] *= 1e6
    elif case == "k hidden":              # the scale comes from a key that most rows do not see
        k[:, :, Sq - 2] *= 1e9
        causal = True
    elif case == "k zeros of q":          # ... from a channel that meets zeros
        k[..., 3] = 1e9
        q[..., 3] = 0.0
    elif case == "v column":              # columns far below the rest
        v[..., 5] *= 1e-7
    elif case == "v tiny column":
        v[..., 5] *= 1e-30
    elif case == "v zero column":
        v[..., 5] = 0.0
    elif case == "first tile zero":
        k[:, :, :64] = 0.0
        v[:, :, :64] = 0.0
    elif case == "scaled":
        q, k, v = q * 1e-20, k * 1e20, v * 1e-33
    elif case == "large logits":
        q, k = q * 60, k * 60
    hidden = causal_mask(Sq, Sk, 0) if causal else torch.zeros(Sq, Sk, dtype=torch.bool, device="cuda")
    want, lse, w = exact(q, k, v, 1 / math.sqrt(D), hidden)
    o, l = eng.FlashAttention(q, k, v, isCausal=causal)
    p = None if causal else eng.ScaledDotProductAttention(q, k, v)[1]
    if case in ("k later", "large logits"):          # (logits of thousands: 2^-24 of one is a relative error of its probability)
        big = float(torch.nan_to_num(torch.matmul(q.double(), k.double().transpose(2, 3).contiguous()) / math.sqrt(D)).abs().max())
        assert float((o.double() - want).norm() / want.norm()) <= 1.5e-6 * max(1.0, big / 4)
        return
    if case == "k hidden":                            # (rows that see the large key: one probability of one)
        seen = Sq - 2
        want, o, lse, l = want[:, :, :seen], o[:, :, :seen], lse[:, :, :seen], l[:, :, :seen]
    assert close(o, want) and float((l.double() - lse).abs().max()) <= 4e-6 * max(1.0, float(lse.abs().max()) / 8)
    assert p is None or close(p, w)
    column = want[..., 5].norm()
    assert float((o[..., 5].double() - want[..., 5]).norm()) <= 3e-6 * float(column)


@pytest.mark.parametrize("block", [1, 16, 24])
@pytest.mark.parametrize("nq,start,D", [(9, 60, 64), (130, 0, 64), (70, 400, 128)])
def test_paged(nq, start, D, block):
    from aidotnet.tensors_amd import Mi355Backend
    be = Mi355Backend()
    H, Hkv, keys = 4, 2, start + nq
    blocks = (keys + block - 1) // block
    q, kp, vp = randn(nq + start, (nq, H, D), (blocks + 3, block, Hkv, D), (blocks + 3, block, Hkv, D))
    table = torch.randperm(blocks + 3, device="cuda")[:blocks].to(torch.int32)
    W = be.WrapTensor
    got = be.PagedAttentionPrefillGqa(W(q), W(kp), W(vp), W(table), H, Hkv, D, block, nq, start, 1 / math.sqrt(D)).tensor.view(nq, H, D)
    flat = lambda p: p[table.long()].reshape(-1, Hkv, D)[:keys].permute(1, 0, 2).contiguous()[None]
    want, _, _ = exact(q.permute(1, 0, 2).contiguous()[None], flat(kp), flat(vp), 1 / math.sqrt(D), causal_mask(nq, keys, start))
    assert close(got.permute(1, 0, 2)[None], want)

"""Attention layers of few rows over a wide model: the output projection runs in K ranges, and, on a captured stream whose workspace was
reserved without room for them, in one launch.

Bound: fp32 1e-4 and 16-bit 2e-2 mixed error against float64 on the same rounded inputs, as for the other sizes of the layer."""
import math

import pytest
import torch

from _util import TORCH16, kernels_of

pytestmark = pytest.mark.gpu


def reference(x, wq, wk, wv, wo, heads):
    B, S, dM = x.shape
    q, k, v = ((x.double() @ w.double()).view(B, S, heads, dM // heads).transpose(1, 2) for w in (wq, wk, wv))
    p = torch.softmax((q @ k.transpose(-1, -2).contiguous()) / math.sqrt(dM // heads), -1)
    return (p @ v).transpose(1, 2).reshape(B, S, dM) @ wo.double()


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("kind,B,S,dM,heads", [("f32", 11, 31, 2048, 16), ("f32", 1, 33, 1536, 12), ("bf16", 2, 128, 2048, 16), ("f16", 3, 21, 2560, 20)])
def test_output_projection_in_ranges(kind, B, S, dM, heads, packed):
    from aidotnet.tensors_amd import Mi355Backend
    be = Mi355Backend(); W = be.WrapTensor
    dt = TORCH16.get(kind, torch.float32)
    gen = torch.Generator(device="cuda").manual_seed(dM + S)
    x = torch.randn(B, S, dM, device="cuda", generator=gen).to(dt)
    ws = [(torch.randn(dM, dM, device="cuda", generator=gen) / math.sqrt(dM)).to(dt) for _ in range(4)]
    out = torch.empty_like(x)
    if packed:
        qkv = be.PackQkvWeights(kind, *(W(w) for w in ws[:3]), dM)
        call = lambda: be.MultiHeadAttentionForwardPacked(kind, W(x), qkv, W(ws[3]), None, W(out), B, S, dM, heads)
    else:
        call = lambda: be.MultiHeadAttentionForward(kind, W(x), *(W(w) for w in ws), None, W(out), B, S, dM, heads)
    names = kernels_of(call)
    assert names[-1].startswith("skinny_reduce_kernel"), names
    want = reference(x, *ws, heads)
    limit = 1e-4 if kind == "f32" else 2e-2
    err = lambda: float(((out.double() - want).abs() / want.abs().clamp(min=1.0)).max())
    assert err() <= limit
    if packed:
        return
    es = x.element_size()
    up = lambda n: (n + 255) // 256 * 256
    be2 = Mi355Backend(synchronous=False)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        be2.ReserveWorkspace(up(B * S * 3 * dM * es) + up(B * S * dM * es))
        graph = torch.cuda.CUDAGraph()
        out.zero_()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=stream):
            be2.MultiHeadAttentionForward(kind, W(x), *(W(w) for w in ws), None, W(out), B, S, dM, heads)
        for _ in range(3):
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert err() <= limit


@pytest.mark.parametrize("kind,B,S,dM,heads", [("f32", 1, 1100, 256, 4), ("f32", 2, 800, 384, 3), ("bf16", 1, 1100, 512, 4), ("f16", 2, 1500, 256, 2)])
def test_attention_of_the_layer_in_key_ranges(kind, B, S, dM, heads):
    """Few heads over a long sequence: the layer's attention cuts its keys too, with a padding mask that hides whole ranges."""
    from aidotnet.tensors_amd import Mi355Backend, Mi355Engine
    eng = Mi355Engine(Mi355Backend())
    dt = TORCH16.get(kind, torch.float32)
    gen = torch.Generator(device="cuda").manual_seed(dM + S)
    x = torch.randn(B, S, dM, device="cuda", generator=gen).to(dt)
    ws = [(torch.randn(dM, dM, device="cuda", generator=gen) / math.sqrt(dM)).to(dt) for _ in range(4)]
    for keep in (None, torch.arange(S, device="cuda")[None, :] < torch.tensor([S // 3, S - 1][:B], device="cuda")[:, None]):
        mask = None if keep is None else keep[:, None, None, :]
        call = lambda: eng.MultiHeadAttentionForward(x, *ws, heads, mask)
        if kind != "f32" or keep is None or dM // heads <= 64:
            assert any(n.startswith("attn_split_merge_kernel") for n in kernels_of(call))
        out = call()
        q, k, v = ((x.double() @ w.double()).view(B, S, heads, dM // heads).transpose(1, 2) for w in ws[:3])
        s = (q @ k.transpose(-1, -2).contiguous()) / math.sqrt(dM // heads)
        if keep is not None:
            s = s.masked_fill(~mask, -math.inf)
        want = (torch.softmax(s, -1) @ v).transpose(1, 2).reshape(B, S, dM) @ ws[3].double()
        assert float(((out.double() - want).abs() / want.abs().clamp(min=1.0)).max()) <= (1e-4 if kind == "f32" else 2e-2)

"""The Q, K and V weights of the attention layer multiplied where they are (three products in one launch) or gathered into one matrix:
widths that take either, with row counts on and around the tiles, weights off the 16-byte grid, and the packed form, which must give the
same bits.  Against a float64 layer.

Bounds: fp32 sums of K products of N(0,1) times N(0,1/K) values, K 2^-24 < 1e-4 relative to the unit-sized results; 16-bit rounds Q, K, V,
P and O once each, 2^-9 relative (bf16), held at 2e-2 as for the layer's other tests."""
import numpy as np
import pytest
import torch

from _util import mixed_err
from test_mha_forward import mha64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("B,S,dM,H,offset", [(1, 1, 64, 1, 0), (2, 33, 128, 4, 0), (1, 257, 192, 3, 0), (3, 100, 320, 5, 0), (2, 65, 768, 12, 0),
                                             (1, 40, 24, 3, 0), (1, 37, 63, 3, 0), (2, 50, 128, 4, 1), (1, 700, 256, 2, 3)])
def test_qkv_weights_in_place(B, S, dM, H, offset, kind):
    from aidotnet.tensors_amd import Mi355Backend, Mi355Engine
    be = Mi355Backend(); eng = Mi355Engine(be)
    dt = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[kind]
    gen = torch.Generator().manual_seed(S + dM)
    x = torch.randn(B, S, dM, generator=gen).to(dt)
    ws = [(torch.randn(dM, dM, generator=gen) / dM ** 0.5).to(dt) for _ in range(4)]
    placed = []
    for w in ws:                                           # offset elements into a buffer: a weight off the 16-byte grid
        raw = torch.zeros(dM * dM + offset, dtype=dt, device="cuda")
        raw[offset:] = w.reshape(-1).cuda()
        placed.append(raw[offset:].view(dM, dM))
    y = eng.MultiHeadAttentionForward(x.cuda(), *placed, H)
    want = mha64(x.float().numpy(), *[w.float().numpy() for w in ws], H)
    assert mixed_err(y.float().cpu().numpy(), want) <= (1e-4 if kind == "f32" else 2e-2)
    W = be.WrapTensor
    packed = be.PackQkvWeights(kind, *[W(w) for w in placed[:3]], dM)
    assert torch.equal(packed.tensor.view(dt).reshape(dM, 3 * dM).cpu(), torch.cat(ws[:3], dim=1))
    y1 = torch.empty_like(y)
    be.MultiHeadAttentionForwardPacked(kind, W(x.cuda()), packed, W(placed[3]), None, W(y1), B, S, dM, H)
    if offset == 0:
        assert torch.equal(y, y1)
    else:
        assert mixed_err(y1.float().cpu().numpy(), want) <= (1e-4 if kind == "f32" else 2e-2)

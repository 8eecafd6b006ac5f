"""The three Q, K and V weights at uneven distances and in any order inside one buffer: the product of three batches reads them by two
strides, and must give the bits it gives for weights of their own."""
import itertools

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("B,S,dM,H", [(2, 65, 128, 2), (1, 300, 256, 4)])
def test_weights_anywhere(B, S, dM, H, kind):
    from aidotnet.tensors_amd import Mi355Engine
    eng = Mi355Engine()
    dt = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[kind]
    gen = torch.Generator(device="cuda").manual_seed(S)
    x = torch.randn(B, S, dM, device="cuda", generator=gen).to(dt)
    ws = [(torch.randn(dM, dM, device="cuda", generator=gen) / dM ** 0.5).to(dt) for _ in range(4)]
    want = eng.MultiHeadAttentionForward(x, *ws, H)
    n = dM * dM
    for order in itertools.permutations(range(3)):
        raw = torch.zeros(3 * n + 1000, dtype=dt, device="cuda")
        at, placed = 0, [None] * 3
        for gap, i in zip((8, 64, 704), order):
            at += gap
            placed[i] = raw[at:at + n].view(dM, dM)
            placed[i].copy_(ws[i])
            at += n
        assert torch.equal(eng.MultiHeadAttentionForward(x, *placed, ws[3], H), want), order

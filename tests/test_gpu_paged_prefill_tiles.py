"""Paged prefill on the direct-to-LDS kernels: key tiles of 64 (fp32 at head dimension 128 on larger grids 32, and head dimension 256:
test_gpu_attention_large_grids.py) fetched block by block, pool rows looked
up 64 tiles at a time, the keys of a few query tiles cut into ranges.  Sizes on both sides of each of those edges, block sizes that are
multiples of 16 (powers of two or not) and one that is not, against a float64 softmax over the gathered cache.

Bounds: fp32 1e-4; 16-bit 2e-2 (probabilities rounded to the storage type: at most 2^-9 (bf16) relative each, on averages of N(0,1)
values), the bars of the contiguous kernels."""
import math

import numpy as np
import pytest
import torch

from _util import TORCH16, mixed_err

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def be():
    from aidotnet.tensors_amd import Mi355Backend
    return Mi355Backend()


# heads, kvHeads, D, block, queries, start
CASES = [
    (4, 2, 128, 16, 1, 0),            # one key  (a single query goes the decode way in 16 bit)
    (4, 2, 128, 16, 64, 0),           # exactly one tile
    (4, 4, 128, 16, 65, 0),           # one key past it
    (8, 2, 128, 32, 130, 61),         # two query tiles, a prefix that is no multiple of anything
    (2, 1, 128, 48, 200, 57),         # blocks of 48: tiles straddle blocks
    (2, 2, 128, 64, 5, 1018),         # 1023 keys: no ranges yet
    (2, 2, 128, 64, 5, 1019),         # 1024 keys: two ranges
    (2, 1, 128, 16, 70, 4050),        # 65 tiles: the row table is read again; ranges
    (2, 1, 128, 128, 33, 2100),       # blocks larger than a tile, ranges
    (4, 2, 64, 16, 63, 2),
    (4, 1, 64, 32, 129, 4090),        # head dimension 64, past 64 tiles
    (2, 2, 128, 8, 40, 100),          # blocks of 8: the general kernel
]


@pytest.mark.parametrize("kind", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("heads,kv,d,block,nq,start", CASES)
def test_paged_prefill_tiles(be, kind, heads, kv, d, block, nq, start):
    gen = torch.Generator(device="cuda").manual_seed(nq * 7919 + start)
    T = torch.float32 if kind == "f32" else TORCH16[kind]
    keys = start + nq
    blocks = (keys + block - 1) // block
    pool = blocks + 3
    randn = lambda *s: torch.randn(*s, device="cuda", generator=gen).to(T)
    q, kp, vp = randn(nq, heads, d), randn(pool, block, kv, d), randn(pool, block, kv, d)
    table = torch.randperm(pool, device="cuda", generator=gen)[:blocks].to(torch.int32)
    spare = torch.ones(pool, dtype=torch.bool, device="cuda"); spare[table.long()] = False
    kp[spare] = float("nan"); vp[spare] = float("nan")                        # blocks of other sequences must not be touched
    if keys % block:
        kp[table[-1].long(), keys % block:] = float("nan"); vp[table[-1].long(), keys % block:] = float("nan")
    scale = 1 / math.sqrt(d)
    W = be.WrapTensor
    args = (W(q), W(kp), W(vp), W(table))
    out = (be.PagedAttentionPrefillGqa(*args, heads, kv, d, block, nq, start, scale) if kind == "f32"
           else be.PagedAttentionHalf(kind, *args, heads, kv, d, block, nq, start, scale))
    got = be.DownloadBuffer(out).numpy().reshape(nq, heads, d)

    K = kp[table.long()].reshape(-1, kv, d)[:keys].double().cpu().numpy(); V = vp[table.long()].reshape(-1, kv, d)[:keys].double().cpu().numpy()
    Q = q.double().cpu().numpy()
    g = heads // kv
    want = np.zeros((nq, heads, d))
    hidden = np.arange(keys)[None, :] > np.arange(nq)[:, None] + start
    for h in range(heads):
        s = Q[:, h] @ K[:, h // g].T * scale
        s[hidden] = -np.inf
        p = np.exp(s - s.max(-1, keepdims=True))
        want[:, h] = p / p.sum(-1, keepdims=True) @ V[:, h // g]
    assert mixed_err(got, want) <= (1e-4 if kind == "f32" else 2e-2)

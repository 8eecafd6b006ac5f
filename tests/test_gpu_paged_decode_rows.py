"""Paged decode: the rows of a load are looked up for the wave (block size a multiple of the keys of a load) or key by key, the loads of
an iteration are asked for one iteration ahead, table entries 16 iterations at a time, and the splits are merged by one or by four waves.
Lengths around one load, one iteration (64 keys at head dimension 128, 128 at 64), two of them and the 17th, with one split (long
chains) and many, against a float64 softmax; every arithmetic step after the load is fp32, held at 1e-4 for every storage type."""
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


# heads, kvHeads, D, block, keys, splits
CASES = [
    (4, 1, 128, 16, 1, 1), (4, 1, 128, 16, 3, 1), (4, 1, 128, 16, 64, 1), (4, 1, 128, 16, 65, 1), (2, 1, 128, 16, 129, 1),
    (8, 2, 128, 16, 64 * 17 + 3, 1),          # the table is read again
    (4, 1, 64, 16, 128 * 17 + 9, 1),
    (4, 4, 128, 48, 1000, 2),                 # blocks of 48
    (8, 2, 128, 4, 700, 2),                   # blocks of one load
    (4, 2, 128, 3, 300, 1),                   # blocks a load straddles: key by key
    (4, 2, 80, 16, 400, 1),                   # head dimension that is no power of two: idle lanes
    (4, 2, 256, 32, 500, 2),                  # two float pairs per lane in the merge
    (4, 1, 128, 16, 256 * 8, 8),              # eight ranges: one wave per row
    (4, 1, 128, 16, 256 * 9, 9),              # nine: four waves
    (4, 1, 128, 16, 256 * 40, 40),            # more than one round of loads per wave
]


@pytest.mark.parametrize("kind", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("heads,kv,d,block,keys,splits", CASES)
def test_paged_decode_rows(be, kind, heads, kv, d, block, keys, splits):
    gen = torch.Generator(device="cuda").manual_seed(keys * 31 + d)
    T = torch.float32 if kind == "f32" else TORCH16[kind]
    blocks = (keys + block - 1) // block
    pool = blocks + 3
    randn = lambda *s: torch.randn(*s, device="cuda", generator=gen).to(T)
    q, kp, vp = randn(1, heads, d), randn(pool, block, kv, d), randn(pool, block, kv, d)
    table = torch.randperm(pool, device="cuda", generator=gen)[:blocks].to(torch.int32)
    spare = torch.ones(pool, dtype=torch.bool, device="cuda"); spare[table.long()] = False
    kp[spare] = float("nan"); vp[spare] = float("nan")
    if keys % block:
        kp[table[-1].long(), keys % block:] = float("nan"); vp[table[-1].long(), keys % block:] = float("nan")
    scale = 1 / math.sqrt(d)
    W = be.WrapTensor
    out = be._paged("decode", kind, W(q), W(kp), W(vp), W(table), heads, kv, d, block, 1, keys, 0, scale, splits, True)
    got = be.DownloadBuffer(out).numpy().reshape(heads, d)

    K = kp[table.long()].reshape(-1, kv, d)[:keys].double().cpu().numpy(); V = vp[table.long()].reshape(-1, kv, d)[:keys].double().cpu().numpy()
    Q = q[0].double().cpu().numpy()
    want = np.zeros((heads, d))
    for h in range(heads):
        s = K[:, h // (heads // kv)] @ Q[h] * scale
        p = np.exp(s - s.max())
        want[h] = p / p.sum() @ V[:, h // (heads // kv)]
    assert mixed_err(got, want) <= 1e-4

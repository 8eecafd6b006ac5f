"""Paged decode on a pool of more than 2^31 rows: one K/V head of eight 16-bit elements makes rows of 16 bytes, so such a pool of K and one
of V take 34 GB each.  Blocks below and above the 2^31st row in one table, against a float64 softmax over the gathered cache.

Bound: operands of 16 bits, everything after the load in fp32, some 200 keys: 200 2^-24, held at 1e-4."""
import pytest
import torch

from _util import mixed_err

pytestmark = pytest.mark.gpu


def test_rows_past_31_bits():
    from aidotnet.tensors_amd import Mi355Backend
    heads, d, block, keys = 4, 8, 16, 203
    pool = (1 << 31) // block + 64
    if torch.cuda.mem_get_info()[0] < 3 * pool * block * d * 2:
        pytest.skip("needs 69 GB of device memory")
    be = Mi355Backend(); W = be.WrapTensor
    gen = torch.Generator(device="cuda").manual_seed(3)
    kp, vp = (torch.empty(pool, block, 1, d, dtype=torch.float16, device="cuda") for _ in range(2))
    # (the first ids, the last ones, and the two on either side of the 2^31st row)
    table = torch.tensor([0, pool - 1, 5, (1 << 27) - 1, 1 << 27, pool - 2, 77, pool - 40, (1 << 26) + 3, (1 << 27) + 9, 1, (1 << 27) + 33, 2], dtype=torch.int32, device="cuda")
    for p in (kp, vp):
        p[table.long()] = torch.randn(len(table), block, 1, d, device="cuda", generator=gen).half()
    q = torch.randn(heads, d, device="cuda", generator=gen).half()
    out = be.PagedAttentionHalf("f16", W(q), W(kp), W(vp), W(table), heads, 1, d, block, 1, keys - 1, d ** -0.5)
    got = be.DownloadBuffer(out).double().view(heads, d)
    flat = lambda p: p[table.long()].reshape(-1, d)[:keys].double().cpu()
    want = torch.softmax(q.double().cpu() @ flat(kp).t() * d ** -0.5, -1) @ flat(vp)
    del kp, vp
    torch.cuda.empty_cache()
    assert mixed_err(got.numpy(), want.numpy()) <= 1e-4

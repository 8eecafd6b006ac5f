"""Projection + rotary embedding of few rows over a short K: one launch (the rotation rides on the stores of the 64 x 64 tile), to the bit
what the product followed by the rotation of its leading columns gives."""
import pytest
import torch

from _util import kernels_of

pytestmark = pytest.mark.gpu

# (M, N, K, head_dim, rotated columns, seq_len, start): first and last K-tile of the range, one and many column tiles, all columns and some,
# every row at its own position and all at one
CASES = [(1, 128, 64, 64, 128, 1, 0), (1, 4096, 512, 128, 4096, 1, 4095), (5, 384, 704, 32, 256, 5, 3), (8, 2048, 704, 128, 1920, 2, 7),
         (9, 1024, 960, 64, 1024, 1, 9), (31, 128, 128, 2, 126, 31, 1), (32, 16384, 64, 256, 512, 8, 0), (32, 1024, 960, 64, 64, 16, 100)]


@pytest.mark.parametrize("kind,dt", [("f16", torch.float16), ("bf16", torch.bfloat16)])
@pytest.mark.parametrize("M,N,K,D,cols,seq_len,start", CASES)
def test_one_launch_same_bits(M, N, K, D, cols, seq_len, start, kind, dt):
    from aidotnet.tensors_amd import Mi355Backend
    be = Mi355Backend(); W = be.WrapTensor
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    a = torch.randn(M, K, device="cuda", generator=gen).to(dt)
    b = (torch.randn(K, N, device="cuda", generator=gen) / K ** 0.5).to(dt)
    angle = torch.rand(start + seq_len, D // 2, device="cuda", generator=gen) * 6.28
    cos, sin = torch.cos(angle).contiguous(), torch.sin(angle).contiguous()
    raw = torch.full((M * N + 64,), -7.0, device="cuda", dtype=dt)
    names = kernels_of(lambda: be.GemmRope(kind, W(a), W(b), W(raw), M, N, K, W(cos), W(sin), D, cols, seq_len, start))
    assert len(names) == 1 and names[0].startswith("gemm_dl_kernel") and "GemmRopeArgs" in names[0], names
    plain = torch.empty(M, N, device="cuda", dtype=dt)
    (be.Hgemm if kind == "f16" else be.Bf16Gemm)(W(a), W(b), W(plain), M, N, K)
    want = plain.clone()
    for m in range(M):                                     # (row by row: the rotation kernel takes dense heads at one position)
        head = plain[m, :cols].reshape(cols // D, D).contiguous()
        at = start + m % seq_len
        be.RopeInterleaved(W(head), W(cos), W(sin), W(head), cols // D, D, 1, at, kind)
        want[m, :cols] = head.reshape(cols)
    torch.cuda.synchronize()
    assert torch.equal(raw[:M * N].view(M, N), want) and bool((raw[M * N:] == -7.0).all())


# 33 to 64 rows: the same tile over a short K, and over a long one K ranges whose summing pass takes the rotation
@pytest.mark.parametrize("kind,dt", [("f16", torch.float16), ("bf16", torch.bfloat16)])
@pytest.mark.parametrize("M,N,K,D,cols,seq_len,start,ranges", [(33, 128, 64, 64, 128, 1, 0, False), (48, 512, 512, 128, 384, 1, 77, False), (64, 1024, 704, 64, 1024, 64, 5, False),
                                                               (33, 2048, 2048, 64, 2048, 1, 300, True), (64, 512, 4160, 128, 256, 8, 9, True), (49, 1536, 1792, 128, 1536, 49, 0, True)])
def test_up_to_64_rows_same_bits(M, N, K, D, cols, seq_len, start, ranges, kind, dt):
    from aidotnet.tensors_amd import Mi355Backend
    be = Mi355Backend(); W = be.WrapTensor
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    a = torch.randn(M, K, device="cuda", generator=gen).to(dt)
    b = (torch.randn(K, N, device="cuda", generator=gen) / K ** 0.5).to(dt)
    angle = torch.rand(start + seq_len, D // 2, device="cuda", generator=gen) * 6.28
    cos, sin = torch.cos(angle).contiguous(), torch.sin(angle).contiguous()
    raw = torch.full((M * N + 64,), -7.0, device="cuda", dtype=dt)
    names = kernels_of(lambda: be.GemmRope(kind, W(a), W(b), W(raw), M, N, K, W(cos), W(sin), D, cols, seq_len, start))
    assert len(names) == (2 if ranges else 1) and names[-1].startswith("skinny_reduce_rope_kernel" if ranges else "gemm_dl_kernel"), names
    want = torch.empty(M, N, device="cuda", dtype=dt)
    (be.Hgemm if kind == "f16" else be.Bf16Gemm)(W(a), W(b), W(want), M, N, K)
    for m in range(M):
        head = want[m, :cols].reshape(cols // D, D).contiguous()
        be.RopeInterleaved(W(head), W(cos), W(sin), W(head), cols // D, D, 1, start + m % seq_len, kind)
        want[m, :cols] = head.reshape(cols)
    torch.cuda.synchronize()
    assert torch.equal(raw[:M * N].view(M, N), want) and bool((raw[M * N:] == -7.0).all())

"""The W6A16 tile kernel (rwkv-infer-next_amd/csrc/w6a16.hip) at the edges of its shapes: every row and column tiling, K
shared by few, many and uneven parts, K split over workgroups, ragged columns, and addresses past 32 bits.  Planes and
packed weights give the same bits, within the kernel tolerance of the oracle (tests/test_gpu_int6.py)."""
import numpy as np
import pytest

from gpu_util import say

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from test_gpu_int6 import DEV, F16_KERNEL_TOL, KERNEL_TOL, _act, _check, _dev, _split, _weights  # noqa: E402


@pytest.mark.parametrize("B,M,N,K,g,split", [
    (1, 1, 16, 64, 64, 16),          # one chunk, one column tile
    (1, 8, 80, 192, 64, 16),         # 8 rows staged, three chunks, a ragged unit of columns
    (1, 9, 208, 1088, 64, 16),       # 16 rows staged; 17 chunks over 16 parts; K split over workgroups on the planes
    (2, 5, 64, 16384, 128, 16),      # deep K: 32 parts over two or four workgroups
    (1, 16, 16384, 320, 64, 8),      # the workgroups fill the chip: four parts, five chunks
    (1, 17, 272, 2048, 256, 16),     # two row tiles, the second with one row
    (1, 32, 48, 16384, 128, 32),     # two row tiles, 32 parts
    (1, 40, 64, 16384, 128, 4),      # above 32 rows, K over four workgroups
    (1, 40, 64, 16384, 128, 2),      # over two
    (1, 33, 144, 1024, 128, 1),      # no split
    (1, 40, 640, 3072, 128, 4),      # planes: three chunks a part, K over as few workgroups as hold the parts
    (1, 40, 640, 6144, 128, 4),      # six chunks a part, over four
    (1, 20, 640, 2560, 128, 16),     # up to 32 rows, five chunks a part
    (1, 203, 2560, 320, 64, 2),      # three row tiles, 64 columns
    (1, 64, 16384, 192, 64, 1),      # four row tiles, 64 columns, three chunks
    (1, 203, 10240, 320, 64, 1),     # three row tiles, 128 columns; five chunks over four parts
    (1, 128, 16336, 576, 64, 1),     # four row tiles, 128 columns, nine chunks, columns that end inside a strip
    (1, 40, 16336, 64, 64, 1),       # one chunk: one row tile
    (1, 200, 16336, 128, 64, 1),     # two chunks, many workgroups: two row tiles
    (1, 20, 33024, 576, 64, 1),      # several rounds: two parts, two row tiles
    (1, 128, 33024, 320, 64, 1),     # one part, four row tiles, 128 columns
    (1, 16, 256, 1088, 64, 1),       # 16 parts, 17 chunks
    (1, 3, 32768, 128, 64, 1),       # planes: eight column tiles a wavefront, two parts of one chunk
    (1, 9, 32784, 320, 64, 1),       # the same, columns that end inside a workgroup's
    (1, 9, 32784, 64, 64, 1),        # one part: four column tiles
    (1, 70, 2752, 16384, 128, 4),    # deep K, one round: planes three row tiles over two workgroups, packed two in one
    (1, 190, 1408, 16384, 128, 2),   # planes four row tiles
    (1, 190, 1408, 16384, 128, 1),   # no room for partial tiles: two row tiles
])
@pytest.mark.parametrize("dtype", ["bf16", "f16"])
def test_tile_shapes(B, M, N, K, g, split, dtype):
    from rwkv_next_amd.kernels import int6_gemm as I6
    say("w6a16 tile", dict(B=B, M=M, N=N, K=K, g=g, split=split, dtype=dtype))
    rng = np.random.default_rng(11000 + M + N + K)
    lo, hi, sc = _weights(rng, B, K, N, g)
    a = _act(rng, B, M, K)
    if dtype == "f16":
        a = a.to(torch.float16)
    Ld, Hd, Sd = _dev(lo, hi, sc)
    C = I6.int6_matmul(a.to(DEV), Ld, Hd, Sd, g, split_k=split, out_dtype=torch.float32)
    Cp = I6.int6_matmul(a.to(DEV), I6.prepack_int6(Ld, Hd, Sd, g), split_k=split, out_dtype=torch.float32)
    again = I6.int6_matmul(a.to(DEV), Ld, Hd, Sd, g, split_k=split, out_dtype=torch.float32)
    torch.cuda.synchronize()
    assert torch.equal(C, Cp) and torch.equal(C, again)
    _check(C, a, lo, hi, sc, g, KERNEL_TOL if dtype == "bf16" else F16_KERNEL_TOL)


@pytest.mark.parametrize("B,M,N,K,g,split", [
    (1, 193, 16384, 512, 128, None),   # chains of two chunks, the last rows' group with one row
    (1, 256, 16336, 576, 64, None),    # chains of one, nine chunks, columns that end inside a strip
    (2, 150, 10896, 640, 128, None),   # a batch, five chains
    (1, 200, 16384, 704, 64, 4),       # eleven chunks; a split beside it changes nothing
])
@pytest.mark.parametrize("dtype", ["bf16", "f16"])
def test_wide_kernel(B, M, N, K, g, split, dtype):
    """145..256 rows over so many columns that 64 x 128 tiles go twice around the CUs."""
    from rwkv_next_amd.kernels import int6_gemm as I6
    say("w6a16 wide", dict(B=B, M=M, N=N, K=K, g=g, split=split, dtype=dtype))
    rng = np.random.default_rng(12000 + M + N + K)
    lo, hi, sc = _weights(rng, B, K, N, g)
    a = _act(rng, B, M, K)
    if dtype == "f16":
        a = a.to(torch.float16)
    Ld, Hd, Sd = _dev(lo, hi, sc)
    split = _split(split, B, M, N, K)
    C = I6.int6_matmul(a.to(DEV), Ld, Hd, Sd, g, split_k=split, out_dtype=torch.float32)
    Cp = I6.int6_matmul(a.to(DEV), I6.prepack_int6(Ld, Hd, Sd, g), split_k=split, out_dtype=torch.float32)
    narrow = I6.int6_matmul(a.to(DEV), Ld, Hd, Sd, g, split_k=split)
    torch.cuda.synchronize()
    assert torch.equal(C, Cp) and torch.equal(narrow, C.to(a.dtype))
    _check(C, a, lo, hi, sc, g, KERNEL_TOL if dtype == "bf16" else F16_KERNEL_TOL)


@pytest.mark.parametrize("B,M,N,K,g,split,stride", [
    (2, 3, 80, 256, 64, None, 1 << 24),      # one row tile, as many parts as chunks
    (1, 40, 144, 2048, 128, None, 1 << 24),  # two row tiles
    (1, 3, 64, 16384, 128, 32, 1 << 24),     # 32 parts over two workgroups
    (1, 17, 80, 16384, 128, 32, 1 << 24),    # two row tiles, 32 parts
    (1, 193, 16384, 512, 128, None, 1 << 24),  # the wide kernel
    (1, 200, 16384, 576, 64, None, 1 << 23),   # the wide kernel, rows that span 2 GB in groups that do not
])
def test_rows_far_apart(B, M, N, K, g, split, stride):
    """Row strides of 2^24 elements: a workgroup's rows span more than its buffer's 32-bit offsets reach.  The same bits
    as the same rows side by side."""
    from rwkv_next_amd.kernels import int6_gemm as I6
    say("w6a16 rows far apart", dict(B=B, M=M, N=N, K=K, stride=stride))
    rng = np.random.default_rng(11 + M)
    lo, hi, sc = _weights(rng, B, K, N, g)
    a = _act(rng, B, M, K)
    Ld, Hd, Sd = _dev(lo, hi, sc)
    far = torch.zeros(B * M, stride, dtype=torch.bfloat16, device=DEV)
    far[:, :K] = a.reshape(B * M, K).to(DEV)
    view = far.view(B, M, stride)[:, :, :K]
    pk = I6.prepack_int6(Ld, Hd, Sd, g)
    split = _split(split, B, M, N, K)
    C = I6.int6_matmul(view, Ld, Hd, Sd, g, split_k=split, out_dtype=torch.float32)
    Cp = I6.int6_matmul(view, pk, split_k=split, out_dtype=torch.float32)
    near = I6.int6_matmul(a.to(DEV), pk, split_k=split, out_dtype=torch.float32)
    torch.cuda.synchronize()
    assert torch.equal(C, Cp) and torch.equal(C, near)
    _check(C, a, lo, hi, sc, g, KERNEL_TOL)


@pytest.mark.parametrize("M,N", [
    (2, (1 << 26) + 80),    # the planes' rows of one chunk span more than 2 GB
    (17, (1 << 26) + 80),   # more rows than one row tile
    (2, (1 << 30) + 80),    # and so do the scales of one group
])
def test_planes_past_2_gb(M, N):
    """Columns from both ends and the middle, against the exact product."""
    from rwkv_next_amd.kernels import int6_gemm as I6
    K, g = 64, 64
    if torch.cuda.mem_get_info()[0] < 96 * N:
        pytest.skip("needs 96 bytes a column of device memory")
    say("w6a16 planes past 2 GB", dict(M=M, N=N))
    gen = torch.Generator(device=DEV).manual_seed(12)
    lo = torch.randint(0, 256, (K // 2, N), device=DEV, dtype=torch.uint8, generator=gen)
    hi = torch.randint(0, 256, (K // 4, N), device=DEV, dtype=torch.uint8, generator=gen)
    sc = torch.empty(K // g, N, dtype=torch.float16, device=DEV).uniform_(0.002, 0.05, generator=gen)
    a = torch.randn(M, K, device=DEV, generator=gen).to(torch.bfloat16)
    C = I6.int6_matmul(a, lo, hi, sc, g, out_dtype=torch.float32)
    torch.cuda.synchronize()
    for n0 in (0, N // 32 * 16, N - 256):
        part = [x[:, n0:n0 + 256].cpu().numpy()[None] for x in (lo, hi, sc)]
        _check(C[None, :, n0:n0 + 256], a.cpu()[None], *part, g, KERNEL_TOL)


@pytest.mark.parametrize("packed", [False, True])
def test_rows_beyond_one_launch(monkeypatch, packed):
    """2^28 + 40 rows of one column tile: more workgroups than one launch takes.  65536 rows, over and over, and 40 others
    at the end equal the same rows multiplied alone."""
    from rwkv_next_amd.kernels import int6_gemm as I6
    monkeypatch.setattr(I6, "MAX_M", 1 << 30)
    N, K, g, R = 16, 64, 64, 1 << 16
    M = (1 << 28) + 40
    if torch.cuda.mem_get_info()[0] < 60 << 30:
        pytest.skip("needs 60 GB of device memory")
    say("w6a16 rows beyond one launch", dict(packed=packed))
    gen = torch.Generator(device=DEV).manual_seed(13)
    lo = torch.randint(0, 256, (K // 2, N), device=DEV, dtype=torch.uint8, generator=gen)
    hi = torch.randint(0, 256, (K // 4, N), device=DEV, dtype=torch.uint8, generator=gen)
    sc = (torch.rand(K // g, N, device=DEV, generator=gen) * 0.05 + 0.002).half()
    w = (I6.prepack_int6(lo, hi, sc, g),) if packed else (lo, hi, sc, g)
    base = torch.randn(R, K, device=DEV, generator=gen).to(torch.bfloat16)
    end = torch.randn(40, K, device=DEV, generator=gen).to(torch.bfloat16)
    a = torch.empty(M, K, dtype=torch.bfloat16, device=DEV)
    a[:M - 40].view(-1, R, K).copy_(base)
    a[M - 40:] = end
    C = I6.int6_matmul(a, *w)
    want, last = I6.int6_matmul(base, lo, hi, sc, g), I6.int6_matmul(end, lo, hi, sc, g)
    torch.cuda.synchronize()
    for part in C[:M - 40].view(-1, R, N).split(256):
        assert bool((part == want).all())
    assert torch.equal(C[M - 40:], last)

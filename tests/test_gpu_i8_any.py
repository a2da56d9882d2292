"""int8 products whose sizes, leading dimensions or bases are not multiples of 16
bytes: exact against float64 products (sums below 2^53)."""
import numpy as np
import pytest

import simplang_amd as sa

pytestmark = pytest.mark.gpu

# K around 16, 32 and the 128-deep step, with remainders; N % 4 of 0 to 3, below
# and above a tile; one and several K splits; 128x128 tiles (2049x2055); operands copied to padded rows
# (the last three: 64x64, 128x128 and 256x256 tiles)
SHAPES = [(1, 5, 17), (2, 3, 40), (3, 4, 16), (5, 6, 15), (33, 67, 31), (40, 64, 129), (64, 131, 255),
          (100, 258, 1533), (7, 4099, 1025), (2049, 2055, 100), (129, 130, 143),
          (717, 803, 1001), (1300, 1283, 2601), (4100, 4097, 260)]


@pytest.mark.parametrize("u8", [False, True])
@pytest.mark.parametrize("nt", [False, True])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_any_size_and_alignment(dev, M, N, K, nt, u8):
    import torch
    rng = np.random.default_rng(M + 3 * N + 5 * K)
    lo, dt = (0, np.uint8) if u8 else (-128, np.int8)
    a = rng.integers(lo, lo + 256, (M, K)).astype(dt)
    b = rng.integers(-128, 128, (N, K) if nt else (K, N)).astype(np.int8)
    fn = {(False, False): sa.tensor_matmul_i8, (False, True): sa.matmul_u8s8_i32,
          (True, False): sa.tensor_matmul_nt_i8, (True, True): sa.matmul_nt_u8s8_i32}[nt, u8]
    want = (a.astype(np.float64) @ (b.T if nt else b).astype(np.float64)).astype(np.int64)
    # dense (the last rows end with the allocation), and views with odd pitches
    for off, pad in ((0, 0), (1, 2), (3, 13)) if M < 4000 else ((1, 2),):
        at = torch.zeros(M, K + off + pad, dtype=torch.uint8 if u8 else torch.int8)
        bt = torch.full((b.shape[0], b.shape[1] + off + pad), 77, dtype=torch.int8)
        at[:, off:off + K] = torch.from_numpy(a)
        bt[:, off:off + b.shape[1]] = torch.from_numpy(b)
        c = torch.full((M + 1, N + 1), 9, dtype=torch.int32, device=dev)
        fn(at.to(dev)[:, off:off + K], bt.to(dev)[:, off:off + b.shape[1]], c[:M, :N])
        got = c.cpu().numpy()
        assert np.array_equal(got[:M, :N], want), (off, pad)
        assert (got[M] == 9).all() and (got[:, N] == 9).all()


# both sides of the lines between padded copies and byte-aligned tiles (rows, tiles,
# size of B, K, products), and more k-rows than a grid of copies has blocks for
PADDED = [(79, 8191, 1001), (80, 8191, 1001), (128, 3001, 1401), (160, 3001, 1401), (33, 3199, 8639),
          (33, 2699, 8639), (191, 1001, 6145), (192, 1001, 6145), (160, 6001, 5101), (64, 9001, 9001),
          (65, 9001, 9001), (32, 64, 8390001)]


@pytest.mark.parametrize("nt", [False, True])
@pytest.mark.parametrize("M,N,K", PADDED)
def test_padded_or_not(dev, M, N, K, nt):
    import torch
    g = torch.Generator(device=dev)
    g.manual_seed(M + N + K)
    small = K > 1 << 20  # sums below 2^31
    a = torch.randint(-2 if small else -128, 3 if small else 128, (M, K), dtype=torch.int8, device=dev,
                      generator=g)
    b = torch.randint(-2 if small else -128, 3 if small else 128, (N, K) if nt else (K, N),
                      dtype=torch.int8, device=dev, generator=g)
    c = torch.empty((M, N), dtype=torch.int32, device=dev)
    (sa.tensor_matmul_nt_i8 if nt else sa.tensor_matmul_i8)(a, b, c)
    step = 1 << 20
    want = torch.zeros((M, N), dtype=torch.float64, device=dev)
    for k in range(0, K, step):
        bk = b[:, k:k + step].double().t().contiguous() if nt else b[k:k + step].double()
        want += a[:, k:k + step].double() @ bk
    assert torch.equal(c, want.int())


def test_rows_near_the_index_limit(dev):
    """2^31 - 1 rows of 17 bytes: past what the tiled kernels index, on the generic
    one, whose rows advance in steps of a grid."""
    import torch
    if torch.cuda.get_device_properties(dev).total_memory < 80 << 30:
        pytest.skip("needs 45 GB")
    M = 2 ** 31 - 1
    a = torch.zeros((M, 17), dtype=torch.int8, device=dev)
    rows = torch.tensor([0, 1, 262139, 2 ** 30, M - 262141, M - 2, M - 1], device=dev)
    a[rows] = torch.arange(1, 8, dtype=torch.int8, device=dev)[:, None]
    b = torch.full((1, 17), 3, dtype=torch.int8, device=dev)
    c = torch.full((M, 1), 9, dtype=torch.int32, device=dev)
    sa.tensor_matmul_nt_i8(a, b, c)
    assert torch.equal(c[rows, 0], torch.arange(1, 8, dtype=torch.int32, device=dev) * 51)
    assert int((c != 0).sum()) == 7
    del a, c
    torch.cuda.empty_cache()


def test_any_batch(dev):
    import torch
    rng = np.random.default_rng(1)
    a = rng.integers(-128, 128, (5, 37, 83)).astype(np.int8)
    b = rng.integers(-128, 128, (5, 83, 45)).astype(np.int8)
    c = torch.empty(5, 37, 45, dtype=torch.int32, device=dev)
    sa.tensor_batch_matmul(torch.from_numpy(a).to(dev), torch.from_numpy(b).to(dev), c)
    assert np.array_equal(c.cpu().numpy(), (a.astype(np.float64) @ b.astype(np.float64)).astype(np.int32))


# B_T with K % 128 == 0 and N % 16 != 0, C of any pitch: tiles with and without K
# splits, one round of 64x64 and 128x128 and two, 256x256 streamed and not
NT = [(100, 260, 256, 0), (512, 1028, 1024, 0), (1024, 1028, 1024, 4), (1024, 3205, 3072, 0),
      (2048, 2052, 1024, 1), (2050, 4100, 8192, 0), (4096, 8196, 256, 0), (4100, 5001, 4096, 3),
      (4096, 8192, 2048, 16), (4096, 8192, 2048, 4)]


@pytest.mark.parametrize("u8", [False, True])
@pytest.mark.parametrize("M,N,K,pad", NT)
def test_nt_columns(dev, M, N, K, pad, u8):
    import torch
    g = torch.Generator(device=dev)
    g.manual_seed(M + N + K)
    a = torch.randint(0, 256, (M, K), dtype=torch.uint8, device=dev, generator=g)
    b = torch.randint(-128, 128, (N, K), dtype=torch.int8, device=dev, generator=g)
    a = a if u8 else a.view(torch.int8)
    c = torch.full((M + 1, N + pad), 9, dtype=torch.int32, device=dev)
    (sa.matmul_nt_u8s8_i32 if u8 else sa.tensor_matmul_nt_i8)(a, b, c[:M, :N])
    rows = torch.tensor([0, 1, M // 2, M - 65, M - 1], device=dev)
    cols = torch.tensor([0, 15, N // 2, N - 17, N - 4, N - 1], device=dev)
    bd = b.double().t().contiguous()
    assert torch.equal(c[rows, :N], (a[rows].double() @ bd).int())
    assert torch.equal(c[:M, cols], (a.double() @ bd[:, cols].contiguous()).int())
    assert bool((c[M] == 9).all()) and bool((c[:, N:] == 9).all())

"""fp32 and W4 products on the bf16 matrix cores (gemm_x3.hip) at the edges of
their tiles, K steps and splits, against float64.

Bound, element by element: every operand is exact in its three parts, a dropped
product is below 2^-25 of its term, and an accumulator is rounded at most six
times per 32 products (W4: three times, then once more for the scale) and once
per part of K, each time by at most 2^-24 of what it holds, itself at most
sum |a||b|:  |error| <= (6 K / 32 + 20) 2^-24 sum |a||b|."""
import numpy as np
import pytest

import simplang_amd as sa

pytestmark = pytest.mark.gpu


def _bound(k):
    return (6 * k / 32 + 20) * 2.0 ** -24


def _check(got, a, b):
    want = a @ b
    err = np.abs(got.astype(np.float64) - want)
    lim = _bound(a.shape[1]) * (np.abs(a) @ np.abs(b)) + 2.0 ** -149
    assert (err <= lim).all(), float((err / lim).max())


# M: the 16-, 32-, 64- and 128-row tiles and their remainders; N: 64, 128 and 256
# columns; K: whole steps, remainders, fewer steps than the pipeline holds, K splits
F32 = [(2, 70, 33), (16, 63, 31), (17, 65, 1), (31, 257, 130), (33, 129, 95), (64, 128, 96),
       (65, 2000, 1025), (100, 300, 4097), (301, 203, 257), (129, 64, 2048), (2048, 8200, 70)]


@pytest.mark.parametrize("nt", [False, True])
@pytest.mark.parametrize("M,N,K", F32)
def test_f32_edges(dev, M, N, K, nt):
    import torch
    g = torch.Generator(device=dev)
    g.manual_seed(M * 7 + N * 3 + K)
    # views with odd leading dimensions and bases that are only 4-byte aligned
    a = torch.randn(M, K + 3, device=dev, generator=g)[:, 1:K + 1]
    b = torch.randn(N if nt else K, (K if nt else N) + 3, device=dev, generator=g)[:, 1:-2]
    c = torch.full((M + 1, N + 3), 7.0, device=dev)
    out = c[:M, 1:N + 1]
    (sa.tensor_matmul_nt_f32 if nt else sa.tensor_matmul_f32)(a, b, out)
    torch.cuda.synchronize()
    bd = b.double().cpu().numpy()
    _check(out.cpu().numpy(), a.double().cpu().numpy(), bd.T if nt else bd)
    full = c.cpu().numpy()
    assert (full[M] == 7).all() and (full[:, 0] == 7).all() and (full[:, N + 1:] == 7).all()


@pytest.mark.parametrize("nt", [False, True])
@pytest.mark.parametrize("K", [1, 2, 3])
def test_f32_shortest_sums(dev, K, nt):
    """Sums of up to three products: one rounding each, by at most 2^-24 of what the
    sum holds (K = 1: the rounded product)."""
    import torch
    g = torch.Generator(device=dev)
    g.manual_seed(K)
    a = torch.randn(1024, K + 1, device=dev, generator=g)[:, 1:]
    b = torch.randn(*((1500, K) if nt else (K, 1500)), device=dev, generator=g)
    c = torch.empty(1024, 1500, device=dev)
    (sa.tensor_matmul_nt_f32 if nt else sa.tensor_matmul_f32)(a, b, c)
    bd = b.double().t().contiguous() if nt else b.double()
    lim = K * 2.0 ** -24 * (a.double().abs() @ bd.abs())
    assert bool(((c - a.double() @ bd).abs() <= lim).all())
    if K == 1:
        assert torch.equal(c, a * (b.t() if nt else b))


@pytest.mark.parametrize("M,N,K", [(40, 100, 70), (70, 130, 2050)])
def test_f32_accumulates(dev, M, N, K):
    """``matmul`` adds to its output, with and without K splits."""
    import torch
    rng = np.random.default_rng(M)
    a, b, c0 = (rng.standard_normal(s).astype(np.float32) for s in ((M, K), (K, N), (M, N)))
    c = torch.from_numpy(c0.ravel()).to(dev)
    sa.matmul(torch.from_numpy(a.ravel()).to(dev), torch.from_numpy(b.ravel()).to(dev), c, M, K, N)
    a1 = np.concatenate([a, c0], 1).astype(np.float64)
    b1 = np.concatenate([b.astype(np.float64), np.eye(N)], 0)
    _check(c.cpu().numpy().reshape(M, N), a1, b1)


@pytest.mark.parametrize("scale_a,scale_b", [(1e-38, 1.0), (1e-44, 1e3), (1e33, 1e-30), (3e38, 1e-20)])
def test_f32_range(dev, scale_a, scale_b):
    """The whole fp32 range keeps its precision: subnormals, and values whose
    scaled parts overflow (formed again in fp32)."""
    import torch
    rng = np.random.default_rng(3)
    M, N, K = 50, 70, 100
    with np.errstate(over="ignore"):
        a = (rng.uniform(-1, 1, (M, K)) * scale_a).astype(np.float32)
        b = (rng.uniform(-1, 1, (K, N)) * scale_b).astype(np.float32)
    c = torch.empty(M, N, device=dev)
    sa.tensor_matmul_f32(torch.from_numpy(a).to(dev), torch.from_numpy(b).to(dev), c)
    _check(c.cpu().numpy(), a.astype(np.float64), b.astype(np.float64))


@pytest.mark.parametrize("nt", [False, True])
def test_f32_non_finite(dev, nt):
    """Infinities and NaN go to the outputs that fp32 arithmetic gives them to."""
    import torch
    rng = np.random.default_rng(5)
    M, N, K = 70, 150, 75
    a = rng.standard_normal((M, K)).astype(np.float32)
    b = rng.standard_normal((K, N)).astype(np.float32)
    a[3, 5], a[40, 74], a[69, 0] = np.inf, np.nan, -np.inf
    b[7, 9], b[74, 149] = np.inf, -np.inf
    a[11] = 0.0  # 0 * inf
    b[:, 20] = 1.0  # exact in one part
    with np.errstate(invalid="ignore"):
        want = a.astype(np.float64) @ b.astype(np.float64)
    bt = torch.from_numpy(np.ascontiguousarray(b.T) if nt else b).to(dev)
    c = torch.empty(M, N, device=dev)
    (sa.tensor_matmul_nt_f32 if nt else sa.tensor_matmul_f32)(torch.from_numpy(a).to(dev), bt, c)
    got = c.cpu().numpy()
    fin = np.isfinite(want)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[~fin & ~np.isnan(want)], want[~fin & ~np.isnan(want)])
    with np.errstate(invalid="ignore"):
        lim = _bound(K) * (np.abs(a).astype(np.float64) @ np.abs(b))[fin]
    assert (np.abs(got[fin] - want[fin]) <= lim).all()


W4 = [(1, 70, 32, 32, 4), (2, 129, 96, 32, 4), (5, 300, 288, 96, 4), (16, 127, 256, 64, 4), (17, 128, 64, 64, 0),
      (33, 257, 160, 32, 0), (65, 100, 2048, 128, 0), (129, 1, 96, 32, 0), (200, 8640, 320, 64, 0),
      (8, 1100, 4096, 128, 0)]


@pytest.mark.parametrize("M,N,K,gs,pad", W4)
def test_w4_edges(dev, M, N, K, gs, pad):
    """pad 4: rows of W that are only 4-byte aligned."""
    import torch
    rng = np.random.default_rng(M + N + K)
    w = rng.integers(0, 256, (N, K // 2 + pad)).astype(np.uint8)
    s = np.abs(rng.standard_normal((N, K // gs + 1))).astype(np.float32)
    x = rng.standard_normal((M, K + 1)).astype(np.float32)
    c = torch.full((M + 1, N + 2), 7.0, device=dev)
    out = c[:M, 1:N + 1]
    sa.matmul_w4s(torch.from_numpy(w).to(dev)[:, pad:], torch.from_numpy(s).to(dev)[:, 1:],
                  torch.from_numpy(x).to(dev)[:, 1:], out, gs)
    q = w[:, pad:]
    wd = np.stack([(q << 4).view(np.int8) >> 4, q.view(np.int8) >> 4], -1).reshape(N, K)
    wd = (wd.reshape(N, -1, gs) * s[:, 1:, None].astype(np.float64)).reshape(N, K)
    _check(out.cpu().numpy(), x[:, 1:].astype(np.float64), wd.T)
    full = c.cpu().numpy()
    assert (full[M] == 7).all() and (full[:, 0] == 7).all() and (full[:, N + 1:] == 7).all()


def test_w4_non_finite(dev):
    import torch
    rng = np.random.default_rng(9)
    M, N, K = 40, 200, 128
    w = rng.integers(0, 256, (N, K // 2)).astype(np.uint8)
    w[5] = 0x11  # no zero weight in this row
    s = np.ones((N, K // 32), np.float32)
    x = rng.standard_normal((M, K)).astype(np.float32)
    x[0, 3], x[20, 64], x[39, 127] = np.inf, np.nan, -np.inf
    c = torch.empty(M, N, device=dev)
    sa.matmul_w4s(torch.from_numpy(w).to(dev), torch.from_numpy(s).to(dev),
                  torch.from_numpy(x).to(dev), c, 32)
    wd = np.stack([(w << 4).view(np.int8) >> 4, w.view(np.int8) >> 4], -1).reshape(N, K)
    with np.errstate(invalid="ignore"):
        want = x.astype(np.float64) @ wd.T.astype(np.float64)
    got = c.cpu().numpy()
    fin = np.isfinite(want)
    assert got[0, 5] == np.inf and np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[~fin & ~np.isnan(want)], want[~fin & ~np.isnan(want)])
    lim = _bound(K) * (np.abs(x[1]).astype(np.float64) @ np.abs(wd.T))
    assert (np.abs(got[1] - want[1]) <= lim).all()


# aligned operands, where the dispatch chooses between the split products and the
# fp32 MFMA kernels by their estimated times: sizes on both sides, 16, 30 and more
# K parts, remainders of K, narrow C, one and several rounds of tiles
CHOICE = [(17, 256, 8640), (33, 256, 4096), (64, 256, 8640), (64, 768, 768), (100, 1536, 900),
          (128, 1024, 512), (200, 640, 2048), (256, 512, 132), (300, 3200, 260), (512, 4096, 48),
          (1024, 128, 512), (1500, 1536, 1000), (2048, 32, 2048), (2048, 4096, 160)]


@pytest.mark.parametrize("nt", [False, True])
@pytest.mark.parametrize("M,N,K", CHOICE)
def test_f32_either_kernel(dev, M, N, K, nt):
    import torch
    g = torch.Generator(device=dev)
    g.manual_seed(M + N + K)
    a = torch.randn(M, K, device=dev, generator=g)
    b = torch.randn(*((N, K) if nt else (K, N)), device=dev, generator=g)
    c = torch.full((M + 1, N + 4), 7.0, device=dev)
    (sa.tensor_matmul_nt_f32 if nt else sa.tensor_matmul_f32)(a, b, c[:M, :N])
    bd = b.double().t().contiguous() if nt else b.double()
    want = a.double() @ bd
    # one rounding per product and sum at most (the fp32 MFMA kernels)
    lim = (K + 40) * 2.0 ** -24 * (a.double().abs() @ bd.abs())
    assert bool(((c[:M, :N] - want).abs() <= lim).all())
    assert float((c[:M, :N] - want).norm() / want.norm()) <= 4 * 2.0 ** -24 * max(K, 16) ** 0.5
    assert bool((c[M] == 7).all()) and bool((c[:, N:] == 7).all())

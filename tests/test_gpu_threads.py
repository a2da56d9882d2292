"""Host threads that share a stream (the default: the null stream): products that
stage operands or partial sums in the library's scratch, of different sizes, at
the same time, each against its exact or float64 result."""
import threading

import numpy as np
import pytest

import simplang_amd as sa

pytestmark = pytest.mark.gpu


def _jobs(dev, seed):
    """(call into a fresh output, check) pairs."""
    import torch
    rng = np.random.default_rng(seed)
    put = lambda a: torch.from_numpy(a).to(dev)
    jobs = []
    # int8 of unaligned sizes above 2^29 products: padded copies, then the product
    for m, n, k in ((600 + 16 * seed, 1001, 1003), (777, 1203 + 8 * seed, 901)):
        a = rng.integers(-128, 128, (m, k)).astype(np.int8)
        b = rng.integers(-128, 128, (k, n)).astype(np.int8)
        want = (a.astype(np.float64) @ b.astype(np.float64)).astype(np.int32)
        jobs.append((lambda a=put(a), b=put(b), s=(m, n): sa.tensor_matmul_i8(
            a, b, torch.empty(s, dtype=torch.int32, device=dev)),
            lambda c, want=want: np.array_equal(c, want)))
    # fp32 of unaligned sizes with K parts, and aligned with few rows
    for m, n, k in ((70 + seed, 201, 4099), (8, 512 + 64 * seed, 4096)):
        a = rng.standard_normal((m, k)).astype(np.float32)
        b = rng.standard_normal((k, n)).astype(np.float32)
        want = a.astype(np.float64) @ b
        jobs.append((lambda a=put(a), b=put(b), s=(m, n): sa.tensor_matmul_f32(
            a, b, torch.empty(s, device=dev)),
            lambda c, want=want: np.abs(c - want).max() < 1e-5 * np.abs(want).max()))
    # W4 of 40 rows with K parts, and of 16
    for m, n, k in ((40 + seed, 600, 4096), (16, 800, 4096 + 1024 * seed)):
        w = rng.integers(0, 256, (n, k // 2)).astype(np.uint8)
        s = rng.uniform(0.5, 1, (n, k // 32)).astype(np.float32)
        x = rng.standard_normal((m, k)).astype(np.float32)
        wd = np.stack([(w << 4).view(np.int8) >> 4, w.view(np.int8) >> 4], -1).reshape(n, -1, 32)
        want = x.astype(np.float64) @ (wd * s[:, :, None].astype(np.float64)).reshape(n, k).T
        jobs.append((lambda w=put(w), s=put(s), x=put(x), o=(m, n): sa.matmul_w4s(
            w, s, x, torch.empty(o, device=dev), 32),
            lambda c, want=want: np.abs(c - want).max() < 1e-4 * np.abs(want).max()))
    return jobs


def test_threads_on_one_stream(dev):
    import torch
    stream = sa.lib.simp_rt_get_stream()
    jobs = [_jobs(dev, t) for t in range(3)]
    torch.cuda.synchronize()
    bad, start = [], threading.Barrier(len(jobs))

    def work(t):
        try:
            torch.cuda.set_device(dev)
            sa.set_stream(stream or 0)
            order = np.random.default_rng(t).integers(0, len(jobs[t]), 60)
            start.wait()
            outs = [(int(j), jobs[t][j][0]()) for j in order]
            sa.sync()
            bad.extend((t, i, j) for i, (j, c) in enumerate(outs)
                       if not jobs[t][j][1](c.cpu().numpy()))
        except Exception as e:  # noqa: BLE001 (reported below)
            bad.append((t, repr(e)))

    ts = [threading.Thread(target=work, args=(t,)) for t in range(len(jobs))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad, bad[:5]

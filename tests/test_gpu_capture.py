"""Products recorded into HIP graphs: replays after other calls on the stream,
against the eager results."""
import numpy as np
import pytest

import simplang_amd as sa
from simplang_amd.llama_synth import make_model

pytestmark = pytest.mark.gpu


def _on_side_stream(record):
    """Calls record() eagerly (the warm-up) and then under capture on a stream of
    its own; returns (graph, stream)."""
    import torch
    main, side = torch.cuda.current_stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    sa.set_stream(side)
    try:
        with torch.cuda.stream(side):
            record()
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=side):
            record()
    finally:
        sa.set_stream(main)
    return g, side


def test_graph_survives_larger_calls(dev):
    """A recorded product with K parts (8x2048x2048), replayed after calls on the
    same stream that want more scratch: a larger fp32 product, a W4 product of
    many rows, a prompt through the engine."""
    import torch
    gen = torch.Generator(device=dev)
    gen.manual_seed(3)
    rnd = lambda *s: torch.randn(*s, device=dev, generator=gen)
    a, b, c = rnd(8, 2048), rnd(2048, 2048), torch.empty(8, 2048, device=dev)
    graph, side = _on_side_stream(lambda: sa.tensor_matmul_f32(a, b, c))
    cfg = dict(dim=1024, hidden_dim=2816, n_layers=2, n_heads=8, n_kv_heads=8, vocab_size=512,
               seq_len=256, eps=1e-5, rope_theta=10000.0, weight_format=1, group_size=32)
    engine = sa.Llama(cfg, make_model(cfg, dev, seed=1))
    x, w = rnd(200, 8640), torch.randint(0, 256, (3200, 4320), dtype=torch.uint8, device=dev)
    s, o = torch.rand(3200, 270, device=dev), torch.empty(200, 3200, device=dev)
    la, lb, lc = rnd(16, 4096), rnd(4096, 8192), torch.empty(16, 8192, device=dev)
    others = [lambda: sa.tensor_matmul_f32(la, lb, lc), lambda: sa.matmul_w4s(w, s, x, o, 32),
              lambda: engine.generate(np.arange(200, dtype=np.int32), 1)]
    main = torch.cuda.current_stream()
    want = torch.empty_like(c)
    for rep in range(6):
        a.copy_(rnd(8, 2048))
        torch.cuda.synchronize()
        sa.set_stream(side)
        with torch.cuda.stream(side):
            others[rep % 3]()
            keep = [torch.full((1 << 20,), 7.0, device=dev) for _ in range(4)]
            graph.replay()
            others[(rep + 1) % 3]()
        sa.set_stream(main)
        torch.cuda.synchronize()
        sa.tensor_matmul_f32(a, b, want)
        torch.cuda.synchronize()
        assert torch.equal(c, want), rep
        assert all(bool((k == 7).all()) for k in keep), rep
    engine.close()


# fp32 [K,N] and B_T: K parts of the split products and of the fp32 MFMA kernel,
# no parts, odd; W4 of many rows and of 5 to 16 with long groups; int8 of
# unaligned sizes that are copied to padded rows
F32 = [(100, 2048, 2048), (64, 768, 768), (48, 4096, 4096), (128, 2048, 8640), (128, 8192, 2048),
       (70, 201, 4099), (8, 2048, 2048)]
W4 = [(200, 3200, 1600, 32), (40, 600, 4096, 64), (16, 3200, 4096, 64)]
I8 = [(700, 1003, 1001), (40, 67, 130)]


def _operands(kind, shape, nt, dev, gen):
    import torch
    rnd = lambda *s: torch.randn(*s, device=dev, generator=gen)
    byte = lambda lo, *s, dt=torch.int8: torch.randint(lo, lo + 256, s, dtype=dt, device=dev,
                                                       generator=gen)
    m, n, k = shape[:3]
    if kind == "f32":
        f = sa.tensor_matmul_nt_f32 if nt else sa.tensor_matmul_f32
        return (rnd(m, k), rnd(*((n, k) if nt else (k, n)))), torch.empty(m, n, device=dev), f
    if kind == "w4":
        w, s = byte(0, n, k // 2, dt=torch.uint8), rnd(n, k // shape[3]).abs()
        return ((rnd(m, k), w, s), torch.empty(m, n, device=dev),
                lambda x, w, s, c: sa.matmul_w4s(w, s, x, c, shape[3]))
    f = sa.tensor_matmul_nt_i8 if nt else sa.tensor_matmul_i8
    return ((byte(-128, m, k), byte(-128, *((n, k) if nt else (k, n)))),
            torch.empty(m, n, dtype=torch.int32, device=dev), f)


CASES = ([("f32", s, nt) for s in F32 for nt in (False, True)] + [("w4", s, False) for s in W4]
         + [("i8", s, nt) for s in I8 for nt in (False, True)])


@pytest.mark.parametrize("kind,shape,nt", CASES)
def test_captured_equals_eager(dev, kind, shape, nt):
    """One uncaptured call of the same size on the stream is all that a captured
    call needs, and it runs the same kernels: equal bits, replay after replay."""
    import torch
    gen = torch.Generator(device=dev)
    gen.manual_seed(sum(shape))
    ops, c, f = _operands(kind, shape, nt, dev, gen)
    graph, _ = _on_side_stream(lambda: f(*ops, c))
    want = torch.empty_like(c)
    for rep in range(3):
        new, _, _ = _operands(kind, shape, nt, dev, gen)
        ops[0].copy_(new[0])
        c.zero_()
        torch.cuda.synchronize()
        graph.replay()
        f(*ops, want)
        torch.cuda.synchronize()
        assert torch.equal(c, want), rep


def test_warm_up_of_another_size(dev):
    """A call that leaves little scratch (the larger product has no K parts) before
    a captured one that would like more: captured without parts, not refused."""
    import torch
    gen = torch.Generator(device=dev)
    gen.manual_seed(2)
    big, cb, f = _operands("f32", (2048, 4096, 512), False, dev, gen)
    ops, c, _ = _operands("f32", (100, 1024, 2048), False, dev, gen)
    main, side = torch.cuda.current_stream(), torch.cuda.Stream()
    errors = sa.lib.simp_rt_error_count()
    sa.set_stream(side)
    try:
        f(*big, cb)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=side):
            f(*ops, c)
    finally:
        sa.set_stream(main)
    assert sa.lib.simp_rt_error_count() == errors
    want = ops[0].double() @ ops[1].double()
    for _ in range(2):
        c.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert float((c - want).norm() / want.norm()) < 1e-6

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

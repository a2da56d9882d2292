"""A prompt taken through the layers together (prefill.hip, inside
simp_rt_llama_generate) against the same prompt fed token by token to the step
(simp_rt_llama_forward), which the oracle pins: the logits after the prompt
read every K/V row it left behind.  Both are fp32 with sums in another order;
the bound, 2e-5 of the largest logit, is a fifth of the bound that either
holds against the oracle."""
import numpy as np
import pytest

import simplang_amd as sa
from simplang_amd.llama_synth import make_model, to_numpy

pytestmark = pytest.mark.gpu


def _cfg(**kw):
    c = dict(dim=256, hidden_dim=512, n_layers=3, n_heads=4, n_kv_heads=2, vocab_size=512,
             seq_len=80, eps=1e-5, rope_theta=10000.0, weight_format=0, group_size=32)
    c.update(kw)
    return c


# prompt lengths: the shortest that is batched, 16-row and 64-key edges, the
# whole context; head sizes 32, 36, 64, 100, 128 (batched) and 136 (not)
CASES = [
    (_cfg(), 9), (_cfg(), 17), (_cfg(), 18), (_cfg(), 65), (_cfg(), 79),
    (_cfg(weight_format=1), 10), (_cfg(weight_format=1, group_size=64), 50),
    (_cfg(dim=128, n_heads=4, n_kv_heads=4), 33),
    (_cfg(dim=144, n_heads=4, n_kv_heads=1, hidden_dim=196), 40),
    (_cfg(dim=400, n_heads=4), 40), (_cfg(dim=256, n_heads=2, n_kv_heads=1), 70),
    (_cfg(dim=272, n_heads=2, n_kv_heads=2), 30),
    (_cfg(rope_theta=0.0), 40),
    (_cfg(n_layers=1), 40),
    (_cfg(seq_len=700, n_layers=2), 690),  # more than one pass of 512 rows
]


@pytest.mark.parametrize("cfg,n", CASES)
def test_prompt_equals_steps(dev, cfg, n):
    import torch
    w = make_model(cfg, dev, seed=n)
    prompt = np.random.default_rng(n).integers(0, cfg["vocab_size"], n).astype(np.int32)
    a, b = sa.Llama(cfg, w), sa.Llama(cfg, w)
    la, lb = (torch.empty(cfg["vocab_size"], device=dev) for _ in range(2))
    got = a.generate(prompt, 0)  # all but the last token
    assert np.array_equal(got, prompt)
    a.forward(int(prompt[-1]), n - 1, la)
    for p, t in enumerate(prompt):
        b.forward(int(t), p, lb)
    ga, gb = la.cpu().numpy(), lb.cpu().numpy()
    assert np.abs(ga - gb).max() <= 2e-5 * np.abs(gb).max()
    # the engine goes on from there as from the steps, with and without graphs
    new = min(6, cfg["seq_len"] - n)
    if new:
        t0 = a.generate(prompt, new)
        assert np.array_equal(t0, a.generate(prompt, new, use_graph=False))
        assert t0[n] == int(np.argmax(gb))
    a.close()
    b.close()


@pytest.mark.parametrize("off", [1, 2, 4, 8])
def test_prompt_with_unaligned_w4_weights(dev, off):
    """W4 matrices that start at any byte: the steps take the prompt where the
    row products (4-byte loads) cannot, and generation is the same."""
    import torch
    cfg = _cfg(weight_format=1)
    w = make_model(cfg, dev, seed=5)
    moved = dict(w)
    for k in w:
        if k.startswith("q_w"):
            buf = torch.empty(w[k].numel() + 16, dtype=torch.uint8, device=dev)
            moved[k] = buf[off:off + w[k].numel()]
            moved[k].copy_(w[k].reshape(-1).view(torch.uint8))
            assert moved[k].data_ptr() % 16 == off
    prompt = np.arange(20, dtype=np.int32)
    a, b = sa.Llama(cfg, w), sa.Llama(cfg, moved)
    la, lb = (torch.empty(cfg["vocab_size"], device=dev) for _ in range(2))
    want, got = a.generate(prompt, 6), b.generate(prompt, 6)
    a.forward(int(want[-1]), len(want) - 1, la)
    b.forward(int(want[-1]), len(want) - 1, lb)
    a.close()
    b.close()
    assert np.array_equal(got, want)
    assert float((la - lb).abs().max()) <= 2e-5 * float(la.abs().max())


@pytest.mark.parametrize("fmt", [0, 1])
def test_prompt_against_oracle(dev, orc, fmt):
    """Greedy tokens and the next logits after a 60-token prompt."""
    import torch
    cfg = _cfg(weight_format=fmt, dim=384, n_heads=4)  # head size 96
    w = make_model(cfg, dev, seed=3 + fmt)
    prompt = np.random.default_rng(fmt).integers(0, cfg["vocab_size"], 60).astype(np.int32)
    m = sa.Llama(cfg, w)
    toks = m.generate(prompt, 8)
    lg = torch.empty(cfg["vocab_size"], device=dev)
    m.forward(int(toks[-1]), len(toks) - 1, lg)
    m.close()
    o = orc.LlamaOracle(cfg, to_numpy(w))
    want, seq = None, list(prompt)
    for p in range(len(toks)):
        want = o.forward(int(seq[p]), p)
        if p + 1 >= len(prompt) and p + 1 < len(toks):
            seq.append(orc.argmax(want))
    assert np.array_equal(toks, np.array(seq, np.int32))
    assert np.abs(lg.cpu().numpy() - want).max() <= 1e-4 * np.abs(want).max()

"""The workloads a user of this library runs, as measurable cases.

Each case is one call (or, for the engine, one request) through the public
Python binding on device-resident operands, the way a SimpLang host, a serving
loop or the benchmark calls it.  Kinds:

  norm   rmsnorm / softmax / silu on one vector: the smallest calls of a decode
         step, and the softmax over a vocabulary that sampling needs
  i8     int8 matmul (u8 x s8 or s8 x s8 -> i32), B as [K,N] or transposed: the
         square benchmark shapes, LLaMA projections at 1 to a few thousand rows
         and sizes that are no multiple of anything
  w4     symmetric W4 matmul: 1 row (decode), up to 16 (batched decode),
         hundreds (prompts), groups of 32, 64 or 128
  f32    fp32 matmul, B as [K,N] or transposed: projections of a prompt through
         fp32 weights, aligned and odd
  llama  a request to the decode engine: a prompt, greedily generated tokens,
         then the logits at the next position (fp32 and W4 weights)
"""
import numpy as np
import torch

import simplang_amd as sa
from simplang_amd.llama_synth import CFG_110M, CFG_3B_W4, kv_bytes, make_model, shapes, weight_bytes

DEV = "cuda:0"


def listed():
    return [
        # The attention RMSNorm of the 3B model, one token: the smallest call.
        dict(name="rmsnorm_3200", kind="norm", op="rmsnorm", n=3200),
        # Probabilities over a 32000-token vocabulary, as a sampler needs them.
        dict(name="softmax_32000", kind="norm", op="softmax", n=32000),
        # The reference's own int8 benchmark at its named size.
        dict(name="i8_square_1024", kind="i8", m=1024, n=1024, k=1024, u8=True, nt=False),
        # The headline of the benchmark: the largest square product.
        dict(name="i8_square_8192", kind="i8", m=8192, n=8192, k=8192, u8=True, nt=False),
        # A prompt of odd length through odd layer sizes, both operands signed.
        dict(name="i8_odd_717x2051x1533", kind="i8", m=717, n=2051, k=1533, u8=False, nt=False),
        # Decode: one token through the 3B model's up projection.
        dict(name="w4_1x3200x8640", kind="w4", m=1, n=8640, k=3200, gs=32),
        # Sixteen concurrent requests through the down projection.
        dict(name="w4_16x8640x3200", kind="w4", m=16, n=3200, k=8640, gs=32),
        # A 200-token prompt through the up projection.
        dict(name="w4_200x3200x8640", kind="w4", m=200, n=8640, k=3200, gs=32),
        # A 128-token prompt through an fp32 FFN matrix.
        dict(name="f32_128x2048x8192", kind="f32", m=128, n=8192, k=2048, nt=False),
        # Odd sizes, weights stored one output per row.
        dict(name="f32_nt_301x1537x2003", kind="f32", m=301, n=2003, k=1537, nt=True),
        # A chat request to the fp32 110M model: 200 prompt tokens, 24 new ones.
        dict(name="llama110m_200p_24n", kind="llama", w4=False, dim=768, hidden=2048, layers=12,
             heads=12, kv_heads=12, prompt=200, new=24),
        # The W4 3B benchmark's request: 32 prompt tokens, then generation.
        dict(name="llama3b_w4_32p_32n", kind="llama", w4=True, dim=3200, hidden=8640, layers=26,
             heads=32, kv_heads=32, prompt=32, new=32),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _size(rng, lo, hi, step):
    """Log-uniform in [lo, hi]; two in three rounded to a multiple of step."""
    v = _log(rng, lo, hi)
    return v if rng.random() < 1 / 3 else max(step, v // step * step)


def draw(rng):
    kind = rng.choice(["norm", "i8", "i8", "w4", "w4", "f32", "f32", "llama"])
    if kind == "norm":
        return dict(kind=kind, op=rng.choice(["rmsnorm", "softmax", "silu"]),
                    n=_size(rng, 288, 131072, 64))
    if kind == "i8":
        return dict(kind=kind, m=_log(rng, 1, 4096), n=_size(rng, 256, 8640, 64),
                    k=_size(rng, 256, 8640, 64), u8=rng.random() < 0.5, nt=rng.random() < 0.5)
    if kind == "w4":
        gs = rng.choice([32, 32, 64, 128])
        n, k = _size(rng, 768, 32000, 64), max(768, _log(rng, 768, 8640) // gs * gs)
        # up to 512 rows, and no more work than the largest listed product
        m = min(_log(rng, 1, 512), max(1, 200 * 8640 * 3200 // (n * k)))
        return dict(kind=kind, m=m, n=n, k=k, gs=gs)
    if kind == "f32":
        return dict(kind=kind, m=_log(rng, 1, 2048), n=_size(rng, 256, 8192, 64),
                    k=_size(rng, 256, 8192, 64), nt=rng.random() < 0.5)
    head = rng.choice([64, 96, 100])
    heads = rng.choice([4, 6, 8, 12])
    kv_heads = rng.choice([heads, heads // 2])
    # rows of a W4 matrix are whole groups of 32
    dim = (head if head * heads % 32 == 0 else 64) * heads
    return dict(kind=kind, w4=rng.random() < 0.5, dim=dim,
                hidden=max(256, int(dim * rng.uniform(2.2, 4)) // 32 * 32),
                layers=rng.randint(4, 12), heads=heads, kv_heads=kv_heads,
                prompt=_log(rng, 8, 256), new=rng.randint(8, 32))


def _cfg(case):
    cfg = dict(CFG_3B_W4 if case["w4"] else CFG_110M)
    cfg.update(dim=case["dim"], hidden_dim=case["hidden"], n_layers=case["layers"],
               n_heads=case["heads"], n_kv_heads=case["kv_heads"],
               weight_format=1 if case["w4"] else 0)
    return cfg


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _inputs(case, seed):
    """The device operands of a case, from the seed alone."""
    g = _gen(seed)
    kind = case["kind"]
    if kind == "norm":
        s = dict(x=torch.randn(case["n"], generator=g, device=DEV))
        if case["op"] == "softmax":
            s["x"] *= 4  # the spread of a trained model's logits
        if case["op"] == "rmsnorm":
            s["w"] = 1 + 0.1 * torch.randn(case["n"], generator=g, device=DEV)
        return s
    if kind == "llama":
        s = make_model(_cfg(case), DEV, seed)
        prompt = np.random.default_rng(seed).integers(0, 32000, case["prompt"])
        return s, prompt.astype(np.int32)
    m, n, k = case["m"], case["n"], case["k"]
    if kind == "i8":
        lo, dt = (0, torch.uint8) if case["u8"] else (-128, torch.int8)
        return dict(a=torch.randint(lo, lo + 256, (m, k), dtype=dt, device=DEV, generator=g),
                    b=torch.randint(-128, 128, (n, k) if case["nt"] else (k, n),
                                    dtype=torch.int8, device=DEV, generator=g))
    if kind == "w4":
        return dict(w=torch.randint(0, 256, (n, k // 2), dtype=torch.uint8, device=DEV,
                                    generator=g),
                    s=torch.randn((n, k // case["gs"]), device=DEV, generator=g).abs()
                    * (0.02 / 7),
                    x=torch.randn((m, k), device=DEV, generator=g))
    return dict(a=torch.randn((m, k), device=DEV, generator=g),
                b=torch.randn((n, k) if case["nt"] else (k, n), device=DEV, generator=g) * 0.02)


def prepare(case, seed):
    sa.set_stream(torch.cuda.current_stream())
    kind = case["kind"]
    if kind == "llama":
        w, prompt = _inputs(case, seed)
        cfg = _cfg(case)
        return dict(case=case, prompt=prompt, engine=sa.Llama(cfg, w),
                    logits=torch.empty(cfg["vocab_size"], device=DEV))
    s = dict(case=case, **_inputs(case, seed))
    if kind == "norm":
        s["out"] = torch.empty(case["n"], device=DEV)
    else:
        s["out"] = torch.empty((case["m"], case["n"]), device=DEV,
                               dtype=torch.int32 if kind == "i8" else torch.float32)
    return s


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "norm":
        if case["op"] == "rmsnorm":
            return sa.rmsnorm(state["x"], state["w"], state["out"], case["n"])
        return (sa.softmax if case["op"] == "softmax" else sa.silu)(state["x"], state["out"],
                                                                   case["n"])
    if kind == "i8":
        if case["nt"]:
            f = sa.matmul_nt_u8s8_i32 if case["u8"] else sa.tensor_matmul_nt_i8
        else:
            f = sa.matmul_u8s8_i32 if case["u8"] else sa.tensor_matmul_i8
        return f(state["a"], state["b"], state["out"])
    if kind == "w4":
        return sa.matmul_w4s(state["w"], state["s"], state["x"], state["out"], case["gs"])
    if kind == "f32":
        f = sa.tensor_matmul_nt_f32 if case["nt"] else sa.tensor_matmul_f32
        return f(state["a"], state["b"], state["out"])
    tokens = state["engine"].generate(state["prompt"], case["new"])
    logits = state["engine"].forward(int(tokens[-1]), len(tokens) - 1, state["logits"])
    return dict(tokens=tokens, logits=logits)


def work(case):
    kind = case["kind"]
    if kind == "norm":
        n = case["n"]
        return dict(bytes=(12 if case["op"] == "rmsnorm" else 8) * n, flops=5 * n)
    if kind == "llama":
        cfg = _cfg(case)
        p, new = case["prompt"], case["new"]
        params = sum(int(np.prod(s)) for k, s in shapes(cfg)[0].items() if k != "wcls")
        head = cfg["dim"] * cfg["vocab_size"]
        # one pass over the weights for the prompt, one per generated token; the
        # last of new + 1 steps gives the logits
        return dict(bytes=(new + 1) * weight_bytes(cfg) + sum(kv_bytes(cfg, p + i)
                                                              for i in range(new + 1)),
                    flops=2 * params * (p + new) + 2 * head * (new + 1)
                    + 4 * cfg["n_layers"] * cfg["dim"] * (p + new) * (p + new + 1) // 2)
    m, n, k = case["m"], case["n"], case["k"]
    flops = 2 * m * n * k
    if kind == "i8":
        return dict(bytes=m * k + n * k + 4 * m * n, flops=flops)
    if kind == "w4":
        return dict(bytes=n * k // 2 + 4 * n * k // case["gs"] + 4 * m * k + 4 * m * n,
                    flops=flops)
    return dict(bytes=4 * (m * k + n * k + m * n), flops=flops)


def tolerance(case):
    kind = case["kind"]
    if kind == "i8":
        return "exact"
    # About four times the error against 64-bit arithmetic that one path shows:
    # norms 4e-8 to 7e-8; fp32 products 8e-7 at k = 2048, growing as its root;
    # W4 products 3e-7 (one row) to 7e-6 (sixteen); logits 2e-7 to 6e-7, where
    # rounding travels through all layers and the cache, and a tie may turn a
    # token.
    if kind == "norm":
        return dict(rel=4e-7, max=4e-6)
    if kind == "f32":
        return dict(rel=6e-6, max=6e-5)
    if kind == "w4":
        return dict(rel=2e-5, max=2e-4)
    return dict(rel=1e-5, max=1e-4, differ=0.01)


def _unpack(q, s, gs):
    """W4 rows as float64: low nibble = even column, signed, times its group's scale."""
    v = torch.stack(((q << 4).view(torch.int8) >> 4, q.view(torch.int8) >> 4), -1)
    v = v.reshape(q.shape[0], -1)
    return (v.double().view(q.shape[0], -1, gs) * s.double()[:, :, None]).view(v.shape)


def _rms(x, w, eps):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def _exact_llama(case, seed):
    w, prompt = _inputs(case, seed)
    cfg = _cfg(case)
    dim, heads, kvh, layers = case["dim"], case["heads"], case["kv_heads"], case["layers"]
    hs = dim // heads
    gs = cfg["group_size"]

    def mat(name, layer):
        if not case["w4"]:
            return (w[name][layer] if layer is not None else w[name]).double()
        rows = {"wk": kvh * hs, "wv": kvh * hs, "w1": case["hidden"], "w3": case["hidden"]}
        r = rows.get(name, dim)
        sl = slice(None) if layer is None else slice(layer * r, (layer + 1) * r)
        return _unpack(w["q_" + name][sl], w["s_" + name][sl], gs)

    total = case["prompt"] + case["new"]
    half = torch.arange(0, hs, 2, dtype=torch.float64, device=DEV)
    ang = (torch.arange(total, dtype=torch.float64, device=DEV)[:, None]
           * cfg["rope_theta"] ** (-half / hs))
    rot = torch.polar(torch.ones_like(ang), ang)  # [pos, hs / 2]
    kc = [torch.empty((total, kvh, hs), dtype=torch.float64, device=DEV) for _ in range(layers)]
    vc = [torch.empty_like(k) for k in kc]
    head = mat("wcls", None)

    def rope(v, p0):
        c = torch.view_as_complex(v.reshape(v.shape[0], v.shape[1], hs // 2, 2).contiguous())
        return torch.view_as_real(c * rot[p0:p0 + v.shape[0], None]).reshape(v.shape)

    def step(toks, p0):
        """Logits after the tokens at positions p0 .. p0 + len(toks) - 1."""
        t = len(toks)
        x = w["token_embedding"][torch.as_tensor(toks, device=DEV).long()].double()
        late = (torch.arange(p0 + t, device=DEV)[None, :]
                > torch.arange(p0, p0 + t, device=DEV)[:, None])
        for i in range(layers):
            h = _rms(x, w["rms_att"][i], cfg["eps"])
            q = rope((h @ mat("wq", i).T).view(t, heads, hs), p0)
            kc[i][p0:p0 + t] = rope((h @ mat("wk", i).T).view(t, kvh, hs), p0)
            vc[i][p0:p0 + t] = (h @ mat("wv", i).T).view(t, kvh, hs)
            out = []
            for a in range(heads):
                b = a * kvh // heads
                att = (q[:, a] @ kc[i][:p0 + t, b].T.contiguous()) / hs ** 0.5
                att = torch.softmax(att.masked_fill(late, float("-inf")), -1)
                out.append(att @ vc[i][:p0 + t, b])
            x = x + torch.cat(out, -1) @ mat("wo", i).T
            h = _rms(x, w["rms_ffn"][i], cfg["eps"])
            g = torch.nn.functional.silu(h @ mat("w1", i).T) * (h @ mat("w3", i).T)
            x = x + g @ mat("w2", i).T
        return _rms(x[-1], w["rms_final"], cfg["eps"]) @ head.T

    logits = step(prompt.tolist(), 0)
    for p in range(case["prompt"], total):
        logits = step([int(torch.argmax(logits))], p)
    return dict(tokens=None, logits=logits)


def exact(case, seed):
    kind = case["kind"]
    if kind == "i8":
        return None  # whole numbers: compared bit for bit
    if kind == "llama":
        return _exact_llama(case, seed)
    s = _inputs(case, seed)
    if kind == "norm":
        x = s["x"].double()
        if case["op"] == "rmsnorm":
            return _rms(x, s["w"], 1e-5)
        return torch.softmax(x, 0) if case["op"] == "softmax" else x * torch.sigmoid(x)
    if kind == "w4":
        return s["x"].double() @ _unpack(s["w"], s["s"], case["gs"]).T
    b = s["b"].double()
    return s["a"].double() @ (b.T if case["nt"] else b)

"""The work that a user of this framework has it do, as cases to be timed.

    listed()             the named cases
    draw(rng)            one more case of the ranges that they stand for
    prepare(case, seed)  what a program has in hand before the call
    run(state)           one pass through the public entry points
    work(case)           the bytes and operations that a pass cannot do without
    tolerance(case)      how far another correct implementation's results may be off
    exact(case, seed)    the same results in 64 bits, without the framework

Sizes are those of the package's own workloads (three-llm_amd/weights.py: the
tiny, Qwen2.5-0.5B, Llama-3.2-1B and Llama-3.2-3B shapes) and what lies between
them.  Two cases are whole replies, a prompt and the tokens after it; the others
are the layers those are made of, each through the entry point of its own that a
host program can call.
"""
import ctypes
import importlib.util
import math
import sys
from pathlib import Path

import numpy as np
import torch

ROOT = Path(__file__).resolve().parents[1]


def _package():
    """three-llm_amd/ (a directory name Python cannot spell) as `three_llm_amd`."""
    if "three_llm_amd" not in sys.modules:
        pkg = ROOT / "three-llm_amd"
        spec = importlib.util.spec_from_file_location("three_llm_amd", pkg / "__init__.py",
                                                      submodule_search_locations=[str(pkg)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["three_llm_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["three_llm_amd"]


P = _package()
tlm, W, R = P.tlm, P.weights, P.runner
FMT = {"q4": tlm.FMT_Q4, "f16": tlm.FMT_F16}
BYTES = {"q4": 0.5 + 2.0 / 32, "f16": 2.0}  # per weight

# (query heads, kv heads, head_dim, RoPE theta) of the package's workloads
HEADS = {"tiny": (4, 2, 64, 1e4), "qwen2.5-0.5b": (14, 2, 64, 1e6), "llama-3.2-1b": (32, 8, 64, 5e5),
         "llama-3.2-3b": (24, 8, 128, 5e5)}


def listed():
    return [
        # A chat turn on the smallest real model: a 128-id prompt, then 32 tokens
        # one at a time, each read back by the host as generate() does.
        {"name": "reply qwen 128+32", "kind": "reply", "model": "qwen2.5-0.5b", "prompt": 128, "new": 32},
        # A long document on the 1B shape: 4096 ids in two batched chunks, then
        # tokens over the long window.
        {"name": "reply llama-1b 4096+16", "kind": "reply", "model": "llama-3.2-1b", "prompt": 4096, "new": 16},
        # One token through one projection, the smallest call there is (Qwen's
        # q|k|v rows with their bias): launches and latency.
        {"name": "linear q4 1152x896", "kind": "linear", "fmt": "q4", "n": 1152, "k": 896, "bias": True},
        # One token through the largest MLP (Llama-3.2-3B): weight streaming.
        {"name": "mlp q4 8192x3072", "kind": "mlp", "fmt": "q4", "inner": 8192, "hidden": 3072},
        # Decode attention early in a chat, and far into a long context.
        {"name": "attention qwen @300", "kind": "attention", "heads": "qwen2.5-0.5b", "pos": 300, "window": 0},
        {"name": "attention llama-3b @16384", "kind": "attention", "heads": "llama-3.2-3b", "pos": 16384, "window": 0},
        # The vocabulary: scores and greedy token, then the sampler's candidates.
        {"name": "logits f16 151936x896", "kind": "logits", "fmt": "f16", "n": 151936, "k": 896},
        {"name": "topk 151936 k8", "kind": "topk", "n": 151936, "k": 8, "softcap": 0.0},
        # Prompt rows through one linear: a short prompt (gate|up of the Qwen
        # shape), a full chunk (gate|up of the 1B shape), and fp16 storage (its
        # down projection for a mid-sized prompt).
        {"name": "rows q4 127 9728x896", "kind": "rows", "fmt": "q4", "rows": 127, "n": 9728, "k": 896, "bias": False},
        {"name": "rows q4 2048 16384x2048", "kind": "rows", "fmt": "q4", "rows": 2048, "n": 16384, "k": 2048,
         "bias": False},
        {"name": "rows f16 512 2048x8192", "kind": "rows", "fmt": "f16", "rows": 512, "n": 2048, "k": 8192,
         "bias": False},
        # A full chunk's causal attention on the 1B shape.
        {"name": "attention rows llama-1b 2048", "kind": "attention_rows", "heads": "llama-3.2-1b", "rows": 2048,
         "pos": 0, "window": 0},
    ]


def _log(rng, lo, hi):
    """A whole number, its logarithm uniform over [lo, hi]."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["reply", "linear", "linear", "mlp", "attention", "attention", "logits", "topk", "rows", "rows",
                       "rows", "attention_rows"])
    fmt = rng.choice(["q4", "q4", "f16"])
    # a contraction length: q4 groups are 32 wide, fp16 rows are read 8 at a time
    k = 32 * _log(rng, 8, 256) if fmt == "q4" else 8 * _log(rng, 32, 1024)
    if kind == "reply":
        model = rng.choice(["qwen2.5-0.5b", "llama-3.2-1b"])
        top = 2048 if model == "qwen2.5-0.5b" else 4096
        return {"kind": kind, "model": model, "prompt": _log(rng, 2, top), "new": _log(rng, 1, 16)}
    if kind == "linear":
        return {"kind": kind, "fmt": fmt, "n": _log(rng, 256, 16384), "k": k, "bias": rng.random() < 0.5}
    if kind == "mlp":
        return {"kind": kind, "fmt": fmt, "inner": 32 * _log(rng, 8, 256), "hidden": 32 * _log(rng, 8, 96)}
    if kind == "attention":
        return {"kind": kind, "heads": rng.choice(sorted(HEADS)), "pos": _log(rng, 1, 16384),
                "window": rng.choice([0, 0, 0, 512, 4096])}
    if kind == "logits":
        return {"kind": kind, "fmt": rng.choice(["f16", "f16", "q4"]), "n": _log(rng, 4096, 151936),
                "k": 32 * _log(rng, 8, 64)}
    if kind == "topk":
        return {"kind": kind, "n": _log(rng, 4096, 151936), "k": rng.randint(1, 16),
                "softcap": rng.choice([0.0, 0.0, 30.0])}
    if kind == "rows":  # batched rows need K % 32 == 0 in both formats
        rows, k = _log(rng, 1, 2048), 32 * _log(rng, 8, 256)
        n = _log(rng, 256, 16384)
        return {"kind": kind, "fmt": fmt, "rows": rows, "n": min(n, max(256, (1 << 36) // (rows * k))), "k": k,
                "bias": rng.random() < 0.3}
    heads = rng.choice(["qwen2.5-0.5b", "llama-3.2-1b", "llama-3.2-3b"])
    return {"kind": kind, "heads": heads, "rows": _log(rng, 1, 2048), "pos": rng.choice([0, 0, _log(rng, 1, 2048)]),
            "window": rng.choice([0, 0, 0, 512])}


# ------------------------------------------------------------------ inputs --

class Dev:
    """A torch tensor as the device buffer that the entry points take."""

    def __init__(self, t):
        self.t = t
        self.ptr = ctypes.c_void_p(t.data_ptr())


class State(dict):
    """What a program holds; its handles are closed with it."""

    def __del__(self):
        for v in self.values():
            if isinstance(v, (tlm.Linear, tlm.Attention)):
                v.close()


_ctx = None


def ctx():
    """One device context, as one program has."""
    global _ctx
    if _ctx is None:
        _ctx = tlm.Context(0)
    return _ctx


def _gen(*key):
    g = torch.Generator(device="cuda")
    s = 0x9E3779B9
    for v in key:
        s = (s * 1000003 + int(v) + 1) % (1 << 62)
    g.manual_seed(s)
    return g


def _normal(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32) * std


def _codes(w):
    """4-bit codes and fp16 scales, 32 weights a group (include/tlm.h)."""
    n, k = w.shape
    v = w.view(n, k // 32, 32)
    s = (v.abs().amax(2) / 7).half()
    q = torch.where(s[:, :, None] > 0, (v / s.float()[:, :, None]).round().clamp(-8, 7), torch.zeros_like(v))
    return q, s


def _host(fmt, w):
    """The bytes that a host hands over for fp32 weights [n][k]: (data, scales)."""
    if fmt == "f16":
        return w.half().view(torch.int16).cpu().numpy().view(np.uint16), None
    q, s = _codes(w)
    c = (q + 8).to(torch.uint8).view(w.shape[0], -1, 2)
    return (c[:, :, 0] | (c[:, :, 1] << 4)).cpu().numpy(), s.view(torch.int16).cpu().numpy().view(np.uint16)


def _stored(fmt, w):
    """The values that those bytes stand for, in 64 bits."""
    if fmt == "f16":
        return w.half().double()
    q, s = _codes(w)
    return (q.double() * s.double()[:, :, None]).view(w.shape)


def _linear(fmt, w):
    return tlm.Linear(ctx(), FMT[fmt], *_host(fmt, w))


def _inv_freq(d, theta):
    return (theta ** (-np.arange(0, d, 2, dtype=np.float64) / d)).astype(np.float32)


def _linear_inputs(case, seed):
    """Weights N(0, 0.02), an activation of unit scale, a bias."""
    n, k = case["n"], case["k"]
    w = _normal(_gen(seed, 1), n, k, std=0.02)
    rows = case.get("rows")
    x = _normal(_gen(seed, 2), *((rows, k) if rows else (k,)))
    b = _normal(_gen(seed, 3), n, std=0.1) if case.get("bias") else None
    return w, x.half() if rows else x, b


def _mlp_inputs(case, seed):
    i, h = case["inner"], case["hidden"]
    return (_normal(_gen(seed, 1), 2 * i, h, std=0.02), _normal(_gen(seed, 2), h, i, std=0.02),
            _normal(_gen(seed, 3), h))


def _scores(case, seed):
    return _normal(_gen(seed, 1), case["n"], std=2.0)


CHUNK = 2048


def _qkv(case, seed, chunk):
    """Projected rows of positions [CHUNK chunk, ...): q, k and v of unit scale."""
    hq, hkv, d, _ = HEADS[case["heads"]]
    return _normal(_gen(seed, 10 + chunk), CHUNK, (hq + 2 * hkv) * d)


def _span(case):
    """(first position of the call, positions it computes)."""
    return case["pos"], case.get("rows", 1)


def _attention_state(case, seed):
    hq, hkv, d, theta = HEADS[case["heads"]]
    p0, rows = _span(case)
    # the cache is as long as a program allots: a power of two above the context
    cap = 1 << max(10, (p0 + rows - 1).bit_length())
    a = tlm.Attention(ctx(), hq, hkv, d, cap, inv_freq=_inv_freq(d, theta), sliding_window=case["window"])
    out16 = torch.empty(CHUNK, hq * d, dtype=torch.float16, device="cuda")
    torch.cuda.synchronize()
    for c in range(0, (p0 + CHUNK - 1) // CHUNK):  # the context so far
        x = _qkv(case, seed, c)
        torch.cuda.synchronize()
        a.rows(Dev(x), min(CHUNK, p0 - c * CHUNK), c * CHUNK, Dev(out16))
    qkv = _qkv(case, seed, 1000)[:rows].contiguous()
    y = (torch.zeros(hq * d, device="cuda") if case["kind"] == "attention"
         else torch.zeros(rows, hq * d, dtype=torch.float16, device="cuda"))
    return State(attn=a, qkv=Dev(qkv), y=Dev(y), rows=rows, pos=p0)


# ------------------------------------------------------------- whole models --

CAP = 4224  # positions the models' caches hold
_runners = {}


def _workload(name):
    wl = W.WORKLOADS[name]
    return W.Workload(wl.name, wl.config, wl.storage, wl.prompt_len, wl.decode_len, CAP, wl.qkv_bias)


def _tensor(hw, model, kind, layer):
    """The model's fp32 tensor: matrices N(0, 0.02), norms near one."""
    g = _gen(sorted(W.WORKLOADS).index(model), sum(kind.encode()), layer)
    shape = hw.shape(kind)
    if len(shape) == 2:
        return _normal(g, *shape, std=0.02)
    return 1 + _normal(g, *shape, std=0.05) if "norm" in kind else _normal(g, *shape, std=0.02)


def _weights(model):
    hw = W.synthetic(_workload(model))

    def tensor(kind, layer=0):
        t = _tensor(hw, model, kind, layer)
        fmt = hw.fmt(kind)
        return _host(fmt, t) if fmt != "f32" else (t.cpu().numpy(), None)

    hw.tensor = tensor
    return hw


def _runner(model):
    """A program loads its model once and serves every prompt with it."""
    if model not in _runners:
        _runners[model] = R.DecoderHIPRunner(_weights(model), {"maxTokens": CAP}, ctx=ctx())
    return _runners[model]


def _ids(case, seed):
    """The prompt and the tokens that follow it."""
    vocab = W.WORKLOADS[case["model"]].config["vocab_size"]
    rng = np.random.default_rng([seed, 77])
    return [int(t) for t in rng.integers(0, vocab, case["prompt"] + case["new"] - 1)]


# ------------------------------------------------------------------ the pass --

def prepare(case, seed):
    kind = case["kind"]
    if kind == "reply":
        return State(kind=kind, runner=_runner(case["model"]), ids=_ids(case, seed), prompt=case["prompt"])
    if kind in ("linear", "rows", "logits"):
        w, x, b = _linear_inputs(case, seed)
        s = State(lin=_linear(case["fmt"], w), x=Dev(x), bias=None if b is None else Dev(b))
        rows = case.get("rows")
        s["y"] = Dev(torch.zeros(*((rows, case["n"]) if rows else (case["n"],)), device="cuda"))
        if kind == "rows":
            s["rows"] = rows
        if kind == "logits":
            s["token"] = Dev(torch.zeros(1, dtype=torch.int32, device="cuda"))
    elif kind == "mlp":
        gu, down, x = _mlp_inputs(case, seed)
        s = State(gu=_linear(case["fmt"], gu), down=_linear(case["fmt"], down), x=Dev(x),
                  y=Dev(torch.zeros(case["hidden"], device="cuda")))
    elif kind == "topk":
        s = State(x=Dev(_scores(case, seed)), n=case["n"], k=case["k"], softcap=case["softcap"],
                  tokens=Dev(torch.zeros(case["k"], dtype=torch.int32, device="cuda")),
                  y=Dev(torch.zeros(case["k"], device="cuda")))
    else:
        s = _attention_state(case, seed)
    s["kind"] = kind
    torch.cuda.synchronize()  # the inputs are there before the library's stream reads them
    return s


def run(s):
    kind = s["kind"]
    if kind == "linear":
        return s["lin"](s["x"], s["y"], s["bias"]).t
    if kind == "rows":
        return s["lin"].rows(s["x"], s["rows"], s["y"], s["bias"]).t
    if kind == "mlp":
        return tlm.gated_mlp(s["gu"], s["down"], s["x"], s["y"]).t
    if kind == "logits":
        return {"token": tlm.logits(s["lin"], s["x"], s["y"], s["token"]).t, "logits": s["y"].t}
    if kind == "topk":
        tlm.check(tlm.lib().tlm_op_topk(ctx().ptr, s["x"].ptr, s["n"], s["k"], s["softcap"], s["tokens"].ptr,
                                        s["y"].ptr))
        return {"tokens": s["tokens"].t, "scores": s["y"].t}
    if kind == "attention":
        return s["attn"](s["qkv"], s["pos"], s["y"]).t
    if kind == "attention_rows":
        return s["attn"].rows(s["qkv"], s["rows"], s["pos"], s["y"]).t
    # reply: the prompt without logits, then token by token (given ids, so that
    # a tie in one token does not decide what the next ones are)
    r, ids, last = s["runner"], s["ids"], s["prompt"] - 1
    r.prefillTokens(ids, 0, last)
    for pos in range(last, len(ids)):
        r.computeToken(ids[pos], pos, True)
        r.sampleToken(1, {"temperature": 0})
    return r.readLogits()


# ------------------------------------------------------------------- figures --

def _attended(p0, rows, window):
    """Key positions attended by the queries at p0 .. p0 + rows - 1, in all."""
    return sum(min(p + 1, window) if window else p + 1 for p in range(p0, p0 + rows))


def work(case):
    kind = case["kind"]
    if kind == "reply":
        r = _weights(case["model"]).recipe
        h, i, v, layers = r.hidden_size, r.inner_size, r.vocab_size, r.layer_count
        lin = layers * (h * (r.q_size + 2 * r.kv_size) + r.q_size * h + 3 * h * i)
        kv_row = layers * 2 * r.kv_size * 2
        p, n = case["prompt"] - 1, case["new"]
        # the prompt's rows read the layers once and write their cache rows;
        # every later token reads the layers, the head and the cache
        keys = _attended(p, n, 0)
        byts = (lin * BYTES["q4"] + p * kv_row if p else 0) + n * (lin * BYTES["q4"] + v * h * 2 + v * 4) + keys * kv_row
        flops = 2.0 * lin * (p + n) + 2.0 * v * h * n + 4.0 * r.q_size * layers * _attended(0, p + n, 0)
        return {"bytes": byts, "flops": flops}
    if kind in ("linear", "rows", "logits"):
        rows, n, k = case.get("rows", 1), case["n"], case["k"]
        byts = n * k * BYTES[case["fmt"]] + rows * (k * (2 if "rows" in case else 4) + n * 4)
        return {"bytes": byts + (n * 4 if case.get("bias") else 0), "flops": 2.0 * rows * n * k}
    if kind == "mlp":
        n = 3 * case["inner"] * case["hidden"]
        return {"bytes": n * BYTES[case["fmt"]] + 8 * case["hidden"], "flops": 2.0 * n}
    if kind == "topk":
        return {"bytes": 4 * case["n"] + 8 * case["k"], "flops": case["n"]}
    hq, hkv, d, _ = HEADS[case["heads"]]
    p0, rows = _span(case)
    first = max(0, p0 - case["window"] + 1) if case["window"] else 0
    byts = (p0 - first) * 2 * hkv * d * 2 + rows * ((hq + 2 * hkv) * d * 4 + 2 * hkv * d * 2)
    byts += rows * hq * d * (4 if kind == "attention" else 2)
    return {"bytes": byts, "flops": 4.0 * hq * d * _attended(p0, rows, case["window"])}


def tolerance(case):
    kind = case["kind"]
    if kind == "topk":
        # which scores are the best, and the scores themselves, are no sums; the
        # softcap's tanh is a 32-bit function
        return "exact" if not case["softcap"] else {"rel": 2e-6}
    if kind in ("linear", "mlp", "logits", "attention"):
        return {"rel": 1e-5, "max": 2e-4}  # 32-bit sums (a tie of two logits does not arise: they are not rounded)
    if kind == "rows":
        # q4 weights are rounded to fp16 once (1.8e-4 from 64 bits), the sums are 32-bit
        return {"rel": 8e-4, "max": 8e-3} if case["fmt"] == "q4" else {"rel": 1e-5, "max": 2e-4}
    if kind == "attention_rows":
        return {"rel": 2e-3, "max": 4e-2}  # fp16 queries, probabilities and outputs (4.2e-4 from 64 bits)
    # whole replies: fp16 activations in the prompt's rows and in the q4 dot
    # products of every token, carried through all layers (1.6e-3 from 64 bits;
    # two such roundings differ by more than either is off)
    return {"rel": 1e-2, "max": 0.1}


# ------------------------------------------------------------------- 64 bits --

def _rope(x, p0, inv):
    """Rotate-half RoPE of x [rows][heads][d] at positions p0.."""
    pos = torch.arange(p0, p0 + x.shape[0], device="cuda", dtype=torch.float64)
    ang = pos[:, None] * torch.from_numpy(inv).cuda().double()[None, :]
    c, s = ang.cos()[:, None, :], ang.sin()[:, None, :]
    a, b = x[..., : x.shape[-1] // 2], x[..., x.shape[-1] // 2:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _attend(q, k, v, p0, window, scale):
    """Causal attention of q [rows][hq][d] at positions p0.. over k, v [keys][hkv][d]."""
    rows, hq, d = q.shape
    hkv, keys = k.shape[1], k.shape[0]
    pos = torch.arange(p0, p0 + rows, device="cuda")[:, None]
    key = torch.arange(keys, device="cuda")[None, :]
    hidden = key > pos
    if window:
        hidden |= key <= pos - window
    out = torch.empty(rows, hq, d, dtype=torch.float64, device="cuda")
    for h in range(hq):
        kh, vh = k[:, h // (hq // hkv)].contiguous(), v[:, h // (hq // hkv)].contiguous()
        sc = (q[:, h].contiguous() @ kh.t().contiguous()) * scale
        out[:, h] = torch.softmax(sc.masked_fill(hidden, -math.inf), 1) @ vh
    return out


def _split(x, hq, hkv, d, p0, inv):
    """Projected rows -> rotated q, and the k and v rows as an fp16 cache holds them."""
    x = x.double()
    n = x.shape[0]
    q = _rope(x[:, : hq * d].view(n, hq, d), p0, inv)
    k = _rope(x[:, hq * d: (hq + hkv) * d].view(n, hkv, d), p0, inv)
    return q, k.half().double(), x[:, (hq + hkv) * d:].view(n, hkv, d).half().double()


def _exact_attention(case, seed):
    hq, hkv, d, theta = HEADS[case["heads"]]
    inv = _inv_freq(d, theta)
    p0, rows = _span(case)
    ks, vs = [], []
    for c in range(0, (p0 + CHUNK - 1) // CHUNK):
        _, k, v = _split(_qkv(case, seed, c)[: min(CHUNK, p0 - c * CHUNK)], hq, hkv, d, c * CHUNK, inv)
        ks.append(k)
        vs.append(v)
    q, k, v = _split(_qkv(case, seed, 1000)[:rows], hq, hkv, d, p0, inv)
    o = _attend(q, torch.cat(ks + [k]), torch.cat(vs + [v]), p0, case["window"], d ** -0.5)
    return o.reshape(rows, hq * d) if case["kind"] == "attention_rows" else o.reshape(-1)


def _silu(x):
    return x / (1 + torch.exp(-x))


def _exact_reply(case, seed):
    model = case["model"]
    hw = W.synthetic(_workload(model))
    r = hw.recipe
    hq, hkv, d, theta = HEADS[model]
    inv = _inv_freq(d, theta)
    ids = torch.tensor(_ids(case, seed), device="cuda")

    def mat(kind, layer=0):
        return _stored(hw.fmt(kind), _tensor(hw, model, kind, layer))

    def vec(kind, layer=0):
        return _tensor(hw, model, kind, layer).double()

    def norm(x, w):
        return x * torch.rsqrt(x.square().mean(1, keepdim=True) + r.norm_eps) * w

    emb = _tensor(hw, model, W.EMBED, 0).half()
    x = emb[ids].double()
    for l in range(r.layer_count):
        qkv = norm(x, vec(W.ATTN_NORM, l)) @ mat(W.WQKV, l).t()
        if r.qkv_bias:
            qkv = qkv + vec(W.BQKV, l)
        q, k, v = _split(qkv, hq, hkv, d, 0, inv)
        x = x + _attend(q, k, v, 0, 0, d ** -0.5).reshape(x.shape[0], -1) @ mat(W.WO, l).t()
        n = norm(x, vec(W.FFN_NORM, l))
        x = x + (_silu(n @ mat(W.WGATE, l).t()) * (n @ mat(W.WUP, l).t())) @ mat(W.WDOWN, l).t()
    last = norm(x[-1:], vec(W.FINAL_NORM))[0]
    return torch.cat([part.double() @ last for part in emb.split(16384)])


def exact(case, seed):
    kind = case["kind"]
    if kind == "reply":
        return _exact_reply(case, seed)
    if kind in ("linear", "rows"):
        w, x, b = _linear_inputs(case, seed)
        y = x.double() @ _stored(case["fmt"], w).t()
        return y if b is None else y + b.double()
    if kind == "logits":
        w, x, _ = _linear_inputs(case, seed)
        y = torch.cat([_stored(case["fmt"], part) @ x.double() for part in w.split(16384)])
        return {"token": y.argmax().to(torch.int32).reshape(1), "logits": y}
    if kind == "mlp":
        gu, down, x = _mlp_inputs(case, seed)
        g, u = (_stored(case["fmt"], gu) @ x.double()).chunk(2)
        return _stored(case["fmt"], down) @ (_silu(g) * u)
    if kind == "topk":
        y = _scores(case, seed).double()
        if case["softcap"]:
            y = case["softcap"] * torch.tanh(y / case["softcap"])
        v, i = torch.topk(y, case["k"])
        return {"tokens": i.to(torch.int32), "scores": v}
    return _exact_attention(case, seed)

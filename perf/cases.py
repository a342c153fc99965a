"""The work that programs have jasmine_amd do, as measurable cases through the public C ABI
binding (jasmine_amd.lib / Lm): decoder language models from prompt to tokens, one encoder
layer, and the single operations a program composes (linear layers, attention, expressions
with row normalisations, reductions).  Sizes are those of this repository's configurations,
tests and benchmark.  Device buffers are torch tensors; every call goes to the library's own
stream, as a program that passes no stream does."""
import ctypes as C
import math

import numpy as np
import torch

import jasmine_amd
from jasmine_amd import expr as E
from jasmine_amd.capi import JAS_BF16, JAS_F32, Ins, Leaf, Lm, LmConfig, check, lib

DEV = "cuda"
ACT_NONE, ACT_RELU = 0, 1
GPT2, LLAMA = 0, 1


# ------------------------------------------------------------------ the cases
def _lm(name, kind, layers, d, heads, ff, vocab, batch, prompt, steps, bf16=0):
    return {"name": name, "op": "lm", "kind": kind, "layers": layers, "d": d, "heads": heads, "ff": ff,
            "vocab": vocab, "batch": batch, "prompt": prompt, "steps": steps, "bf16": bf16}


def listed():
    return [
        # one short request to a tiny model: prompt of 32 tokens, 32 greedy tokens, batch 1;
        # every kernel is a few microseconds, so launches and latency are all of it
        _lm("tiny_gpt2_request", GPT2, 2, 128, 4, 512, 256, 1, 32, 31),
        # a batch of 8 requests to a GPT-2-small shape: 512-token prompts, then greedy decode
        # with the KV cache -- the everyday serving call
        _lm("gpt2_small_request", GPT2, 12, 768, 12, 3072, 50257, 8, 512, 31),
        # prompt processing at LLaMA-7B width (one layer and the head): large matrix products
        # and causal attention over two 1024-token prompts, logits of the last position
        _lm("llama_prefill", LLAMA, 1, 4096, 32, 11008, 32000, 2, 1024, 0),
        # the same width stored as bf16 (weights and KV cache), batch 16: 16 short prompts,
        # then decode steps that stream the weights
        _lm("llama_bf16_request", LLAMA, 1, 4096, 32, 11008, 32000, 16, 128, 7, 1),
        # one linear layer / mat_dot_t product, large and square
        {"name": "linear_4096", "op": "linear", "m": 4096, "k": 4096, "t": 4096, "act": ACT_NONE},
        # a feed-forward layer (768 -> 3072, ReLU) on feature-major activations of an odd
        # number of tokens, so that the activations' rows are not 16-byte aligned
        {"name": "linear_ragged", "op": "linear", "m": 3072, "k": 768, "t": 509, "act": ACT_RELU},
        # a Transformer-base encoder layer of the C++ API (512 features, 8 heads, 512 tokens):
        # the kernel sequence its fused heads issue, all of it short launches
        {"name": "encoder_layer", "op": "encoder", "d": 512, "heads": 8, "t": 512},
        # causal attention forward, fp32, GPT-2-small heads
        {"name": "attention_f32", "op": "attention", "b": 8, "h": 12, "s": 1024, "dh": 64, "dtype": "f32", "causal": 1},
        # causal attention forward, bf16 in and out, LLaMA heads over one 2048-token prompt
        {"name": "attention_bf16", "op": "attention", "b": 1, "h": 32, "s": 2048, "dh": 128, "dtype": "bf16", "causal": 1},
        # one decode step's attention over the KV caches of 16 LLaMA-7B sequences of about
        # 2000 tokens, each of its own length
        {"name": "attention_decode", "op": "decode", "b": 16, "h": 32, "dh": 128, "ctx": 2304},
        # the fused expression A*B + 0.5*C - tanh(A) over 8192 x 8192, then row softmax,
        # LayerNorm and RMSNorm of it: pure memory traffic
        {"name": "expression_norms", "op": "expr", "rows": 8192, "cols": 8192},
        # hsum, hmax, vmean and the mean of a whole matrix (losses and statistics)
        {"name": "reductions", "op": "reduce", "rows": 8192, "cols": 8192},
    ]


def _log(rng, lo, hi, step=1):
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(lo, min(hi, (v + step // 2) // step * step))


def draw(rng):
    op = rng.choice(["lm", "lm", "linear", "linear", "encoder", "attention", "attention", "decode", "expr", "reduce"])
    if op == "lm":
        dh = rng.choice([32, 64, 64, 128])
        d = _log(rng, 128, 2048, max(64, dh))
        kind = rng.choice([GPT2, LLAMA])
        steps = rng.choice([0, rng.randint(1, 31)])
        c = _lm("", kind, rng.randint(1, 4), d, d // dh, _log(rng, 256, 8192, 16), _log(rng, 250, 50257),
                rng.randint(1, 16), _log(rng, 16, 512), steps, rng.choice([0, 0, 1]))
    elif op == "linear":
        c = {"op": op, "m": _log(rng, 64, 4096), "k": _log(rng, 64, 4096), "t": _log(rng, 16, 4096),
             "act": rng.choice([ACT_NONE, ACT_RELU])}
        if rng.random() < 0.6:  # feature widths are round numbers more often than not
            c["m"], c["k"] = (c["m"] + 63) // 64 * 64, (c["k"] + 63) // 64 * 64
        if rng.random() < 0.4:
            c["t"] = (c["t"] + 31) // 32 * 32
    elif op == "encoder":
        dh = rng.choice([32, 64, 128])
        d = _log(rng, 256, 1024, dh)
        c = {"op": op, "d": d, "heads": d // dh, "t": _log(rng, 32, 1024)}
    elif op == "attention":
        h = rng.choice([8, 12, 16, 32])
        c = {"op": op, "b": rng.randint(1, 8), "h": h, "s": _log(rng, 64, 1536), "dh": rng.choice([32, 64, 128]),
             "dtype": rng.choice(["f32", "bf16"]), "causal": rng.choice([1, 1, 0])}
    elif op == "decode":
        c = {"op": op, "b": rng.randint(1, 16), "h": rng.choice([8, 12, 16, 32]), "dh": rng.choice([32, 64, 128]),
             "ctx": _log(rng, 64, 2304)}
    else:
        c = {"op": op, "rows": _log(rng, 128, 8192), "cols": _log(rng, 128, 8192)}
    c.pop("name", None)
    return c


# ------------------------------------------------------------------ inputs
def _gen(seed, k):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed * 64 + k)
    return g


def _normal(seed, k, shape, std=1.0, mean=0.0):
    x = torch.randn(shape, generator=_gen(seed, k), device=DEV, dtype=torch.float32)
    return x.mul_(std).add_(mean)


def _shapes(c):
    """Weight tensors of a decoder model: name -> (layers, rows, cols, std, mean, stored as bf16)."""
    n, d, f, v, b = c["layers"], c["d"], c["ff"], c["vocab"], c["bf16"]
    s = {"ln1_g": (n, 1, d, 0.02, 1.0, 0), "ln2_g": (n, 1, d, 0.02, 1.0, 0), "lnf_g": (1, 1, d, 0.02, 1.0, 0),
         "w_qkv": (n, 3 * d, d, 0.02, 0.0, b), "w_o": (n, d, d, 0.02, 0.0, b)}
    if c["kind"] == GPT2:
        s.update({"wte": (1, v, d, 0.02, 0.0, b), "wpe": (1, _ctx(c), d, 0.02, 0.0, 0), "ln1_b": (n, 1, d, 0.02, 0.0, 0),
                  "ln2_b": (n, 1, d, 0.02, 0.0, 0), "lnf_b": (1, 1, d, 0.02, 0.0, 0),
                  "b_qkv": (n, 1, 3 * d, 0.02, 0.0, 0), "b_o": (n, 1, d, 0.02, 0.0, 0),
                  "w_fc": (n, f, d, 0.02, 0.0, b), "b_fc": (n, 1, f, 0.02, 0.0, 0), "w_proj": (n, d, f, 0.02, 0.0, b),
                  "b_proj": (n, 1, d, 0.02, 0.0, 0)})
    else:
        s.update({"wte": (1, v, d, 0.02, 0.0, 0), "w_gate": (n, f, d, 0.02, 0.0, b), "w_up": (n, f, d, 0.02, 0.0, b),
                  "w_down": (n, d, f, 0.02, 0.0, b), "w_head": (1, v, d, 0.02, 0.0, b)})
    return s


def _weights(c, seed):
    """Yields (name, fp32 tensor [layers, rows, cols]); values stored as bf16 are bf16 numbers already."""
    for k, (name, (n, r, cols, std, mean, b)) in enumerate(sorted(_shapes(c).items())):
        w = _normal(seed, k, (n, r, cols), std, mean)
        yield name, w.bfloat16().float() if b else w


def _ctx(c):
    return c["prompt"] + c["steps"] + 1


def _prompt(c, seed):
    return np.random.default_rng(seed).integers(0, c["vocab"], (c["batch"], c["prompt"]), dtype=np.int32)


def _eps(c):
    return 1e-5 if c["kind"] == GPT2 else 1e-6


def _dense_leaf(t):
    r, c = t.shape
    return E.Node("leaf", E.F32, r, c, leaf=Leaf(t.data_ptr(), JAS_F32, r, c, 1, 0, 0, 0, r, c), owner=t)


def _empty(*shape, dtype=torch.float32):
    return torch.empty(shape, device=DEV, dtype=dtype)


def _lens(c, seed):
    lo = max(1, c["ctx"] * 3 // 4)
    lens = np.random.default_rng(seed).integers(lo, c["ctx"] + 1, c["b"], dtype=np.int32)
    lens[0] = c["ctx"]
    return torch.from_numpy(lens).to(DEV)


def prepare(case, seed):
    c = dict(case)
    check(lib.jas_init(0))
    s = {"case": c}
    op = c["op"]
    if op == "lm":
        lm = Lm(LmConfig(c["kind"], c["layers"], c["d"], c["heads"], c["ff"], c["vocab"], _ctx(c), c["batch"], _eps(c),
                         10000.0, c["bf16"], c["bf16"]))
        for name, w in _weights(c, seed):
            lm.set_weight(name, w.cpu().numpy())
        s.update(lm=lm, ids=_prompt(c, seed))
    elif op == "linear":
        s.update(w=_normal(seed, 0, (c["m"], c["k"]), 0.02), x=_normal(seed, 1, (c["k"], c["t"])),
                 b=_normal(seed, 2, (c["m"],), 0.02), y=_empty(c["m"], c["t"]))
    elif op == "encoder":
        d, t = c["d"], c["t"]
        dh = d // c["heads"]
        s.update(x=_normal(seed, 0, (d, t)), wqkv=_normal(seed, 1, (c["heads"], 3 * dh, dh), 0.1),
                 bqkv=_normal(seed, 2, (c["heads"], 3 * dh), 0.02), wo=_normal(seed, 3, (d, d), 0.05),
                 bo=_normal(seed, 4, (d,), 0.02), wf=_normal(seed, 5, (d, d), 0.05), bf=_normal(seed, 6, (d,), 0.02),
                 g1=_normal(seed, 7, (d,), 0.02, 1.0), b1=_normal(seed, 8, (d,), 0.02),
                 g2=_normal(seed, 9, (d,), 0.02, 1.0), b2=_normal(seed, 10, (d,), 0.02),
                 qkv=_empty(t, 3 * d), att=_empty(t, d), r1=_empty(d, t), h=_empty(d, t), r2=_empty(d, t), y=_empty(d, t))
    elif op == "attention":
        shape = (c["b"], c["h"], c["s"], c["dh"])
        dt = torch.float32 if c["dtype"] == "f32" else torch.bfloat16
        s.update({n: _normal(seed, k, shape).to(dt) for k, n in enumerate("qkv")}, o=_empty(*shape, dtype=dt))
    elif op == "decode":
        b, h, dh, ctx = c["b"], c["h"], c["dh"], c["ctx"]
        s.update(q=_normal(seed, 0, (b, h, dh)), k=_normal(seed, 1, (b, h, ctx, dh)), v=_normal(seed, 2, (b, h, ctx, dh)),
                 o=_empty(b, h, dh), lens=_lens(c, seed),
                 work=_empty(max(1, lib.jas_attn_decode_workspace(b, h, dh, ctx) // 4)))
    elif op == "expr":
        shape = (c["rows"], c["cols"])
        a, b, m = (_normal(seed, k, shape) for k in range(3))
        node = _dense_leaf(a)
        tree = node * _dense_leaf(b) + 0.5 * _dense_leaf(m) - E.un("tanh", node)
        prog, leaves = E.lower(tree)
        s.update(tree=tree, prog=(Ins * len(prog))(*[Ins(o, t, g, 0, i) for o, t, g, i in prog]),
                 leaves=(Leaf * len(leaves))(*leaves), d=_empty(*shape), sm=_empty(*shape), ln=_empty(*shape), rms=_empty(*shape))
    else:
        x = _normal(seed, 0, (c["rows"], c["cols"]), 1.0, 0.25)
        s.update(x=x, leaf=_dense_leaf(x).leaf, hsum=_empty(c["rows"], 1), hmax=_empty(c["rows"], 1),
                 vmean=_empty(1, c["cols"]), mean=_empty(1))
    torch.cuda.synchronize()
    return s


# ------------------------------------------------------------------ one pass
def run(s):
    c = s["case"]
    op = c["op"]
    if op == "lm":
        lm, steps = s["lm"], c["steps"]
        if steps == 0:
            first, logits = lm.prefill(s["ids"], want_logits=True)
            return {"first": first, "logits": logits}
        first, _ = lm.prefill(s["ids"])
        ids = lm.generate(steps, c["batch"])
        last, logits = lm.decode(B=c["batch"], want_logits=True)
        return {"first": first, "ids": ids, "last": last, "logits": logits}
    if op == "linear":
        m, k, t = c["m"], c["k"], c["t"]
        check(lib.jas_gemm(m, t, k, s["w"].data_ptr(), k, 1, s["x"].data_ptr(), t, 1, s["y"].data_ptr(), t, 1,
                           s["b"].data_ptr(), 1, c["act"], 0, 1, 0, 0, 0, 0, None))
        return s["y"]
    if op == "encoder":
        d, t, nh = c["d"], c["t"], c["heads"]
        dh = d // nh
        p = {n: v.data_ptr() for n, v in s.items() if isinstance(v, torch.Tensor)}
        check(lib.jas_gemm(3 * dh, t, dh, p["wqkv"], dh, 1, p["x"], t, 1, p["qkv"], 1, 3 * d, p["bqkv"], 1, ACT_NONE, 0, nh,
                           3 * dh * dh, dh * t, 3 * dh, 3 * dh, None))
        check(lib.jas_attn_prefill(p["qkv"], p["qkv"] + 4 * dh, p["qkv"] + 8 * dh, p["att"], 1, nh, t, t, dh, t * 3 * d, 3 * dh,
                                   3 * d, t * 3 * d, 3 * dh, 3 * d, t * d, dh, d, 1.0 / math.sqrt(dh), 0, JAS_F32, None))
        check(lib.jas_gemm_residual(d, t, d, p["wo"], d, 1, p["att"], 1, d, p["r1"], t, 1, p["bo"], 1, ACT_NONE, p["x"], t, 1,
                                    None))
        check(lib.jas_layernorm(p["r1"], p["h"], t, d, 1, 1, t, 0.0, p["g1"], p["b1"], None))
        check(lib.jas_gemm_residual(d, t, d, p["wf"], d, 1, p["h"], t, 1, p["r2"], t, 1, p["bf"], 1, ACT_RELU, p["h"], t, 1,
                                    None))
        check(lib.jas_layernorm(p["r2"], p["y"], t, d, 1, 1, t, 0.0, p["g2"], p["b2"], None))
        return s["y"]
    if op == "attention":
        st = (c["h"] * c["s"] * c["dh"], c["s"] * c["dh"], c["dh"])
        check(lib.jas_attn_prefill(s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(), s["o"].data_ptr(), c["b"], c["h"],
                                   c["s"], c["s"], c["dh"], *st, *st, *st, 1.0 / math.sqrt(c["dh"]), c["causal"],
                                   JAS_F32 if c["dtype"] == "f32" else JAS_BF16, None))
        return s["o"]
    if op == "decode":
        b, h, dh, ctx = c["b"], c["h"], c["dh"], c["ctx"]
        check(lib.jas_attn_decode(s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(), s["o"].data_ptr(),
                                  s["lens"].data_ptr(), b, h, dh, ctx, h * ctx * dh, ctx * dh, 1.0 / math.sqrt(dh),
                                  s["work"].data_ptr(), None))
        return s["o"]
    r, n = c["rows"], c["cols"]
    if op == "expr":
        d = s["d"].data_ptr()
        check(lib.jas_ew_eval(s["prog"], len(s["prog"]), s["leaves"], len(s["leaves"]), d, JAS_F32, r, n, None))
        check(lib.jas_softmax(d, s["sm"].data_ptr(), r, n, n, n, 1, None))
        check(lib.jas_layernorm(d, s["ln"].data_ptr(), r, n, n, n, 1, 1e-5, None, None, None))
        check(lib.jas_rmsnorm(d, s["rms"].data_ptr(), r, n, n, n, 1, 1e-6, None, None))
        return {"d": s["d"], "softmax": s["sm"], "layernorm": s["ln"], "rmsnorm": s["rms"]}
    lf = C.byref(s["leaf"])
    check(lib.jas_reduce(lf, 0, 0, s["hsum"].data_ptr(), JAS_F32, None))
    check(lib.jas_reduce(lf, 1, 0, s["hmax"].data_ptr(), JAS_F32, None))
    check(lib.jas_reduce(lf, 2, 1, s["vmean"].data_ptr(), JAS_F32, None))
    check(lib.jas_reduce(lf, 2, 2, s["mean"].data_ptr(), JAS_F32, None))
    return {"hsum": s["hsum"], "hmax": s["hmax"], "vmean": s["vmean"], "mean": s["mean"]}


# ------------------------------------------------------------------ what a pass cannot do without
def work(case):
    c, op = case, case["op"]
    if op == "lm":
        proj = [v for k, v in _shapes(c).items() if k.startswith("w_") and k != "w_head"]
        per_token = sum(n * r * k for n, r, k, *_ in proj)  # weights each token is multiplied with
        head = c["vocab"] * c["d"]
        es = 2 if c["bf16"] else 4
        passes = 1 + (c["steps"] + 1 if c["steps"] else 0)
        tokens = c["batch"] * (c["prompt"] + passes - 1)
        keys = c["batch"] * sum(c["prompt"] + i for i in range(1, passes))  # cached keys the decode steps read
        causal = c["batch"] * c["prompt"] * (c["prompt"] + 1) // 2
        kv = 2 * c["layers"] * c["d"] * es
        return {"bytes": passes * (per_token + head) * es + kv * (keys + tokens) + 4 * c["batch"] * c["vocab"],
                "flops": 2 * per_token * tokens + 2 * head * c["batch"] * passes + 4 * c["layers"] * c["d"] * (causal + keys)}
    if op == "linear":
        m, k, t = c["m"], c["k"], c["t"]
        return {"bytes": 4 * (m * k + k * t + m * t + m), "flops": 2 * m * k * t}
    if op == "encoder":
        d, t, dh = c["d"], c["t"], c["d"] // c["heads"]
        return {"bytes": 4 * (2 * d * t + 3 * d * dh + 2 * d * d + 9 * d), "flops": 2 * t * (3 * d * dh + 2 * d * d) + 4 * t * t * d}
    if op == "attention":
        es = 4 if c["dtype"] == "f32" else 2
        n = c["b"] * c["h"] * c["s"] * c["dh"]
        pairs = c["s"] * (c["s"] + 1) // 2 if c["causal"] else c["s"] * c["s"]
        return {"bytes": 4 * n * es, "flops": 4 * c["b"] * c["h"] * pairs * c["dh"]}
    if op == "decode":
        keys = int(c["ctx"] * (1 + (c["b"] - 1) * 0.875))  # mean length of the drawn ones: 7/8 of the cache
        return {"bytes": 4 * c["h"] * c["dh"] * (2 * keys + 2 * c["b"]), "flops": 4 * keys * c["h"] * c["dh"]}
    n = c["rows"] * c["cols"]
    if op == "expr":  # three inputs read, four results written
        return {"bytes": 4 * 7 * n, "flops": 20 * n}
    return {"bytes": 4 * (n + 2 * c["rows"] + c["cols"]), "flops": 4 * n}


def tolerance(case):
    op = case["op"]
    if op == "lm":  # whole models: rounding of one layer travels through the next; a rounded
        # bf16 cache entry may fall to either side, and a greedy tie to either token
        return {"rel": 1e-3 if case["bf16"] else 2e-5, "differ": 0.01}
    if op == "attention" and case["dtype"] == "bf16":
        return {"rel": 1e-2}
    return {"rel": 1e-5}


# ------------------------------------------------------------------ the same results in 64 bits
def _norm64(c, x, g, b):
    if c["kind"] == GPT2:
        x = x - x.mean(-1, keepdim=True)
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + _eps(c)) * g + (0 if b is None else b)


def _rope64(x, pos):
    dh = x.shape[-1]
    a = pos[:, None].double() * 10000.0 ** (-2.0 * torch.arange(dh // 2, device=DEV, dtype=torch.float64) / dh)
    cs, sn = torch.cos(a), torch.sin(a)
    x0, x1 = x[..., 0::2], x[..., 1::2]
    return torch.stack((x0 * cs - x1 * sn, x0 * sn + x1 * cs), -1).flatten(-2)


def _step64(c, w, x, cache, pos):
    """x [B, T, d] at positions pos [T] through every layer; cache[l] = (K, V) of the positions before."""
    b, t, d = x.shape
    nh = c["heads"]
    dh = d // nh
    for l in range(c["layers"]):
        lw = lambda n: w[n][l, 0] if w[n].shape[1] == 1 else w[n][l]  # noqa: E731
        lb = lambda n: lw(n) if n in w else None  # noqa: E731
        h = _norm64(c, x, lw("ln1_g"), lb("ln1_b"))
        qkv = h @ lw("w_qkv").T + (lw("b_qkv") if "b_qkv" in w else 0)
        q, k, v = (z.reshape(b, t, nh, dh).transpose(1, 2) for z in qkv.split(d, -1))
        if c["kind"] == LLAMA:
            q, k = _rope64(q, pos), _rope64(k, pos)
        k0, v0 = cache[l] if cache[l] is not None else (k[:, :, :0], v[:, :, :0])
        # a prompt attends over the keys just computed; a bf16 cache keeps them rounded, and a
        # decode step attends over the rounded cache, its own entry included
        kr, vr = (k.float().bfloat16().double(), v.float().bfloat16().double()) if c["bf16"] else (k, v)
        cache[l] = (torch.cat((k0, kr), 2), torch.cat((v0, vr), 2))
        ka, va = (k, v) if k0.shape[2] == 0 else cache[l]
        sc = (q @ ka.transpose(-1, -2)) / math.sqrt(dh)
        if t > 1:
            sc = sc.masked_fill(torch.ones(t, t, device=DEV, dtype=torch.bool).triu(1), -math.inf)
        o = (torch.softmax(sc, -1) @ va).transpose(1, 2).reshape(b, t, d)
        x = x + o @ lw("w_o").T + (lw("b_o") if "b_o" in w else 0)
        h = _norm64(c, x, lw("ln2_g"), lb("ln2_b"))
        if c["kind"] == GPT2:
            u = h @ lw("w_fc").T + lw("b_fc")
            u = 0.5 * u * (1 + torch.tanh(math.sqrt(2 / math.pi) * (u + 0.044715 * u ** 3)))
            x = x + u @ lw("w_proj").T + lw("b_proj")
        else:
            x = x + (torch.nn.functional.silu(h @ lw("w_gate").T) * (h @ lw("w_up").T)) @ lw("w_down").T
    return x


def _lm64(c, seed):
    w = {n: v.double() for n, v in _weights(c, seed)}
    head = w["wte" if c["kind"] == GPT2 else "w_head"][0]
    cache = [None] * c["layers"]
    ids = torch.from_numpy(_prompt(c, seed)).long().to(DEV)

    def logits(ids, start):
        pos = torch.arange(start, start + ids.shape[1], device=DEV)
        x = w["wte"][0][ids]
        if c["kind"] == GPT2:
            x = x + w["wpe"][0][pos]
        x = _step64(c, w, x, cache, pos)[:, -1]
        return _norm64(c, x, w["lnf_g"][0, 0], w["lnf_b"][0, 0] if "lnf_b" in w else None) @ head.T

    lg = logits(ids, 0)
    if c["steps"] == 0:
        return {"first": None, "logits": lg}
    for i in range(c["steps"] + 1):
        lg = logits(lg.argmax(-1, keepdim=True), c["prompt"] + i)
    return {"first": None, "ids": None, "last": None, "logits": lg}


def _attend64(q, k, v, scale, causal):
    out = torch.empty_like(q)
    for b in range(q.shape[0]):  # one batch entry at a time: the scores are held in 64 bits
        sc = (q[b] @ k[b].transpose(-1, -2)) * scale
        if causal:
            sc = sc.masked_fill(torch.ones(sc.shape[-2:], device=DEV, dtype=torch.bool).triu(1), -math.inf)
        out[b] = torch.softmax(sc, -1) @ v[b]
    return out


def _collnorm64(x, g, b):
    z = x - x.mean(0, keepdim=True)
    return z / torch.sqrt((z * z).mean(0, keepdim=True)) * g[:, None] + b[:, None]


def exact(case, seed):
    c, op = dict(case), case["op"]
    if op == "lm":
        return _lm64(c, seed)
    s = prepare(c, seed)
    if op == "linear":
        y = s["w"].double() @ s["x"].double() + s["b"].double()[:, None]
        return y.clamp_min(0) if c["act"] == ACT_RELU else y
    if op == "encoder":
        f = {n: v.double() for n, v in s.items() if isinstance(v, torch.Tensor)}
        d, t, nh = c["d"], c["t"], c["heads"]
        dh = d // nh
        x = f["x"]
        qkv = f["wqkv"] @ x.reshape(nh, dh, t) + f["bqkv"][..., None]  # [heads, 3 dh, t]
        q, k, v = (z.transpose(-1, -2).contiguous()[None] for z in qkv.split(dh, 1))
        o = _attend64(q, k, v, 1.0 / math.sqrt(dh), 0)[0]  # [heads, t, dh]
        h = _collnorm64(f["wo"] @ o.transpose(-1, -2).reshape(d, t) + f["bo"][:, None] + x, f["g1"], f["b1"])
        return _collnorm64((f["wf"] @ h + f["bf"][:, None]).clamp_min(0) + h, f["g2"], f["b2"])
    if op == "attention":
        return _attend64(s["q"].double(), s["k"].double(), s["v"].double(), 1.0 / math.sqrt(c["dh"]), c["causal"])
    if op == "decode":
        out = torch.empty(c["b"], c["h"], c["dh"], device=DEV, dtype=torch.float64)
        for b, n in enumerate(s["lens"].tolist()):
            k, v = s["k"][b, :, :n].double(), s["v"][b, :, :n].double()
            p = torch.softmax((k @ s["q"][b].double()[..., None])[..., 0] / math.sqrt(c["dh"]), -1)
            out[b] = (p[:, None, :] @ v)[:, 0]
        return out
    if op == "expr":
        a, b, m = (_normal(seed, k, (c["rows"], c["cols"])) for k in range(3))
        d = a.double() * b.double() + 0.5 * m.double() - torch.tanh(a.double())
        sm = torch.softmax(d, -1)
        z = d - d.mean(-1, keepdim=True)
        z /= torch.sqrt((z * z).mean(-1, keepdim=True) + 1e-5)
        rms = d / torch.sqrt((d * d).mean(-1, keepdim=True) + 1e-6)
        return {"d": d, "softmax": sm, "layernorm": z, "rmsnorm": rms}
    x = s["x"].double()
    return {"hsum": x.sum(1, keepdim=True), "hmax": x.max(1, keepdim=True).values, "vmean": x.mean(0, keepdim=True),
            "mean": x.mean().reshape(1)}

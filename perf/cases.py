"""Performance cases: the work a program built on zinc_amd has the GPU do.

Kernel-level cases call the C ABI's operations through zinc_amd.Context, with
weights and activations resident on the device and the results left there;
engine-level cases run whole prefill and decode calls and read the logits
back, as a program that samples does. Weights, norms and KV rows come from
the library's seeded synthetic generator, whose definition is restated below
in torch, so exact() can compute every case's result in 64 bits without the
library.

Ranges the cases stand for (draw() samples them):
  dmmv          one-vector mat-vecs, the decode step of one sequence: Q4_K,
                Q6_K, Q8_0, MXFP4; 256..151936 rows, 512..12288 columns
  batched       mat-vecs over 2..16 activation columns (a decode batch), plain
                (Q4_K, Q6_K) and gate/up + SwiGLU (Q4_K)
  gemm          prompt projections over 2..512 tokens, Q4_K and Q6_K
  flash_decode  decode attention over 1..32768 cached tokens through a page table
  attention     causal prompt attention: 1..512 queries after 0..4096 tokens
  decode        greedy decode through an engine, dense and MoE
  prefill       prompts of 2..1024 tokens through an engine
  batch_decode  2..16 sequences in lockstep over one copy of the weights
"""
import math

import numpy as np
import torch

import zinc_amd
from zinc_amd import MXFP4, Q4_K, Q6_K, Q8_0

TYPES = {"Q4_K": Q4_K, "Q6_K": Q6_K, "Q8_0": Q8_0, "MXFP4": MXFP4}
BLOCK = {"Q4_K": (256, 144), "Q6_K": (256, 210), "Q8_0": (32, 34), "MXFP4": (32, 17)}
_DEVICE = "cuda"
HEAD = 128  # head dimension of every model here

# The dense decoder layer of zinc_amd.DENSE_8B and the MoE one of
# zinc_amd.MOE_48L, as cases name them: hidden, q heads, kv heads, FFN rows.
DENSE = dict(hidden=4096, heads=32, kv_heads=8, ffn=12288)
MOE = dict(hidden=2048, heads=32, kv_heads=4, experts=128, used=8, ffn=768)


def listed():
    return [
        # one attention projection of a decode step: the smallest call, where
        # launch and latency count
        dict(name="dmmv_q4k_4096", kind="dmmv", type="Q4_K", rows=4096, cols=4096),
        # a projection whose width is no multiple of 256, in 4-bit floats
        dict(name="dmmv_mxfp4_2880", kind="dmmv", type="MXFP4", rows=2880, cols=2880),
        # the output head over the whole vocabulary: the largest single read
        dict(name="dmmv_q6k_head", kind="dmmv", type="Q6_K", rows=151936, cols=4096),
        # gate and up of a decode batch of six sequences
        dict(name="batched_gate_up_6", kind="batched", op="gate_up", type="Q4_K", rows=12288, cols=4096, vectors=6),
        # one FFN projection of a 512-token prompt chunk
        dict(name="gemm_q4k_512", kind="gemm", type="Q4_K", rows=12288, cols=4096, tokens=512),
        # the down projection of a short, ragged prompt
        dict(name="gemm_q6k_77", kind="gemm", type="Q6_K", rows=4096, cols=12288, tokens=77),
        # one layer's attention late in a long conversation, pages in pool order
        dict(name="flash_decode_32k", kind="flash_decode", heads=32, kv_heads=8, context=32768),
        # one layer's attention of the third chunk of a prompt, ragged at both ends
        dict(name="attention_509_at_1031", kind="attention", heads=32, kv_heads=8, queries=509, start=1031),
        # greedy decode of the whole 8B-shaped model at a 4K context
        dict(name="decode_8b_4k", kind="decode", model="dense", layers=36, vocab=151936, context=4096, tokens=4),
        # greedy decode of MoE layers (128 experts, top 8) at an 8K context
        dict(name="decode_moe_8k", kind="decode", model="moe", layers=4, vocab=8192, context=8192, tokens=4),
        # a 512-token prompt through 8B-shaped layers
        dict(name="prefill_512", kind="prefill", layers=4, vocab=8192, tokens=512),
        # eight sequences decoding in lockstep through 8B-shaped layers
        dict(name="batch_decode_8", kind="batch_decode", layers=8, vocab=8192, context=4096, sequences=8, tokens=8),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["dmmv", "batched", "gemm", "flash_decode", "attention", "decode", "prefill", "batch_decode"])
    if kind == "dmmv":
        t = rng.choice(["Q4_K", "Q6_K", "Q8_0", "MXFP4"])
        unit = 256 if t in ("Q4_K", "Q6_K") else 32
        rows, cols = _log_int(rng, 256, 151936), max(1, _log_int(rng, 512, 12288) // unit) * unit
        return dict(kind=kind, type=t, rows=max(256, min(rows, 151936 * 4096 // cols)), cols=cols)
    if kind == "batched":
        op = rng.choice(["plain", "gate_up"])
        return dict(kind=kind, op=op, type="Q4_K" if op == "gate_up" else rng.choice(["Q4_K", "Q6_K"]),
                    rows=_log_int(rng, 256, 24576), cols=_log_int(rng, 2, 48) * 256, vectors=rng.randint(2, 16))
    if kind == "gemm":
        return dict(kind=kind, type=rng.choice(["Q4_K", "Q6_K"]), rows=_log_int(rng, 256, 12288),
                    cols=_log_int(rng, 4, 48) * 256, tokens=_log_int(rng, 2, 512))
    if kind == "flash_decode":
        return dict(kind=kind, heads=32, kv_heads=rng.choice([4, 8]), context=_log_int(rng, 1, 32768))
    if kind == "attention":
        return dict(kind=kind, heads=32, kv_heads=rng.choice([4, 8]), queries=_log_int(rng, 1, 512),
                    start=rng.choice([0, rng.randint(1, 4096)]))
    if kind == "decode":
        m = rng.choice(["dense", "moe"])
        return dict(kind=kind, model=m, layers=rng.randint(1, 4), vocab=rng.choice([4096, 8192, 32000]),
                    context=_log_int(rng, 16, 16384), tokens=rng.randint(1, 4))
    if kind == "prefill":
        return dict(kind=kind, layers=rng.randint(1, 4), vocab=rng.choice([4096, 8192, 32000]),
                    tokens=_log_int(rng, 2, 1024))
    return dict(kind=kind, layers=rng.randint(1, 4), vocab=rng.choice([4096, 8192, 32000]),
                context=_log_int(rng, 16, 4096), sequences=rng.randint(2, 16), tokens=rng.randint(1, 4))


# ---------------------------------------------------------------------------
# Device state. One context (device + stream) for a program's single-sequence
# work and one for its decode batches, each kept for the process.
# ---------------------------------------------------------------------------
_contexts = {}


def _context(name="solo"):
    if name not in _contexts:
        _contexts[name] = zinc_amd.Context(0)
    return _contexts[name]


class _Buffer(zinc_amd.Buffer):
    """A device buffer given back with its last reference."""

    def __del__(self):
        if getattr(self, "h", None):
            self.free()


class _View:
    """The library's buffer as an array on the device (kept alive by it)."""

    def __init__(self, buf, shape, typestr):
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "version": 2, "strides": None,
                                         "data": (int(buf.device_ptr), False)}


def _tensor(buf, shape, typestr="<f4"):
    return torch.as_tensor(_View(buf, shape, typestr), device=_DEVICE)


class _Engines:
    """An engine and those sharing its weights, destroyed in order."""

    def __init__(self, engines):
        self.engines = engines

    def __del__(self):
        for e in reversed(self.engines):
            e.deinit()


def _upload(ctx, a):
    a = np.ascontiguousarray(a)
    return _Buffer(ctx, a.nbytes).upload(a)


def _weight_bytes(t, rows, cols):
    n, b = BLOCK[t]
    return rows * (cols // n) * b


def _weights(ctx, t, rows, cols, seed, stream):
    buf = _Buffer(ctx, _weight_bytes(t, rows, cols))
    ctx.synth_tensor(buf, 0, TYPES[t] | (0x100 if t == "Q4_K" else 0), rows, cols, seed, stream)
    return buf


def _normals(shape, seed, dtype=np.float32):
    return np.random.default_rng(seed).standard_normal(shape, dtype=np.float32).astype(dtype)


def _pages(n, seed):
    """A page table in the order a used pool hands pages out."""
    return np.random.default_rng(seed).permutation(n).astype(np.uint32)


def _tokens(case, seed, n):
    return np.random.default_rng(seed).integers(0, case["vocab"], n).astype(np.uint32)


def _config(case, seed, context):
    moe = case.get("model") == "moe"
    m = MOE if moe else DENSE
    cfg = dict(zinc_amd.MOE_48L if moe else zinc_amd.DENSE_8B)
    cfg.update(n_layers=case["layers"], hidden=m["hidden"], vocab=case["vocab"], seed=seed,
               max_ctx=(context + 15) // 16 * 16)
    return cfg


def _cache_tokens(n):
    return (n + 15) // 16 * 16


def prepare(case, seed):
    kind = case["kind"]
    ctx = _context("batch" if kind == "batch_decode" else "solo")
    s = {"case": case, "ctx": ctx}
    if kind in ("dmmv", "batched", "gemm"):
        M, K, t = case["rows"], case["cols"], case["type"]
        n = case.get("vectors", case.get("tokens", 1))
        s["W"] = _weights(ctx, t, M, K, seed, 1)
        if case.get("op") == "gate_up":
            s["W2"] = _weights(ctx, t, M, K, seed, 2)
        s["x"] = _upload(ctx, _normals((n, K), seed, np.float16 if kind == "gemm" else np.float32))
        y = _Buffer(ctx, 4 * n * M)
        s["y"], s["out"] = y, _tensor(y, (n, M) if kind != "dmmv" else (M,))
    elif kind in ("flash_decode", "attention"):
        nh, nkv = case["heads"], case["kv_heads"]
        n = case.get("queries", 1)
        total = case["context"] if kind == "flash_decode" else case["start"] + n
        s["cache"] = cache = _cache_tokens(total)
        for which, stream in (("k", 11), ("v", 12)):
            s[which] = _Buffer(ctx, 2 * nkv * cache * HEAD)
            ctx.synth_vector(s[which], 0, 1, nkv * cache * HEAD, 1.0, seed, stream)
        s["pages"] = _upload(ctx, _pages(cache // 16, seed))
        s["q"] = _upload(ctx, _normals((n, nh * HEAD), seed))
        y = _Buffer(ctx, (4 if kind == "flash_decode" else 2) * n * nh * HEAD)
        s["y"] = y
        s["out"] = _tensor(y, (nh * HEAD,)) if kind == "flash_decode" else _tensor(y, (n, nh * HEAD), "<f2")
    elif kind == "decode":
        L = case["context"]
        e = zinc_amd.InferenceEngine(ctx, _config(case, seed, L + case["tokens"]))
        s["engines"] = _Engines([e])
        e.prefill_kv_random(L, seed)
        s["prompt"] = _tokens(case, seed, 1)
    elif kind == "prefill":
        e = zinc_amd.InferenceEngine(ctx, _config(case, seed, case["tokens"]))
        s["engines"] = _Engines([e])
        s["prompt"] = _tokens(case, seed, case["tokens"])
    else:
        L, n = case["context"], case["sequences"]
        e = zinc_amd.InferenceEngine(ctx, _config(case, seed, L + case["tokens"]))
        s["engines"] = _Engines([e] + [e.share(ctx) for _ in range(n - 1)])
        for v, ev in enumerate(s["engines"].engines):
            ev.prefill_kv_random(L, seed + 1000 * v)
        s["prompt"] = _tokens(case, seed, n).reshape(n, 1)
    ctx.sync()
    return s


def run(s):
    case, ctx = s["case"], s["ctx"]
    kind = case["kind"]
    if kind == "dmmv":
        ctx.dmmv(TYPES[case["type"]], s["W"], 0, s["x"], 0, s["y"], 0, case["rows"], case["cols"])
        return s["out"]
    if kind == "batched":
        t, M, K, n = TYPES[case["type"]], case["rows"], case["cols"], case["vectors"]
        if case["op"] == "gate_up":
            ctx.dmmv_fused_gate_up_swiglu_batched(t, s["W"], 0, s["W2"], 0, s["x"], 0, s["y"], 0, M, K, n)
        else:
            ctx.dmmv_batched(t, s["W"], 0, s["x"], 0, s["y"], 0, M, K, n)
        return s["out"]
    if kind == "gemm":
        ctx.gemm_xw(TYPES[case["type"]], s["W"], 0, s["x"], 0, s["y"], 0, case["rows"], case["cols"], case["tokens"])
        return s["out"]
    if kind == "flash_decode":
        ctx.flash_decode(s["q"], s["k"], s["v"], s["pages"], s["cache"] // 16, s["cache"], s["y"], case["heads"],
                         case["kv_heads"], HEAD, case["context"])
        return s["out"]
    if kind == "attention":
        ctx.flash_attn_batched(s["q"], s["k"], s["v"], s["pages"], s["cache"] // 16, s["cache"], s["y"],
                               case["heads"], case["kv_heads"], HEAD, case["start"], case["queries"])
        return s["out"]
    es = s["engines"].engines
    if kind == "decode":
        toks = es[0].generate(s["prompt"], case["tokens"], start_pos=case["context"])
        return {"tokens": np.array(toks, dtype=np.int64), "logits": es[0].logits()}
    if kind == "prefill":
        es[0].prefill(s["prompt"])
        return {"logits": es[0].logits(), "hidden": es[0].hidden()}
    toks = zinc_amd.InferenceEngine.generate_batch(es, s["prompt"], case["tokens"], start_pos=case["context"])
    return {"tokens": np.array(toks, dtype=np.int64), "logits": [e.logits() for e in es]}


def _layer_bytes(moe):
    """Weight bytes a decode step reads of one layer: (projections and norms, FFN)."""
    m = MOE if moe else DENSE
    H, qd, kvd = m["hidden"], m["heads"] * HEAD, m["kv_heads"] * HEAD
    t = "Q8_0" if moe else "Q4_K"
    attn = _weight_bytes(t, qd + 2 * kvd, H) + _weight_bytes(t, H, qd) + 4 * (2 * H + 2 * HEAD)
    if moe:
        return attn, _weight_bytes("Q8_0", m["experts"], H) + m["used"] * 3 * _weight_bytes("Q4_K", m["ffn"], H)
    return attn, 2 * _weight_bytes("Q4_K", m["ffn"], H) + _weight_bytes("Q6_K", H, m["ffn"])


def _layer_macs(moe):
    m = MOE if moe else DENSE
    H, qd, kvd = m["hidden"], m["heads"] * HEAD, m["kv_heads"] * HEAD
    ffn = 3 * m["ffn"] * H * m.get("used", 1) + m.get("experts", 0) * H
    return H * (2 * qd + 2 * kvd) + ffn


def work(case):
    kind = case["kind"]
    if kind in ("dmmv", "batched", "gemm"):
        M, K = case["rows"], case["cols"]
        n = case.get("vectors", case.get("tokens", 1))
        mats = 2 if case.get("op") == "gate_up" else 1
        return {"bytes": mats * _weight_bytes(case["type"], M, K) + n * (K * (2 if kind == "gemm" else 4) + 4 * M),
                "flops": 2.0 * mats * M * K * n}
    if kind == "flash_decode":
        nh, nkv, L = case["heads"], case["kv_heads"], case["context"]
        return {"bytes": 4 * nkv * HEAD * L + 8 * nh * HEAD + L // 4, "flops": 4.0 * nh * HEAD * L}
    if kind == "attention":
        nh, nkv, n, p = case["heads"], case["kv_heads"], case["queries"], case["start"]
        return {"bytes": 4 * nkv * HEAD * (p + n) + 6 * n * nh * HEAD,
                "flops": 4.0 * nh * HEAD * (n * p + n * (n + 1) / 2)}
    moe = case.get("model") == "moe"
    m = MOE if moe else DENSE
    H, V, nl = m["hidden"], case["vocab"], case["layers"]
    attn, ffn = _layer_bytes(moe)
    head = _weight_bytes("Q6_K", V, H) + 4 * V
    kv = 4 * m["kv_heads"] * HEAD  # bytes of one cached token of one layer
    if kind == "prefill":
        n = case["tokens"]
        return {"bytes": nl * (attn + ffn + kv * n) + head + n * _weight_bytes("Q4_K", 1, H),
                "flops": 2.0 * nl * n * _layer_macs(moe) + 2.0 * nl * m["heads"] * HEAD * n * (n + 1) + 2.0 * V * H}
    n, T, L = case.get("sequences", 1), case["tokens"], case["context"]
    ctx = sum(L + t + 1 for t in range(T))
    return {"bytes": T * (nl * (attn + ffn) + head) + n * nl * kv * ctx,
            "flops": 2.0 * n * T * (nl * _layer_macs(moe) + V * H) + 4.0 * n * nl * m["heads"] * HEAD * ctx}


def tolerance(case):
    # about four times each path's distance from exact()
    kind = case["kind"]
    if kind in ("dmmv", "batched"):  # 32-bit sums over a 24-bit image of x: 2.5e-7 .. 4e-7
        return {"rel": 2e-6, "max": 2e-5}
    if kind == "gemm":  # weights rounded to 16 bits, 32-bit sums: 2.1e-4
        return {"rel": 1e-3, "max": 1e-2}
    if kind == "flash_decode":  # 16-bit cache as stored, 32-bit softmax and sums: 3.1e-7
        return {"rel": 2e-6, "max": 2e-5}
    if kind == "attention":  # q, probabilities and result in 16 bits: 3.5e-4
        return {"rel": 1.5e-3, "max": 1.5e-2}
    if kind == "prefill":  # 16-bit operands through every layer: 1.3e-3
        return {"rel": 5e-3, "max": 5e-2}
    # decode: 32-bit rounding grows with the layers it passes: 3.6e-4 after
    # 36, 1.1e-4 after 8, 2.3e-5 after 1
    rel = 1e-4 if case["layers"] == 1 else 5e-5 * case["layers"]
    return {"rel": rel, "max": 10 * rel, "differ": 0.0}


# ---------------------------------------------------------------------------
# The results in 64 bits: the synthetic generator and the block formats in
# torch, then plain float64 arithmetic.
# ---------------------------------------------------------------------------
_M64 = (1 << 64) - 1


def _s64(v):
    v &= _M64
    return v - (1 << 64) if v >> 63 else v


def _shr(z, n):
    return (z >> n) & ((1 << (64 - n)) - 1)


def _mix(z):
    z = (z ^ _shr(z, 30)) * _s64(0xBF58476D1CE4E5B9)
    z = (z ^ _shr(z, 27)) * _s64(0x94D049BB133111EB)
    return z ^ _shr(z, 31)


def _key(seed, stream):
    z = (seed ^ (stream * 0xD1B54A32D192ED03)) & _M64
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & _M64
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & _M64
    return z ^ (z >> 31)


def _rand(key, ctr):
    """64 random bits for each counter of an int64 tensor."""
    return _mix((ctr + 1) * _s64(0x9E3779B97F4A7C15) + _s64(key))


def _normal(r):
    sm = (r & 0xFFFF) + (_shr(r, 16) & 0xFFFF) + (_shr(r, 32) & 0xFFFF) + (_shr(r, 48) & 0xFFFF) - 131070
    return sm.to(torch.float32) * torch.tensor(2.6429573e-05, dtype=torch.float32, device=r.device)


def _scale(r):
    return (_normal(r).abs() * torch.tensor(0.02, dtype=torch.float32, device=r.device)).half()


def _bytes(key, base, first, n):
    """n bytes per block from the words first, first + 1, ... after `base`."""
    w = torch.stack([_rand(key, base + first + i) for i in range((n + 7) // 8)], 1)
    sh = torch.arange(8, device=w.device) * 8
    return ((w[:, :, None] >> sh) & 0xFF).reshape(w.shape[0], -1)[:, :n]


def _rows(t, r0, rows, cols, seed, stream, router=False):
    """Rows r0 .. r0+rows of a synthetic matrix, dequantised, in float64."""
    n, _ = BLOCK[t]
    nb, key = cols // n, _key(seed, stream)
    b = torch.arange(r0 * nb, (r0 + rows) * nb, device=_DEVICE)
    if t == "Q4_K":
        d = _scale(_rand(key, b * 32))
        dmin = (d.float() * 7.5).half().double()
        d = d.double()
        raw = _bytes(key, b * 32, 2, 140)
        s, q = raw[:, :12], raw[:, 12:].reshape(-1, 4, 1, 32)
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1)
        m = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
        q = torch.cat([q & 15, q >> 4], 2).reshape(-1, 8, 32)
        w = (d[:, None] * sc)[:, :, None] * q - (dmin[:, None] * m)[:, :, None]
    elif t == "Q6_K":
        raw = _bytes(key, b * 32, 1, 192)
        d = _scale(_rand(key, b * 32)).double()
        ql, qh = raw[:, :128].reshape(-1, 2, 2, 32), raw[:, 128:].reshape(-1, 2, 32)
        sc = ((_bytes(key, b * 32, 25, 16) & 63) - 32).reshape(-1, 2, 4, 2)
        q = torch.stack([(ql[:, :, g & 1] >> (4 * (g >> 1))) & 15 | ((qh >> (2 * g)) & 3) << 4 for g in range(4)], 2)
        w = (d[:, None, None, None] * sc)[..., None] * (q.reshape(-1, 2, 4, 2, 16) - 32)
    elif t == "Q8_0":
        d = _scale(_rand(key, b * 16))
        if router:  # logits of about unit variance
            d = (d.float() * 2.0 ** -round(math.log2(1.466 * math.sqrt(cols)))).half()
        words = torch.stack([_rand(key, b * 16 + 1 + i) for i in range(8)], 1)
        u = (words[:, :, None] >> (torch.arange(4, device=_DEVICE) * 16)) & 0xFFFF
        w = d.double()[:, None] * (u.reshape(-1, 32) % 255 - 127)
    else:
        r = _rand(key, b * 4)
        e = 118 + (_shr(r, 32) % 13 * ((1 << 32) % 13) + (r & 0xFFFFFFFF) % 13) % 13
        c = _bytes(key, b * 4, 1, 16)
        c = torch.cat([c & 15, c >> 4], 1)
        val = torch.tensor([0, .5, 1, 1.5, 2, 3, 4, 6], dtype=torch.float64, device=_DEVICE)
        val = torch.cat([val, -val])
        w = torch.ldexp(val[c], (e - 127)[:, None])
    return w.reshape(rows, cols)


def _matmul(x, t, rows, cols, seed, stream, r0=0, router=False):
    """x (n, cols) against rows of a synthetic matrix: (n, rows)."""
    step = max(1, (1 << 26) // cols)
    return torch.cat([x @ _rows(t, r0 + r, min(step, rows - r), cols, seed, stream, router).T
                      for r in range(0, rows, step)], 1)


def _vector(kind, n, seed, stream):
    r = _rand(_key(seed, stream), torch.arange(n, device=_DEVICE))
    if kind == 1:
        return _normal(r).half()
    u = ((r & 0xFFFF) - 32768).to(torch.float32)
    return (1.0 + u * torch.tensor(3.0517578e-07, dtype=torch.float32, device=_DEVICE)).double()


def _silu(g):
    return g / (1 + torch.exp(-g))


def _attend(q, k, v, pos):
    """q (n, heads, d) at positions pos (n) over k, v (tokens, kv_heads, d)."""
    nh, nkv = q.shape[1], k.shape[1]
    out = torch.empty_like(q)
    hide = torch.arange(k.shape[0], device=_DEVICE)[None] > pos[:, None]
    for h in range(nh):
        s = q[:, h] @ k[:, h // (nh // nkv)].double().T / math.sqrt(q.shape[2])
        out[:, h] = torch.softmax(s.masked_fill(hide, -math.inf), 1) @ v[:, h // (nh // nkv)].double()
    return out


class _Model:
    """The engine's synthetic model in float64: K and V rows rounded to the
    16 bits they are stored in, everything else unrounded."""

    def __init__(self, case, seed):
        self.moe = case.get("model") == "moe"
        self.m = MOE if self.moe else DENSE
        self.case, self.seed, self.kept = case, seed, {}
        half = HEAD // 2
        base = np.float32(1e6)
        self.inv = torch.tensor(np.array([np.float32(1) / np.power(base, np.float32(2 * i) / np.float32(HEAD))
                                          for i in range(half)], np.float32), device=_DEVICE)

    def weight(self, t, rows, cols, stream, r0=0, router=False):
        k = (stream, r0)
        if k not in self.kept:  # each value is one of 32 bits
            self.kept[k] = _rows(t, r0, rows, cols, self.seed, stream, router).float()
        return self.kept[k].double()

    def norm(self, x, stream):
        k = ("n", stream)
        if k not in self.kept:
            self.kept[k] = _vector(2, x.shape[-1], self.seed, stream)
        return self.kept[k] * (x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6))

    def rope(self, x, pos):
        th = (pos.to(torch.float32)[:, None] * self.inv[None]).double()[:, None]
        a, b = x[..., :HEAD // 2], x[..., HEAD // 2:]
        return torch.cat([a * torch.cos(th) - b * torch.sin(th), a * torch.sin(th) + b * torch.cos(th)], -1)

    def ffn(self, l, x):
        H, F, s = self.m["hidden"], self.m["ffn"], (l + 1) << 8
        if not self.moe:
            h = _silu(x @ self.weight("Q4_K", F, H, s | 9).T) * (x @ self.weight("Q4_K", F, H, s | 10).T)
            return h @ self.weight("Q6_K", H, F, s | 11).T
        logits = x @ self.weight("Q8_0", self.m["experts"], H, s | 12, router=True).T
        out = torch.zeros_like(x)
        for i in range(x.shape[0]):
            top = torch.topk(logits[i], self.m["used"])
            for w, e in zip(torch.softmax(top.values, 0), top.indices.tolist()):
                g = x[i] @ self.weight("Q4_K", F, H, s | 13, e * F).T
                u = x[i] @ self.weight("Q4_K", F, H, s | 14, e * F).T
                out[i] += w * ((_silu(g) * u) @ self.weight("Q4_K", H, F, s | 15, e * H).T)
        return out

    def embed(self, tokens):
        return torch.cat([_rows("Q4_K", int(t), 1, self.m["hidden"], self.seed, 1) for t in tokens])

    def layers(self, tokens, pos, caches):
        """tokens (n) at positions pos. caches[l][i]: (k, v) of the sequence
        that token i belongs to, its own row already made room for."""
        m, case = self.m, self.case
        H, nh, nkv = m["hidden"], m["heads"], m["kv_heads"]
        t = "Q8_0" if self.moe else "Q4_K"
        x = self.embed(tokens)
        n = x.shape[0]
        for l in range(case["layers"]):
            s = (l + 1) << 8
            a = self.norm(x, s | 1)
            q = self.norm((a @ self.weight(t, nh * HEAD, H, s | 2).T).view(n, nh, HEAD), s | 6)
            k = self.norm((a @ self.weight(t, nkv * HEAD, H, s | 3).T).view(n, nkv, HEAD), s | 7)
            v = (a @ self.weight(t, nkv * HEAD, H, s | 4).T).view(n, nkv, HEAD)
            q, k, v = self.rope(q, pos), self.rope(k, pos).half(), v.half()
            o = torch.empty_like(q)
            if case["kind"] == "prefill":
                o = _attend(q, k, v, pos)
            else:
                for i in range(n):
                    kc, vc = caches[l][i]
                    kc[pos[i]], vc[pos[i]] = k[i], v[i]
                    o[i:i + 1] = _attend(q[i:i + 1], kc, vc, pos[i:i + 1])
            x = x + o.reshape(n, nh * HEAD) @ self.weight(t, H, nh * HEAD, s | 5).T
            x = x + self.ffn(l, self.norm(x, s | 8))
        return x

    def head(self, x):
        H, V = self.m["hidden"], self.case["vocab"]
        return self.norm(x, 2) @ self.weight("Q6_K", V, H, 3).T

    def cache(self, l, kv_seed):
        """A layer's pre-filled (k, v), with room for the decoded tokens."""
        nkv, L = self.m["kv_heads"], self.case["context"]
        got = []
        for which in (0, 1):
            c = torch.zeros(L + self.case["tokens"], nkv, HEAD, dtype=torch.float16, device=_DEVICE)
            r = _rand(_key(kv_seed, 0x100000 + 2 * l + which), torch.arange(L * nkv * HEAD, device=_DEVICE))
            c[:L] = _normal(r).half().view(L, nkv, HEAD)
            got.append(c)
        return tuple(got)


def _cached(flat, nkv, cache, pages, n):
    """Tokens 0 .. n-1 of a paged [kv_heads][cache][d] cache, token-major."""
    t = torch.arange(n, device=_DEVICE)
    phys = torch.tensor(pages.astype(np.int64), device=_DEVICE)[t // 16] * 16 + t % 16
    return flat.view(nkv, cache, HEAD)[:, phys].transpose(0, 1)


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    if kind in ("dmmv", "batched", "gemm"):
        M, K, t = case["rows"], case["cols"], case["type"]
        n = case.get("vectors", case.get("tokens", 1))
        x = torch.tensor(_normals((n, K), seed, np.float16 if kind == "gemm" else np.float32), device=_DEVICE).double()
        y = _matmul(x, t, M, K, seed, 1)
        if case.get("op") == "gate_up":
            y = _silu(y) * _matmul(x, t, M, K, seed, 2)
        return y if kind != "dmmv" else y[0]
    if kind in ("flash_decode", "attention"):
        nh, nkv = case["heads"], case["kv_heads"]
        n = case.get("queries", 1)
        total = case["context"] if kind == "flash_decode" else case["start"] + n
        cache = _cache_tokens(total)
        pages = _pages(cache // 16, seed)
        k, v = (_cached(_vector(1, nkv * cache * HEAD, seed, st), nkv, cache, pages, total) for st in (11, 12))
        q = torch.tensor(_normals((n, nh * HEAD), seed), device=_DEVICE).double().view(n, nh, HEAD)
        y = _attend(q, k, v, torch.arange(total - n, total, device=_DEVICE)).reshape(n, nh * HEAD)
        return y if kind == "attention" else y[0]
    model = _Model(case, seed)
    if kind == "prefill":
        n = case["tokens"]
        x = model.layers(_tokens(case, seed, n), torch.arange(n, device=_DEVICE), None)[-1:]
        return {"logits": model.head(x)[0], "hidden": x[0]}
    n = case.get("sequences", 1)
    caches = [[model.cache(l, seed + 1000 * v) for v in range(n)] for l in range(case["layers"])]
    tokens, got = _tokens(case, seed, n), []
    for step in range(case["tokens"]):
        pos = torch.full((n,), case["context"] + step, device=_DEVICE)
        logits = model.head(model.layers(tokens, pos, caches))
        tokens = logits.argmax(1).cpu().numpy()
        got.append(tokens)
    if kind == "decode":
        return {"tokens": None, "logits": logits[0]}
    return {"tokens": None, "logits": [row for row in logits]}

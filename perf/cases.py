"""Timed workloads of the attention path, through the ``ema_attn`` Python binding.

Each case is one piece of work that a serving program has this library do: the attention
layers of one decoded token, a batched decode step over each cache format, a prompt or a
chunk of one, the quantised projections at decode and prompt sizes, and the Gated DeltaNet
step and scan. ``listed()`` holds fixed sizes, ``draw()`` others of the same ranges,
``exact()`` the same results from plain torch in float64.

Kinds (the ``kind`` field):

``token``    attention of one decoded token in every layer of a model: q|k|v projection,
             fused decode step, o projection per layer, each layer with its own weights and
             cache. Captured in a HIP graph once and replayed, as a decode loop does.
``step``     one fused decode step (q/k norm, RoPE, K/V row written, attention) of a batch.
``prefill``  pre-attention and causal prefill of a chunk at an offset into the cache.
``proj``     q|k|v and o projections of several layers for M rows; in a graph where the rows
             are a decode batch (``graph``), eager where they are a prompt's.
``gdn``      Gated DeltaNet recurrence over T tokens, state updated in place (T = 1: decode).
"""
import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "engine-mlx_amd"))
import ema_attn as ema  # noqa: E402

EPS, THETA, D = 1e-6, 1e6, 128
# hidden size, query heads, kv heads: the 0.6B-, 1.7B-, 8B- and 14B-size layers, head_dim 128
SHAPES = [(1024, 16, 8), (2048, 16, 8), (4096, 32, 8), (5120, 40, 8)]


def listed():
    return [
        # One token of one user over the 28 layers of a 1.7B-size model, 1024 tokens in: the
        # smallest kernels there are, where latency and launches decide.
        dict(name="token_b1_1p7b", kind="token", batch=1, hidden=2048, n_heads=16, n_kv=8, layers=28, cap=4096,
             lmin=1024, lmax=1024, bits=4, group=64, lens=1),
        # A serving batch of an 8B-size model at mixed lengths: the decode step's main workload.
        dict(name="step_b32_8b_bf16", kind="step", cache="bf16", ring=False, batch=32, n_heads=32, n_kv=8, cap=8192,
             lmin=512, lmax=8192, lens=3),
        # The same batch over the FP8 cache.
        dict(name="step_b32_8b_fp8", kind="step", cache="fp8", ring=False, batch=32, n_heads=32, n_kv=8, cap=8192,
             lmin=512, lmax=8192, lens=3),
        # Long documents over the int4 cache, kept to fit more of them.
        dict(name="step_b8_32k_int4", kind="step", cache="int4", ring=False, batch=8, n_heads=32, n_kv=4, cap=32768,
             lmin=32000, lmax=32768, lens=4),
        # A chat turn: a short, odd-sized message appended to a history of 3000 tokens.
        dict(name="prefill_turn_157", kind="prefill", cache="bf16", ring=False, batch=1, tokens=157, n_heads=32,
             n_kv=8, cap=4096, offset=3000),
        # A 2048-token prompt from the start, 8B-size layer.
        dict(name="prefill_2k_8b", kind="prefill", cache="bf16", ring=False, batch=1, tokens=2048, n_heads=32,
             n_kv=8, cap=4096, offset=0),
        # The last 2048-token chunk of a 16k prompt, 64 query heads: the largest call.
        dict(name="prefill_chunk_16k", kind="prefill", cache="bf16", ring=False, batch=1, tokens=2048, n_heads=64,
             n_kv=8, cap=16384, offset=14336),
        # Projections of a decode batch of 32, 8B-size layers, 4 bits.
        dict(name="proj_m32_8b", kind="proj", rows=32, hidden=4096, n_heads=32, n_kv=8, layers=12, bits=4, group=64,
             dtype="bf16", graph=True),
        # Projections of a chat turn's 157 rows.
        dict(name="proj_m157_8b", kind="proj", rows=157, hidden=4096, n_heads=32, n_kv=8, layers=12, bits=4, group=64,
             dtype="bf16", graph=False),
        # Projections of a long, odd-sized prompt, 8 bits.
        dict(name="proj_m1531_8b_8bit", kind="proj", rows=1531, hidden=4096, n_heads=32, n_kv=8, layers=4, bits=8,
             group=64, dtype="bf16", graph=False),
        # Gated DeltaNet: a decode batch's step (HBM-bound) and a prompt's scan (serial).
        dict(name="gdn_step_b32", kind="gdn", batch=32, tokens=1, k_heads=16, v_heads=32),
        dict(name="gdn_scan_2k", kind="gdn", batch=1, tokens=2048, k_heads=16, v_heads=32),
    ]


def _log(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["token", "step", "step", "prefill", "prefill", "proj", "proj", "gdn"])
    hidden, n_heads, n_kv = rng.choice(SHAPES)
    if kind == "token":
        lmax = _log(rng, 16, 4096)
        return dict(kind=kind, batch=rng.choice([1, 1, 2, 3, 4, 8]), hidden=hidden, n_heads=n_heads, n_kv=n_kv,
                    layers=rng.randint(6, 16), cap=4096, lmin=max(1, lmax // rng.choice([1, 2, 8])), lmax=lmax,
                    bits=rng.choice([4, 4, 8]), group=64, lens=rng.randint(1, 10**6))
    if kind == "step":
        cache = rng.choice(["bf16", "fp8", "int4"])
        n_kv = rng.choice([4, 8, 8])
        batch = _log(rng, 2, 64)
        cap = 32 * _log(rng, 32, min(1024, 32 * 256 * 8 // (batch * n_kv)))
        lmax = rng.randint(cap // 2, cap)
        ring = rng.random() < 0.2
        return dict(kind=kind, cache=cache, ring=ring, batch=batch, n_heads=n_heads // 8 * 8, n_kv=n_kv, cap=cap,
                    lmin=max(1, lmax // rng.choice([1, 2, 16])), lmax=lmax * (2 if ring else 1),
                    lens=rng.randint(1, 10**6))
    if kind == "prefill":
        tokens = _log(rng, 16, 2048)
        batch = rng.randint(1, 4) if tokens < 600 else 1
        offset = rng.choice([0, 0, _log(rng, 16, 12000)])
        cache = rng.choice(["bf16", "bf16", "fp8"])
        ring = rng.random() < 0.15
        cap = 32 * (_log(rng, max(tokens, 512), 4096) // 32 + 1) if ring else 32 * ((offset + tokens) // 32 + 8)
        return dict(kind=kind, cache=cache, ring=ring, batch=batch, tokens=tokens, n_heads=n_heads, n_kv=n_kv,
                    cap=cap, offset=offset)
    if kind == "proj":
        rows = _log(rng, 2, 2048)
        return dict(kind=kind, rows=rows, hidden=hidden, n_heads=n_heads, n_kv=n_kv,
                    layers=rng.randint(6, 12) if rows < 512 else 4, bits=rng.choice([4, 4, 4, 8]),
                    group=rng.choice([64, 64, 64, 32, 128]), dtype=rng.choice(["bf16", "bf16", "bf16", "f16"]),
                    graph=rows <= 64)
    if rng.random() < 0.4:
        return dict(kind=kind, batch=_log(rng, 2, 64), tokens=1, k_heads=16, v_heads=rng.choice([16, 32, 32]))
    tokens = _log(rng, 40, 4000)
    return dict(kind=kind, batch=rng.randint(1, max(1, min(4, 4000 // tokens))), tokens=tokens, k_heads=16,
                v_heads=rng.choice([16, 32, 32]))


# ---------------------------------------------------------------- inputs
class _Gen:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, shape, mean=0.0, std=1.0, dtype=torch.bfloat16):
        t = torch.empty(shape, dtype=dtype, device="cuda")
        flat = t.view(-1)
        for i in range(0, flat.numel(), 1 << 28):  # large tensors in pieces
            n = min(1 << 28, flat.numel() - i)
            flat[i:i + n] = torch.randn(n, generator=self.g, device="cuda").mul_(std).add_(mean).to(dtype)
        return t

    def uniform(self, shape, lo, hi, dtype=torch.float32):
        return (torch.rand(shape, generator=self.g, device="cuda") * (hi - lo) + lo).to(dtype)

    def ints(self, shape, lo, hi, dtype):
        return torch.randint(lo, hi, shape, generator=self.g, device="cuda", dtype=torch.int64).to(dtype)


def _lengths(case):
    r = random.Random(case["lens"])
    return [r.randint(case["lmin"], case["lmax"]) for _ in range(case["batch"])]


def _i32(values):
    return torch.tensor(values, dtype=torch.int32, device="cuda")


def _weights(g, n, k, bits, group, dtype=torch.bfloat16):
    """One affine-quantised layer: random codes, scales that give weights of about
    1/sqrt(k), biases that centre them."""
    w = g.ints((n, k * bits // 32), -2**31, 2**31, torch.int32)
    top = (1 << bits) - 1
    unit = 3.4 / (math.sqrt(k) * top)
    sc = g.uniform((n, k // group), 0.6 * unit, 1.4 * unit)
    bi = -sc * (top / 2) + g.uniform((n, k // group), -0.1, 0.1) * unit * top / 2
    return w, sc.to(dtype), bi.to(dtype)


def _cache(g, case):
    """A cache whose rows all hold values of N(0, 1) size."""
    b, n_kv, cap = case["batch"], case["n_kv"], case["cap"]
    kind = case["cache"]
    if kind == "bf16":
        kw = dict(k=g.normal((b, n_kv, cap, D)), v=g.normal((b, n_kv, cap, D)))
    elif kind == "fp8":
        def codes():
            c = g.ints((b, n_kv, cap, D), 0, 254, torch.uint8)
            return c + (c >= 0x7F).to(torch.uint8)  # no NaN codes

        kw = dict(k=codes(), v=codes(), k_exp=g.ints((b, n_kv, cap, D // 64), -8, -6, torch.int8),
                  v_exp=g.ints((b, n_kv, cap, D // 64), -8, -6, torch.int8))
    else:
        words, meta = (b, n_kv, cap, D // 8), (b, n_kv, cap, D // 64)
        kw = dict(k=g.ints(words, -2**31, 2**31, torch.int32), v=g.ints(words, -2**31, 2**31, torch.int32),
                  k_scales=g.normal(meta, 0.3, 0.03), k_biases=g.normal(meta, -2.2, 0.1),
                  v_scales=g.normal(meta, 0.3, 0.03), v_biases=g.normal(meta, -2.2, 0.1))
    return ema.StaticCache(b, n_kv, cap, D, dtype=kind, rotating=case["ring"], **kw)


def _stored(cache):
    if cache.dtype == "bf16":
        return [cache.k, cache.v]
    if cache.dtype == "fp8":
        return [cache.k, cache.v, cache.k_exp, cache.v_exp]
    return [cache.k, cache.v, cache.k_scales, cache.k_biases, cache.v_scales, cache.v_biases]


def _captured(call):
    """call() recorded into a HIP graph after one eager pass."""
    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    return graph


def _proj_sizes(case):
    q_dim, kv_dim = case["n_heads"] * D, case["n_kv"] * D
    return (case["hidden"], q_dim + 2 * kv_dim), (q_dim, case["hidden"])


def _inputs(case, seed):
    """Inputs and weights of a case, from the seed alone."""
    g, kind = _Gen(seed), case["kind"]
    s = dict(case=case)
    if kind in ("token", "step", "prefill"):
        s["qw"], s["kw"] = g.normal((D,), 1.0, 0.1), g.normal((D,), 1.0, 0.1)
    row = (case["n_heads"] + 2 * case["n_kv"]) * D if kind != "gdn" else 0
    if kind == "token":
        n, b = case["layers"], case["batch"]
        (k1, n1), (k2, n2) = _proj_sizes(case)
        s["x"] = g.normal((n, b, case["hidden"]))
        s["w_qkv"] = [_weights(g, n1, k1, case["bits"], case["group"]) for _ in range(n)]
        s["w_o"] = [_weights(g, n2, k2, case["bits"], case["group"]) for _ in range(n)]
        s["k"] = g.normal((n, b, case["n_kv"], case["cap"], D))
        s["v"] = g.normal((n, b, case["n_kv"], case["cap"], D))
        s["offsets"] = _i32([x - 1 for x in _lengths(case)])
    elif kind == "step":
        s["cache"] = _cache(g, case)
        s["qkv"] = g.normal((case["batch"], row))
        s["offsets"] = _i32([x - 1 for x in _lengths(case)])
    elif kind == "prefill":
        s["cache"] = _cache(g, case)
        s["qkv"] = g.normal((case["batch"], case["tokens"], row))
        s["offsets"] = _i32([case["offset"]] * case["batch"])
    elif kind == "proj":
        dt = torch.bfloat16 if case["dtype"] == "bf16" else torch.float16
        (k1, n1), (k2, n2) = _proj_sizes(case)
        n = case["layers"]
        s["x"] = g.normal((n, case["rows"], k1), dtype=dt)
        s["a"] = g.normal((n, case["rows"], k2), std=0.5, dtype=dt)
        s["w_qkv"] = [_weights(g, n1, k1, case["bits"], case["group"], dt) for _ in range(n)]
        s["w_o"] = [_weights(g, n2, k2, case["bits"], case["group"], dt) for _ in range(n)]
    else:
        b, t, hk, hv = case["batch"], case["tokens"], case["k_heads"], case["v_heads"]
        s["q"] = g.normal((b, t, hk, D), std=1.0 / D)
        k = g.normal((b, t, hk, D), dtype=torch.float32)
        s["k"] = (k / k.norm(dim=-1, keepdim=True)).to(torch.bfloat16)
        s["v"] = g.normal((b, t, hv, D))
        s["g"] = g.uniform((b, t, hv), 0.5, 1.0)
        s["beta"] = g.uniform((b, t, hv), 0.0, 1.0)
        s["state"] = g.normal((b, hv, D, D), std=0.5, dtype=torch.float32)
    return s


def prepare(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    if kind == "token":
        n, b, h, n_kv = case["layers"], case["batch"], case["n_heads"], case["n_kv"]
        caches = [ema.StaticCache(b, n_kv, case["cap"], D, k=s["k"][i], v=s["v"][i]) for i in range(n)]
        s["ws"] = ema.decode_workspace(b, h, n_kv, D, case["cap"])
        s["qkv"] = torch.empty((b, (h + 2 * n_kv) * D), dtype=torch.bfloat16, device="cuda")
        s["attn"] = torch.empty((b, h * D), dtype=torch.bfloat16, device="cuda")
        s["out"] = torch.empty((n, b, case["hidden"]), dtype=torch.bfloat16, device="cuda")

        def token():
            for i in range(n):
                ema.quantized_matmul(s["x"][i], *s["w_qkv"][i], case["group"], case["bits"], out=s["qkv"])
                ema.decode_step(s["qkv"], s["qw"], s["kw"], EPS, THETA, s["offsets"], h, caches[i], case["cap"],
                                out=s["attn"], workspace=s["ws"])
                ema.quantized_matmul(s["attn"], *s["w_o"][i], case["group"], case["bits"], out=s["out"][i])

        s["caches"] = caches
        s["graph"] = _captured(token)
    elif kind == "step":
        s["ws"] = ema.decode_workspace(case["batch"], case["n_heads"], case["n_kv"], D, case["cap"])
        s["out"] = torch.empty((case["batch"], case["n_heads"] * D), dtype=torch.bfloat16, device="cuda")
    elif kind == "prefill":
        b, t, h = case["batch"], case["tokens"], case["n_heads"]
        s["q"] = torch.empty((b, h, t, D), dtype=torch.bfloat16, device="cuda")
        s["out"] = torch.empty((b, t, h * D), dtype=torch.bfloat16, device="cuda")
        s["pre"], s["att"] = {}, {}
        if case["cache"] == "fp8":  # the bf16 copy of the attended rows that a program keeps
            rows = case["cap"] if case["ring"] else case["offset"] + t
            ws = torch.empty(ema.prefill_workspace_size(s["cache"], rows), dtype=torch.uint8, device="cuda")
            s["pre"] = dict(prefill_workspace=ws, max_kv_len=rows)
            s["att"] = dict(workspace=ws, max_kv_len=rows, rows_decoded=True,
                            chunk_only=case["offset"] == 0 and not case["ring"])
    elif kind == "proj":
        dt = s["x"].dtype
        (_, n1), (_, n2) = _proj_sizes(case)
        s["qkv"] = torch.empty((case["layers"], case["rows"], n1), dtype=dt, device="cuda")
        s["out"] = torch.empty((case["layers"], case["rows"], n2), dtype=dt, device="cuda")
        if case["graph"]:
            s["graph"] = _captured(lambda: _projections(s))
    else:
        s["y"] = torch.empty_like(s["v"])
        s["ws"] = None
        if case["tokens"] > 1:
            s["ws"] = ema.gdn_workspace(case["batch"], case["tokens"], case["k_heads"], case["v_heads"], D, D)
    return s


def _projections(s):
    case = s["case"]
    for i in range(case["layers"]):
        ema.quantized_matmul(s["x"][i], *s["w_qkv"][i], case["group"], case["bits"], out=s["qkv"][i])
        ema.quantized_matmul(s["a"][i], *s["w_o"][i], case["group"], case["bits"], out=s["out"][i])


def run(state):
    s, case = state, state["case"]
    kind = case["kind"]
    if kind == "token":
        s["graph"].replay()
        return [s["out"], s["k"], s["v"]]
    if kind == "step":
        ema.decode_step(s["qkv"], s["qw"], s["kw"], EPS, THETA, s["offsets"], case["n_heads"], s["cache"],
                        case["cap"], out=s["out"], workspace=s["ws"])
        return [s["out"]] + _stored(s["cache"])
    if kind == "prefill":
        ema.pre_attention(s["qkv"], s["qw"], s["kw"], EPS, THETA, s["offsets"], case["n_heads"], s["cache"],
                          q_out=s["q"], **s["pre"])
        ema.prefill_attention(s["q"], s["cache"], s["offsets"], out=s["out"], **s["att"])
        return [s["out"], s["q"]] + _stored(s["cache"])
    if kind == "proj":
        if case["graph"]:
            s["graph"].replay()
        else:
            _projections(s)
        return [s["qkv"], s["out"]]
    ema.gdn_scan(s["q"], s["k"], s["v"], s["g"], s["beta"], s["state"], y=s["y"], workspace=s["ws"])
    return [s["y"], s["state"]]


# ---------------------------------------------------------------- work
_ROW = {"bf16": 2 * D, "fp8": D + D // 64, "int4": D // 2 + 4 * (D // 64)}  # bytes of one K or V row


def _weight_bytes(n, k, bits, group):
    return n * k * bits // 8 + 4 * n * (k // group)


def work(case):
    kind = case["kind"]
    if kind == "gdn":
        b, t, hk, hv = case["batch"], case["tokens"], case["k_heads"], case["v_heads"]
        return {"bytes": 8 * b * hv * D * D + 2 * b * t * (2 * hk * D + 2 * hv * D) + 8 * b * t * hv,
                "flops": 6 * b * t * hv * D * D}
    h, n_kv = case["n_heads"], case["n_kv"]
    if kind == "prefill":
        b, t = case["batch"], case["tokens"]
        past = min(case["offset"], case["cap"] - t) if case["ring"] else case["offset"]
        rows = _ROW[case["cache"]]
        # qkv in, out out, the chunk's K/V rows written, the older ones read
        return {"bytes": b * (t * (h + 2 * n_kv) * D * 2 + t * h * D * 2 + 2 * n_kv * (t + past) * rows),
                "flops": 4 * b * h * D * (t * past + t * (t + 1) // 2)}
    if kind == "proj":
        m, n_bytes, flops = case["rows"], 0, 0
        for k, n in _proj_sizes(case):
            n_bytes += _weight_bytes(n, k, case["bits"], case["group"]) + 2 * m * (k + n)
            flops += 2 * m * n * k
        return {"bytes": case["layers"] * n_bytes, "flops": case["layers"] * flops}
    lens = [min(x, case["cap"]) for x in _lengths(case)]
    b = case["batch"]
    if kind == "step":
        rows = _ROW[case["cache"]]
        return {"bytes": 2 * n_kv * sum(lens) * rows + b * (2 * h + 2 * n_kv) * D * 2,
                "flops": 4 * h * D * sum(lens)}
    n_bytes, flops = 2 * n_kv * sum(lens) * _ROW["bf16"] + 4 * b * case["hidden"], 4 * h * D * sum(lens)
    for k, n in _proj_sizes(case):
        n_bytes += _weight_bytes(n, k, case["bits"], case["group"])
        flops += 2 * b * n * k
    return {"bytes": case["layers"] * n_bytes, "flops": case["layers"] * flops}


def tolerance(case):
    """About four times what a change of summation order or of a split shows at the same
    precision. Measured against float64: projections 1.7e-3 to 2.3e-3 (the bf16 output and
    bf16 dequantised weights), attention 3e-3 to 4.2e-3 (bf16 q and probabilities too), the
    Gated DeltaNet output 1.7e-3. Quantised caches: a new row's value at a rounding edge moves
    by one code, which a short context shows (1.4e-2 over 16 tokens). `differ`: such codes, of
    all codes in the cache."""
    kind = case["kind"]
    if kind in ("step", "prefill") and case["cache"] != "bf16":
        return {"rel": 2e-2, "max": 0.3, "differ": 2e-3}
    if kind in ("token", "step", "prefill"):
        return {"rel": 1.5e-2, "max": 0.2}
    return {"rel": 1e-2, "max": 0.05}


# ---------------------------------------------------------------- float64
def _dequant(w, sc, bi, bits, group):
    n = w.shape[0]
    shifts = torch.arange(0, 32, bits, device=w.device)
    codes = (w.to(torch.int64)[:, :, None] >> shifts) & ((1 << bits) - 1)
    codes = codes.reshape(n, -1, group).double()
    return (codes * sc.double()[..., None] + bi.double()[..., None]).reshape(n, -1)


def _norm_rope(x, w, pos):
    """x [..., D] float64, pos broadcastable to x's leading shape."""
    x = x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()
    i = torch.arange(D // 2, dtype=torch.float64, device=x.device)
    angle = pos.double()[..., None] * THETA ** (-i / (D // 2))
    c, s = torch.cos(angle), torch.sin(angle)
    a, b = x[..., :D // 2], x[..., D // 2:]
    return torch.cat([a * c - b * s, a * s + b * c], -1)


def _fp8_values(codes, exp):
    v = codes.view(torch.float8_e4m3fn).float().double()
    return v * torch.exp2(exp.double()).repeat_interleave(64, -1)


def _fp8_round(x):
    """The values an FP8 cache holds for rows x: 64-value blocks, a power-of-two scale."""
    blocks = x.reshape(*x.shape[:-1], -1, 64)
    amax = blocks.abs().amax(-1, keepdim=True).clamp(min=1e-4)
    scale = torch.exp2(torch.ceil(torch.log2(amax / 448)))
    codes = (blocks / scale).clamp(-448, 448).float().to(torch.float8_e4m3fn).float().double()
    return (codes * scale).reshape(x.shape)


def _int4_values(words, sc, bi):
    codes = (words.to(torch.int64)[..., None] >> torch.arange(0, 32, 4, device=words.device)) & 15
    codes = codes.reshape(*words.shape[:-1], -1, 64).double()
    return (codes * sc.double()[..., None] + bi.double()[..., None]).reshape(*words.shape[:-1], -1)


def _int4_round(x):
    """The values an int4 cache holds for rows x: 64-value groups, affine, the end of larger
    magnitude on the grid."""
    g = x.reshape(*x.shape[:-1], -1, 64)
    lo, hi = g.amin(-1, keepdim=True), g.amax(-1, keepdim=True)
    scale = ((hi - lo) / 15).clamp(min=1e-7)
    scale = torch.where(lo.abs() > hi.abs(), scale, -scale)
    edge = torch.where(lo.abs() > hi.abs(), lo, hi)
    q0 = torch.round(edge / scale)
    scale = torch.where(q0 != 0, edge / q0, scale)
    bias = torch.where(q0 != 0, edge, torch.zeros_like(edge))
    codes = torch.floor((g - bias) / scale + 0.5).clamp(0, 15)
    return (codes * scale + bias).reshape(x.shape)


def _split_row(qkv, case):
    h, n_kv = case["n_heads"], case["n_kv"]
    return qkv.reshape(*qkv.shape[:-1], h + 2 * n_kv, D).double().split([h, n_kv, n_kv], -2)


def _attend(q, k, v, mask=None):
    """q [H, T, D], k and v [Hkv, L, D], float64; mask [T, L] of the keys each row sees."""
    per = q.shape[0] // k.shape[0]
    out = torch.empty_like(q)
    for j in range(k.shape[0]):
        for h in range(j * per, (j + 1) * per):
            s = (q[h] @ k[j].T) / math.sqrt(D)
            if mask is not None:
                s = s.masked_fill(~mask, -math.inf)
            out[h] = torch.softmax(s, -1) @ v[j]
    return out


def _rows(cache, b):
    """K and V of sequence b as float64 values."""
    if cache.dtype == "bf16":
        return cache.k[b].double(), cache.v[b].double()
    if cache.dtype == "fp8":
        return _fp8_values(cache.k[b], cache.k_exp[b]), _fp8_values(cache.v[b], cache.v_exp[b])
    return (_int4_values(cache.k[b], cache.k_scales[b], cache.k_biases[b]),
            _int4_values(cache.v[b], cache.v_scales[b], cache.v_biases[b]))


_KEEP = {"bf16": lambda x: x, "fp8": _fp8_round, "int4": _int4_round}


def _exact_step(s, case):
    cache, lens, cap = s["cache"], _lengths(case), case["cap"]
    keep = _KEEP[case["cache"]]
    q, k, v = _split_row(s["qkv"], case)
    out, new_k, new_v = [], [], []
    for b, n in enumerate(lens):
        pos = torch.full((1,), n - 1, device="cuda")
        qb, kb = _norm_rope(q[b], s["qw"], pos), _norm_rope(k[b], s["kw"], pos)
        kc, vc = _rows(cache, b)
        row = (n - 1) % cap
        kc[:, row], vc[:, row] = keep(kb), keep(v[b])
        held = min(n, cap)
        out.append(_attend(qb[:, None], kc[:, :held], vc[:, :held]).reshape(-1))
        if case["cache"] == "bf16":
            new_k.append(kc)
            new_v.append(vc)
    out = torch.stack(out)
    if case["cache"] == "bf16":
        return [out, torch.stack(new_k), torch.stack(new_v)]
    return [out] + [None] * (len(_stored(cache)) - 1)


def _exact_prefill(s, case):
    cache, t, off, cap = s["cache"], case["tokens"], case["offset"], case["cap"]
    keep = _KEEP[case["cache"]]
    q, k, v = _split_row(s["qkv"], case)
    pos = torch.arange(off, off + t, device="cuda")
    q, k = _norm_rope(q, s["qw"], pos[:, None]), _norm_rope(k, s["kw"], pos[:, None])
    end = off + t
    outs, ks, vs = [], [], []
    for b in range(case["batch"]):
        kc, vc = _rows(cache, b)
        rows = pos % cap
        kc[:, rows], vc[:, rows] = keep(k[b]).transpose(0, 1), keep(v[b]).transpose(0, 1)
        held = min(end, cap)
        at = torch.arange(held, device="cuda")
        if case["ring"] and end > cap:
            at = at + (end - 1 - at) // cap * cap
        mask = at[None, :] <= pos[:, None]
        o = _attend(q[b].transpose(0, 1), kc[:, :held], vc[:, :held], mask)
        outs.append(o.transpose(0, 1).reshape(t, -1))
        ks.append(kc)
        vs.append(vc)
    got = [torch.stack(outs), q.transpose(1, 2).contiguous()]
    if case["cache"] == "bf16":
        return got + [torch.stack(ks), torch.stack(vs)]
    return got + [None] * (len(_stored(cache)))


def exact(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    if kind == "step":
        return _exact_step(s, case)
    if kind == "prefill":
        return _exact_prefill(s, case)
    if kind == "proj":
        pairs = [(s["x"], s["w_qkv"]), (s["a"], s["w_o"])]
        return [torch.stack([x[i].double() @ _dequant(*w[i], case["bits"], case["group"]).T
                             for i in range(case["layers"])]) for x, w in pairs]
    if kind == "token":
        lens, out = _lengths(case), []
        ks, vs = s["k"].double(), s["v"].double()
        for i in range(case["layers"]):
            qkv = s["x"][i].double() @ _dequant(*s["w_qkv"][i], case["bits"], case["group"]).T
            q, k, v = _split_row(qkv, case)
            attn = []
            for b, n in enumerate(lens):
                pos = torch.full((1,), n - 1, device="cuda")
                ks[i, b, :, n - 1], vs[i, b, :, n - 1] = _norm_rope(k[b], s["kw"], pos), v[b]
                attn.append(_attend(_norm_rope(q[b], s["qw"], pos)[:, None], ks[i, b, :, :n],
                                    vs[i, b, :, :n]).reshape(-1))
            out.append(torch.stack(attn) @ _dequant(*s["w_o"][i], case["bits"], case["group"]).T)
        return [torch.stack(out), ks, vs]
    b, t, hv = case["batch"], case["tokens"], case["v_heads"]
    q, k = (s[x].double().repeat_interleave(hv // case["k_heads"], 2) for x in ("q", "k"))
    v, g, beta, state = s["v"].double(), s["g"].double(), s["beta"].double(), s["state"].double()
    y = torch.empty_like(v)
    for i in range(t):
        state = state * g[:, i, :, None, None]
        recall = (state @ k[:, i, :, :, None])[..., 0]
        delta = (v[:, i] - recall) * beta[:, i, :, None]
        state = state + delta[..., None] * k[:, i, :, None, :]
        y[:, i] = (state @ q[:, i, :, :, None])[..., 0]
    return [y, state]

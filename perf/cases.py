"""The work that a user of the framework has it do, as measurable cases over the public entry points.

A case is a dict of plain values; `path` says which entry point it goes through:

  host    one matvec on host slices (`q4k_matvec`, `q8_0_gemv`, `mxfp4_gemv`, `bf16_gemv_force`)
  head    the lm_head on host slices with the top-K kept on the device (`q8_0_gemv_topk`)
  token   a decode token's matvecs in dependency order, recorded once as a sequence (`sequence_run`)
  knn     gate-KNN over one layer's resident gate (`dev_gate_knn`)
  walk    gate-KNN over all layers in one submission (`dev_gate_walk`)
  moe     an MXFP4 expert block with its routing (`dev_moe_mxfp4_routed`)
  moe_kq  a MoE layer over a k-quant expert bank, router projection included (`dev_moe_layer_forward`)
  gemm    prefill GEMM over a Q4_K matrix (`dev_q4k_gemm`, `dev_q4k_gemm_prepared`)
  encode  a block encoder over a resident f32 matrix (`dev_quantize_*`)

Weights are N(0, 1/k) and activations N(0, 1), so that a chain of matvecs keeps its scale as a normalised network does.
"""
import math

import numpy as np
import torch

import larql_amd as fmt

FORMATS = {"q4k": fmt.FMT_Q4_K, "q6k": fmt.FMT_Q6_K, "q8_0": fmt.FMT_GGML_Q8_0, "q4_0": fmt.FMT_Q4_0, "mxfp4": fmt.FMT_MXFP4,
           "bf16": fmt.FMT_BF16, "f16": fmt.FMT_F16, "f32": fmt.FMT_F32}
# format -> (elements a block, bytes a block)
BLOCK = {"q4k": (256, 144), "q6k": (256, 210), "q8_0": (32, 34), "q4_0": (32, 18), "mxfp4": (32, 17), "bf16": (1, 2), "f16": (1, 2),
         "f32": (1, 4)}


def _bytes(f, n):
    return n // BLOCK[f][0] * BLOCK[f][1]


# ---- the cases ------------------------------------------------------------------------------------------------------

def listed():
    return [
        # The smallest call a backend gets from the trait: one Q4_K matvec on host slices, its weights in a registered region.
        {"name": "host_q4k_3072x1024", "path": "host", "format": "q4k", "rows": 3072, "k": 1024, "registered": True},
        # Sampling a token from a 262144-row vocabulary: scores and their 64 largest, from and to host memory.
        {"name": "head_q8_0_262144x2560", "path": "head", "rows": 262144, "k": 2560, "top_k": 64},
        # One decode token of the 34-layer stack: each stage reads what the one before wrote.
        {"name": "token_q4k_34_layers", "path": "token", "layers": 34, "hidden": 2560, "q_rows": 2048, "kv_rows": 1024, "inter": 10240,
         "vocab": 262144, "down": "q4k"},
        # One layer's features for one residual, f16 gate as an index keeps it.
        {"name": "knn_f16_10240x2560", "path": "knn", "format": "f16", "batch": 1, "features": 10240, "hidden": 2560, "top_k": 64},
        # A query walked over every layer of an index (one position, quantised gates)...
        {"name": "walk_q4k_34_layers", "path": "walk", "format": "q4k", "layers": 34, "batch": 1, "features": 10240, "hidden": 2560,
         "top_k": 64},
        # ...and the last eight positions of a prompt over bf16 gates.
        {"name": "walk_bf16_34_layers_8", "path": "walk", "format": "bf16", "layers": 34, "batch": 8, "features": 10240, "hidden": 2560,
         "top_k": 64},
        # Decode and prefill through a GPT-OSS-shaped expert block (fused gate_up rows, biases).
        {"name": "moe_mxfp4_1_token", "path": "moe", "tokens": 1, "experts": 32, "top_k": 4, "hidden": 2880, "inter": 2880,
         "interleaved": True, "biases": True},
        {"name": "moe_mxfp4_128_tokens", "path": "moe", "tokens": 128, "experts": 32, "top_k": 4, "hidden": 2880, "inter": 2880,
         "interleaved": True, "biases": True},
        # A batch of decode tokens through a 128-expert Q4_K layer.
        {"name": "moe_q4k_16_tokens", "path": "moe_kq", "format": "q4k", "tokens": 16, "experts": 128, "top_k": 8, "hidden": 2816,
         "inter": 704, "rule": "gelu_tanh"},
        # A short, ragged prompt through a down projection, and a long prefill chunk through a gate projection.
        {"name": "gemm_3840x15360_77_tokens", "path": "gemm", "rows": 3840, "k": 15360, "tokens": 77, "prepared": True},
        {"name": "gemm_15360x3840_2048_tokens", "path": "gemm", "rows": 15360, "k": 3840, "tokens": 2048, "prepared": True},
        # Quantising one feed-forward matrix while a model is loaded.
        {"name": "encode_q4k_10240x2560", "path": "encode", "format": "q4k", "rows": 10240, "k": 2560},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _log_mult(rng, lo, hi, of):
    return _log_int(rng, lo // of, hi // of) * of


def _one(rng):
    path = rng.choice(["host", "head", "token", "knn", "walk", "moe", "moe", "moe_kq", "gemm", "gemm", "encode"])
    if path == "host":
        return {"path": path, "format": rng.choice(["q4k", "q4k", "q8_0", "mxfp4", "bf16"]), "rows": _log_int(rng, 64, 16384),
                "k": _log_mult(rng, 256, 10240, 256), "registered": rng.random() < 0.75}
    if path == "head":
        return {"path": path, "rows": _log_int(rng, 16384, 262144), "k": _log_mult(rng, 1024, 4096, 256), "top_k": rng.choice([1, 40, 64, 200])}
    if path == "token":
        hidden = rng.randint(4, 15) * 256
        return {"path": path, "layers": rng.randint(2, 34), "hidden": hidden, "q_rows": rng.randint(4, 16) * 256,
                "kv_rows": rng.choice([256, 512, 1024]), "inter": rng.randint(8, 40) * 256, "vocab": _log_int(rng, 16384, 262144),
                "down": rng.choice(["q4k", "q6k"])}
    if path == "knn":
        return {"path": path, "format": rng.choice(["f16", "bf16", "f32", "q4k", "q4_0"]), "batch": _log_int(rng, 1, 16),
                "features": _log_int(rng, 1000, 16384), "hidden": _log_mult(rng, 512, 5120, 256), "top_k": rng.choice([8, 64, 64, 256])}
    if path == "walk":
        return {"path": path, "format": rng.choice(["bf16", "q4k"]), "layers": rng.randint(8, 34), "batch": _log_int(rng, 1, 8),
                "features": _log_int(rng, 4000, 12288), "hidden": _log_mult(rng, 1024, 3840, 256), "top_k": rng.choice([16, 64])}
    if path == "moe":
        return {"path": path, "tokens": _log_int(rng, 1, 256), "experts": rng.choice([16, 32, 64]), "top_k": rng.choice([2, 4]),
                "hidden": rng.randint(24, 48) * 64, "inter": rng.randint(24, 48) * 64, "interleaved": rng.random() < 0.7,
                "biases": rng.random() < 0.5}
    if path == "moe_kq":
        return {"path": path, "format": rng.choice(["q4k", "q4k", "q6k"]), "tokens": _log_int(rng, 1, 64), "experts": rng.choice([32, 64, 128]),
                "top_k": rng.choice([4, 8]), "hidden": rng.randint(6, 12) * 256, "inter": rng.randint(8, 24) * 32,
                "rule": rng.choice(["gelu_tanh", "silu"])}
    if path == "gemm":
        return {"path": path, "rows": _log_int(rng, 1000, 15360), "k": _log_mult(rng, 1024, 15360, 256), "tokens": _log_int(rng, 16, 2048),
                "prepared": rng.random() < 0.75}
    return {"path": path, "format": rng.choice(["q4k", "q6k", "q8_0", "q4_0", "mxfp4", "bf16"]), "rows": _log_int(rng, 64, 10240),
            "k": _log_mult(rng, 1024, 10240, 256)}


def draw(rng):
    big = [work(c) for c in listed()]
    while True:
        c = _one(rng)
        w = work(c)
        if w["bytes"] <= max(b["bytes"] for b in big) and w["flops"] <= max(b["flops"] for b in big):
            return c


# ---- what a pass cannot do without ----------------------------------------------------------------------------------

def _token_stages(c):
    """The stages of one layer: [(buffer read, [(buffer written, format, rows, k)])]."""
    h, q, kv, i = c["hidden"], c["q_rows"], c["kv_rows"], c["inter"]
    return [("h", [("q", "q4k", q, h), ("k", "q4k", kv, h), ("v", "q4k", kv, h)]), ("q", [("o", "q4k", h, q)]),
            ("o", [("gate", "q4k", i, h), ("up", "q4k", i, h)]), ("gate", [("down", c["down"], h, i)])]


def _kq_inter(c):
    return -(-c["inter"] // 256) * 256


def work(c):
    p = c["path"]
    if p in ("host", "head"):
        n, f = c["rows"] * c["k"], c.get("format", "q8_0")
        return {"bytes": _bytes(f, n) + 4 * c["k"] + (4 * c["rows"] if p == "host" else 8 * c["top_k"]), "flops": 2.0 * n}
    if p == "token":
        mats = [(f, r, k) for _, jobs in _token_stages(c) for _, f, r, k in jobs] * c["layers"] + [("q8_0", c["vocab"], c["hidden"])]
        return {"bytes": sum(_bytes(f, r * k) + 4 * r + 4 * k for f, r, k in mats), "flops": sum(2.0 * r * k for _, r, k in mats)}
    if p in ("knn", "walk"):
        layers = c.get("layers", 1)
        n, b = layers * c["features"] * c["hidden"], c["batch"]
        out = layers * b * (4 * c["features"] + 8 * min(c["top_k"], c["features"]))
        return {"bytes": _bytes(c["format"], n) + 4 * b * c["hidden"] + out, "flops": 2.0 * n * b}
    if p in ("moe", "moe_kq"):
        t, e, k, h, i = c["tokens"], c["experts"], c["top_k"], c["hidden"], c["inter"]
        read = e * (1 - (1 - k / e) ** t)  # distinct experts that t tokens choose
        expert = _bytes("mxfp4", 3 * h * i) if p == "moe" else _bytes(c["format"], 2 * i * h + h * _kq_inter(c))
        return {"bytes": read * expert + 8 * t * h + (4 * t * e if p == "moe" else 4 * e * h), "flops": 6.0 * t * k * h * i}
    if p == "gemm":
        n, k, t = c["rows"], c["k"], c["tokens"]
        return {"bytes": _bytes("q4k", n * k) + 2 * t * k + 4 * t * n, "flops": 2.0 * n * k * t}
    n = c["rows"] * c["k"]
    return {"bytes": 4 * n + _bytes(c["format"], n), "flops": 0}


def tolerance(c):
    p = c["path"]
    if p == "encode":
        return "exact"
    if p == "gemm":      # f16 operands with one rounding per weight: 2.9e-4 from the f64 product
        return {"rel": 1.2e-3}
    if p == "moe_kq":    # up to 6e-5: an activation code moves by one step where expf / tanhf differ in the last place
        return {"rel": 2e-4, "max": 2e-2, "differ": 0.01}
    if p == "token":     # a stage is off by 1e-6, and up to 137 of them follow one another
        return {"rel": 2e-5}
    if p == "moe":       # 1.5e-6 from the f64 block: two f32 contractions with an exponential between them
        return {"rel": 6e-6, "differ": 0.01}
    return {"rel": 4e-6, "differ": 0.01}  # f32 sums of one contraction: up to 1e-6 from f64


# ---- inputs ---------------------------------------------------------------------------------------------------------

_BACKEND = []


def _backend():
    """The process's context for resident operands, as a serving program has one."""
    if not _BACKEND:
        _BACKEND.append(fmt.HipBackend(0))
    return _BACKEND[0]


class State:
    """What a program holds between calls; handles of the library are given back with it."""

    def __init__(self, case, seed):
        self.case, self.be, self.seed, self.stream = case, _backend(), seed, 0
        self.keep, self.own, self.plans, self.seq, self.layer = [], None, [], None, None

    def normal(self, n, sigma=1.0):
        t = torch.empty(n + 16, dtype=torch.float32, device="cuda")
        self.stream += 1
        self.be.dev_fill_normal(t.data_ptr(), n, (self.seed * 1000003 + self.stream * 7919) & 0xFFFFFFFFFFFF, sigma)
        return t

    def empty(self, n, dtype=torch.float32):
        t = torch.zeros(n, dtype=dtype, device="cuda")
        self.keep.append(t)
        return t

    def encoded(self, f, rows, k, into=None):
        """A [rows, k] matrix of N(0, 1/k) in format f: (bytes, e8m0 stream or None)."""
        be, step, aux = self.be, max(1, (1 << 26) // k), None
        w = into if into is not None else torch.empty(_bytes(f, rows * k) + 64 if f != "mxfp4" else rows * k // 2 + 64, dtype=torch.uint8, device="cuda")
        if f == "mxfp4":
            aux = torch.empty(rows * k // 32 + 64, dtype=torch.uint8, device="cuda")
        for r in range(0, rows, step):
            n = min(step, rows - r) * k
            src = self.normal(n, 1.0 / math.sqrt(k))
            if f == "mxfp4":
                be.dev_quantize_mxfp4(src.data_ptr(), n // k, k, w.data_ptr() + r * k // 2, aux.data_ptr() + r * k // 32)
            elif f == "f32":
                w[4 * r * k: 4 * (r * k + n)] = src[:n].view(torch.uint8)
            elif f == "f16":
                w[2 * r * k: 2 * (r * k + n)] = src[:n].half().view(torch.uint8)
            else:
                _encoder(be, f)(src.data_ptr(), n, w.data_ptr() + _bytes(f, r * k))
            be.synchronize()
        if into is None:
            self.keep.append(w)
        self.keep.append(aux)
        return w, aux

    def host(self, t, n):
        self.be.synchronize()
        return t[:n].cpu().numpy()

    def __del__(self):
        if self.seq is not None:
            self.be.sequence_destroy(self.seq)
        for p in self.plans:
            self.be.plan_destroy(p)
        if self.layer is not None:
            self.be.moe_layer_destroy(self.layer)
        if self.own is not None:
            self.own.close()


def _encoder(be, f):
    return {"q4k": be.dev_quantize_q4_k, "q6k": be.dev_quantize_q6_k, "q8_0": be.dev_quantize_q8_0, "q4_0": be.dev_quantize_q4_0,
            "bf16": be.dev_f32_to_bf16}[f]


def prepare(case, seed):
    s = State(case, seed)
    _PREPARE[case["path"]](s, case)
    s.be.synchronize()
    torch.cuda.synchronize()
    return s


def run(state):
    return _RUN[state.case["path"]](state, state.case)


# host slices: a context of its own holds the registered region

def _prepare_host(s, c):
    f, rows, k = c.get("format", "q8_0"), c["rows"], c["k"]
    w, aux = s.encoded(f, rows, k)
    s.w = s.host(w, rows * k // 2 if f == "mxfp4" else _bytes(f, rows * k))
    s.aux = s.host(aux, rows * k // 32) if f == "mxfp4" else None
    s.x = s.host(s.normal(k), k)
    s.keep.clear()
    s.own = fmt.HipBackend(0)
    if c.get("registered", True):
        for a in (s.w, s.aux):
            if a is not None:
                s.own.register_weight_region(a)
        s.own.seal_weight_regions()


def _run_host(s, c):
    f, rows, k = c["format"], c["rows"], c["k"]
    if f == "q4k":
        return s.own.q4k_matvec(s.w, s.x, rows, k)
    if f == "q8_0":
        return s.own.q8_0_gemv(s.w, s.x, rows, k)
    if f == "mxfp4":
        return s.own.mxfp4_gemv(s.w, s.aux, s.x, rows, k)
    return s.own.bf16_gemv_force(s.w, s.x, rows, k)


def _run_head(s, c):
    hits = s.own.q8_0_gemv_topk(s.w, s.x, c["rows"], c["k"], c["top_k"])
    return np.array([i for i, _ in hits], np.int64), np.array([v for _, v in hits], np.float32)


# a decode token

def _prepare_token(s, c):
    sizes = {"q": c["q_rows"], "k": c["kv_rows"], "v": c["kv_rows"], "o": c["hidden"], "gate": c["inter"], "up": c["inter"],
             "down": c["hidden"]}
    per, at = sum(sizes.values()), {}
    for n, r in sizes.items():
        at[n] = sum(v for m, v in sizes.items() if list(sizes).index(m) < list(sizes).index(n))
    s.acts = s.empty(c["layers"] * per)
    s.logits = s.empty(c["vocab"])
    x0 = s.normal(c["hidden"])
    s.keep.append(x0)
    x = x0.data_ptr()

    def plan(jobs):
        p = s.be.plan_create(jobs)
        assert p, s.be.last_error()
        s.plans.append(p)

    for layer in range(c["layers"]):
        buf = {n: s.acts.data_ptr() + 4 * (layer * per + o) for n, o in at.items()}
        buf["h"] = x
        for src, jobs in _token_stages(c):
            plan([(FORMATS[f], s.encoded(f, r, k)[0].data_ptr(), None, buf[src], buf[dst], r, k) for dst, f, r, k in jobs])
        x = buf["down"]
    plan([(fmt.FMT_GGML_Q8_0, s.encoded("q8_0", c["vocab"], c["hidden"])[0].data_ptr(), None, x, s.logits.data_ptr(), c["vocab"],
           c["hidden"])])
    s.seq = s.be.sequence_create(s.plans)
    assert s.seq, s.be.last_error()


def _run_token(s, c):
    s.be.sequence_run(s.seq)
    return s.acts, s.logits


# gate-KNN

def _prepare_gates(s, c):
    layers, b, n, k = c.get("layers", 1), c["batch"], c["features"], c["top_k"]
    s.gates = [s.encoded(c["format"], n, c["hidden"])[0].data_ptr() for _ in range(layers)]
    s.x = s.normal(b * c["hidden"])
    s.scores = s.empty(layers * b * n)
    s.idx, s.val, s.count = s.empty(layers * b * k, torch.int32), s.empty(layers * b * k), s.empty(layers * b, torch.int32)


def _run_knn(s, c):
    s.be.dev_gate_knn(FORMATS[c["format"]], s.gates[0], s.x.data_ptr(), c["batch"], c["features"], c["hidden"], c["top_k"],
                      s.scores.data_ptr(), s.idx.data_ptr(), s.val.data_ptr(), s.count.data_ptr())
    return s.scores, s.idx, s.val, s.count


def _run_walk(s, c):
    s.be.dev_gate_walk(FORMATS[c["format"]], s.gates, s.x.data_ptr(), 0, c["batch"], c["features"], c["hidden"], c["top_k"],
                       s.scores.data_ptr(), s.idx.data_ptr(), s.val.data_ptr(), s.count.data_ptr())
    return s.scores, s.idx, s.val, s.count


# experts

def _prepare_moe(s, c):
    t, e, k, h, i = c["tokens"], c["experts"], c["top_k"], c["hidden"], c["inter"]
    if c["interleaved"]:
        gate, up = s.encoded("mxfp4", e * 2 * i, h), (None, None)
    else:
        gate, up = s.encoded("mxfp4", e * i, h), s.encoded("mxfp4", e * i, h)
    down = s.encoded("mxfp4", e * h, i)
    bias = [s.normal(n, 0.1) if c["biases"] else None for n in (e, 2 * e * i, e * h)]
    ptr = [None if a is None else a.data_ptr() for a in (*gate, *up, *down, *bias)]
    s.keep.extend(bias)
    s.bank = fmt.Mxfp4Experts(*ptr[:6], e, h, i, 7.0, 1.702, int(c["interleaved"]), *ptr[6:])
    s.x, s.router = s.normal(t * h), s.normal(t * e)
    s.chosen, s.weights, s.out = s.empty(t * k, torch.int32), s.empty(t * k), s.empty(t * h)
    s.ws_bytes = s.be.moe_mxfp4_workspace_bytes(t, k, h, i)
    s.ws = s.empty(s.ws_bytes, torch.uint8)


def _run_moe(s, c):
    s.be.dev_moe_mxfp4_routed(s.bank, s.x.data_ptr(), c["tokens"], c["top_k"], s.router.data_ptr(), 1, s.chosen.data_ptr(),
                              s.weights.data_ptr(), s.out.data_ptr(), s.ws.data_ptr(), s.ws_bytes)
    return s.chosen, s.weights, s.out


def _prepare_moe_kq(s, c):
    t, e, k, h, i, f = c["tokens"], c["experts"], c["top_k"], c["hidden"], c["inter"], c["format"]
    gu_n, dn_n = _bytes(f, 2 * i * h), _bytes(f, h * _kq_inter(c))
    gu, dn = s.host(s.encoded(f, e * 2 * i, h)[0], e * gu_n), s.host(s.encoded(f, e * h, _kq_inter(c))[0], e * dn_n)
    router = s.host(s.normal(e * h, 1.0 / math.sqrt(h)), e * h).reshape(e, h)
    s.keep.clear()
    rule = {"gelu_tanh": fmt.MOE_GATE_GELU_TANH, "silu": fmt.MOE_GATE_SILU}[c["rule"]]
    s.layer = s.be.moe_layer_create([gu[n * gu_n: (n + 1) * gu_n] for n in range(e)], [dn[n * dn_n: (n + 1) * dn_n] for n in range(e)], None,
                                    None, router, k, h, i, fmt.MOE_ROWS_CONTIGUOUS_HALVES, expert_scales=fmt.MOE_SCALES_INLINE,
                                    expert_data_format=FORMATS[f], gate_rule=rule)
    assert s.layer, s.be.last_error()
    s.x = s.normal(t * h)
    s.chosen, s.weights, s.out = s.empty(t * k, torch.int32), s.empty(t * k), s.empty(t * h)


def _run_moe_kq(s, c):
    s.be.dev_moe_layer_forward(s.layer, s.x.data_ptr(), s.x.data_ptr(), c["tokens"], s.out.data_ptr(), s.chosen.data_ptr(),
                               s.weights.data_ptr())
    return s.chosen, s.weights, s.out


# prefill

def _prepare_gemm(s, c):
    n, k, t = c["rows"], c["k"], c["tokens"]
    s.w = s.encoded("q4k", n, k)[0]
    x = s.normal(t * k)
    s.x = s.empty(t * k + 32, torch.int16)
    s.be.dev_f32_to_bf16(x.data_ptr(), t * k, s.x.data_ptr())
    s.be.synchronize()
    s.out = s.empty(t * n)
    if c["prepared"]:
        s.exponents = s.empty(n, torch.int32)
        s.be.dev_q4k_row_exponents(s.w.data_ptr(), n, k, s.exponents.data_ptr())


def _run_gemm(s, c):
    n, k, t = c["rows"], c["k"], c["tokens"]
    if c["prepared"]:
        s.be.dev_q4k_gemm_prepared(s.w.data_ptr(), s.exponents.data_ptr(), s.x.data_ptr(), n, k, t, s.out.data_ptr())
    else:
        s.be.dev_q4k_gemm(s.w.data_ptr(), s.x.data_ptr(), n, k, t, s.out.data_ptr())
    return s.out


# encoders

def _prepare_encode(s, c):
    n = c["rows"] * c["k"]
    s.src = s.normal(n, 1.0 / math.sqrt(c["k"]))
    s.out = s.empty(n // 2 if c["format"] == "mxfp4" else _bytes(c["format"], n), torch.uint8)
    s.exp = s.empty(n // 32, torch.uint8) if c["format"] == "mxfp4" else None


def _run_encode(s, c):
    if c["format"] == "mxfp4":
        s.be.dev_quantize_mxfp4(s.src.data_ptr(), c["rows"], c["k"], s.out.data_ptr(), s.exp.data_ptr())
        return s.out, s.exp
    _encoder(s.be, c["format"])(s.src.data_ptr(), c["rows"] * c["k"], s.out.data_ptr())
    return s.out


_PREPARE = {"host": _prepare_host, "head": _prepare_host, "token": _prepare_token, "knn": _prepare_gates, "walk": _prepare_gates,
            "moe": _prepare_moe, "moe_kq": _prepare_moe_kq, "gemm": _prepare_gemm, "encode": _prepare_encode}
_RUN = {"host": _run_host, "head": _run_head, "token": _run_token, "knn": _run_knn, "walk": _run_walk, "moe": _run_moe,
        "moe_kq": _run_moe_kq, "gemm": _run_gemm, "encode": _run_encode}

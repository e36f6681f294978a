"""The work that a user of this framework has it do, as measurable cases: mixture-of-experts layers in decode and in
prefill, the dense quantized projections beside them, and the activation-quantized forms, each through the public
entry points (dgpp_amd.moe_layer, dgpp_amd.launch) and eagerly, as a serving program's step calls them.

A case is a dict of plain values; listed() names the cases, draw() gives more of the same ranges, prepare() builds the
weights, handles and inputs from a seed, run() is one pass, work() what a pass cannot do without, tolerance() how far
two correct implementations may lie apart.
"""
from __future__ import annotations

import math

import torch

from dgpp_amd import launch as L, moe_layer as ML

DEV = "cuda:0"
WEIGHT_STD = 0.02          # of the matrices before they are quantized
INF = float("inf")

# Contraction lengths that the FP4 forms accept (hidden and intermediate widths in use); block FP8 takes any multiple of
# 16 and is laid out in 128-blocks, MXFP8 any multiple of 32.
FP4_K = {"mxfp4": (512, 576, 1024, 1152, 2048, 2304, 4096, 5120),
         "nvfp4": (512, 640, 768, 1024, 1536, 2048, 2560, 3072, 4096, 5120, 6144, 7168)}
FORMATS = {"fp8": ML.EXPERTS_FP8, "nvfp4": ML.EXPERTS_NVFP4, "mxfp4": ML.EXPERTS_MXFP4}


# ---- the cases ----------------------------------------------------------------------------------------------------

def _moe(name, step, fmt, experts, hidden, inter, tokens, layers=1, top_k=8, shared="none", shared_inter=0, w4a4=False):
    return {"name": name, "kind": "moe", "step": step, "format": fmt, "experts": experts, "hidden": hidden,
            "inter": inter, "top_k": top_k, "tokens": tokens, "layers": layers, "shared": shared,
            "shared_inter": shared_inter, "w4a4": w4a4}


def _dense(name, fmt, m, n, k, layers):
    return {"name": name, "kind": "dense", "format": fmt, "m": m, "n": n, "k": k, "layers": layers}


def listed():
    return [
        # One user generating: a token through the expert layers of a model (each layer has its own weights and rows,
        # so what a layer reads is not in a cache). The smallest calls: launches and latency count.
        _moe("decode_mxfp4_t1", "decode", "mxfp4", 256, 4096, 1024, 1, layers=4),
        # A small serving batch on the same model: the headline of the benchmark.
        _moe("decode_mxfp4_t8", "decode", "mxfp4", 256, 4096, 1024, 8, layers=4),
        # Speculative or few-user decoding of a tensor-parallel slice with a block-FP8 shared expert beside NVFP4 experts.
        _moe("decode_nvfp4_fp8shared_t3", "decode", "nvfp4", 288, 4096, 512, 3, layers=4, shared="fp8", shared_inter=512),
        # A large decode batch: wide NVFP4 experts with an MXFP8 shared expert of its own width.
        _moe("decode_nvfp4_mxfp8shared_t64", "decode", "nvfp4", 256, 6144, 2048, 64, shared="mxfp8", shared_inter=4096),
        # A prompt chunk of a ragged length through block-FP8 experts.
        _moe("prefill_fp8_t777", "prefill", "fp8", 128, 2048, 768, 777, layers=2),
        # A long prompt through the headline model's layer.
        _moe("prefill_mxfp4_t2048", "prefill", "mxfp4", 256, 4096, 1024, 2048),
        # The longest prompt chunk, the tensor-parallel slice with its shared expert.
        _moe("prefill_nvfp4_fp8shared_t4096", "prefill", "nvfp4", 288, 4096, 512, 4096, shared="fp8", shared_inter=512),
        # A prompt chunk with the activations quantized to NVFP4 as well.
        _moe("prefill_w4a4_t512", "prefill", "nvfp4", 256, 6144, 2048, 512, w4a4=True),
        # A single row through an attention-sized FP8 projection, one such matrix per layer.
        _dense("dense_fp8_m1", "fp8", 1, 4096, 4096, 8),
        # A small batch through a dense NVFP4 gate/up projection.
        _dense("dense_nvfp4_m8", "nvfp4", 8, 17408, 5120, 4),
        # A prompt chunk through a large FP8 projection.
        _dense("dense_fp8_m1000", "fp8", 1000, 12288, 6144, 1),
        # The shared expert's MLP with MXFP8 activations, a prompt chunk.
        {"name": "mlp_w8a8_t300", "kind": "mlp_w8a8", "tokens": 300, "hidden": 6144, "inter": 4096, "layers": 2},
    ]


def _cost(case):
    """Roughly the time of a pass at rates that the path reaches with ease: bounds what draw() gives."""
    w = work(case)
    return w["bytes"] / 3e12 + w["flops"] / 60e12


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_once(rng):
    kind = rng.choice(("decode", "decode", "prefill", "prefill", "dense", "dense", "w4a4", "mlp_w8a8"))
    if kind == "mlp_w8a8":
        return {"kind": kind, "tokens": _log_int(rng, 1, 1024), "hidden": 64 * _log_int(rng, 16, 96),
                "inter": 64 * _log_int(rng, 16, 96), "layers": rng.choice((1, 2, 3))}
    if kind == "dense":
        fmt = rng.choice(("fp8", "mxfp8", "nvfp4", "mxfp4"))
        k = rng.choice([v for v in FP4_K[fmt] if v >= 1024]) if fmt in FP4_K else 32 * _log_int(rng, 32, 256)
        n = _log_int(rng, 512, 17408)
        return {"kind": kind, "format": fmt, "m": _log_int(rng, 1, 1024), "n": n, "k": k,
                "layers": max(1, min(8, (128 << 20) // (n * k)))}
    fmt = "nvfp4" if kind == "w4a4" else rng.choice(("fp8", "nvfp4", "mxfp4"))
    if fmt == "fp8":
        hidden, inter = 128 * rng.randint(12, 48), 128 * rng.randint(3, 16)
    else:
        hidden = rng.choice([v for v in FP4_K[fmt] if v >= 1536])
        inter = rng.choice([v for v in FP4_K[fmt] if v <= 2048])
    top_k = rng.choice((4, 6, 8, 8, 10))
    experts = _log_int(rng, 32, 288)
    if kind == "decode":
        tokens, layers = _log_int(rng, 1, 64), rng.choice((1, 2, 3, 4))
    else:
        tokens, layers = _log_int(rng, 17, 4096), rng.choice((1, 1, 2))
    shared, shared_inter = "none", 0
    if kind != "w4a4":
        shared = rng.choice(("none", "none", "fp8", "mxfp8"))
        if shared == "mxfp8" and fmt != "nvfp4":
            shared = "fp8"
        if shared != "none":
            shared_inter = inter if shared == "fp8" and inter % 128 == 0 else 128 * rng.randint(4, 32)
            if shared == "fp8":
                shared_inter = max(128, min(shared_inter, 2048) // 128 * 128)
    case = _moe("", "decode" if kind == "decode" else "prefill", fmt, experts, hidden, inter, tokens, layers, top_k,
                shared, shared_inter, kind == "w4a4")
    del case["name"]
    return case


def draw(rng):
    """A case of the listed ones' ranges: decode batches of 1 to 64 tokens, prompt chunks up to 4096, projections of 1
    to 1024 rows, 32 to 288 experts, ragged sizes among them, no dearer than the dearest listed one."""
    most = max(_cost(c) for c in listed())
    while True:
        case = _draw_once(rng)
        layer_bytes = case["layers"] * (_layer_weight_bytes(case) if case["kind"] == "moe" else 0)
        if _cost(case) <= most and layer_bytes <= 8 << 30:
            return case


# ---- what a pass needs --------------------------------------------------------------------------------------------

def _matrix_bytes(fmt, n, k):
    if fmt == "fp8":
        return n * k + 4 * ((n + 127) // 128) * ((k + 127) // 128)
    if fmt == "mxfp8":
        return n * k + n * (k // 32)
    return n * k // 2 + n * (k // (16 if fmt == "nvfp4" else 32))


def _expert_bytes(fmt, hidden, inter):
    return 2 * _matrix_bytes(fmt, inter, hidden) + _matrix_bytes(fmt, hidden, inter)


def _layer_weight_bytes(c):
    return c["experts"] * _expert_bytes(c["format"], c["hidden"], c["inter"])


def work(case):
    """The bytes (distinct weights, scales, activation rows in and out, each once) and operations of one pass."""
    c = case
    if c["kind"] == "dense":
        m, n, k = c["m"], c["n"], c["k"]
        return {"bytes": c["layers"] * (_matrix_bytes(c["format"], n, k) + 2 * m * (n + k)),
                "flops": c["layers"] * 2.0 * m * n * k}
    T, H = c["tokens"], c["hidden"]
    if c["kind"] == "mlp_w8a8":
        return {"bytes": c["layers"] * (_expert_bytes("mxfp8", H, c["inter"]) + 4 * T * H),
                "flops": c["layers"] * 6.0 * T * H * c["inter"]}
    E, K = c["experts"], c["top_k"]
    distinct = E * (1.0 - (1.0 - K / E) ** T)   # experts that T tokens reach when every expert is as likely
    shared = c["shared_inter"]
    nbytes = distinct * _expert_bytes(c["format"], H, c["inter"]) + 2 * E * H + 4 * T * H
    if shared:
        nbytes += _expert_bytes(c["shared"], H, shared)
    return {"bytes": c["layers"] * nbytes,
            "flops": c["layers"] * (6.0 * T * H * (K * c["inter"] + shared) + 2.0 * T * H * E)}


def tolerance(case):
    """Outputs are BF16 after FP32 sums. Measured between two orders of summation (vector core against matrix core, or
    against float64 products of the same quantized operands): up to 2.2e-4 and one BF16 step (0.8 %) on single values;
    with MXFP8 activations, whose codes step where the BF16 rows between the projections do, 1.6e-3 and 2.8 %."""
    if case["kind"] == "mlp_w8a8":
        return {"rel": 7e-3, "max": 0.12}
    return {"rel": 1e-3, "max": 0.035}


# ---- weights: normally distributed matrices in their published quantized layouts --------------------------------------

def _pow2_exponent(amax, top):
    """ceil(log2(amax / top)) of positive values, as e8m0 exponents."""
    return torch.ceil(torch.log2(torch.clamp(amax, min=1e-30) / top)).clamp(-127, 127)


def _fp4_bytes(q):
    """e2m1 codes (nearest) of values within [-6, 6], two to a byte, the even element in the low nibble."""
    edges = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device=q.device)
    code = torch.bucketize(q.abs(), edges).to(torch.uint8) + (q < 0).to(torch.uint8) * 8
    return code[..., 0::2] | (code[..., 1::2] << 4)


class _Rows:
    """Quantized rows of width k to build matrices of: a matrix takes rows of this pool in a random order, so that
    every expert has memory of its own and payload, scales and their statistics belong together."""

    POOL = 1024

    def __init__(self, g, fmt, k):
        self.fmt, self.k, self.g = fmt, k, g
        w = torch.randn((self.POOL, k), generator=g, device=DEV) * WEIGHT_STD
        self.glob = None
        if fmt == "fp8":
            # one f32 scale per 128 x 128 block: the largest of a block's 16384 normal values on the largest code
            self.payload = torch.clamp(w * (448.0 / (4.4 * WEIGHT_STD)), -448, 448).to(torch.float8_e4m3fn).view(torch.uint8)
            return
        if fmt == "mxfp8":
            v = w.view(self.POOL, k // 32, 32)
            e = _pow2_exponent(v.abs().amax(-1), 448.0)
            self.payload = (v / torch.exp2(e)[..., None]).to(torch.float8_e4m3fn).view(torch.uint8).view(self.POOL, k)
            self.scales = (e + 127).to(torch.uint8)
        elif fmt == "mxfp4":
            v = w.view(self.POOL, k // 32, 32)
            e = _pow2_exponent(v.abs().amax(-1), 6.0)
            self.payload = _fp4_bytes((v / torch.exp2(e)[..., None]).view(self.POOL, k))
            self.scales = (e + 127).to(torch.uint8)
        else:
            v = w.view(self.POOL, k // 16, 16)
            ws2 = v.abs().max() / (6.0 * 448.0)
            s = (v.abs().amax(-1) / 6.0 / ws2).to(torch.float8_e4m3fn)
            self.payload = _fp4_bytes((v / (s.float() * ws2)[..., None]).clamp(-6, 6).view(self.POOL, k))
            self.scales = s.view(torch.uint8)
            self.glob = (1.0 / ws2).reshape(1).float()   # a finished dot is divided by it

    def matrix(self, n):
        """(payload, scales, global or None) of an [n, k] matrix."""
        at = torch.randint(0, self.POOL, (n,), generator=self.g, device=DEV)
        if self.fmt == "fp8":
            jitter = torch.randn(((n + 127) // 128, (self.k + 127) // 128), generator=self.g, device=DEV)
            return self.payload[at], (4.0 + 0.2 * jitter) * (WEIGHT_STD / 448.0), None
        return self.payload[at], self.scales[at], self.glob


def _view(fmt, mat):
    v = L.MoeExpertView()
    v.payload = mat[0].data_ptr()
    if fmt == "fp8":
        v.scales = mat[1].data_ptr()
    else:
        v.fp4_scales = mat[1].data_ptr()
        v.fp4_global = mat[2].data_ptr() if mat[2] is not None else None
    v.scale_shift_rows = v.scale_shift_cols = 7
    v.fp4_group = 32 if fmt == "mxfp4" else 16
    return v


# ---- states --------------------------------------------------------------------------------------------------------

class _MoeLayer:
    """One expert layer as a serving program holds it: weights, layer driver, its batch's rows and output buffer."""

    def __init__(self, c, g, pools):
        fmt, E, H, I, K, T = c["format"], c["experts"], c["hidden"], c["inter"], c["top_k"], c["tokens"]
        self.c, self.keep, views = c, [], []
        gate_up = pools[0].matrix(2 * E * I) if fmt != "fp8" else None
        down = pools[1].matrix(E * H) if fmt != "fp8" else None
        for e in range(E):
            for j in range(3):
                if fmt == "fp8":   # one scale grid per matrix
                    mat = pools[0].matrix(I) if j < 2 else pools[1].matrix(H)
                else:              # rows of one allocation
                    src, n = (gate_up, I) if j < 2 else (down, H)
                    r0 = (2 * e + j) * I if j < 2 else e * H
                    mat = (src[0][r0:r0 + n], src[1][r0:r0 + n], src[2])
                self.keep.append(mat)
                views.append(_view(fmt, mat))
        # Hidden rows have a common part besides what tells them apart: some experts are more popular than others.
        common = 0.5 * torch.randn((1, H), generator=g, device=DEV)
        self.x = (torch.randn((T, H), generator=g, device=DEV) + common).to(torch.bfloat16)
        self.gate = (torch.randn((E, H), generator=g, device=DEV) / math.sqrt(H)).to(torch.bfloat16)
        sigmoid = c["shared"] != "none"   # the families with a shared expert route by sigmoid scores with a bias
        self.bias = 0.05 * torch.randn((E,), generator=g, device=DEV) if sigmoid else None
        self.out = torch.empty((T, H), dtype=torch.bfloat16, device=DEV)
        self.cfg = L.make_config(H, I, E, K, n_shared_experts=1 if c["shared"] != "none" else 0,
                                 routed_scaling_factor=2.5 if sigmoid else 1.0, swiglu_limit=10.0 if sigmoid else INF,
                                 router_mode=L.ROUTER_SIGMOID_BIAS if sigmoid else L.ROUTER_SOFTMAX_TOPK)
        more = {}
        if c["shared"] != "none":
            SI, sh = c["shared_inter"], c["shared"]
            up, dn = _Rows(g, sh, H), _Rows(g, sh, SI)
            mats = [up.matrix(SI), up.matrix(SI), dn.matrix(H)]
            self.keep.append(mats)
            more = {"shared_inter": SI, "sh_payload": tuple(m[0] for m in mats),
                    ("sh_scales" if sh == "fp8" else "sh_scales_e8m0"): tuple(m[1] for m in mats)}
        self.layer = ML.MoeLayer(self.cfg, FORMATS[fmt], views, T, router_gate=self.gate, router_bias=self.bias, **more)
        if c["w4a4"]:
            self.ids = torch.empty((T, K), dtype=torch.int32, device=DEV)
            self.weights = torch.empty((T, K), dtype=torch.float32, device=DEV)
            self.scores, self.biased = (torch.empty((T, E), dtype=torch.float32, device=DEV) for _ in range(2))

    def step(self):
        c, T, H = self.c, self.c["tokens"], self.c["hidden"]
        if c["w4a4"]:
            L.launch_moe_router(self.x, self.gate, self.bias, self.ids, self.weights, self.scores, self.biased, self.cfg, T)
            self.layer.enqueue_prefill_routed_w4a4(self.x, H, self.ids, self.weights, self.out, T)
        elif c["step"] == "decode":
            self.layer.enqueue_decode(self.x, H, self.out, T)
        else:
            self.layer.enqueue_prefill(self.x, H, self.out, T)
        return self.out


class _Dense:
    """One dense projection: out[m, n] = act[m, k] * W[n, k]^T over a quantized W."""

    def __init__(self, c, g, pools):
        m, n, k = c["m"], c["n"], c["k"]
        self.c = c
        self.w = pools[0].matrix(n)
        self.x = torch.randn((m, k), generator=g, device=DEV).to(torch.bfloat16)
        self.out = torch.empty((m, n), dtype=torch.bfloat16, device=DEV)
        if c["format"] in FP4_K:
            group = 16 if c["format"] == "nvfp4" else 32
            glob = self.w[2].data_ptr() if self.w[2] is not None else None
            self.mat = L.Fp4Matrix(self.w[0].data_ptr(), self.w[1].data_ptr(), glob, n, k, group, 0, None)

    def step(self):
        c, m, n, k = self.c, self.c["m"], self.c["n"], self.c["k"]
        if c["format"] in FP4_K:
            L.launch_fp4_gemv_bf16(self.x, k, self.mat, self.out, m, n, k)
        elif c["format"] == "fp8":
            L.launch_scale_gemm_bf16(self.x, k, self.w[0], self.w[1], self.out, m, n, k)
        else:
            L.launch_scale_gemm_grid_e8m0_bf16(self.x, k, self.w[0], self.w[1], self.out, m, n, k, None, n, 0, 5)
        return self.out


class _MlpW8A8:
    """An MLP with MXFP8 weights and activations: quantize, gate, up, SwiGLU + quantize, down."""

    def __init__(self, c, g, pools):
        T, H, I = c["tokens"], c["hidden"], c["inter"]
        self.c = c
        self.w = [pools[0].matrix(I), pools[0].matrix(I), pools[1].matrix(H)]
        self.x = torch.randn((T, H), generator=g, device=DEV).to(torch.bfloat16)
        self.xq, self.aq = (torch.empty((T, d), dtype=torch.uint8, device=DEV) for d in (H, I))
        self.xs, self.as_ = (torch.empty((T, d // 32), dtype=torch.uint8, device=DEV) for d in (H, I))
        self.g, self.u = (torch.empty((T, I), dtype=torch.bfloat16, device=DEV) for _ in range(2))
        self.out = torch.empty((T, H), dtype=torch.bfloat16, device=DEV)

    def step(self):
        T, H, I = self.c["tokens"], self.c["hidden"], self.c["inter"]
        (wg, sg, _), (wu, su, _), (wd, sd, _) = self.w
        L.launch_mxfp8_quantize_rows(self.x, H, T, H, self.xq, self.xs)
        L.launch_mxfp8_gemm_bf16(self.xq, self.xs, wg, sg, self.g, T, I, H)
        L.launch_mxfp8_gemm_bf16(self.xq, self.xs, wu, su, self.u, T, I, H)
        L.launch_minimax_swiglu_mxfp8_rows(self.g, self.u, I, T, I, 1.702, 7.0, self.aq, self.as_)
        L.launch_mxfp8_gemm_bf16(self.aq, self.as_, wd, sd, self.out, T, H, I)
        return self.out


def prepare(case, seed):
    """A model's worth of the case: `layers` layers, each with weights, rows and buffers of its own."""
    c = dict(case)
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    if c["kind"] == "dense":
        pools, make = [_Rows(g, c["format"], c["k"])], _Dense
    elif c["kind"] == "mlp_w8a8":
        pools, make = [_Rows(g, "mxfp8", c["hidden"]), _Rows(g, "mxfp8", c["inter"])], _MlpW8A8
    else:
        pools, make = [_Rows(g, c["format"], c["hidden"]), _Rows(g, c["format"], c["inter"])], _MoeLayer
    return [make(c, g, pools) for _ in range(c["layers"])]


def run(state):
    """One pass: every layer's step over its own rows, on the current stream, nothing waited for."""
    return [layer.step() for layer in state]

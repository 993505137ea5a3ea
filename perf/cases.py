"""Performance cases: the calls a program on libfmx makes, with their inputs.

Every case is one call of the C ABI (include/fmx.h) through freemoe_amd.fmx on
tensors resident on the GPU:

  decode     fmx_moe_decode, one token through one MoE layer
  prefill    fmx_moe_prefill, a prompt's tokens through one MoE layer
  matvec     fmx_matvec, one projection of one token (attention projections,
             the output head)
  gemm       fmx_gemm_quant, one projection of a prompt (the dense batched
             prefill)
  attention  fmx_attention_decode, one token over its cached positions

Weights are quantised blocks whose values are centred with a standard
deviation near 1 / sqrt(inputs), as trained projections are; activations are
N(0, 1) before the layer's RMSNorm and 0.5 N(0, 1) in attention.
"""
import ctypes
import math

import torch

from freemoe_amd import fmx
from freemoe_amd.device import pack

F32, Q4_0, Q8_0, Q4_K, Q6_K = 0, 2, 8, 12, 14
TYPES = {"f32": F32, "q4_0": Q4_0, "q8_0": Q8_0, "q4_k": Q4_K, "q6_k": Q6_K}
BLOCK = {"f32": (1, 4), "q4_0": (32, 18), "q8_0": (32, 34), "q4_k": (256, 144), "q6_k": (256, 210)}
RMS_EPS = 1e-5
WEIGHT_EPS = 6.103515625e-5

TINY = dict(hidden=64, ffn=128, experts=4, top_k=2, zipf=0.0)
MIXTRAL = dict(hidden=4096, ffn=14336, experts=8, top_k=2, zipf=0.0)
FINE = dict(hidden=2048, ffn=768, experts=128, top_k=8, zipf=1.2)


def _layer_case(name, kind, shape, gate, down, tokens):
    return dict(name=name, kind=kind, gate=gate, down=down, tokens=tokens, **shape)


def listed():
    return [
        # the smallest call: one token of the freemoe-tiny-v1 block, all latency
        _layer_case("decode_tiny_f32", "decode", TINY, "f32", "f32", 1),
        # the headline: one token of a Mixtral-shaped layer with Q4_0 experts
        _layer_case("decode_mixtral_q4_0", "decode", MIXTRAL, "q4_0", "q4_0", 1),
        # the mixed k-quant files: Q4_K gate / up with Q6_K down
        _layer_case("decode_mixtral_q4_k_q6_k", "decode", MIXTRAL, "q4_k", "q6_k", 1),
        # one token of a fine-grained layer: many small experts, launch bound
        _layer_case("decode_finegrained_q4_k", "decode", FINE, "q4_k", "q4_k", 1),
        # a short chat turn's prompt: a few rows per expert, every expert read
        _layer_case("prefill_mixtral_q4_0_33", "prefill", MIXTRAL, "q4_0", "q4_0", 33),
        # an ordinary prompt on the largest layer
        _layer_case("prefill_mixtral_q8_0_512", "prefill", MIXTRAL, "q8_0", "q8_0", 512),
        # a long prompt on the fine-grained layer: ragged, 0 to 2000 rows per expert
        _layer_case("prefill_finegrained_q4_k_2048", "prefill", FINE, "q4_k", "q4_k", 2048),
        # an attention projection of one token
        dict(name="matvec_q8_0_4096x4096", kind="matvec", type="q8_0", rows=4096, cols=4096),
        # the same in F32, as the 8-layer decoder keeps them
        dict(name="matvec_f32_4096x4096", kind="matvec", type="f32", rows=4096, cols=4096),
        # the output head over a 32000-entry vocabulary
        dict(name="matvec_q6_k_32000x4096", kind="matvec", type="q6_k", rows=32000, cols=4096),
        # an attention projection of a prompt
        dict(name="gemm_q8_0_4096x4096_256", kind="gemm", type="q8_0", rows=4096, cols=4096, tokens=256),
        # one token's attention in the middle of a long conversation
        dict(name="attention_32_of_8x128_2000", kind="attention", heads=32, kv_heads=8, head_dim=128, positions=2000),
    ]


def _log_int(rng, lo, hi, unit=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / unit)) * unit))


# Multiply-adds of the largest listed case, and its expert elements: what a
# drawn case may reach.
MAX_MACS = 512 * 2 * 3 * 4096 * 14336
MAX_ELEMENTS = 8 * 3 * 4096 * 14336


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "prefill", "matvec", "matvec", "gemm",
                       "attention"])
    if kind in ("decode", "prefill"):
        gate, down = rng.choice([("q4_0", "q4_0"), ("q4_0", "q4_0"), ("q8_0", "q8_0"), ("q4_k", "q4_k"),
                                 ("q4_k", "q6_k"), ("q6_k", "q6_k")])
        unit = max(BLOCK[gate][0], BLOCK[down][0])
        if kind == "prefill":
            unit = 256
        if rng.random() < 0.5:  # few large experts
            hidden, ffn = _log_int(rng, 1024, 4096, unit), _log_int(rng, 2048, 14336, unit)
            experts, top_k, zipf = rng.choice([4, 8, 16]), rng.choice([1, 2, 2, 4]), 0.0
        else:  # many small ones
            hidden, ffn = _log_int(rng, 1024, 4096, unit), _log_int(rng, 512, 2048, unit)
            experts, top_k, zipf = rng.choice([32, 60, 64, 128]), rng.choice([4, 6, 8]), rng.choice([0.0, 1.2])
        while experts * 3 * hidden * ffn > MAX_ELEMENTS:
            experts //= 2
        tokens = 1
        if kind == "prefill":
            tokens = _log_int(rng, 2, 2048)
            tokens = max(1, min(tokens, MAX_MACS // (top_k * 3 * hidden * ffn)))
        return dict(kind=kind, hidden=hidden, ffn=ffn, experts=experts, top_k=min(top_k, experts), zipf=zipf,
                    gate=gate, down=down, tokens=tokens)
    if kind in ("matvec", "gemm"):
        t = rng.choice(["f32", "q4_0", "q8_0", "q4_k", "q6_k"])
        unit = 4 if t == "f32" else BLOCK[t][0]
        case = dict(kind=kind, type=t, rows=_log_int(rng, 256, 32000), cols=_log_int(rng, 512, 14336, unit))
        if kind == "gemm":
            case["rows"] = min(case["rows"], 14336)
            case["tokens"] = max(1, min(_log_int(rng, 2, 512), (1 << 34) // (case["rows"] * case["cols"])))
        return case
    kv_heads = rng.choice([1, 2, 4, 8, 32])
    heads = kv_heads * rng.choice([1, 4]) if kv_heads < 32 else 32
    return dict(kind="attention", heads=heads, kv_heads=kv_heads, head_dim=rng.choice([64, 96, 128, 256]),
                positions=_log_int(rng, 16, 8192))


# ------------------------------------------------------------------ inputs --

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _half_bytes(v):
    return v.to(torch.float16).view(torch.uint8).reshape(-1, 2)


def _matrix(t, g, rows, cols):
    """A [rows x cols] matrix as raw GGUF bytes (uint8 [rows, row bytes]),
    values of standard deviation about 1 / sqrt(cols)."""
    sigma = 1.0 / math.sqrt(cols)
    if t == "f32":
        return (_randn(g, rows, cols) * sigma).view(torch.uint8)
    bs, bb = BLOCK[t]
    n = rows * cols // bs
    jitter = 1.0 + 0.2 * torch.rand(n, generator=g, device="cuda")
    w = torch.empty((n, bb), dtype=torch.uint8, device="cuda")
    if t == "q8_0":
        w[:, :2] = _half_bytes(jitter * (sigma / 40.0))
        w[:, 2:] = (_randn(g, n, 32) * 40.0).round_().clamp_(-127, 127).to(torch.int8).view(torch.uint8)
    elif t == "q4_0":
        w[:, :2] = _half_bytes(jitter * (sigma / 2.7))
        q = (_randn(g, n, 32) * 2.7).round_().clamp_(-8, 7).add_(8).to(torch.uint8)
        w[:, 2:] = q[:, :16] | (q[:, 16:] << 4)
    elif t == "q4_k":
        # value d sc q - dmin m: sc and m uniform in 0..63, q in 0..15
        w[:, :] = torch.randint(0, 256, (n, bb), generator=g, device="cuda", dtype=torch.uint8)
        w[:, :2] = _half_bytes(jitter * (sigma / 257.0))
        w[:, 2:4] = _half_bytes(jitter * (7.5 * sigma / 257.0))
    else:  # q6_k: value d sc (q - 32): sc uniform int8, q uniform in 0..63
        w[:, :] = torch.randint(0, 256, (n, bb), generator=g, device="cuda", dtype=torch.uint8)
        w[:, 208:] = _half_bytes(jitter * (sigma / (73.0 * 18.5)))
    return w.reshape(rows, -1)


class _Layer:
    """One MoE layer's raw weights and inputs, all made from the seed."""

    def __init__(self, case, seed):
        g = _generator(seed)
        H, F, E, T = case["hidden"], case["ffn"], case["experts"], case["tokens"]
        self.x = _randn(g, T, H)
        self.norm = 1.0 + 0.02 * _randn(g, H)
        self.router = _randn(g, E, H) / math.sqrt(H)
        self.bias = None
        if case["zipf"]:
            ranks = torch.randperm(E, generator=g, device="cuda").to(torch.float32) + 1.0
            self.bias = -case["zipf"] * torch.log(ranks)
        self.g = g
        self.shapes = (("gate", case["gate"], F, H), ("up", case["gate"], F, H), ("down", case["down"], H, F))
        self.experts = E

    def matrices(self):
        """(expert, projection, type, rows, cols, raw) in a fixed order."""
        for e in range(self.experts):
            for name, t, rows, cols in self.shapes:
                yield e, name, t, rows, cols, _matrix(t, self.g, rows, cols)


def _prepare_layer(case, seed):
    layer = _Layer(case, seed)
    slots = {"gate": [], "up": [], "down": []}
    for _, name, t, rows, cols, raw in layer.matrices():
        slots[name].append(pack(TYPES[t], raw, rows, cols))
    table = torch.tensor([[m.data_ptr() for m in slots[n]] for n in ("gate", "up", "down")], dtype=torch.int64,
                         device="cuda")
    gate, down = TYPES[case["gate"]], TYPES[case["down"]]
    desc = fmx.MoELayer(case["hidden"], case["ffn"], case["experts"], case["top_k"], layer.norm.data_ptr(), RMS_EPS,
                        0.0, F32, layer.router.data_ptr(), fmx.ptr(layer.bias), 1, 0, WEIGHT_EPS, 1.0, gate, gate,
                        down, table[0].data_ptr(), table[1].data_ptr(), table[2].data_ptr())
    T, K = case["tokens"], case["top_k"]
    prefill = case["kind"] == "prefill"
    need = fmx.lib().fmx_moe_prefill_workspace_bytes if prefill else fmx.lib().fmx_moe_workspace_bytes
    nbytes = need(ctypes.byref(desc), T)
    return dict(entry="fmx_moe_prefill" if prefill else "fmx_moe_decode", desc=desc, tokens=T, x=layer.x,
                out=torch.empty_like(layer.x), ids=torch.empty((T, K), dtype=torch.int32, device="cuda"),
                weights=torch.empty((T, K), dtype=torch.float32, device="cuda"),
                workspace=torch.zeros(nbytes, dtype=torch.uint8, device="cuda"), workspace_bytes=nbytes,
                held=(slots, table, layer.norm, layer.router, layer.bias))


def _matrix_inputs(case, seed):
    g = _generator(seed)
    raw = _matrix(case["type"], g, case["rows"], case["cols"])
    return raw, _randn(g, case.get("tokens", 1), case["cols"])


def _attention_inputs(case, seed):
    g = _generator(seed)
    kv_dim = case["kv_heads"] * case["head_dim"]
    kv = 0.5 * _randn(g, case["positions"], 2 * kv_dim)
    return kv, 0.5 * _randn(g, case["heads"] * case["head_dim"])


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        return dict(kind=kind, **_prepare_layer(case, seed))
    if kind == "attention":
        kv, q = _attention_inputs(case, seed)
        return dict(kind=kind, kv=kv, q=q, case=dict(case), out=torch.empty_like(q),
                    workspace=torch.zeros(256, dtype=torch.uint8, device="cuda"))
    raw, x = _matrix_inputs(case, seed)
    t = TYPES[case["type"]]
    if kind == "matvec":
        raw = pack(t, raw, case["rows"], case["cols"])
    return dict(kind=kind, type=t, rows=case["rows"], cols=case["cols"], w=raw, x=x,
                y=torch.empty((x.shape[0], case["rows"]), dtype=torch.float32, device="cuda"))


def run(state):
    kind = state["kind"]
    if kind in ("decode", "prefill"):
        fmx.call(state["entry"], ctypes.byref(state["desc"]), state["x"].data_ptr(), state["out"].data_ptr(),
                 state["tokens"], state["ids"].data_ptr(), state["weights"].data_ptr(),
                 state["workspace"].data_ptr(), state["workspace_bytes"], fmx.stream_handle())
        return {"out": state["out"], "ids": state["ids"], "weights": state["weights"]}
    if kind == "matvec":
        fmx.call("fmx_matvec", state["type"], state["w"].data_ptr(), state["x"].data_ptr(), state["y"].data_ptr(),
                 state["rows"], state["cols"], fmx.stream_handle())
        return state["y"]
    if kind == "gemm":
        fmx.call("fmx_gemm_quant", state["type"], state["w"].data_ptr(), state["x"].data_ptr(),
                 state["y"].data_ptr(), state["x"].shape[0], state["rows"], state["cols"], fmx.stream_handle())
        return state["y"]
    c, kv = state["case"], state["kv"]
    fmx.call("fmx_attention_decode", state["q"].data_ptr(), kv.data_ptr(), kv.shape[1], kv.shape[1] // 2, c["heads"],
             c["kv_heads"], c["head_dim"], c["positions"], 1.0 / math.sqrt(c["head_dim"]), state["out"].data_ptr(),
             state["workspace"].data_ptr(), 256, fmx.stream_handle())
    return state["out"]


# -------------------------------------------------------------------- work --

def _bytes(t, rows, cols):
    bs, bb = BLOCK[t]
    return rows * (cols // bs) * bb


def work(case):
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        H, F, E, K, T = (case[k] for k in ("hidden", "ffn", "experts", "top_k", "tokens"))
        expert = 2 * _bytes(case["gate"], F, H) + _bytes(case["down"], H, F)
        hit = K if T == 1 else E * (1.0 - (1.0 - K / E) ** T)  # experts some token chose
        return {"bytes": int(hit * expert) + 4 * E * H + 8 * T * H + 8 * T * K,
                "flops": 2 * T * (3 * K * H * F + E * H)}
    if kind in ("matvec", "gemm"):
        R, C, T = case["rows"], case["cols"], case.get("tokens", 1)
        return {"bytes": _bytes(case["type"], R, C) + 4 * T * (R + C), "flops": 2 * T * R * C}
    n = case["head_dim"] * case["positions"]
    return {"bytes": 8 * case["kv_heads"] * n + 8 * case["heads"] * case["head_dim"], "flops": 4 * case["heads"] * n}


def tolerance(case):
    # Prefill multiplies in bf16 (8-bit significands of weights and
    # activations) with f32 sums: 1.4e-3 to 2.1e-3 from exact() over the listed
    # and a few drawn cases. Every other path reproduces the reference's order
    # of operations bit for bit, whatever the kernel.
    if case["kind"] == "prefill":
        return {"rel": 8e-3}
    return "exact"


# ------------------------------------------------------------------- exact --

def _dequantize(t, raw):
    """Raw GGUF rows (uint8 [rows, row bytes]) -> float64 [rows, cols]."""
    rows = raw.shape[0]
    if t == "f32":
        return raw.view(torch.float32).to(torch.float64)
    b = raw.reshape(-1, BLOCK[t][1])

    def half(o):
        return b[:, o:o + 2].contiguous().view(torch.float16).to(torch.float64)

    if t == "q8_0":
        v = half(0) * b[:, 2:].contiguous().view(torch.int8).to(torch.float64)
    elif t == "q4_0":
        q = torch.cat((b[:, 2:] & 15, b[:, 2:] >> 4), dim=1).to(torch.float64)
        v = half(0) * (q - 8.0)
    elif t == "q4_k":
        s = b[:, 4:16]
        sc = torch.cat((s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)), dim=1).to(torch.float64)
        m = torch.cat((s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)), dim=1).to(torch.float64)
        qs = b[:, 16:].reshape(-1, 4, 32)
        q = torch.stack((qs & 15, qs >> 4), dim=2).reshape(-1, 8, 32).to(torch.float64)
        v = (half(0) * sc)[:, :, None] * q - (half(2) * m)[:, :, None]
    else:  # q6_k: per half, low nibbles of 64 bytes then high, two more bits from qh
        ql = b[:, :128].reshape(-1, 2, 64)
        qh = b[:, 128:192].reshape(-1, 2, 1, 32)
        low = torch.cat((ql & 15, ql >> 4), dim=2).reshape(-1, 2, 4, 32)
        shift = torch.tensor([0, 2, 4, 6], dtype=torch.uint8, device=raw.device).reshape(1, 1, 4, 1)
        q = (low | (((qh >> shift) & 3) << 4)).reshape(-1, 16, 16).to(torch.float64) - 32.0
        sc = b[:, 192:208].contiguous().view(torch.int8).to(torch.float64)
        v = (half(208) * sc)[:, :, None] * q
    return v.reshape(rows, -1)


def _exact_layer(case, seed):
    layer = _Layer(case, seed)
    K = case["top_k"]
    x = layer.x.to(torch.float64)
    h = x / torch.sqrt((x * x).mean(dim=1, keepdim=True) + RMS_EPS) * layer.norm.to(torch.float64)
    logits = h @ layer.router.to(torch.float64).t()
    if layer.bias is not None:
        logits = logits + layer.bias.to(torch.float64)
    probs, ids = torch.topk(torch.softmax(logits, dim=1), K, dim=1)
    weights = probs / probs.sum(dim=1, keepdim=True).clamp_min(WEIGHT_EPS)
    out = x.clone()
    held = {}
    for e, name, t, _, _, raw in layer.matrices():
        token, rank = torch.nonzero(ids == e, as_tuple=True)
        if token.numel() == 0:
            continue
        held[name] = _dequantize(t, raw)
        if name == "down":
            he = h[token]
            gate, up = he @ held["gate"].t(), he @ held["up"].t()
            y = (gate * torch.sigmoid(gate) * up) @ held["down"].t()
            out.index_add_(0, token, y * weights[token, rank][:, None])
            held = {}
    return {"out": out, "ids": None, "weights": weights}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        return _exact_layer(case, seed)
    if kind in ("matvec", "gemm"):
        raw, x = _matrix_inputs(case, seed)
        return x.to(torch.float64) @ _dequantize(case["type"], raw).t()
    kv, q = _attention_inputs(case, seed)
    D, KV = case["head_dim"], case["kv_heads"]
    kv = kv.to(torch.float64).reshape(case["positions"], 2, KV, D)
    q = q.to(torch.float64).reshape(case["heads"], D)
    group = case["heads"] // KV
    rows = []
    for head in range(case["heads"]):
        keys, values = kv[:, 0, head // group].contiguous(), kv[:, 1, head // group].contiguous()
        p = torch.softmax(keys @ q[head] / math.sqrt(D), dim=0)
        rows.append(values.t().contiguous() @ p)
    return torch.cat(rows)

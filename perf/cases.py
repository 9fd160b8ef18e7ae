"""Workloads of the weight-only quantized matmul path, as a program that serves or prefills with it calls it.

A case is a dict of plain values; `prepare` builds its weights and inputs from a seed, `run` makes one pass through the
public wrappers (`qengine_amd.ops`), `exact` is the same pass in 64-bit torch arithmetic, `work` the bytes and
operations the pass cannot do without, `tolerance` what two correct implementations at the same precision may differ by.

Kinds:
  mlp     a gated MLP block of INT4 matrices: gate_up (GLU) then down, 1 row (decode) to thousands (prefill)
  linear  one INT4 matrix through the row-count dispatch (decode up to 64 rows, the prefill GEMM above)
  w8      one INT8 matrix, bf16 activations: decode up to 16 rows, the GEMM above
  w8a8    one INT8 matrix with activations quantized per (row, 128 k), the row GEMM used for prefill
  w4a8    one INT4 matrix with activations quantized per (token, G k), the reference's default prefill numerics
  moe     one layer of INT4 experts: top-k routing, gate_up, down, combine

Sizes: hidden 5120 / intermediate 17408 (and their C0 / C2 matrices), INT8 8192 x 2048 and the 512-expert top-10 layer
are the workloads of bench.py; the drawn ones are generic sizes around them.
"""
import math

import torch

from qengine_amd import ops

DEV = "cuda"


# ------------------------------------------------------------------------------------------------ cases
def listed():
    return [
        # one sequence generating: each token passes every block's MLP with one row, the latency of a token
        {"name": "mlp_decode_1", "kind": "mlp", "hidden": 5120, "inter": 17408, "rows": 1, "scales": "f16"},
        # a dozen sequences decoded together (an odd batch, not a power of two)
        {"name": "mlp_decode_12", "kind": "mlp", "hidden": 5120, "inter": 17408, "rows": 12, "scales": "f16"},
        # a full decode batch of a busy server
        {"name": "mlp_decode_48", "kind": "mlp", "hidden": 5120, "inter": 17408, "rows": 48, "scales": "f16"},
        # the prefill of one short chat turn, or a decode batch past 64 sequences
        {"name": "mlp_prefill_200", "kind": "mlp", "hidden": 5120, "inter": 17408, "rows": 200, "scales": "f16"},
        # a chunk of a chunked prefill, ragged at its end
        {"name": "mlp_prefill_1000", "kind": "mlp", "hidden": 5120, "inter": 17408, "rows": 1000, "scales": "f16"},
        # a long prompt in one call, bench.py's prefill matrix
        {"name": "linear_prefill_8192", "kind": "linear", "n": 17408, "k": 5120, "rows": 8192, "scales": "f16",
         "out": "bf16"},
        # the smallest call: one row of an INT8 matrix
        {"name": "w8_decode_1", "kind": "w8", "n": 8192, "k": 2048, "rows": 1, "per_channel": True, "out": "bf16"},
        # prefill of the same INT8 matrix with bf16 activations
        {"name": "w8_prefill_4096", "kind": "w8", "n": 8192, "k": 2048, "rows": 4096, "per_channel": True,
         "out": "bf16"},
        # prefill of the same INT8 matrix with the reference's INT8 row numerics
        {"name": "w8a8_prefill_4096", "kind": "w8a8", "n": 8192, "k": 2048, "rows": 4096, "per_channel": True,
         "out": "f32"},
        # a prompt with the reference's default INT4 prefill numerics (activation groups of 64)
        {"name": "w4a8_prefill_2048", "kind": "w4a8", "n": 17408, "k": 5120, "rows": 2048, "group": 64,
         "scales": "f16", "out": "bf16"},
        # a small decode batch of a mixture-of-experts layer: about 140 of the 512 experts are hit
        {"name": "moe_decode_16", "kind": "moe", "experts": 512, "topk": 10, "hidden": 2048, "inter": 512,
         "rows": 16},
        # a prompt through the same layer: every expert gets about 80 rows
        {"name": "moe_prefill_4096", "kind": "moe", "experts": 512, "topk": 10, "hidden": 2048, "inter": 512,
         "rows": 4096},
    ]


MOST_FLOPS = 2.0 * 8192 * 17408 * 5120  # of the largest listed case
MOST_MOE_FLOPS = 6.0 * 4096 * 10 * 2048 * 512
MOST_MOE_WEIGHTS = 512 * 3 * 2048 * 512


def _log(rng, lo, hi, step=1):
    """a multiple of `step` in [lo, hi], spread over the logarithm"""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return int(min(hi, max(lo, step * round(v / step))))


def draw(rng):
    kind = rng.choice(["mlp", "mlp", "mlp", "linear", "linear", "w8", "w8a8", "w4a8", "moe", "moe"])
    while True:
        if kind == "mlp":
            c = {"kind": kind, "hidden": _log(rng, 1024, 8192, 128), "inter": _log(rng, 1024, 24576, 128),
                 "rows": _log(rng, 1, 8192), "scales": rng.choice(["f16", "bf16"])}
        elif kind == "linear":
            c = {"kind": kind, "n": _log(rng, 1024, 34816, 16), "k": _log(rng, 1024, 17408, 128),
                 "rows": _log(rng, 1, 8192), "scales": rng.choice(["f16", "bf16"]), "out": rng.choice(["bf16", "f32"])}
        elif kind == "w8":
            c = {"kind": kind, "n": _log(rng, 1024, 16384, 16), "k": _log(rng, 1024, 8192, 128),
                 "rows": _log(rng, 1, 4096), "per_channel": rng.random() < 0.5, "out": rng.choice(["bf16", "f32"])}
        elif kind == "w8a8":
            c = {"kind": kind, "n": _log(rng, 1024, 16384, 16), "k": _log(rng, 1024, 4096, 128),
                 "rows": _log(rng, 64, 4096), "per_channel": rng.random() < 0.5, "out": rng.choice(["bf16", "f32"])}
        elif kind == "w4a8":
            c = {"kind": kind, "n": _log(rng, 1024, 17408, 16), "k": _log(rng, 1024, 17408, 128),
                 "rows": _log(rng, 65, 8192), "group": rng.choice([32, 64, 64, 128]),
                 "scales": rng.choice(["f16", "bf16"]), "out": rng.choice(["bf16", "f32"])}
        else:
            c = {"kind": kind, "experts": rng.choice([32, 64, 128, 256, 512]), "topk": rng.randint(2, 10),
                 "hidden": _log(rng, 1024, 4096, 512), "inter": rng.choice([256, 384, 512, 640, 768, 896, 1024, 2048]),
                 "rows": _log(rng, 1, 4096)}
            if (work(c)["flops"] > MOST_MOE_FLOPS
                    or c["experts"] * 3 * c["hidden"] * c["inter"] > MOST_MOE_WEIGHTS):
                continue
        # INT8 matrices and activation groups of 32 run at about half the rate of the largest case
        if work(c)["flops"] <= MOST_FLOPS / (1 if kind in ("mlp", "linear", "moe") else 2):
            return c


# ------------------------------------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _x(g, rows, k):
    return torch.randn(rows, k, device=DEV, generator=g).bfloat16()


def _int4(g, n, k, dtype, lead=()):
    """weights N(0, 1 / k) rounded to INT4 with one scale per (row, 128 k): (u = w + 8 packed as compressed-tensors
    int32 [.., n, k / 8], scales [.., n, k / 128])"""
    w = torch.randn(*lead, n, k // 128, 128, device=DEV, generator=g) * (k ** -0.5)
    s = (w.abs().amax(-1) / 7.5).to(dtype)
    u = (w / s.float().unsqueeze(-1)).round_().clamp_(-8, 7).add_(8).to(torch.int32).view(*lead, n, k // 8, 8)
    q = u[..., 0].clone()
    for j in range(1, 8):
        q |= u[..., j] << (4 * j)
    return q, s


def _int8(g, n, k, per_channel):
    """weights N(0, 1 / k) rounded to INT8 with one fp16 scale per row, or bf16 per (row, 128 k)"""
    w = torch.randn(n, 1 if per_channel else k // 128, k if per_channel else 128, device=DEV, generator=g) * (k ** -0.5)
    s = (w.abs().amax(-1) / 127).to(torch.float16 if per_channel else torch.bfloat16)
    q = (w / s.float().unsqueeze(-1)).round_().clamp_(-127, 127).to(torch.int8).view(n, k)
    return q, s.view(n) if per_channel else s


SCALES = {"f16": torch.float16, "bf16": torch.bfloat16}
OUT = {"bf16": torch.bfloat16, "f32": torch.float32}


def _sources(case, seed):
    """the matrices and activations as a checkpoint and a producing layer hold them"""
    g = _gen(seed)
    kind, rows = case["kind"], case["rows"]
    if kind == "mlp":
        h, i = case["hidden"], case["inter"]
        gu = _int4(g, 2 * i, h, SCALES[case["scales"]])
        dn = _int4(g, h, i, SCALES[case["scales"]])
        return {"gu": gu, "dn": dn, "x": _x(g, rows, h)}
    if kind in ("linear", "w4a8"):
        return {"w": _int4(g, case["n"], case["k"], SCALES[case["scales"]]), "x": _x(g, rows, case["k"])}
    if kind in ("w8", "w8a8"):
        return {"w": _int8(g, case["n"], case["k"], case["per_channel"]), "x": _x(g, rows, case["k"])}
    e, h, i = case["experts"], case["hidden"], case["inter"]
    step = max(1, (64 << 20) // (2 * i * h))  # experts made at a time
    parts = []
    for e0 in range(0, e, step):
        ne = min(step, e - e0)
        parts.append(_int4(g, 2 * i, h, torch.float16, (ne,)) + _int4(g, h, i, torch.float16, (ne,)))
    gq, gs, dq, ds = (torch.cat(p) for p in zip(*parts))
    return {"gq": gq, "gs": gs, "dq": dq, "ds": ds, "logits": torch.randn(rows, e, device=DEV, generator=g),
            "x": _x(g, rows, h)}


def prepare(case, seed):
    src = _sources(case, seed)
    kind, rows = case["kind"], case["rows"]
    st = {"kind": kind, "rows": rows, "x": src["x"], "bf16": case.get("out", "bf16") == "bf16"}
    if kind == "mlp":
        st["gu"] = ops.repack_w4(*ops.glu_rows(*src["gu"]), glu=True)
        st["dn"] = ops.repack_w4(*src["dn"])
        st["act"] = torch.empty(rows, case["inter"], dtype=torch.bfloat16, device=DEV)
        st["y"] = torch.empty(rows, case["hidden"], dtype=torch.bfloat16, device=DEV)
    elif kind in ("linear", "w4a8"):
        st["w"] = ops.repack_w4(*src["w"])
        st["group"] = case.get("group")
        st["y"] = torch.empty(rows, case["n"], dtype=OUT[case["out"]], device=DEV)
    elif kind in ("w8", "w8a8"):
        st["w"] = ops.tile_w8(*src["w"], per_channel=case["per_channel"])
        st["y"] = torch.empty(rows, case["n"], dtype=OUT[case["out"]], device=DEV)
    else:
        st["moe"] = ops.MoE.pack(src["gq"], src["gs"], src["dq"], src["ds"], case["topk"])
        st["logits"] = src["logits"]
        st["y"] = torch.empty(rows, case["hidden"], dtype=torch.bfloat16, device=DEV)
    return st


# ------------------------------------------------------------------------------------------------ the pass
def run(st):
    kind, x, bf16, y = st["kind"], st["x"], st["bf16"], st["y"]
    if kind == "mlp":
        act = ops.matmul_w4(st["gu"], x, out_bf16=True, y=st["act"])
        return {"act": act, "y": ops.matmul_w4(st["dn"], act, out_bf16=True, y=y)}
    if kind == "linear":
        return ops.matmul_w4(st["w"], x, out_bf16=bf16, y=y)
    if kind == "w8":
        return (ops.gemv_w8 if st["rows"] <= 16 else ops.gemm_w8)(st["w"], x, out_bf16=bf16, y=y)
    if kind == "w8a8":
        return ops.gemm_w8a8(st["w"], x, out_bf16=bf16, y=y)
    if kind == "w4a8":
        return ops.gemm_w4_i8(st["w"], x, G=st["group"], out_bf16=bf16, y=y)
    return st["moe"](st["logits"], x, out_bf16=True, out=y)


# ------------------------------------------------------------------------------------------------ work
def _w4_bytes(n, k):
    return n * k // 2 + n * (k // 128) * 2


def work(case):
    kind, t = case["kind"], case["rows"]
    if kind == "mlp":
        h, i = case["hidden"], case["inter"]
        return {"bytes": _w4_bytes(2 * i, h) + _w4_bytes(h, i) + 2 * t * (2 * h + i), "flops": 6.0 * t * h * i}
    if kind == "moe":
        e, h, i, topk = case["experts"], case["hidden"], case["inter"], case["topk"]
        hit = e * (1.0 - (1.0 - topk / e) ** t)  # expected number of experts with a row
        per = _w4_bytes(2 * i, h) + _w4_bytes(h, i)
        return {"bytes": hit * per + 4 * t * e + 4 * t * h, "flops": 6.0 * t * topk * h * i}
    n, k = case["n"], case["k"]
    out = 2 if case["out"] == "bf16" else 4
    if kind in ("linear", "w4a8"):
        wb = _w4_bytes(n, k)
    else:
        wb = n * k + 2 * n * (1 if case["per_channel"] else k // 128)
    return {"bytes": wb + 2 * t * k + out * t * n, "flops": 2.0 * t * n * k}


def tolerance(case):
    """Relative 2-norm differences. The bf16 rounding of an output is 1.7e-3 of it, that of a weight operand
    (prefill multiplies bf16_rn((u - 8) s), decode the unrounded product) 1.6e-3 in a sum of independent terms, so two
    correct implementations differ by up to about 2.5e-3; stated is four times that. fp32 outputs of exact integer
    products, or of unrounded weights, differ by the order of their sums only."""
    kind, t = case["kind"], case["rows"]
    if kind in ("w8a8", "w4a8") and case["out"] == "f32":
        return {"rel": 1e-5}
    if kind == "linear" and case["out"] == "f32" and t <= 64:
        return {"rel": 1e-5}
    if kind == "w8" and case["out"] == "f32" and t <= 16:
        return {"rel": 1e-5}
    return {"rel": 1e-2}


# ------------------------------------------------------------------------------------------------ 64-bit result
def _w4_64(q, s):
    """[n, k] float64 weights (u - 8) s"""
    n, k = q.shape[0], q.shape[1] * 8
    u = torch.stack([(q >> (4 * j)) & 15 for j in range(8)], -1).view(n, k // 128, 128)
    return ((u - 8).double() * s.double().unsqueeze(-1)).view(n, k)


def _w8_64(q, s, per_channel):
    n, k = q.shape
    if per_channel:
        return q.double() * s.double().unsqueeze(-1)
    return (q.view(n, k // 128, 128).double() * s.double().unsqueeze(-1)).view(n, k)


def _quantized(x, group):
    """the activations the INT8 numerics multiply: per (row, group) sx = amax / 127 with its two lowest mantissa bits
    cleared, q = round(x fp32(1 / sx)); returns q sx in float64"""
    t, k = x.shape
    xg = x.float().view(t, k // group, group)
    amax = xg.abs().amax(-1)
    # (a division by a tensor: by a number, torch multiplies with the rounded reciprocal)
    sx = ((amax / torch.full_like(amax, 127)).view(torch.int32) & -4).view(torch.float32)
    sx = torch.where(amax > 0, sx, torch.ones_like(sx))
    q = (xg * (torch.ones_like(sx) / sx).unsqueeze(-1)).round().clamp(-127, 127)
    return (q.double() * sx.double().unsqueeze(-1)).view(t, k)


def _silu_mul(g, u):
    return g / (1.0 + torch.exp(-g)) * u


def exact(case, seed):
    src = _sources(case, seed)
    kind = case["kind"]
    x = src["x"].double()
    if kind == "mlp":
        i = case["inter"]
        gu = x @ _w4_64(*src["gu"]).t()
        act = _silu_mul(gu[:, :i], gu[:, i:])
        return {"act": act, "y": act @ _w4_64(*src["dn"]).t()}
    if kind == "linear":
        return x @ _w4_64(*src["w"]).t()
    if kind == "w8":
        return x @ _w8_64(*src["w"], case["per_channel"]).t()
    if kind == "w8a8":
        return _quantized(src["x"], 128) @ _w8_64(*src["w"], case["per_channel"]).t()
    if kind == "w4a8":
        return _quantized(src["x"], case["group"]) @ _w4_64(*src["w"]).t()
    i = case["inter"]
    val, sel = torch.topk(src["logits"], case["topk"], dim=1)
    wgt = torch.softmax(val.double(), dim=1)
    out = torch.zeros_like(x)
    for e in torch.unique(sel).tolist():
        tok, pos = torch.nonzero(sel == e, as_tuple=True)
        gu = x[tok] @ _w4_64(src["gq"][e], src["gs"][e]).t()
        act = _silu_mul(gu[:, :i], gu[:, i:]) * wgt[tok, pos].unsqueeze(1)
        out[tok] += act @ _w4_64(src["dq"][e], src["ds"][e]).t()
    return out

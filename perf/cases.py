"""The workloads that the performance of this package is followed on.

Four kinds of work, all through the public entry points:

  layer     a mixture-of-experts block as a serving program runs it: routing of the logits, up projection (gathered
            rows, bias, SwiGLU), down projection (bias, gate weights, scatter), sum over the picked experts;
  dense     one product with a bias: a gate, a shared expert, an unrouted layer;
  routing   the routing alone, with every table that it hands on;
  convert   weights or activations to a microscaled type and back, as quantisation-aware fine-tuning and the
            preparation of a checkpoint do.

Activations and weights are named by their types: "bf16", "f16", "fp8" (float8_e4m3fn with per-tensor scales),
"mxfp8", "mxfp4" (microscaled: one e8m0 byte per 32 values along K).
"""
import math

import torch

from triton_amd.matmul import (Epilogue, FlexCtx, FnSpecs, FusedActivation, InFlexData, OutFlexData, PrecisionConfig,
                               matmul)
from triton_amd.numerics_details.mxfp import downcast_to_mxfp, upcast_from_mxfp
from triton_amd.reduce import reduce
from triton_amd.routing import routing
from triton_amd.swiglu import swiglu_fn
from triton_amd.tensor import FP4, convert_layout, wrap_torch_tensor
from triton_amd.tensor_details.layout import CDNA4MXScaleLayout, CDNA4MXValueLayout

SIXTEEN_BIT = {"bf16": torch.bfloat16, "f16": torch.float16}
SWIGLU = FusedActivation(FnSpecs("swiglu", swiglu_fn, ("alpha", "limit"), reduction_n=2), (1.702, 7.0))
TO_MXFP8 = Epilogue(FnSpecs("QUANTIZE_MXFP8", None, (), ()), (), (), 6.0)

# bytes of one stored value; microscaled ones with their share of the scale byte
BYTES = {"f32": 4.0, "bf16": 2.0, "f16": 2.0, "fp8": 1.0, "mxfp8": 1 + 1 / 32, "mxfp4": 0.5 + 1 / 32}


def _layer(name, tokens, hidden, inter, experts, k, acts, weights, layout="blocks"):
    return {"name": name, "kind": "layer", "tokens": tokens, "hidden": hidden, "inter": inter, "experts": experts, "k": k,
            "acts": acts, "weights": weights, "layout": layout}


def listed():
    return [
        # decoding for one user: four experts of 128 are read, launches and host time count
        _layer("decode_1", 1, 2880, 2880, 128, 4, "bf16", "mxfp4"),
        # decoding for a batch: about 110 experts with two rows each
        _layer("decode_64", 64, 2880, 2880, 128, 4, "bf16", "mxfp4"),
        # a prefill chunk of a smaller model in float16, weights as the quantiser leaves them, no size round
        _layer("chunk_333_f16", 333, 2016, 1056, 32, 4, "f16", "mxfp4", "strided"),
        # a wide layer in fp8 between decoding and prefill: about 16 rows per expert, every weight is read
        _layer("layer_509_fp8", 509, 5760, 2880, 128, 4, "fp8", "mxfp4"),
        # prefill of a batch of prompts
        _layer("prefill_4096", 4096, 2880, 2880, 128, 4, "bf16", "mxfp4"),
        # the same with activations in the weights' own format, quantised between the products
        _layer("prefill_2048_mxfp4", 2048, 2880, 2880, 128, 4, "mxfp4", "mxfp4"),
        # the largest: long prompts in fp8, experts with thousands of rows each
        _layer("prefill_16384_fp8", 16384, 2880, 2880, 32, 4, "fp8", "mxfp4"),
        # experts that were not quantised, a ragged chunk
        _layer("chunk_1021_bf16", 1021, 2880, 2880, 32, 4, "bf16", "bf16"),
        # an unrouted layer with quantised weights
        {"name": "dense_256_mxfp4", "kind": "dense", "rows": 256, "inner": 2048, "columns": 4096, "acts": "bf16", "weights": "mxfp4",
         "layout": "blocks"},
        # an unrouted layer with both sides in fp8
        {"name": "dense_1024_fp8", "kind": "dense", "rows": 1024, "inner": 8192, "columns": 8192, "acts": "fp8", "weights": "fp8",
         "layout": "strided"},
        {"name": "routing_4096", "kind": "routing", "tokens": 4096, "experts": 128, "k": 4, "logits": "f32"},
        # weights of eight experts quantised along their inner axis and brought back
        {"name": "convert_weights", "kind": "convert", "batch": 8, "rows": 2880, "columns": 5760, "axis": -2, "source": "f32",
         "values": "mxfp4", "back": "bf16"},
    ]


def _spread(rng, low, high, step=1):
    """A whole multiple of `step` between `low` and `high`, even over the logarithm."""
    v = math.exp(rng.uniform(math.log(low), math.log(high)))
    return min(high, max(low, round(v / step) * step))


def draw(rng):
    kind = rng.choices(("layer", "dense", "routing", "convert"), (6, 2, 1, 1))[0]
    if kind == "layer":
        acts, weights = rng.choice((("bf16", "mxfp4"), ("bf16", "mxfp4"), ("f16", "mxfp4"), ("fp8", "mxfp4"), ("mxfp8", "mxfp4"),
                                    ("mxfp4", "mxfp4"), ("bf16", "bf16"), ("f16", "f16")))
        hidden, inter = _spread(rng, 512, 5760, 32), _spread(rng, 512, 2880, 32)
        most = 3.7e9 / (3 * hidden * inter * BYTES[weights])            # bytes of the weights: those of the widest listed layer
        if weights != "mxfp4":
            most /= 2
        experts = rng.choice([e for e in (8, 16, 32, 60, 64, 128) if e <= most] or [8])
        k = rng.choice((1, 2, 4, 4, 6, 8))
        flops = 0.75e12 if weights != "mxfp4" else 1.5e12 if acts == "fp8" else 0.8e12
        tokens = _spread(rng, 1, max(1, min(16384, int(flops / (6.0 * k * hidden * inter)))))
        return {"kind": kind, "tokens": tokens, "hidden": hidden, "inter": inter, "experts": experts, "k": k, "acts": acts,
                "weights": weights, "layout": rng.choice(("blocks", "blocks", "strided")) if weights == "mxfp4" else "strided"}
    if kind == "dense":
        acts, weights = rng.choice((("bf16", "mxfp4"), ("f16", "mxfp4"), ("fp8", "mxfp4"), ("bf16", "bf16"), ("fp8", "fp8")))
        rows, inner, columns = _spread(rng, 1, 4096), _spread(rng, 512, 8192, 32), _spread(rng, 128, 8192, 8)
        return {"kind": kind, "rows": rows, "inner": inner, "columns": columns, "acts": acts, "weights": weights,
                "layout": rng.choice(("blocks", "strided")) if weights == "mxfp4" else "strided"}
    if kind == "routing":
        return {"kind": kind, "tokens": _spread(rng, 1, 32768), "experts": rng.choice((8, 32, 60, 64, 128, 256)),
                "k": rng.choice((1, 2, 4, 6, 8)), "logits": rng.choice(("f32", "bf16"))}
    if rng.random() < 0.5:      # weights, quantised along K
        return {"kind": kind, "batch": rng.choice((1, 2, 5, 8)), "rows": _spread(rng, 512, 2880, 32), "columns": _spread(rng, 512, 5760, 8),
                "axis": -2, "source": rng.choice(("f32", "bf16")), "values": "mxfp4", "back": "bf16"}
    return {"kind": kind, "batch": 1, "rows": _spread(rng, 1, 16384), "columns": _spread(rng, 512, 5760, 32), "axis": -1,
            "source": rng.choice(("bf16", "f16")), "values": rng.choice(("mxfp4", "mxfp8")), "back": "bf16"}


# ---------------------------------------------------------------------------------------------------------------------


def _weights(E, K, N, kind, layout, g):
    """Weights [E, K, N] ~ N(0, 0.02), unit stride along K: (what `matmul` takes, precision options that go with it)."""
    n = max(1, min(E, (1 << 28) // (K * N)))    # experts made together
    parts, scales = [], []
    for e in range(0, E, n):
        w = torch.randn((min(n, E - e), N, K), generator=g, device="cuda", dtype=torch.bfloat16).mul_(0.02)
        if kind == "mxfp4":
            v, s = downcast_to_mxfp(w, torch.uint8, axis=-1)
            scales.append(s)
        elif kind == "fp8":
            v = (w.float() * 2048.0).to(torch.float8_e4m3fn)
        else:
            v = w.to(SIXTEEN_BIT[kind])
        parts.append(v)
    w = torch.cat(parts).transpose(-1, -2)
    if kind == "fp8":
        return w, {"scale": torch.full((1,), 1 / 2048.0, device="cuda")}
    if kind != "mxfp4":
        return w, {}
    s = torch.cat(scales).transpose(-1, -2)
    if layout == "blocks":
        w = convert_layout(wrap_torch_tensor(w, dtype=FP4), CDNA4MXValueLayout())
        s = convert_layout(wrap_torch_tensor(s), CDNA4MXScaleLayout())
    return w, {"b_mx_scale": s, "b_microblock_size": 32}


def _rows(M, K, kind, g):
    """Normalised activations [M, K]: (what `matmul` or the quantiser takes, per-tensor scale or None)."""
    x = torch.randn((M, K), generator=g, device="cuda", dtype=torch.float32)
    if kind == "fp8":
        scale = (x.abs().amax() / 448.0).reshape(1)
        return (x / scale).to(torch.float8_e4m3fn), scale
    return x.to(SIXTEEN_BIT.get(kind, torch.bfloat16)), None


def _logits(T, E, dtype, g):
    """Router outputs: tokens differ, and some experts are picked more often than others."""
    return (torch.randn((T, E), generator=g, device="cuda") + 0.2 * torch.randn(E, generator=g, device="cuda")).to(dtype)


def prepare(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    c = case
    if c["kind"] == "routing":
        dtype = torch.float32 if c["logits"] == "f32" else torch.bfloat16
        return {"kind": "routing", "k": c["k"], "logits": _logits(c["tokens"], c["experts"], dtype, g)}
    if c["kind"] == "convert":
        shape = (c["batch"], c["rows"], c["columns"]) if c["axis"] == -2 else (c["rows"], c["columns"])
        x = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).mul_(0.02 if c["axis"] == -2 else 1.0)
        return {"kind": "convert", "x": x if c["source"] == "f32" else x.to(SIXTEEN_BIT[c["source"]]), "axis": c["axis"],
                "values": torch.uint8 if c["values"] == "mxfp4" else torch.float8_e4m3fn, "back": torch.bfloat16}
    if c["kind"] == "dense":
        w, pw = _weights(1, c["inner"], c["columns"], c["weights"], c["layout"], g)
        if not isinstance(w, torch.Tensor):
            pass                                                        # the block layout keeps its leading axis
        elif c["weights"] == "mxfp4":
            w, pw["b_mx_scale"] = w[0], pw["b_mx_scale"][0]
        else:
            w = w[0]
        x, xs = _rows(c["rows"], c["inner"], c["acts"], g)
        bias = torch.randn((c["columns"],), generator=g, device="cuda").mul_(0.01).to(torch.bfloat16)
        flex = FlexCtx(InFlexData(x.dtype, xs) if xs is not None else InFlexData(),
                       InFlexData(w.dtype, pw.pop("scale")) if "scale" in pw else InFlexData())
        out = torch.bfloat16 if c["acts"] == "fp8" else None
        return {"kind": "dense", "x": x, "w": w, "bias": bias, "pc": PrecisionConfig(flex_ctx=flex, out_dtype=out, **pw)}
    T, H, I, E, k = c["tokens"], c["hidden"], c["inter"], c["experts"], c["k"]
    w1, pw1 = _weights(E, H, 2 * I, c["weights"], c["layout"], g)
    w2, pw2 = _weights(E, I, H, c["weights"], c["layout"], g)
    b1 = torch.randn((E, 2 * I), generator=g, device="cuda").mul_(0.1).to(torch.bfloat16)
    b2 = torch.randn((E, H), generator=g, device="cuda").mul_(0.1).to(torch.bfloat16)
    x, xs = _rows(T, H, c["acts"], g)
    st = {"kind": "layer", "acts": c["acts"], "k": k, "T": T, "H": H, "I": I, "x": x, "logits": _logits(T, E, torch.float32, g),
          "w1": w1, "w2": w2, "b1": b1, "b2": b2, "pw1": pw1, "pw2": pw2}
    if c["acts"] == "fp8":
        # the rows between the products are fp8 as well, with a scale from calibration
        mid = torch.full((1,), 1 / 32.0, device="cuda")
        st["pc1"] = PrecisionConfig(out_dtype=torch.float8_e4m3fn, flexpoint_saturate_inf=True,
                                    flex_ctx=FlexCtx(lhs_data=InFlexData(x.dtype, xs), out_data=OutFlexData(x.dtype, mid)), **pw1)
        st["pc2"] = PrecisionConfig(out_dtype=torch.bfloat16, flex_ctx=FlexCtx(lhs_data=InFlexData(x.dtype, mid)), **pw2)
    elif c["acts"] in SIXTEEN_BIT:
        st["pc1"], st["pc2"] = PrecisionConfig(**pw1), PrecisionConfig(**pw2)
    return st


def _run_layer(s):
    x, k, acts = s["x"], s["k"], s["acts"]
    r = routing(s["logits"], k)
    if acts == "mxfp4":
        xq, xs = downcast_to_mxfp(x, torch.uint8, axis=-1)
        h = matmul(xq, s["w1"], s["b1"], r.ragged_metadata, gather_indx=r.gather_indx, fused_activation=SWIGLU,
                   precision_config=PrecisionConfig(a_mx_scale=xs, a_microblock_size=32, **s["pw1"]))
        h, hs = downcast_to_mxfp(h, torch.uint8, axis=-1)
        pc2 = PrecisionConfig(a_mx_scale=hs, a_microblock_size=32, **s["pw2"])
    elif acts == "mxfp8":
        xq, xs = downcast_to_mxfp(x, torch.float8_e4m3fn, axis=-1)
        hs = torch.empty((s["T"] * k, s["I"] // 32), dtype=torch.uint8, device=x.device)
        h = matmul(xq, s["w1"], s["b1"], r.ragged_metadata, gather_indx=r.gather_indx, fused_activation=SWIGLU, epilogue=TO_MXFP8,
                   precision_config=PrecisionConfig(a_mx_scale=xs, a_microblock_size=32, c_mx_scale=hs, **s["pw1"]))
        pc2 = PrecisionConfig(a_mx_scale=hs, a_microblock_size=32, **s["pw2"])
    else:
        h = matmul(x, s["w1"], s["b1"], r.ragged_metadata, gather_indx=r.gather_indx, fused_activation=SWIGLU,
                   precision_config=s["pc1"])
        pc2 = s["pc2"]
    y = matmul(h, s["w2"], s["b2"], r.ragged_metadata, scatter_indx=r.scatter_indx, gammas=r.expert_sorted_gate_weights,
               precision_config=pc2)
    z, _ = reduce(y.view(s["T"], k, s["H"]), dim=1)
    return z


def run(state):
    s = state
    if s["kind"] == "layer":
        return _run_layer(s)
    if s["kind"] == "dense":
        return matmul(s["x"], s["w"], s["bias"], precision_config=s["pc"])
    if s["kind"] == "routing":
        r = routing(s["logits"], s["k"])
        md = r.ragged_metadata
        return {"indx": r.indx, "vals": r.vals, "col_sum": r.col_sum, "gather": r.gather_indx, "scatter": r.scatter_indx,
                "row_sorted": r.row_sorted_indx, "slice_offs": md.slice_offs, "block_offs": md.block_offs_data,
                "block_schedule": md.block_schedule_data}
    v, sc = downcast_to_mxfp(s["x"], s["values"], axis=s["axis"])
    return {"values": v, "scales": sc, "back": upcast_from_mxfp(v, sc, s["back"], axis=s["axis"])}


# ---------------------------------------------------------------------------------------------------------------------


def work(case):
    c = case
    if c["kind"] == "layer":
        T, H, I, E, k = c["tokens"], c["hidden"], c["inter"], c["experts"], c["k"]
        active = E * (1.0 - (1.0 - min(1.0, k / E)) ** T)               # experts with rows, expected
        weights = active * (3.0 * H * I * BYTES[c["weights"]] + 2.0 * (2 * I + H))
        x = 1.0 if c["acts"] == "fp8" else 2.0                          # microscaled activations are given in bf16
        return {"bytes": weights + T * H * (x + 2.0) + T * E * 4.0, "flops": 6.0 * T * k * H * I}
    if c["kind"] == "dense":
        M, K, N = c["rows"], c["inner"], c["columns"]
        return {"bytes": M * K * BYTES[c["acts"]] + K * N * BYTES[c["weights"]] + N * 2.0 + M * N * 2.0, "flops": 2.0 * M * K * N}
    if c["kind"] == "routing":
        T, E, k = c["tokens"], c["experts"], c["k"]
        logit = BYTES[c["logits"]]
        # logits in; picks, gate weights, bit matrix, three index arrays, histogram and tables out
        return {"bytes": T * E * logit + T * k * (2.0 + logit) + T * math.ceil(E / 32) * 4.0 + 12.0 * T * k + 4.0 * E + 24.0 * (E + 1),
                "flops": 0.0}
    n = float(c["batch"] * c["rows"] * c["columns"])
    packed = BYTES[c["values"]]
    return {"bytes": n * (BYTES[c["source"]] + 2.0 * packed + BYTES[c["back"]]), "flops": 0.0}


def tolerance(case):
    if case["kind"] == "convert":
        return "exact"
    if case["kind"] == "routing":
        return {"rel": 1e-5, "differ": 0.0}                             # the softmax over the picks; whole numbers are exact
    if case["kind"] == "dense":
        return {"rel": 4e-3, "max": 0.05}                               # 16-bit results of 32-bit sums
    if case["acts"] in ("bf16", "f16"):
        return {"rel": 1e-2, "max": 0.1}                                # 16-bit rows between the two products
    return {"rel": 1e-2, "max": 0.5}                                    # rows of 8 or 4 bits between them: a rounding may flip

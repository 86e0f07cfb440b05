"""GPU: what the routing kernels leave in expert-sorted order, on every launch form of the routing, against the oracle; what the
host code of the entry points hands out and keeps."""
import sys

import pytest
import torch

from oracle import routing_ref as RR
from triton_amd import _native
from triton_amd.matmul import (Epilogue, FlexCtx, FnSpecs, FusedActivation, InFlexData, OutFlexData, PrecisionConfig, matmul)
from triton_amd.numerics_details.mxfp import downcast_to_mxfp, upcast_from_mxfp
from triton_amd.reduce import reduce
from triton_amd.routing import routing
from triton_amd.swiglu import swiglu_fn
from triton_amd.tensor import FP4, convert_layout, wrap_torch_tensor
from triton_amd.tensor_details.layout import CDNA4MXScaleLayout, CDNA4MXValueLayout

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,E,k", [
    (1, 128, 4), (128, 128, 4), (129, 128, 4), (64, 500, 1),  # one launch, its last row count, the two launches after it
    (8192, 128, 4), (8193, 128, 4),                           # two launches, more blocks than they cover
    (300, 128, 3), (5000, 33, 3), (5, 600, 2),                # rows that make no whole chunks; columns past one launch
])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_expert_sorted_gate_weights(T, E, k, dtype, device):
    torch.manual_seed(0)
    logits = torch.randn(T, E).to(dtype)
    r = routing(logits.to(device), k)
    ref = RR.routing_ref(logits, k)
    assert torch.equal(r.scatter_indx.cpu(), ref["scatter_indx"])
    gates = r.expert_sorted_gate_weights
    assert gates.dtype == dtype and torch.equal(gates.cpu(), r.vals.cpu().flatten()[ref["scatter_indx"].long()])


@pytest.mark.parametrize("T,E,k", [(1, 1, 1), (3, 64, 2), (16, 500, 4), (700, 33, 3), (9000, 128, 4)])
def test_routing_tables_of_one_call(T, E, k, device):
    """Each table against the oracle, whichever is asked for first, by the call that lays a shape out and by the next one, and
    after so many other shapes that the layouts were dropped."""
    module = sys.modules["triton_amd.routing"]
    torch.manual_seed(T)
    logits = torch.randn(T, E)
    ref = RR.routing_ref(logits, k)
    dev = logits.to(device)
    module._layouts.clear()
    for i in range(3):
        if i == 2:
            module._layouts.update({(j, 0, 0, 0): {} for j in range(600)})   # (600 entries of no shape: the next new shape drops all)
            routing(torch.randn(T + 1, E, device=device), k)
            assert len(module._layouts) == 1
        r = routing(dev, k)
        if i == 1:
            assert torch.equal(r.gather_indx.cpu(), ref["gather_indx"])
        md = r.ragged_metadata
        assert torch.equal(r.scatter_indx.cpu(), ref["scatter_indx"]) and torch.equal(r.gather_indx.cpu(), ref["gather_indx"])
        assert torch.equal(r.col_sum.cpu(), ref["col_sum"]) and md.slice_sizes is r.col_sum
        inverse = torch.empty_like(ref["scatter_indx"])
        inverse[ref["scatter_indx"].long()] = torch.arange(T * k, dtype=inverse.dtype)
        assert torch.equal(r.row_sorted_indx.cpu(), inverse)
        sizes = ref["col_sum"].long()
        assert torch.equal(md.slice_offs.cpu().long(), torch.cat([torch.zeros(1, dtype=torch.long), sizes.cumsum(0)]))
        for b in md.block_sizes():
            blocks = (sizes + b - 1) // b
            assert torch.equal(md.block_offs(b).cpu().long(), torch.cat([torch.zeros(1, dtype=torch.long), blocks.cumsum(0)]))
            want = [(j << 16) | e for e in range(E) for j in range(int(blocks[e]))]
            got = md.block_schedule(b).cpu().tolist()
            assert got[:len(want)] == want and all(v == -1 for v in got[len(want):])


@pytest.mark.parametrize("inference", [False, True])
def test_gate_weights_are_the_callers_own(inference, device):
    """Scaling the gate weights in place changes neither later accesses nor vals; scaling vals changes later accesses."""
    with torch.inference_mode(inference):
        torch.manual_seed(3)
        logits = torch.randn(65, 32, device=device)
        r = routing(logits, 4)
        want = r.vals.clone().reshape(-1)[r.scatter_indx.long()]
        first = routing(logits, 4).expert_sorted_gate_weights   # (vals not touched before: the kernel's own copy)
        assert torch.equal(first, want)
        g = r.expert_sorted_gate_weights
        g.mul_(3.0)
        assert torch.equal(r.expert_sorted_gate_weights, want)
        r.vals.mul_(2.0)
        assert torch.equal(r.expert_sorted_gate_weights, want * 2)
        q = routing(logits, 4)
        q.vals.mul_(2.0)
        assert torch.equal(q.expert_sorted_gate_weights, want * 2)
        q = routing(logits, 4)
        q.expert_sorted_gate_weights.zero_()
        assert torch.equal(q.expert_sorted_gate_weights, want)


def gate(device, seed):
    """A gate product whose weights have unit stride along N: they are turned, and the copy is kept."""
    g = torch.Generator().manual_seed(seed)
    x, w = torch.randn(48, 256, generator=g).bfloat16(), (torch.randn(256, 32, generator=g) * 0.1).bfloat16()
    return x.to(device), w.to(device), x.float() @ w.float()


def close(y, ref):
    torch.testing.assert_close(y.cpu().float(), ref, rtol=1e-2, atol=1e-2)


def test_turned_weights_on_another_stream(device):
    x, w, ref = gate(device, 0)
    first, second = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(first):
        torch.cuda._sleep(200_000_000)      # the copy is made about 0.1 s from now
        y1 = matmul(x, w, None)
    with torch.cuda.stream(second):
        y2 = matmul(x, w, None)
    torch.cuda.synchronize()
    close(y1, ref)
    close(y2, ref)


def test_turned_weights_in_a_graph(device):
    x, w, ref = gate(device, 1)
    warm = gate(device, 2)
    matmul(warm[0], warm[1], None)
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        y = matmul(x, w, None)              # the first call on these weights is only recorded
    close(matmul(x, w, None), ref)          # ... and leaves nothing behind
    for scale in (1.0, 2.0, 0.5):
        w.mul_(scale)
        ref = x.cpu().float() @ w.cpu().float()
        graph.replay()
        torch.cuda.synchronize()
        close(y, ref)
        close(matmul(x, w, None), ref)


def test_turned_weights_in_inference_mode(device):
    with torch.inference_mode():
        x, w, ref = gate(device, 3)
        close(matmul(x, w, None), ref)
        w.mul_(2.0)
        close(matmul(x, w, None), 2 * ref)


class BothPaths:
    """Runs a call as it is and with the native function switched off, says which path the first took, compares the results
    bit for bit."""

    def __init__(self, monkeypatch, name):
        _native.load()
        self.mp, self.name, self.fn, self.covered = monkeypatch, name, getattr(_native, name), None

    def __call__(self, call):
        def spy(*args):
            done = self.fn(*args)
            if self.covered is None:   # (the general path may call itself with a form that is covered)
                self.covered = done is not None and type(done) is not int
            return done
        self.mp.setattr(_native, self.name, spy)
        native = call()
        self.mp.setattr(_native, self.name, lambda *args: None)
        general = call()
        for a, b in zip(native, general):
            assert a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride()
            assert torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8))
        return self.covered


SWIGLU = FusedActivation(FnSpecs("swiglu", swiglu_fn, ("alpha", "limit"), reduction_n=2), (1.702, 7.0))
F8 = torch.float8_e4m3fn
# rows, weights, weight layout, options, whether the native path takes the call
FORMS = [(a, w, lay, opts, True) for a, w, lays in (("bf16", "mxfp4", ("strided", "blocks")), ("f16", "mxfp4", ("strided", "blocks")),
                                                   ("fp8", "mxfp4", ("strided", "blocks")), ("mxfp8", "mxfp4", ("strided", "blocks")),
                                                   ("bf16", "bf16", ("strided", )), ("f16", "f16", ("strided", )),
                                                   ("fp8", "fp8", ("strided", )))
         for lay in lays for opts in ((), ("gather", "swiglu"), ("scatter", "gammas"), ("dense", ), ("pitch", "c"))] + [
    ("bf16", "mxfp4", "strided", ("betas", "bias f32"), True), ("bf16", "mxfp4", "strided", ("no bias", "f32 out"), True),
    ("fp8", "mxfp4", "strided", ("swiglu", "flex out"), True), ("fp8", "mxfp4", "blocks", ("dense", "flex out"), True),
    ("mxfp8", "mxfp4", "blocks", ("swiglu", "mx out"), True), ("bf16", "mxfp4", "strided", ("out_alpha", "expected"), True),
    ("bf16", "bf16", "strided", ("2-D", "dense"), True), ("bf16", "mxfp4", "strided", ("2-D", "dense"), True),
    # conversions, other layouts and long splits are the general path's
    ("mxfp4", "mxfp4", "strided", ("gather", "swiglu"), False), ("bf16", "mxfp8", "strided", (), False),
    ("bf16", "mxfp4", "strided", ("scatter", "gammas bf16"), False), ("bf16", "bf16", "along N", (), False),
    ("fp8", "fp8", "along N", (), False), ("bf16", "mxfp4", "strided", ("dense", "long K"), False),
    ("bf16", "mxfp4", "strided", ("int64 indices", "gather"), False), ("bf16", "mxfp4", "strided", ("no rows", ), False)]


@pytest.mark.parametrize("acts,weights,layout,opts,covered", FORMS)
def test_native_matmul_is_the_general_path(acts, weights, layout, opts, covered, device, monkeypatch):
    g = torch.Generator(device=device).manual_seed(7)
    rnd = lambda *s: torch.randn(s, generator=g, device=device)
    T, E, k, K, N = (0 if "no rows" in opts else 37), 8, 4, 8192 if "long K" in opts else 160, 192
    dense = "dense" in opts
    E = 1 if dense else E
    r = None if dense else routing(rnd(T, E), k)
    gathered = "gather" in opts
    rows = T if dense or gathered else T * k
    one = lambda v: torch.full((1,), v, device=device)
    # ---- weights
    w = rnd(E, N, K) * 0.1
    pw, lhs, rhs = {}, InFlexData(), InFlexData()
    if weights[:2] == "mx":
        v, s = downcast_to_mxfp(w.bfloat16(), torch.uint8 if weights == "mxfp4" else F8, axis=-1)
        w, s = v.transpose(-1, -2), s.transpose(-1, -2)
        if layout == "blocks":
            w, s = (convert_layout(wrap_torch_tensor(w, dtype=FP4), CDNA4MXValueLayout()),
                    convert_layout(wrap_torch_tensor(s), CDNA4MXScaleLayout()))
        pw = {"b_mx_scale": s, "b_microblock_size": 32}
    else:
        w = w.to({"bf16": torch.bfloat16, "f16": torch.float16, "fp8": F8}[weights]).transpose(-1, -2)
        if layout == "along N":
            w = w.contiguous()
        if weights == "fp8":
            rhs = InFlexData(F8, one(0.5))
    if "2-D" in opts:
        w = w[0]
        if pw:
            pw["b_mx_scale"] = pw["b_mx_scale"][0]
    # ---- rows
    x = rnd(rows, K + (32 if "pitch" in opts else 0))[:, :K]
    if acts[:2] == "mx":
        x, xs = downcast_to_mxfp(x.bfloat16().contiguous(), torch.uint8 if acts == "mxfp4" else F8, axis=-1)
        pw.update(a_mx_scale=xs, a_microblock_size=32)
    else:
        dt = {"bf16": torch.bfloat16, "f16": torch.float16, "fp8": F8}[acts]
        full = rnd(rows, K + 32).to(dt)
        x = full[:, :K] if "pitch" in opts else x.to(dt)
        if acts == "fp8":
            lhs = InFlexData(F8, one(0.25))
    # ---- the rest
    red = 2 if "swiglu" in opts else 1
    M = T if dense else T * k
    out_type = torch.float32 if "f32 out" in opts else F8 if "flex out" in opts or "mx out" in opts else None
    out = OutFlexData(F8, one(0.1), one(0.0)) if "flex out" in opts else OutFlexData(torch.bfloat16, one(0.1)) if "expected" in opts else OutFlexData()
    if acts == "fp8" and out_type is None:
        out_type = torch.bfloat16
    bias = rnd(E, N) if not dense else rnd(N)
    if "no bias" in opts:
        bias = None
    elif "bias f32" not in opts:
        bias = bias.bfloat16()
    gammas = torch.rand(M, generator=g, device=device) if "gammas" in opts else torch.rand(M, generator=g, device=device).bfloat16() if "gammas bf16" in opts else None
    betas = torch.rand(M, generator=g, device=device) if "betas" in opts else None
    gather = r.gather_indx if gathered else None
    if "int64 indices" in opts:
        gather = gather.long()

    def call():
        if "flex out" in opts:
            out.actual_scale.zero_()
        extra = {}
        if "mx out" in opts:
            extra["c_mx_scale"] = torch.zeros((M, N // red // 32), dtype=torch.uint8, device=device)
        pc = PrecisionConfig(flex_ctx=FlexCtx(lhs, rhs, out), out_dtype=out_type, c_microblock_size=32 if extra else None,
                             flexpoint_saturate_inf="flex out" in opts, **pw, **extra)
        c = torch.zeros((M, N // red + 8), dtype=out_type or x.dtype, device=device)[:, :N // red] if "c" in opts and acts != "mxfp8" else None
        y = matmul(x, w, bias, None if dense else r.ragged_metadata, gather_indx=gather,
                   scatter_indx=r.scatter_indx if "scatter" in opts else None, precision_config=pc, betas=betas, gammas=gammas,
                   out_alpha=0.5 if "out_alpha" in opts else None, c=c, fused_activation=SWIGLU if red == 2 else None,
                   epilogue=Epilogue(FnSpecs("QUANTIZE_MXFP8", None, (), ()), (), (), 6.0) if extra else None)
        return [y, *extra.values(), *([out.actual_scale.clone()] if "flex out" in opts else [])]

    assert BothPaths(monkeypatch, "matmul")(call) == covered


@pytest.mark.parametrize("shape,axis,values,covered", [
    ((33, 96), -1, torch.uint8, True), ((33, 96), 1, F8, True), ((3, 40, 64), 2, torch.float8_e5m2, True),
    ((2, 64, 24), -2, torch.uint8, True), ((64, 24), 0, torch.uint8, True),
    ((2, 64, 24), 1, F8, False), ((2, 64, 24), 0, torch.uint8, False), ((64, 24, 2), 0, torch.uint8, False), ((2, 3, 5, 32), -1, F8, False)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_native_conversions_are_the_general_path(shape, axis, values, covered, dtype, device, monkeypatch):
    torch.manual_seed(8)
    if shape[axis] % 32:
        shape = tuple(64 if d == axis % len(shape) else n for d, n in enumerate(shape))
    x = torch.randn(shape, device=device).to(dtype)
    assert BothPaths(monkeypatch, "downcast")(lambda: downcast_to_mxfp(x, values, axis=axis)) == covered
    monkeypatch.undo()
    v, s = downcast_to_mxfp(x, values, axis=axis)
    assert BothPaths(monkeypatch, "upcast")(lambda: [upcast_from_mxfp(v, s, dtype, axis=axis)]) == covered
    monkeypatch.undo()
    part = x[..., :-1] if axis % x.ndim != x.ndim - 1 else x[..., :-32]     # rows with gaps between them
    if part.shape[axis] and part.numel():
        assert BothPaths(monkeypatch, "downcast")(lambda: downcast_to_mxfp(part, values, axis=axis)) in (False, part.is_contiguous())


@pytest.mark.parametrize("shape,dim", [((5, 4, 24), 1), ((4, 7, 9), 0), ((3, 5, 33), -1), ((2, 600, 8), 1)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_native_reduce_is_the_general_path(shape, dim, dtype, device, monkeypatch):
    torch.manual_seed(9)
    x = torch.randn(shape, device=device).to(dtype)
    for t in (x, x.transpose(0, 2).contiguous().transpose(0, 2)):
        assert BothPaths(monkeypatch, "reduce")(lambda: [reduce(t, dim=dim)[0]]) == (shape[dim] < 512)
        monkeypatch.undo()


@pytest.mark.parametrize("layout", ["strided", "blocks"])
@pytest.mark.parametrize("form,covered", [("gather swiglu", True), ("scatter", True), ("dense", True), ("out type", True), ("c", True),
                                          ("short", False),
                                          ("lhs type", False), ("pitch", False), ("split_k", False)])
def test_native_matmul_of_packed_rows(form, covered, layout, device, monkeypatch):
    """Packed e2m1 rows: what their kernel reads as it is goes the native way."""
    g = torch.Generator(device=device).manual_seed(11)
    T, E, k, K, N = 37, 1 if form in ("dense", "split_k") else 8, 4, {"short": 96, "split_k": 8192}.get(form, 288), 192
    rnd = lambda *s: torch.randn(s, generator=g, device=device).bfloat16()
    v, s = downcast_to_mxfp(rnd(E, N, K) * 0.1, torch.uint8, axis=-1)
    w, s = v.transpose(-1, -2), s.transpose(-1, -2)
    if layout == "blocks":
        w, s = (convert_layout(wrap_torch_tensor(w, dtype=FP4), CDNA4MXValueLayout()),
                convert_layout(wrap_torch_tensor(s), CDNA4MXScaleLayout()))
    r = None if E == 1 else routing(torch.randn((T, E), generator=g, device=device), k)
    gathered = form == "gather swiglu"
    x, xs = downcast_to_mxfp(rnd(T if r is None or gathered else T * k, K), torch.uint8, axis=-1)
    if form == "pitch":
        x = torch.cat([x, x[:, :8]], dim=1)[:, :K // 2]
    bias, M = rnd(E, N), T if r is None else T * k
    lhs = InFlexData(F8) if form == "lhs type" else InFlexData()

    def call():
        pc = PrecisionConfig(flex_ctx=FlexCtx(lhs_data=lhs), a_mx_scale=xs, a_microblock_size=32, b_mx_scale=s, b_microblock_size=32,
                             out_dtype=torch.float32 if form == "out type" else None)
        c = torch.zeros((M, N), dtype=torch.bfloat16, device=device) if form == "c" else None
        return [matmul(x, w, bias if r is not None else bias[0], r.ragged_metadata if r is not None else None,
                       gather_indx=r.gather_indx if gathered else None, scatter_indx=r.scatter_indx if form == "scatter" else None,
                       precision_config=pc, c=c, fused_activation=SWIGLU if gathered else None)]

    assert BothPaths(monkeypatch, "matmul")(call) == covered


def test_native_matmul_fills_in_the_output_block_size(device, monkeypatch):
    torch.manual_seed(12)
    x, xs = downcast_to_mxfp(torch.randn(5, 64, device=device).bfloat16(), F8, axis=-1)
    v, s = downcast_to_mxfp(torch.randn(96, 64, device=device).bfloat16(), torch.uint8, axis=-1)

    def call():
        ys = torch.zeros((5, 3), dtype=torch.uint8, device=device)
        pc = PrecisionConfig(a_mx_scale=xs, a_microblock_size=32, b_mx_scale=s.t(), b_microblock_size=32, c_mx_scale=ys)
        y = matmul(x, v.t(), None, precision_config=pc, epilogue=Epilogue(FnSpecs("QUANTIZE_MXFP8", None, (), ()), (), (), 6.0))
        assert pc.c_microblock_size == 32
        return [y, ys]

    assert BothPaths(monkeypatch, "matmul")(call)


def test_routing_in_threads(device):
    """Four threads that meet more shapes than are kept, and one that all of them come back to: every call is answered, each with its own tables."""
    import threading
    logits = torch.randn(900, 16, generator=torch.Generator().manual_seed(1)).to(device)
    want = {T: RR.routing_ref(logits[:T].cpu(), 2)["col_sum"] for T in (3, 333)}
    errors = []

    def work(first):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for T in range(first, 900, 4):
                    r, again = routing(logits[:T], 2), routing(logits[:3], 2)
                    assert r.col_sum.sum().item() == 2 * T and torch.equal(again.col_sum.cpu(), want[3])
                assert torch.equal(routing(logits[:333], 2).col_sum.cpu(), want[333])
        except Exception as e:
            errors.append(e)
    torch.cuda.synchronize()
    threads = [threading.Thread(target=work, args=(i + 1,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors

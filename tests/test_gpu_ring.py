"""GPU: the persistent kernel of few rows per slice (weights in 4 KB blocks, pre-shuffled scales) at the sizes where it can go wrong: K below a stage, below the
ring and off both, columns off strips and tiles, empty slices and slices of several blocks, with gathered and scattered rows that are not
there, every kind of row and of output.  Rows of 8 and 4 bits give the bits of the tiled kernels, which strided weights take; 16-bit
rows are held against float32 products."""
import ctypes

import pytest
import torch

from triton_amd import _lib, _native
from triton_amd.matmul import Epilogue, FlexCtx, FnSpecs, FusedActivation, InFlexData, OutFlexData, PrecisionConfig, matmul
from triton_amd.numerics_details.mxfp import downcast_to_mxfp, upcast_from_mxfp
from triton_amd.swiglu import swiglu_fn
from triton_amd.tensor import FP4, convert_layout, make_ragged_tensor_metadata, wrap_torch_tensor
from triton_amd.tensor_details.layout import CDNA4MXScaleLayout, CDNA4MXValueLayout

SWIGLU = FusedActivation(FnSpecs("swiglu", swiglu_fn, ("alpha", "limit"), reduction_n=2), (1.702, 7.0))
TO_MXFP8 = Epilogue(FnSpecs("QUANTIZE_MXFP8", None, (), ()), (), (), 6.0)
TYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "fp8": torch.float8_e4m3fn}


def ring_rows(m, n, k, e, kind, out="16", swiglu=False, **changed):
    bag = _lib.MatmulArgBag()
    bag.x_dtype = {"bf16": _lib.BF16, "f16": _lib.F16, "mxfp4": _lib.MXFP4}.get(kind, _lib.FP8_E4M3)
    bag.y_dtype = _lib.FP8_E4M3 if out != "16" else _lib.F16 if kind == "f16" else _lib.BF16
    bag.M, bag.N, bag.K, bag.n_experts, bag.w_dtype = m, n, k, e, _lib.MXFP4
    bag.w_layout, bag.w_mx_layout, bag.block_schedule = _lib.W_CDNA4_BLOCKS, _lib.SCALE_CDNA4, 1 << 20
    bag.activation = _lib.ACT_SWIGLU if swiglu else _lib.ACT_NONE
    bag.y, bag.y_rows, bag.y_stride_m = 1 << 20, m, n // 2 if swiglu else n
    if kind[:2] == "mx":
        bag.x_mx_scale = 1 << 20
    if out == "mx":
        bag.y_mx_scale, bag.y_mx_stride_m = 1 << 20, -(-n // 32)
    for name, value in changed.items():
        setattr(bag, name, value)
    packed = bag.pack()
    return _native.ring_rows(ctypes.addressof(packed), 256)


def test_where_it_is_taken():
    """Layers timed with both: large ones of few rows, by the block that covers their slices; not what the kernel does not cover."""
    assert ring_rows(2036, 11520, 5760, 128, "fp8") == 64 and ring_rows(512, 5760, 2880, 128, "fp8") == 32
    assert ring_rows(8192, 5760, 2880, 128, "mxfp4", swiglu=True) == 96 and ring_rows(2048, 5760, 2880, 128, "mxfp8") == 32
    for M, N, K, E, kind in ((256, 5760, 2880, 128, "bf16"), (16384, 5760, 2880, 128, "bf16"), (65536, 5760, 2880, 32, "fp8"),
                             (1, 5760, 2880, 128, "fp8"), (2048, 5760, 512, 128, "mxfp4")):
        assert ring_rows(M, N, K, E, kind) == 0
    for changed in (dict(w_layout=_lib.W_STRIDED), dict(w_mx_layout=_lib.SCALE_STRIDED), dict(block_schedule=None), dict(n_experts=257),
                    dict(x_dtype=_lib.FP8_E5M2), dict(y_dtype=_lib.F32), dict(y_dtype=_lib.F16), dict(y_rows=0), dict(y_rows=1 << 20),
                    dict(y_expected_scale=1 << 20), dict(N=5759), dict(y=(1 << 20) + 2), dict(y_stride_m=5761)):
        assert ring_rows(512, 5760, 2880, 128, "fp8", **changed) == 0, changed


def blocks(w, ws):
    return convert_layout(wrap_torch_tensor(w, dtype=FP4), CDNA4MXValueLayout()), convert_layout(wrap_torch_tensor(ws), CDNA4MXScaleLayout())


# (rows per slice, slices, K, columns): blocks of 32 alone on their CUs (K of one stage and less, of fewer stages than the ring, off the
# stages), in several rounds; of 64; of 96
SIZES = [(9, 10, 96, 2832), (4, 12, 352, 1872), (14, 16, 736, 1296), (20, 16, 1440, 1392), (5, 128, 1056, 1184), (11, 64, 2144, 2320),
         (40, 16, 608, 2608), (30, 60, 1248, 2320), (72, 32, 1056, 4368)]


@pytest.mark.gpu
@pytest.mark.parametrize("rows,E,K,N", SIZES)
@pytest.mark.parametrize("kind", ["bf16", "f16", "fp8", "mxfp8", "mxfp4"])
@pytest.mark.parametrize("out", ["16", "16 swiglu", "fp8 swiglu", "mx swiglu"])
def test_edges(rows, E, K, N, kind, out, device):
    swiglu, to = out.endswith("swiglu"), out.split()[0]
    sizes = torch.randint(max(0, rows - 9), rows + 10, (E,), generator=torch.Generator().manual_seed(rows), dtype=torch.int32)
    sizes[1], sizes[E // 2] = 0, 3 * rows
    M, T = int(sizes.sum()), 50
    used = ring_rows(M, N, K, E, kind, to, swiglu)
    if not used:
        pytest.skip("another kernel's")
    torch.manual_seed(K)
    gather, scatter = torch.randint(0, T, (M,), dtype=torch.int32), torch.randperm(M, dtype=torch.int32)
    gather[3], scatter[5] = -1, -1
    x = torch.randn(T, K, device=device)
    w, ws = downcast_to_mxfp((torch.randn(E, N, K, device=device) * 0.1).bfloat16(), torch.uint8, axis=-1)
    w, ws = w.transpose(1, 2), ws.transpose(1, 2)
    wb, wsb = blocks(w, ws)
    bias, gammas = torch.randn(E, N, device=device), torch.rand(M, device=device)
    opts = {}
    if kind[:2] == "mx":
        a, s = downcast_to_mxfp(x, torch.uint8 if kind == "mxfp4" else torch.float8_e4m3fn, axis=-1)
        opts.update(a_mx_scale=s, a_microblock_size=32)
    else:
        a = x.to(TYPES[kind])
    scale = torch.full((1,), 0.25, device=device)
    lhs = InFlexData(a.dtype, scale) if kind == "fp8" else InFlexData()
    if to == "fp8":
        opts.update(flex_ctx=FlexCtx(lhs_data=lhs, out_data=OutFlexData(torch.float8_e4m3fn, torch.full((1,), 0.125, device=device))),
                    out_dtype=torch.float8_e4m3fn, flexpoint_saturate_inf=True)
    else:
        opts.update(flex_ctx=FlexCtx(lhs_data=lhs), out_dtype=torch.float8_e4m3fn if to == "mx" else torch.float16 if kind == "f16" else torch.bfloat16)
    md = make_ragged_tensor_metadata(sizes.to(device), M)

    def run(weights, scales):
        c = torch.zeros(M, -(-N // (64 if swiglu else 32)), dtype=torch.uint8, device=device) if to == "mx" else None
        pc = PrecisionConfig(b_mx_scale=scales, b_microblock_size=32, c_mx_scale=c, **opts)
        y = matmul(a, weights, bias, md, gather_indx=gather.to(device), scatter_indx=None if to == "mx" else scatter.to(device),
                   gammas=gammas, precision_config=pc, fused_activation=SWIGLU if swiglu else None, **({"epilogue": TO_MXFP8} if to == "mx" else {}))
        rows_of = torch.arange(M) if to == "mx" else scatter.long()
        there = torch.arange(M)[rows_of >= 0]
        return y[rows_of[there].to(device)], None if c is None else c, there

    got, got_scales, there = run(wb, wsb)
    if kind not in ("bf16", "f16"):
        ref, ref_scales, _ = run(w, ws)
        assert torch.equal(got.view(torch.uint8), ref.view(torch.uint8))
        assert got_scales is None or torch.equal(got_scales, ref_scales)
        return
    wf = upcast_from_mxfp(w, ws, torch.float32, axis=1)
    expert = torch.repeat_interleave(torch.arange(E), sizes.long())
    xf = torch.where((gather >= 0)[:, None].to(device), a.float()[gather.clamp(min=0).long().to(device)], 0.0)
    full = torch.empty(M, N // 2 if swiglu else N, device=device)
    slack = torch.empty_like(full)
    for e in range(E):
        r = (expert == e).to(device)
        v, mag = xf[r] @ wf[e] + bias[e], K * 2.0 ** -23 * (xf[r].abs() @ wf[e].abs())
        if swiglu:
            g, l = v[:, 0::2].clamp(max=7.0), v[:, 1::2].clamp(-7.0, 7.0)
            s = g * torch.sigmoid(1.702 * g)
            v, mag = s * (l + 1), 1.2 * mag[:, 0::2] * (l.abs() + 1) + s.abs() * mag[:, 1::2]   # (|d swish| <= 1.1)
        full[r], slack[r] = v * gammas[r, None], mag
    full, slack = full[there.to(device)], slack[there.to(device)]
    # a 16-bit result (2^-8) of K float32 additions, and the hardware's exponential and reciprocal (2^-20)
    assert bool(((got.float() - full).abs() <= 2.0 ** -8 * full.abs() + slack + 1e-5).all())

"""GPU: MXFP4 weights with few tiles.  16-bit rows: eight K groups on tiles of 128 columns, at the lines of its K (928 to 7168: groups of one pair of stages, groups
beyond the end of K, the last scales that fit) and at the edges of its columns, against float32 products.  Rows of 8 and 4 bits: four groups, from K 769 on, likewise."""
import pytest
import torch

from triton_amd.matmul import FnSpecs, FusedActivation, PrecisionConfig, matmul
from triton_amd.matmul_details.opt_flags import scoped_opt_flags_constraints
from triton_amd.numerics_details.mxfp import downcast_to_mxfp, upcast_from_mxfp
from triton_amd.swiglu import swiglu_fn
from triton_amd.tensor import FP4, convert_layout, make_ragged_tensor_metadata, wrap_torch_tensor
from triton_amd.tensor_details.layout import CDNA4MXScaleLayout, CDNA4MXValueLayout

pytestmark = pytest.mark.gpu
SWIGLU = FusedActivation(FnSpecs("swiglu", swiglu_fn, ("alpha", "limit"), reduction_n=2), (1.702, 7.0))


@pytest.mark.parametrize("K,N", [(896, 264), (928, 264), (1024, 128), (1056, 130), (1152, 8), (2080, 392), (7168, 136), (7200, 136)])
@pytest.mark.parametrize("layout", ["blocks", "strided", "strided, odd"])
@pytest.mark.parametrize("mode", ["dense", "ragged", "ragged swiglu"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_edges(K, N, layout, mode, dtype, device):
    torch.manual_seed(K + N)
    ragged, swiglu = mode != "dense", mode.endswith("swiglu")
    sizes = [33, 0, 24] if ragged else [70]
    E, M = len(sizes), sum(sizes)
    w, ws = downcast_to_mxfp((torch.randn(E, N, K, device=device) * torch.exp(torch.randn(E, N, 1, device=device))).bfloat16(), torch.uint8, axis=-1)
    wf = upcast_from_mxfp(w, ws, torch.float32, axis=-1).transpose(1, 2)
    if layout == "strided, odd":   # (scales that no copy of 16 bytes can take)
        ws = torch.empty(ws.numel() + 4, dtype=torch.uint8, device=device)[4:].view(ws.shape).copy_(ws)
    w, ws = w.transpose(1, 2), ws.transpose(1, 2)
    if not ragged:
        w, ws = w[0], ws[0]
    if layout == "blocks":
        w, ws = convert_layout(wrap_torch_tensor(w, dtype=FP4), CDNA4MXValueLayout()), convert_layout(wrap_torch_tensor(ws), CDNA4MXScaleLayout())
    x = torch.randn(50 if ragged else M, K, device=device).to(dtype)
    gather = torch.randint(-1, 50, (M,), dtype=torch.int32, device=device) if ragged else None
    bias = torch.randn(E, N, device=device)
    md = make_ragged_tensor_metadata(torch.tensor(sizes, dtype=torch.int32, device=device), M) if ragged else None
    with scoped_opt_flags_constraints({"block_m": 32}):
        got = matmul(x, w, bias if ragged else bias[0], md, gather_indx=gather, fused_activation=SWIGLU if swiglu else None,
                     precision_config=PrecisionConfig(b_mx_scale=ws, b_microblock_size=32))
    rows = x.float() if gather is None else torch.where((gather >= 0)[:, None], x.float()[gather.clamp(min=0).long()], 0.0)
    at = 0
    for e, n in enumerate(sizes):
        r = rows[at:at + n]
        v, slack = r @ wf[e] + bias[e], K * 2.0 ** -23 * (r.abs() @ wf[e].abs())
        if swiglu:
            g, l = v[:, 0::2].clamp(max=7.0), v[:, 1::2].clamp(-7.0, 7.0)
            s = g * torch.sigmoid(1.702 * g)
            v, slack = s * (l + 1), 1.2 * slack[:, 0::2] * (l.abs() + 1) + s.abs() * slack[:, 1::2]   # (|d swish| <= 1.1)
        # a 16-bit result (2^-8) of K float32 additions on either side
        assert bool(((got[at:at + n].float() - v).abs() <= 2.0 ** -8 * v.abs() + 2 * slack + 1e-5).all())
        at += n


@pytest.mark.parametrize("K,N", [(768, 264), (800, 264), (1024, 128), (1056, 130), (1312, 8), (2112, 392), (8192, 136)])
@pytest.mark.parametrize("layout", ["blocks", "strided, odd"])
@pytest.mark.parametrize("mode", ["dense", "ragged", "ragged swiglu"])
@pytest.mark.parametrize("kind", ["fp8", "fp8e5", "mxfp8", "mxfp4"])
def test_edges_of_8_and_4_bits(K, N, layout, mode, kind, device):
    torch.manual_seed(K + N)
    ragged, swiglu = mode != "dense", mode.endswith("swiglu")
    sizes = [33, 0, 24] if ragged else [70]
    E, M = len(sizes), sum(sizes)
    w, ws = downcast_to_mxfp((torch.randn(E, N, K, device=device) * 0.1).bfloat16(), torch.uint8, axis=-1)
    wf = upcast_from_mxfp(w, ws, torch.float32, axis=-1).transpose(1, 2)
    if layout != "blocks":   # (scales at an odd address between others that are NaN)
        room = torch.full((ws.numel() + 65,), 255, dtype=torch.uint8, device=device)
        ws = room[1:1 + ws.numel()].view(ws.shape).copy_(ws)
    w, ws = w.transpose(1, 2), ws.transpose(1, 2)
    if not ragged:
        w, ws = w[0], ws[0]
    if layout == "blocks":
        w, ws = convert_layout(wrap_torch_tensor(w, dtype=FP4), CDNA4MXValueLayout()), convert_layout(wrap_torch_tensor(ws), CDNA4MXScaleLayout())
    x, opts = torch.randn(50 if ragged else M, K, device=device), {}
    if kind[:2] == "mx":
        x, s = downcast_to_mxfp(x, torch.uint8 if kind == "mxfp4" else torch.float8_e4m3fn, axis=-1)
        xf = upcast_from_mxfp(x, s, torch.float32, axis=-1)
        opts.update(a_mx_scale=s, a_microblock_size=32)
    else:
        x = x.to(torch.float8_e4m3fn if kind == "fp8" else torch.float8_e5m2)
        xf = x.float()
    gather = torch.randint(-1, 50, (M,), dtype=torch.int32, device=device) if ragged else None
    bias = torch.randn(E, N, device=device)
    md = make_ragged_tensor_metadata(torch.tensor(sizes, dtype=torch.int32, device=device), M) if ragged else None
    with scoped_opt_flags_constraints({"block_m": 32}):
        got = matmul(x, w, bias if ragged else bias[0], md, gather_indx=gather, fused_activation=SWIGLU if swiglu else None,
                     precision_config=PrecisionConfig(b_mx_scale=ws, b_microblock_size=32, out_dtype=torch.float32, **opts))
    rows = xf if gather is None else torch.where((gather >= 0)[:, None], xf[gather.clamp(min=0).long()], 0.0)
    at = 0
    for e, n in enumerate(sizes):
        r = rows[at:at + n]
        # float32 sums of products that the instruction aligns at the largest of 64 (off by up to 6e-5 of the result); 1e-4 of the sum of magnitudes
        v, slack = r @ wf[e] + bias[e], 1e-4 * (r.abs() @ wf[e].abs())
        if swiglu:
            g, l = v[:, 0::2].clamp(max=7.0), v[:, 1::2].clamp(-7.0, 7.0)
            s = g * torch.sigmoid(1.702 * g)
            v, slack = s * (l + 1), 1.2 * slack[:, 0::2] * (l.abs() + 1) + s.abs() * slack[:, 1::2]   # (|d swish| <= 1.1)
        assert bool(((got[at:at + n] - v).abs() <= slack + 1e-5 + 2.0 ** -20 * v.abs()).all())
        at += n

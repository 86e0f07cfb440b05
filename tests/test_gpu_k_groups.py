"""GPU: 16-bit rows x MXFP4 weights with few tiles: eight K groups on tiles of 128 columns, at the lines of its K (928 to 7168: groups of one pair of stages, groups
beyond the end of K, the last scales that fit) and at the edges of its columns, against float32 products."""
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

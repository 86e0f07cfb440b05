"""GPU: MXFP8 activations against MXFP4 weights where the number of 32-K groups decides how the rows' block scales are copied
(four, two or one byte at a time), for every row block and both scale layouts, against float32 products of the same values."""
import pytest
import torch

from triton_amd.matmul import PrecisionConfig, matmul
from triton_amd.matmul_details.opt_flags import scoped_opt_flags_constraints
from triton_amd.numerics_details.mxfp import downcast_to_mxfp, upcast_from_mxfp
from triton_amd.tensor import convert_layout, make_ragged_tensor_metadata, wrap_torch_tensor
from triton_amd.tensor_details.layout import CDNA4MXScaleLayout

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [32, 320, 352, 384, 2880])
@pytest.mark.parametrize("block_m", [32, 64, 128])
@pytest.mark.parametrize("swizzled", [False, True])
def test_block_scales_of_rows(K, block_m, swizzled, device):
    torch.manual_seed(0)
    sizes = torch.tensor([70, 1, 0, 129], dtype=torch.int32)
    M, N, E = int(sizes.sum()), 264, 4
    x = torch.randn(M, K, device=device) * torch.exp(torch.randn(M, K // 32, device=device)).repeat_interleave(32, dim=1)
    xq, xs = downcast_to_mxfp(x, torch.float8_e4m3fn, axis=-1)
    wq, ws = downcast_to_mxfp(torch.randn(E, K, N, device=device) * 0.1, torch.uint8, axis=1)
    xf = upcast_from_mxfp(xq, xs, torch.float32, axis=-1).cpu()
    wf = upcast_from_mxfp(wq, ws, torch.float32, axis=1).cpu()
    scales = convert_layout(wrap_torch_tensor(ws), CDNA4MXScaleLayout()) if swizzled else ws
    pc = PrecisionConfig(a_mx_scale=xs, a_microblock_size=32, b_mx_scale=scales, b_microblock_size=32, out_dtype=torch.bfloat16)
    gather = torch.randperm(M).int()
    md = make_ragged_tensor_metadata(sizes.to(device), M)
    with scoped_opt_flags_constraints({"block_m": block_m}):
        y = matmul(xq, wq, None, md, gather_indx=gather.to(device), precision_config=pc)
    rows = xf[gather.long()].split(sizes.tolist())
    ref = torch.cat([part @ wf[e] for e, part in enumerate(rows)])
    torch.testing.assert_close(y.cpu().float(), ref, rtol=1e-2, atol=1e-2 * float(ref.abs().mean()) + 1e-3)

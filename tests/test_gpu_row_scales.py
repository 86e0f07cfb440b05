"""GPU: block scales of float8_e5m2 rows (float8_e4m3fn tensors whose bytes the flex options name as e5m2) enter the product in every
kernel that such rows can take."""
import pytest
import torch

from triton_amd.matmul import FlexCtx, InFlexData, PrecisionConfig, matmul
from triton_amd.matmul_details.opt_flags import scoped_opt_flags_constraints
from triton_amd.numerics_details.mxfp import downcast_to_mxfp, upcast_from_mxfp
from triton_amd.tensor import make_ragged_tensor_metadata

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [64, 736])
@pytest.mark.parametrize("block_m", [None, 16, 32, 64, 128])
@pytest.mark.parametrize("ragged", [False, True])
def test_e5m2_rows(ragged, block_m, K, device):
    torch.manual_seed(K)
    M, N = 37, 272
    x = torch.randn(M, K, device=device).to(torch.float8_e5m2)
    s = torch.randint(118, 134, (M, K // 32), dtype=torch.uint8, device=device)
    w, ws = downcast_to_mxfp(torch.randn(1, K, N, device=device), torch.uint8, axis=1)
    wf = upcast_from_mxfp(w, ws, torch.float32, axis=1)[0].double()
    pc = PrecisionConfig(a_mx_scale=s, a_microblock_size=32, b_mx_scale=ws, b_microblock_size=32, out_dtype=torch.float32,
                         flex_ctx=FlexCtx(lhs_data=InFlexData(torch.float8_e5m2)))
    md = make_ragged_tensor_metadata(torch.tensor([M], dtype=torch.int32, device=device), M) if ragged else None
    with scoped_opt_flags_constraints({} if block_m is None else {"block_m": block_m}):
        y = matmul(x.view(torch.float8_e4m3fn), w if ragged else w[0], None, md, precision_config=pc).double()
    xf = x.double() * (2.0 ** (s.double() - 127)).repeat_interleave(32, dim=1)
    # (the scaled MFMA drops parts of its products, 6e-5 of the result; a group's scale is a factor of 2^-9 to 2^6)
    assert float((y - xf @ wf).norm() / (xf @ wf).norm()) <= 2.0 ** -13

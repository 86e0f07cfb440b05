"""GPU: outputs that the tiled kernels store pair by pair through 32-bit offsets, and those they store element by element
(odd column counts, an output that starts on an odd element, odd row pitches), against the oracle."""
import pytest
import torch

from oracle import matmul_ref as MR
from oracle.mxfp_ref import downcast_to_mxfp_ref
from triton_amd.matmul import PrecisionConfig, matmul
from triton_amd.matmul_details.opt_flags import scoped_opt_flags_constraints
from triton_amd.numerics_details.mxfp import downcast_to_mxfp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("block_m,M", [(32, 33), (128, 160)])
@pytest.mark.parametrize("N,first,pitch", [(202, 0, 202), (201, 0, 201), (202, 1, 202), (202, 0, 203), (64, 0, 64)])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
def test_output_alignment(block_m, M, N, first, pitch, out_dtype, device):
    torch.manual_seed(0)
    K = 96
    x, w, bias = torch.randn(M, K).to(torch.bfloat16), torch.randn(K, N) * 0.1, torch.randn(N)
    v, s = downcast_to_mxfp(w.to(device), torch.uint8, axis=0)
    rv, rs = downcast_to_mxfp_ref(w, torch.uint8, 0)
    flat = torch.full((first + M * pitch + 8, ), -7.0, dtype=out_dtype, device=device)
    y = flat[first:first + M * pitch].view(M, pitch)[:, :N]
    with scoped_opt_flags_constraints({"block_m": block_m}):
        matmul(x.to(device), v, bias.to(device), precision_config=PrecisionConfig(b_mx_scale=s, b_microblock_size=32), c=y)
    ref = MR.matmul_ref(x, rv, bias, b_mx_scale=rs)
    torch.testing.assert_close(y.cpu().float(), ref.float(), rtol=1e-2, atol=1e-2)
    untouched = torch.ones_like(flat, dtype=torch.bool)
    untouched[first:first + M * pitch].view(M, pitch)[:, :N] = False
    assert (flat[untouched] == -7.0).all()

"""GPU: strided MXFP4 weights, which come 256 K at a time, give the bits of pre-shuffled ones, which come by the stage (the same
products in the same order), with the last piece of K whole, half and partial and columns past the end of a tile."""
import pytest
import torch

from triton_amd.matmul import PrecisionConfig, matmul
from triton_amd.matmul_details.opt_flags import scoped_opt_flags_constraints
from triton_amd.numerics_details.mxfp import downcast_to_mxfp
from triton_amd.tensor import FP4, convert_layout, make_ragged_tensor_metadata, wrap_torch_tensor
from triton_amd.tensor_details.layout import CDNA4MXScaleLayout, CDNA4MXValueLayout

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [32, 128, 160, 256, 288, 384, 416, 672])
@pytest.mark.parametrize("dtype,block_m", [(torch.bfloat16, 32), (torch.float16, 64), (torch.float8_e4m3fn, 32),
                                           (torch.float8_e4m3fn, 128), (torch.float8_e5m2, 128)])
def test_same_bits(K, dtype, block_m, device):
    torch.manual_seed(K)
    sizes = torch.tensor([70, 1, 0, 129], dtype=torch.int32)
    M, N, E = int(sizes.sum()), 266, 4
    x = torch.randn(M, K, device=device).to(dtype)
    w, s = downcast_to_mxfp(torch.randn(E, K, N, device=device) * torch.exp(torch.randn(E, 1, N, device=device)), torch.uint8, axis=1)
    md = make_ragged_tensor_metadata(sizes.to(device), M)

    def product(w, s):
        pc = PrecisionConfig(b_mx_scale=s, b_microblock_size=32, out_dtype=torch.float32)
        with scoped_opt_flags_constraints({"block_m": block_m}):
            return matmul(x, w, None, md, precision_config=pc)

    blocks = convert_layout(wrap_torch_tensor(w, dtype=FP4), CDNA4MXValueLayout())
    assert torch.equal(product(w, s), product(blocks, convert_layout(wrap_torch_tensor(s), CDNA4MXScaleLayout())))


@pytest.mark.parametrize("K", [1056, 1312, 1952, 4256])
@pytest.mark.parametrize("dtype,block_m", [(torch.bfloat16, 32), (torch.float16, 32), (torch.float8_e4m3fn, 32)])
def test_same_bits_of_one_block_per_slice(K, dtype, block_m, device):
    """Columns that do not start on 64 bytes, more tiles than CUs, slices of up to one row block: 16-bit rows take the kernel with pieces
    of 64 bytes."""
    torch.manual_seed(K)
    E, N = 44, 1544
    sizes = torch.randint(0, 33, (E,), dtype=torch.int32)
    sizes[0], sizes[1], sizes[2] = 32, 33, 0
    M = int(sizes.sum())
    x = torch.randn(M + 5, K, device=device).to(dtype)
    gather = torch.randint(-1, M + 5, (M,), dtype=torch.int32, device=device)
    w, s = downcast_to_mxfp(torch.randn(E, K, N, device=device), torch.uint8, axis=1)
    md = make_ragged_tensor_metadata(sizes.to(device), M)

    def product(w, s):
        pc = PrecisionConfig(b_mx_scale=s, b_microblock_size=32, out_dtype=torch.float32)
        with scoped_opt_flags_constraints({"block_m": block_m}):
            return matmul(x, w, None, md, gather_indx=gather, precision_config=pc)

    blocks = convert_layout(wrap_torch_tensor(w, dtype=FP4), CDNA4MXValueLayout())
    assert torch.equal(product(w, s), product(blocks, convert_layout(wrap_torch_tensor(s), CDNA4MXScaleLayout())))

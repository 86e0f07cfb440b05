"""GPU: 16-bit weights that a call reads more of than the caches keep are copied non-temporally, by the persistent kernel and, for products that
it does not take, by the tiled one; the bits are those of the ordinary copies, which weights with columns off whole lines take."""
import ctypes
import sys

import pytest
import torch

from triton_amd import _native
from triton_amd.matmul import PrecisionConfig, matmul
from triton_amd.matmul_details.opt_flags import scoped_opt_flags_constraints
from triton_amd.tensor import make_ragged_tensor_metadata

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [3, 20, 45, 90])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_same_bits(rows, dtype, device):
    """In the persistent kernel (its blocks are 64 and 160 rows here)."""
    torch.manual_seed(rows)
    E, K, N = 5, 2048, 20016
    sizes = torch.tensor([rows, 0, 3 * rows, 1, rows], dtype=torch.int32, device=device)   # (empty, and several blocks)
    M = 5 * rows + 1
    w = torch.randn(E, N, K, device=device, dtype=dtype)
    off_lines = torch.zeros(E, N, K + 8, device=device, dtype=dtype)
    off_lines[:, :, :K] = w
    x = torch.randn(M, K, device=device, dtype=dtype)
    md = make_ragged_tensor_metadata(sizes, M)
    y = [matmul(x, v.transpose(1, 2), None, md, precision_config=PrecisionConfig()) for v in (w, off_lines[:, :, :K])]
    assert torch.equal(y[0], y[1])


@pytest.mark.parametrize("rows", [3, 20, 90, "dense"])
def test_same_bits_in_tiles(rows, monkeypatch, device):
    """float32 outputs and dense products are the tiled kernel's."""
    torch.manual_seed(1)
    E, K, N = 5, 2048, 20016
    dense = rows == "dense"
    if dense:
        E, K, N, M, md = 1, 4096, 41008, 20, None
    else:
        sizes = torch.tensor([rows, 0, 3 * rows, 1, rows], dtype=torch.int32, device=device)
        M = 5 * rows + 1
        md = make_ragged_tensor_metadata(sizes, M)
    w = torch.randn(E, N, K, device=device, dtype=torch.bfloat16)
    off_lines = torch.zeros(E, N, K + 8, device=device, dtype=torch.bfloat16)
    off_lines[:, :, :K] = w
    x = torch.randn(M, K, device=device, dtype=torch.bfloat16)
    seen = []
    module = sys.modules["triton_amd.matmul"]
    launch = module._launch
    monkeypatch.setattr(module, "_launch", lambda args, dev: seen.append(args) or launch(args, dev))
    with scoped_opt_flags_constraints({"num_warps": 4}):   # (asks for nothing, through the general host path)
        y = [matmul(x, v[0] if dense else v, None, md, precision_config=PrecisionConfig(out_dtype=torch.float32))
             for v in (w.transpose(1, 2), off_lines[:, :, :K].transpose(1, 2))]
    assert torch.equal(y[0], y[1])
    for args in seen:
        assert not _native.ring_rows(ctypes.addressof(args), 256)
    block_m = seen[0].block_m if not dense else _native.dense_block_m(ctypes.addressof(seen[0]), 256)
    live = E if dense else E * (1 - 0.8 ** M)
    assert 4 * (M // E) <= 3 * block_m and live * N * K * 2 >= 320 << 20   # (what the tiled kernel asks for)

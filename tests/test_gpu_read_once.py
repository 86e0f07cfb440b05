"""GPU: 16-bit weights that a call reads more of than the caches keep are copied non-temporally; the bits are those of the ordinary copies, which
weights with columns off whole lines take."""
import pytest
import torch

from triton_amd.matmul import PrecisionConfig, matmul
from triton_amd.tensor import make_ragged_tensor_metadata

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [3, 20, 45, 90])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_same_bits(rows, dtype, device):
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

"""GPU: tiles of ragged problems found from the slice sizes: numbers of slices around the lanes of a wave and past what they hold,
empty slices, slices of many row blocks (walked in groups), for every row block, against float32 products."""
import pytest
import torch

from triton_amd.matmul import PrecisionConfig, matmul
from triton_amd.matmul_details.opt_flags import scoped_opt_flags_constraints
from triton_amd.numerics_details.mxfp import downcast_to_mxfp, upcast_from_mxfp
from triton_amd.tensor import make_ragged_tensor_metadata

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E", [1, 63, 64, 65, 200, 512, 513])
@pytest.mark.parametrize("block_m", [16, 32, 64, 128])
@pytest.mark.parametrize("kind", ["bf16", "fp8", "mxfp4"])
def test_slices(E, block_m, kind, device):
    torch.manual_seed(E)
    K, N = 256, 272
    sizes = torch.randint(0, 5, (E,), dtype=torch.int32)
    sizes[:: max(1, E // 3)] = 7 * block_m + 5      # several groups of row blocks, a remainder
    M = int(sizes.sum())
    w, ws = downcast_to_mxfp(torch.randn(E, K, N, device=device) * 0.1, torch.uint8, axis=1)
    x = torch.randn(M, K, device=device)
    pc = dict(b_mx_scale=ws, b_microblock_size=32, out_dtype=torch.bfloat16)
    if kind == "mxfp4":
        a, s = downcast_to_mxfp(x, torch.uint8, axis=-1)
        x, pc["a_mx_scale"], pc["a_microblock_size"] = upcast_from_mxfp(a, s, torch.float32, axis=-1), s, 32
    else:
        a = x.to(torch.bfloat16 if kind == "bf16" else torch.float8_e4m3fn)
        x = a.float()
    md = make_ragged_tensor_metadata(sizes.to(device), M)
    with scoped_opt_flags_constraints({"block_m": block_m}):
        y = matmul(a, w, None, md, precision_config=PrecisionConfig(**pc)).float()
    wf = upcast_from_mxfp(w, ws, torch.float32, axis=1)
    for e, (rows, got) in enumerate(zip(x.split(sizes.tolist()), y.split(sizes.tolist()))):
        ref = rows @ wf[e]
        # a 16-bit result (2^-8) of K float32 additions
        bound = 2.0 ** -8 * ref.abs() + K * 2.0 ** -23 * (rows.abs() @ wf[e].abs())
        assert bool(((got - ref).abs() <= bound + 1e-6).all()), e

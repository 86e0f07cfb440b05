"""GPU: gathered rows whose index is -1 are rows of zeros in every kernel, whatever lies in front of the activations and of their
block scales: the product's row is the bias, and the other rows are what float32 gives."""
import pytest
import torch

from triton_amd.matmul import PrecisionConfig, matmul
from triton_amd.matmul_details.opt_flags import scoped_opt_flags_constraints
from triton_amd.numerics_details.mxfp import downcast_to_mxfp, upcast_from_mxfp
from triton_amd.tensor import make_ragged_tensor_metadata

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("block_m", [16, 32, 64, 128])
@pytest.mark.parametrize("K", [640, 1440])   # (1440: K groups for blocks of 16 and 32)
@pytest.mark.parametrize("kind", ["bf16", "f16", "fp8", "mxfp8", "mxfp4", "bf16 w along K", "bf16 w along N"])
def test_no_row(kind, K, block_m, device):
    torch.manual_seed(block_m)
    T, E, N = 40, 3, 272
    sizes = torch.tensor([block_m + 3, 5, 0], dtype=torch.int32)
    M = int(sizes.sum())
    gather = torch.randint(1, T - 1, (M,), dtype=torch.int32)
    none = torch.rand(M) < 0.3
    none[0] = none[M - 1] = True
    gather[none] = -1
    x, w, bias = torch.randn(T, K, device=device), torch.randn(E, K, N, device=device) * 0.1, torch.randn(E, N, device=device)
    pc = {"out_dtype": torch.bfloat16}
    if kind.startswith("bf16 w"):
        w = w.bfloat16()
        w = w.transpose(1, 2).contiguous().transpose(1, 2) if kind.endswith("K") else w
        wf = w.float()
    else:
        w, ws = downcast_to_mxfp(w, torch.uint8, axis=1)
        wf = upcast_from_mxfp(w, ws, torch.float32, axis=1)
        pc.update(b_mx_scale=ws, b_microblock_size=32)
    if kind[:2] == "mx":
        a, s = downcast_to_mxfp(x, torch.uint8 if kind == "mxfp4" else torch.float8_e4m3fn, axis=-1)
        x = upcast_from_mxfp(a, s, torch.float32, axis=-1)
        s[0] = s[T - 1] = 255                       # (NaN: the rows at the ends are not gathered, and stand for no other)
        pc.update(a_mx_scale=s, a_microblock_size=32)
    else:
        a = x.to({"f16": torch.float16, "fp8": torch.float8_e4m3fn}.get(kind, torch.bfloat16))
        x = a.float()
    md = make_ragged_tensor_metadata(sizes.to(device), M)
    with scoped_opt_flags_constraints({"block_m": block_m}):
        y = matmul(a, w, bias, md, gather_indx=gather.to(device), precision_config=PrecisionConfig(**pc)).float()
    none = none.to(device)
    rows = torch.where(none[:, None], 0.0, x[gather.clamp(min=0).long().to(device)])
    expert = torch.repeat_interleave(torch.arange(E), sizes.long()).to(device)
    assert torch.equal(y[none], bias[expert][none].bfloat16().float())
    for e in range(2):
        ref, mag = rows[expert == e] @ wf[e] + bias[e], rows[expert == e].abs() @ wf[e].abs() + bias[e].abs()
        # a 16-bit result (2^-8) of K float32 additions
        assert bool(((y[expert == e] - ref).abs() <= 2.0 ** -8 * ref.abs() + K * 2.0 ** -23 * mag + 1e-6).all()), e

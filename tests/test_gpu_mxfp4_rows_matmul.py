"""GPU: the kernel for packed e2m1 rows x MXFP4 weights where it can go wrong -- K of less than a stage, one stage and ragged last stages
(whose block scales are read eight at a time), few and odd numbers of rows, column tails, every row block, both layouts of codes and scales --
bit for bit against the same numbers as float8_e4m3fn rows (whose kernel takes the same products in the same steps), and its
precision against 64-bit sums."""
import pytest
import torch

from triton_amd.matmul import PrecisionConfig, matmul
from triton_amd.matmul_details.opt_flags import scoped_opt_flags_constraints
from triton_amd.numerics_details.mxfp import downcast_to_mxfp, upcast_from_mxfp
from triton_amd.tensor import FP4, convert_layout, make_ragged_tensor_metadata, wrap_torch_tensor
from triton_amd.tensor_details.layout import CDNA4MXScaleLayout, CDNA4MXValueLayout

pytestmark = pytest.mark.gpu


def _rows(M, K, device):
    x = torch.randn(M, K, device=device) * torch.exp(torch.randn(M, K // 32, device=device)).repeat_interleave(32, dim=1)
    q, s = downcast_to_mxfp(x, torch.uint8, axis=-1)
    values = upcast_from_mxfp(q, torch.full_like(s, 127), torch.float32, axis=-1)
    return q, s, values.to(torch.float8_e4m3fn)


def _weights(E, K, N, blocks, device):
    w, s = downcast_to_mxfp(torch.randn(E, K, N, device=device) * 0.1, torch.uint8, axis=1)
    if not blocks:
        return w, s, w, s
    return (convert_layout(wrap_torch_tensor(w, dtype=FP4), CDNA4MXValueLayout()),
            convert_layout(wrap_torch_tensor(s), CDNA4MXScaleLayout()), w, s)


@pytest.mark.parametrize("K", [32, 64, 224, 256, 288, 480, 512, 736, 2880])
@pytest.mark.parametrize("block_m", [16, 32, 64, 128])
@pytest.mark.parametrize("blocks", [False, True])
def test_same_bits_as_widened_rows(K, block_m, blocks, device):
    torch.manual_seed(0)
    sizes = torch.tensor([70, 1, 0, 129, 33], dtype=torch.int32)
    M, N, E = int(sizes.sum()), 328, 5
    xq, xs, x8 = _rows(M, K, device)
    w, ws, *_ = _weights(E, K, N, blocks, device)
    bias = torch.randn(E, N, device=device)
    gather = torch.randperm(M).int().to(device)
    md = make_ragged_tensor_metadata(sizes.to(device), M)
    out = []
    with scoped_opt_flags_constraints({"block_m": block_m}):
        for x in (xq, x8):
            pc = PrecisionConfig(a_mx_scale=xs, a_microblock_size=32, b_mx_scale=ws, b_microblock_size=32, out_dtype=torch.float32)
            out.append(matmul(x, w, bias, md, gather_indx=gather, precision_config=pc))
    assert torch.equal(out[0], out[1])


@pytest.mark.parametrize("rows", [1, 33, 300])
@pytest.mark.parametrize("K", [256, 928, 4096])
def test_precision(rows, K, device):
    """Products of e2m1 numbers and powers of two are exact; each of the K additions rounds once in float32 (an MFMA adds 64
    products with no more roundings than that)."""
    torch.manual_seed(1)
    N = 256
    xq, xs, _ = _rows(rows, K, device)
    w, ws, wq, wss = _weights(1, K, N, True, device)
    pc = PrecisionConfig(a_mx_scale=xs, a_microblock_size=32, b_mx_scale=ws, b_microblock_size=32, out_dtype=torch.float32)
    y = matmul(xq, w, None, precision_config=pc).double()
    xf = upcast_from_mxfp(xq, xs, torch.float32, axis=-1).double()
    wf = upcast_from_mxfp(wq, wss, torch.float32, axis=1)[0].double()
    assert bool(((y - xf @ wf).abs() <= K * 2.0 ** -24 * (xf.abs() @ wf.abs())).all())


@pytest.mark.parametrize("view", ["misaligned", "pitch"])
def test_other_rows_are_widened(view, device):
    """Rows that the kernel does not read as they are give the same result through float8_e4m3fn."""
    torch.manual_seed(2)
    K, N = 512, 192
    xq, xs, _ = _rows(40, K, device)
    w, ws, *_ = _weights(1, K, N, False, device)
    pc = PrecisionConfig(a_mx_scale=xs, a_microblock_size=32, b_mx_scale=ws, b_microblock_size=32, out_dtype=torch.float32)
    want = matmul(xq.clone(), w, None, precision_config=pc)
    if view == "misaligned":
        buf = torch.empty(xq.numel() + 1, dtype=torch.uint8, device=device)
        x = buf[1:].view(xq.shape)
    else:
        x = torch.empty((40, K // 2 + 8), dtype=torch.uint8, device=device)[:, :K // 2]
    x.copy_(xq)
    assert torch.equal(matmul(x, w, None, precision_config=pc), want)

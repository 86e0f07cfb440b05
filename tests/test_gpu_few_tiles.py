"""GPU: ragged products of few tiles, whose row blocks are smaller than the slices' sizes ask for (or, for fp8 rows, the streaming
kernel's): around the lines of the rule, against float32 products of the same values; block scales over their whole range, which only
the scaled MFMA takes, whatever the number of tiles; the weight scales that the streaming kernel holds exactly."""
import pytest
import torch

from triton_amd.matmul import Epilogue, FnSpecs, PrecisionConfig, matmul
from triton_amd.matmul_details.opt_flags import scoped_opt_flags_constraints
from triton_amd.numerics_details.mxfp import downcast_to_mxfp, upcast_from_mxfp
from triton_amd.tensor import make_ragged_tensor_metadata

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,E,N", [(150, 8, 272), (40, 8, 1552), (20, 3, 304), (9, 12, 256), (2, 16, 1552), (1, 1, 16)])
@pytest.mark.parametrize("kind", ["bf16", "f16", "fp8", "mxfp8", "mxfp4", "bf16 w"])
@pytest.mark.parametrize("K", [512, 640, 4096, 4128])
def test_few_tiles(rows, E, N, kind, K, device):
    torch.manual_seed(rows)
    sizes = torch.randint(max(0, rows - 3), rows + 4, (E,), dtype=torch.int32)
    M = max(1, int(sizes.sum()))
    sizes[0] += M - int(sizes.sum())
    x, w = torch.randn(M, K, device=device), torch.randn(E, K, N, device=device) * 0.1
    pc = {"out_dtype": torch.bfloat16}
    if kind == "bf16 w":
        w = w.bfloat16().transpose(1, 2).contiguous().transpose(1, 2)
        wf = w.float()
    else:
        w, ws = downcast_to_mxfp(w, torch.uint8, axis=1)
        wf = upcast_from_mxfp(w, ws, torch.float32, axis=1)
        pc.update(b_mx_scale=ws, b_microblock_size=32)
    if kind[:2] == "mx":
        a, s = downcast_to_mxfp(x, torch.uint8 if kind == "mxfp4" else torch.float8_e4m3fn, axis=-1)
        x = upcast_from_mxfp(a, s, torch.float32, axis=-1)
        pc.update(a_mx_scale=s, a_microblock_size=32)
    else:
        a = x.to({"bf16": torch.bfloat16, "f16": torch.float16, "fp8": torch.float8_e4m3fn, "bf16 w": torch.bfloat16}[kind])
        x = a.float()
    md = make_ragged_tensor_metadata(sizes.to(device), M)
    y = matmul(a, w, None, md, precision_config=PrecisionConfig(**pc)).float()
    for e, (part, got) in enumerate(zip(x.split(sizes.tolist()), y.split(sizes.tolist()))):
        ref = part @ wf[e]
        # a 16-bit result (2^-8) of K float32 additions
        assert bool(((got - ref).abs() <= 2.0 ** -8 * ref.abs() + K * 2.0 ** -23 * (part.abs() @ wf[e].abs()) + 1e-6).all()), e


@pytest.mark.parametrize("byte", [0, 1, 238, 255])
def test_special_block_scales(byte, device):
    """Scale bytes of a row: blocks of 16 and of 32 rows agree (NaN for 255; 0 stands for 2^-127, against weights that make sums of it)."""
    torch.manual_seed(0)
    K, N = 640, 256
    a, s = downcast_to_mxfp(torch.randn(4, K, device=device), torch.float8_e4m3fn, axis=-1)
    s[1, 3] = byte
    s[2] = byte
    w, ws = downcast_to_mxfp(torch.randn(1, K, N, device=device), torch.uint8, axis=1)
    codes = upcast_from_mxfp(w, torch.full_like(ws, 127), torch.float32, axis=1)
    ws = (ws.int() - 40).clamp(min=1).to(torch.uint8) if byte == 238 else torch.full_like(ws, 230) if byte < 2 else ws.clone()   # (finite products)
    md = make_ragged_tensor_metadata(torch.tensor([4], dtype=torch.int32, device=device), 4)
    out = []
    for block_m in (16, 32):
        with scoped_opt_flags_constraints({"block_m": block_m}):
            pc = PrecisionConfig(a_mx_scale=s, a_microblock_size=32, b_mx_scale=ws.transpose(1, 2).contiguous().transpose(1, 2),
                                 b_microblock_size=32, out_dtype=torch.float32)
            out.append(matmul(a, w, None, md, precision_config=pc))
    assert torch.equal(out[0].isnan(), out[1].isnan()) and bool(out[0][2].isnan().all()) == (byte == 255)
    torch.testing.assert_close(out[0], out[1], rtol=1e-3, atol=1e-3, equal_nan=True)
    if byte < 2:   # (2^-13: see below; twice or half the scale, or none, is far off)
        ref = scaled_sums(a, s, codes[0], ws[0])
        for y in out:
            assert float((y[2].double().cpu() - ref[2]).norm() / ref[2].norm()) <= 2.0 ** -13


def scaled_sums(x8, xs, codes, ws):
    """The product in 64 bits: values and e8m0 bytes [M, K], [M, K/32] against [K, N], [K/32, N]."""
    two = torch.tensor(2.0, dtype=torch.float64)
    x = x8.double().cpu() * (two ** (xs.double().cpu() - 127)).repeat_interleave(32, dim=1)
    return x @ (codes.double().cpu() * (two ** (ws.double().cpu() - 127)).repeat_interleave(32, dim=0))


@pytest.mark.parametrize("ragged", [True, False])
@pytest.mark.parametrize("byte,shift", [(2, 100), (119, 0), (247, -100), (254, -100)])
def test_block_scales_of_the_whole_range(byte, shift, ragged, device):
    """Few tiles of rows with block scales that bf16 does not hold the scaled values of: the sums are those of the whole range."""
    torch.manual_seed(byte)
    M, K, N = 4, 640, 256
    a, s = downcast_to_mxfp(torch.randn(M, K, device=device), torch.float8_e4m3fn, axis=-1)
    s = (s.int() - s.int().max(dim=1, keepdim=True).values + byte).clamp(0, 254).to(torch.uint8)
    w, _ = downcast_to_mxfp(torch.randn(1, K, N, device=device), torch.uint8, axis=1)
    ws = torch.randint(120 + shift, 128 + shift, (1, N, K // 32), dtype=torch.uint8, device=device).transpose(1, 2)
    codes = upcast_from_mxfp(w, torch.full_like(ws, 127), torch.float32, axis=1)
    pc = PrecisionConfig(a_mx_scale=s, a_microblock_size=32, b_mx_scale=ws if ragged else ws[0], b_microblock_size=32, out_dtype=torch.float32)
    md = make_ragged_tensor_metadata(torch.tensor([M], dtype=torch.int32, device=device), M) if ragged else None
    y = matmul(a, w if ragged else w[0], None, md, precision_config=pc).double().cpu()
    ref = scaled_sums(a, s, codes[0], ws[0])
    # (the scaled MFMA's sums are off by up to 6e-5 of the result; values that bf16 loses are at least 2^-9 of it)
    assert float((y - ref).norm() / ref.norm()) <= 2.0 ** -13


@pytest.mark.parametrize("byte", [0, 1, 127, 252])
@pytest.mark.parametrize("block_m", [16, 32])
def test_weight_scales_that_16_bit_operands_hold(byte, block_m, device):
    """fp8 rows without block scales: weights of scale bytes up to 252 (6 * 2^125 is a bf16 number) are exact in the streaming kernel
    (blocks of 16) as in the scaled MFMA; 0 stands for 2^-127."""
    torch.manual_seed(byte)
    M, K, N = 4, 640, 256
    a = (torch.randn(M, K, device=device) * (2.0 ** -6 if byte > 200 else 8.0)).to(torch.float8_e4m3fn)
    w, _ = downcast_to_mxfp(torch.randn(1, K, N, device=device), torch.uint8, axis=1)
    ws = torch.full((1, N, K // 32), byte, dtype=torch.uint8, device=device).transpose(1, 2)
    codes = upcast_from_mxfp(w, torch.full_like(ws, 127), torch.float32, axis=1)
    md = make_ragged_tensor_metadata(torch.tensor([M], dtype=torch.int32, device=device), M)
    with scoped_opt_flags_constraints({"block_m": block_m}):
        y = matmul(a, w, None, md, precision_config=PrecisionConfig(b_mx_scale=ws, b_microblock_size=32, out_dtype=torch.float32))
    ref = scaled_sums(a, torch.full((M, K // 32), 127, dtype=torch.uint8), codes[0], ws[0])
    assert float((y.double().cpu() - ref).norm() / ref.norm()) <= 2.0 ** -13


@pytest.mark.parametrize("form,block_m", [("dense", 16), ("padded codes", 32), ("padded scales", 32), ("odd start", 32)])
def test_blocks_of_16_only_where_they_stream(form, block_m, device):
    """Weights that the streaming kernel does not read run in blocks of 32 rows, one pass over them, with the same results."""
    torch.manual_seed(3)
    E, K, N = 3, 1280, 256
    sizes = torch.tensor([20, 18, 22], dtype=torch.int32)
    M = int(sizes.sum())
    x = torch.randn(M, K, device=device).bfloat16()
    w, ws = downcast_to_mxfp(torch.randn(E, K, N, device=device) * 0.1, torch.uint8, axis=1)
    wf = upcast_from_mxfp(w, ws, torch.float32, axis=1)

    def pitched(t, pitch, start=0):   # the same values, [E, N, pitch] in memory
        room = torch.zeros(start + E * N * pitch, dtype=torch.uint8, device=device)
        view = room[start:].view(E, N, pitch)[..., :t.shape[1]]
        view.copy_(t.transpose(1, 2))
        return view.transpose(1, 2)

    if form == "padded codes":
        w = pitched(w, K // 2 + 16)
    elif form != "dense":
        ws = pitched(ws, K // 32 + (8 if form == "padded scales" else 0), 4 if form == "odd start" else 0)
    md = make_ragged_tensor_metadata(sizes.to(device), M)
    asked = []

    class Seen(type(md)):
        def block_schedule(self, size):
            asked.append(size)
            return super().block_schedule(size)

    seen = Seen(**{f: getattr(md, f) for f in md.__dataclass_fields__})
    pc = PrecisionConfig(b_mx_scale=ws, b_microblock_size=32)
    with scoped_opt_flags_constraints({"split_k": 1}):       # (a constraint: the general host path)
        y = matmul(x, w, None, seen, precision_config=pc)
    assert set(asked) == {block_m}
    assert torch.equal(y, matmul(x, w, None, md, precision_config=pc))
    for e, (rows, got) in enumerate(zip(x.float().split(sizes.tolist()), y.float().split(sizes.tolist()))):
        ref = rows @ wf[e]
        # a 16-bit result (2^-8) of K float32 additions
        assert bool(((got - ref).abs() <= 2.0 ** -8 * ref.abs() + K * 2.0 ** -23 * (rows.abs() @ wf[e].abs()) + 1e-6).all()), e


def test_microscaled_output_keeps_its_kernel(device):
    torch.manual_seed(1)
    K, N, M = 640, 256, 12
    a, s = downcast_to_mxfp(torch.randn(M, K, device=device), torch.float8_e4m3fn, axis=-1)
    w, ws = downcast_to_mxfp(torch.randn(2, K, N, device=device) * 0.1, torch.uint8, axis=1)
    md = make_ragged_tensor_metadata(torch.tensor([5, 7], dtype=torch.int32, device=device), M)
    ys = torch.zeros((M, N // 32), dtype=torch.uint8, device=device)
    pc = PrecisionConfig(a_mx_scale=s, a_microblock_size=32, b_mx_scale=ws, b_microblock_size=32, c_mx_scale=ys, c_microblock_size=32)
    y = matmul(a, w, None, md, precision_config=pc, epilogue=Epilogue(FnSpecs("QUANTIZE_MXFP8", None, (), ()), (), (), 6.0))
    pc = PrecisionConfig(a_mx_scale=s, a_microblock_size=32, b_mx_scale=ws, b_microblock_size=32, out_dtype=torch.float32)
    with scoped_opt_flags_constraints({"block_m": 32}):
        want = downcast_to_mxfp(matmul(a, w, None, md, precision_config=pc), torch.float8_e4m3fn, axis=-1)
    assert torch.equal(y.view(torch.uint8), want[0].view(torch.uint8)) and torch.equal(ys, want[1])


@pytest.mark.parametrize("M,N", [(257, 448), (700, 272), (1500, 128), (161, 2560), (161, 2576), (2100, 1600), (33, 16)])
@pytest.mark.parametrize("kind", ["bf16", "f16", "fp8", "mxfp4", "bf16 w", "fp8 w", "bf16 along N w"])
def test_dense(M, N, kind, device):
    """Dense products around the lines between the streaming kernel's units, blocks of 32, 64 and 128 rows."""
    torch.manual_seed(M)
    K = 608
    x, w = torch.randn(M, K, device=device), torch.randn(K, N, device=device) * 0.1
    bias = torch.randn(N, device=device)
    pc = {"out_dtype": torch.bfloat16}
    if kind[-1] == "w":
        w = w.to(torch.float8_e4m3fn if kind == "fp8 w" else torch.bfloat16)
        w = w if "along N" in kind else w.t().contiguous().t()
        wf = w.float()
    else:
        w, ws = downcast_to_mxfp(w, torch.uint8, axis=0)
        wf = upcast_from_mxfp(w, ws, torch.float32, axis=0)
        pc.update(b_mx_scale=ws, b_microblock_size=32)
    if kind == "mxfp4":
        a, s = downcast_to_mxfp(x, torch.uint8, axis=-1)
        x = upcast_from_mxfp(a, s, torch.float32, axis=-1)
        pc.update(a_mx_scale=s, a_microblock_size=32)
    else:
        a = x.to(torch.float16 if kind == "f16" else torch.float8_e4m3fn if kind[:3] == "fp8" else torch.bfloat16)
        x = a.float()
    y = matmul(a, w, bias, precision_config=PrecisionConfig(**pc)).float()
    ref = x @ wf + bias
    assert bool(((y - ref).abs() <= 2.0 ** -8 * ref.abs() + K * 2.0 ** -23 * (x.abs() @ wf.abs() + bias.abs()) + 1e-6).all())

"""GPU parity (bit-exact) of the microscaled row kernels where a thread takes two groups: 131072 groups and more, the last
workgroup partly filled, a batch axis, groups with infinities or a NaN among ordinary ones; just below that the one-group form."""
import pytest
import torch

from oracle.mxfp_ref import downcast_to_mxfp_ref, upcast_from_mxfp_ref
from triton_amd.numerics_details.mxfp import downcast_to_mxfp, upcast_from_mxfp

pytestmark = pytest.mark.gpu

SHAPES = [(2, 1031, 2080), (2, 1007, 2080)]      # 134030 and 130910 groups


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("vdt", [torch.uint8, torch.float8_e4m3fn, torch.float8_e5m2])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_rows_both_ways(shape, vdt, dtype, device):
    torch.manual_seed(3)
    x = (torch.randn(shape) * torch.exp(2 * torch.randn(shape[:2] + (1,)))).to(dtype)
    flat = x.view(-1)
    if vdt == torch.uint8:
        flat[9::90001] = float("inf")      # (fp8: infinity times the group's zero multiplier, whose NaN has a sign that processors differ in)
    flat[64:96] = 0
    ref_v, ref_s = downcast_to_mxfp_ref(x, vdt, -1, "up")
    v, s = downcast_to_mxfp(x.to(device), vdt, -1)
    assert torch.equal(s.cpu(), ref_s)
    assert torch.equal(v.cpu().view(torch.uint8), ref_v.contiguous().view(torch.uint8))
    back = upcast_from_mxfp(v, s, torch.bfloat16, -1).cpu().float()
    ref = upcast_from_mxfp_ref(ref_v, ref_s, torch.bfloat16, -1).float()
    assert torch.equal(torch.isnan(back), torch.isnan(ref))
    assert torch.equal(torch.nan_to_num(back), torch.nan_to_num(ref))


@pytest.mark.parametrize("vdt,nan_code", [(torch.uint8, 7), (torch.float8_e4m3fn, 0x7F), (torch.float8_e5m2, 0x7F)])
def test_rows_with_nan(vdt, nan_code, device):
    """A NaN takes the code of its own and leaves the rest of its group as it is."""
    torch.manual_seed(5)
    x = torch.randn(SHAPES[0], device=device)
    x.view(-1)[2::6006] = 0
    v0, s0 = downcast_to_mxfp(x, vdt, -1)
    x.view(-1)[2::6006] = float("nan")
    v1, s1 = downcast_to_mxfp(x, vdt, -1)
    assert torch.equal(s0, s1)
    want = v0.view(torch.uint8).clone()
    if vdt == torch.uint8:
        want.view(-1)[1::3003] |= nan_code        # (even positions: the low nibble)
    else:
        want.view(-1)[2::6006] = nan_code
    assert torch.equal(v1.view(torch.uint8), want)


@pytest.mark.parametrize("rows,row_bytes", [(1031, 4096), (1031, 4080), (3, 24), (5, 13)])
def test_widen_rows(rows, row_bytes, device):
    from triton_amd import _lib
    torch.manual_seed(4)
    src = torch.randint(0, 256, (rows, row_bytes), dtype=torch.uint8)
    table = torch.tensor([0x00, 0x30, 0x38, 0x3C, 0x40, 0x44, 0x48, 0x4C], dtype=torch.uint8)   # 0 .5 1 1.5 2 3 4 6 in e4m3
    table = torch.cat([table, table + 128])
    want = torch.stack([table[(src & 15).long()], table[(src >> 4).long()]], dim=-1).reshape(rows, 2 * row_bytes)
    d, wide = src.to(device), torch.zeros((rows, 2 * row_bytes), dtype=torch.uint8, device=device)
    rc = _lib.lib().tamd_widen_mxfp4_rows(_lib.ptr(d), rows, row_bytes, row_bytes, _lib.ptr(wide), 2 * row_bytes,
                                          _lib.stream_ptr(d.device))
    assert rc == 0
    assert torch.equal(wide.cpu(), want)


@pytest.mark.parametrize("shape", [(5, 2080, 1160), (1, 1664, 2616), (2, 96, 264)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_columns_by_tiles_and_one_by_one(shape, dtype, device):
    """A strided quantised axis: 150 / 125 tiles with partly filled ones, and two sizes with too few tiles; any finite values."""
    torch.manual_seed(6)
    x = torch.randn(shape)
    odd = torch.randint(-2**31, 2**31 - 1, shape, dtype=torch.int64).to(torch.int32).view(torch.float32)
    x = torch.where(torch.rand(shape) < 0.02, odd, x).to(dtype)
    x = torch.where(torch.isfinite(x), x, torch.ones((), dtype=dtype))
    ref_v, ref_s = downcast_to_mxfp_ref(x, torch.uint8, -2, "up")
    v, s = downcast_to_mxfp(x.to(device), torch.uint8, -2)
    assert torch.equal(s.cpu(), ref_s) and torch.equal(v.cpu(), ref_v)
    back = upcast_from_mxfp(v, s, dtype, -2).cpu().float()
    assert torch.equal(back, upcast_from_mxfp_ref(ref_v, ref_s, dtype, -2).float())

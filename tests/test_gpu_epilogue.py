"""GPU: outputs that the tiled kernels store pair by pair through 32-bit offsets, and those they store element by element
(odd column counts, an output that starts on an odd element, odd row pitches), against the oracle."""
import pytest
import torch

from oracle import matmul_ref as MR
from oracle.mxfp_ref import downcast_to_mxfp_ref
from triton_amd import _lib
from triton_amd.matmul import (Epilogue, FlexCtx, FnSpecs, FusedActivation, InFlexData, OutFlexData, PrecisionConfig, matmul)
from triton_amd.matmul_details.opt_flags import scoped_opt_flags_constraints
from triton_amd.numerics_details.mxfp import downcast_to_mxfp
from triton_amd.swiglu import swiglu_fn

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


# half a unit in the last place: 2^-(m + 1) of the value with m stored mantissa bits, and at the smallest exponent
ROUNDING = {torch.float32: (2.0 ** -24, 0.0), torch.bfloat16: (2.0 ** -8, 0.0), torch.float16: (2.0 ** -11, 2.0 ** -25),
            torch.float8_e4m3fn: (2.0 ** -4, 2.0 ** -10), torch.float8_e5m2: (2.0 ** -3, 2.0 ** -17)}


@pytest.mark.parametrize("M,N,pad", [(33, 202, 0), (160, 201, 0), (97, 202, 1), (5, 66, 2)])
@pytest.mark.parametrize("swiglu,flex,known", [(False, False, True), (False, True, True), (True, True, True), (False, True, False)])
@pytest.mark.parametrize("out_dtype", list(ROUNDING))
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float8_e4m3fn])
def test_output_types(M, N, pad, swiglu, flex, known, out_dtype, dtype, device, monkeypatch):
    """Every output type, with and without flexpoint scales, in whole and in cut pairs of columns, rows that are dropped, and
    an output whose number of rows is not given (64-bit addresses)."""
    if swiglu and N % 2:
        N += 1
    if not known:
        pack = _lib.MatmulArgBag.pack

        def without_rows(bag):
            bag.y_rows = 0
            return pack(bag)
        monkeypatch.setattr(_lib.MatmulArgBag, "pack", without_rows)
    g = torch.Generator().manual_seed(5)
    K, n_out = 96, N // 2 if swiglu else N
    x = torch.randn(M, K, generator=g).to(dtype)
    bias, gammas = torch.randn(N, generator=g), torch.rand(M, generator=g) + 0.5
    rv, rs = downcast_to_mxfp_ref(torch.randn(K, N, generator=g) * 0.1, torch.uint8, 0)
    v, s = (t.to(device).t().contiguous().t() for t in (rv, rs))
    scatter = torch.randperm(M, generator=g).int()
    scatter[::9] = -1
    expected, actual = (torch.full((1,), f, device=device) for f in (0.05, 0.0))
    fc = FlexCtx(lhs_data=InFlexData(dtype, torch.ones(1, device=device)) if dtype.itemsize == 1 else InFlexData(),
                 out_data=OutFlexData(out_dtype, expected, actual) if flex else OutFlexData())
    flat = torch.zeros(M * (n_out + pad), dtype=out_dtype, device=device)
    flat.view(torch.uint8).fill_(0x35)
    y = flat.view(M, n_out + pad)[:, :n_out]
    act = FusedActivation(FnSpecs("swiglu", swiglu_fn, ("alpha", "limit"), reduction_n=2), (1.702, 7.0)) if swiglu else None
    with scoped_opt_flags_constraints({"block_m": 128 if M > 64 else 32}):
        matmul(x.to(device), v, bias.to(device), scatter_indx=scatter.to(device), gammas=gammas.to(device), c=y, fused_activation=act,
               precision_config=PrecisionConfig(b_mx_scale=s, b_microblock_size=32, flex_ctx=fc, out_dtype=out_dtype,
                                                flexpoint_saturate_inf=True))
    ref = MR.matmul_ref(x.double(), rv, bias, b_mx_scale=rs, fused_swiglu=(1.702, 7.0) if swiglu else None).double() * gammas[:, None]
    kept = scatter >= 0
    if flex:
        top = torch.finfo(out_dtype).max
        torch.testing.assert_close(actual.cpu().double(), (ref[kept].abs().max() / top + 1e-30)[None], rtol=1e-3, atol=0.0)
        ref = (ref / 0.05).clamp(-top, top)
    rel, least = ROUNDING[out_dtype]
    got = y.cpu().double()[scatter[kept].long()]
    # (the sums of 96 products: 2e-4 with the fp8 MFMA, whose products are not exact)
    bound = (rel + 2e-4) * ref[kept].abs() + least + 2e-4 * ref[kept].abs().mean()
    assert ((got - ref[kept]).abs() <= bound).all()
    bytes_ = flat.cpu().view(torch.uint8).view(M, -1)
    named = torch.zeros(M, dtype=torch.bool)
    named[scatter[kept].long()] = True
    assert (bytes_[~named] == 0x35).all() and (bytes_[:, n_out * out_dtype.itemsize:] == 0x35).all()


def _bytes_of(x):
    return x.contiguous().view(torch.uint8)


@pytest.mark.parametrize("block_m,M", [(32, 33), (128, 127)])
@pytest.mark.parametrize("N,first,pad", [(64, 0, 0), (192, 0, 0), (200, 0, 4), (200, 4, 4), (200, 2, 0), (200, 0, 3), (196, 0, 0), (328, 0, 0)])
@pytest.mark.parametrize("swiglu", [False, True])
@pytest.mark.parametrize("saturate,factors", [(True, False), (False, False), (True, True), (None, True)])
def test_fp8_output_bytes(block_m, M, N, first, pad, swiglu, saturate, factors, device):
    """float8_e4m3fn outputs in whole quads of lanes on whole words and in others, infinite, NaN and overflowing ones among them: the bytes
    that a cast of the float32 output of the same product gives."""
    g = torch.Generator().manual_seed(3)
    K, n_out = 128, N // 2 if swiglu else N
    x = (torch.randn(M, K, generator=g) * 2).to(torch.float8_e4m3fn).to(device)
    rv, rs = downcast_to_mxfp_ref(torch.randn(K, N, generator=g), torch.uint8, 0)
    v, s = (t.to(device).t().contiguous().t() for t in (rv, rs))
    bias = torch.randn(N, generator=g)
    bias[6], bias[9], bias[14], bias[21] = float("inf"), -float("inf"), float("nan"), 3.0e4
    kw = dict(gammas=(torch.rand(M, generator=g) + 0.5).to(device), betas=(torch.rand(M, generator=g) + 0.5).to(device)) if factors else {}
    act = FusedActivation(FnSpecs("swiglu", swiglu_fn, ("alpha", "limit"), reduction_n=2), (1.702, 7.0 if factors else None)) if swiglu else None
    expected, actual = torch.full((1,), 0.25, device=device), torch.zeros(1, device=device)

    def run(dtype, **out):
        fc = FlexCtx(lhs_data=InFlexData(x.dtype, torch.full((1,), 0.5, device=device)), **out)
        flat = torch.zeros(first + M * (n_out + pad) + 16, dtype=dtype, device=device)
        y = flat[first:first + M * (n_out + pad)].view(M, n_out + pad)[:, :n_out]
        with scoped_opt_flags_constraints({"block_m": block_m}):
            matmul(x, v, bias.to(device), c=y, fused_activation=act, precision_config=PrecisionConfig(
                b_mx_scale=s, b_microblock_size=32, flex_ctx=fc, out_dtype=dtype, flexpoint_saturate_inf=bool(saturate)), **kw)
        rest = torch.ones_like(flat, dtype=torch.bool)
        rest[first:first + M * (n_out + pad)].view(M, n_out + pad)[:, :n_out] = False
        assert (_bytes_of(flat[rest]) == 0).all()
        return y
    ref = run(torch.float32)
    if saturate is None:
        got = run(torch.float8_e4m3fn)
    else:
        got = run(torch.float8_e4m3fn, out_data=OutFlexData(torch.float8_e4m3fn, expected, actual if saturate else None))
        if saturate:
            assert float(actual) == float("inf") or torch.isclose(actual, ref.abs().amax() / 448.0 + 1e-30, rtol=1e-6).all()
        ref = ref * 4.0
        if saturate:
            ref = torch.where(ref.isnan(), -448.0, ref.clamp(-448.0, 448.0))   # (a NaN takes the lower bound)
    want = ref.to(torch.float8_e4m3fn)
    over = ref.abs() >= 464.0   # rounds beyond the largest value
    finite = ~(over | ref.isnan())
    assert torch.equal(_bytes_of(got)[finite], _bytes_of(want)[finite])
    assert (_bytes_of(got)[~finite] & 0x7F == 0x7F).all()
    assert torch.equal(_bytes_of(got)[over] >> 7, (ref[over] < 0).to(torch.uint8))


@pytest.mark.parametrize("block_m,M", [(32, 5), (128, 127)])
@pytest.mark.parametrize("N", [64, 192, 256, 448])
@pytest.mark.parametrize("swiglu", [False, True])
def test_mxfp8_output_specials(block_m, M, N, swiglu, device):
    """MXFP8 outputs whose groups hold zeros only, tiny and infinite values and NaNs: a NaN does not count for its group's scale and
    stays one, an infinity makes the scale 255 and the other values zero."""
    g = torch.Generator().manual_seed(4)
    K, n_out = 128, N // 2 if swiglu else N
    x = torch.randn(M, K, generator=g)
    x[0] = 0.0
    x[1] = 2.0 ** -6 * torch.sign(x[1])
    x = x.to(torch.float8_e4m3fn).to(device)
    xs = torch.full((M, K // 32), 127, dtype=torch.uint8)
    xs[2], xs[3] = 7, 240
    rv, rs = downcast_to_mxfp_ref(torch.randn(K, N, generator=g), torch.uint8, 0)
    v, s = (t.to(device).t().contiguous().t() for t in (rv, rs))
    bias = torch.zeros(N)
    if n_out >= 96:
        bias[70], bias[130 if swiglu else 40] = float("nan"), float("inf")
    act = FusedActivation(FnSpecs("swiglu", swiglu_fn, ("alpha", "limit"), reduction_n=2), (1.702, None)) if swiglu else None
    ys = torch.empty((M, n_out // 32), dtype=torch.uint8, device=device)
    kw = dict(b_mx_scale=s, b_microblock_size=32, a_mx_scale=xs.to(device), a_microblock_size=32)
    with scoped_opt_flags_constraints({"block_m": block_m}):
        ref = matmul(x, v, bias.to(device), fused_activation=act, precision_config=PrecisionConfig(out_dtype=torch.float32, **kw)).cpu()
        got = matmul(x, v, bias.to(device), fused_activation=act, precision_config=PrecisionConfig(c_mx_scale=ys, **kw),
                     epilogue=Epilogue(FnSpecs("QUANTIZE_MXFP8", None, (), ()), (), (), 6.0)).cpu()
    groups = ref.view(M, n_out // 32, 32)
    top = groups.abs().nan_to_num(nan=0.0, posinf=float("inf")).amax(-1)
    exponent = torch.ceil(torch.log2(top.double() / 448.0)).clamp(-126, 127)
    byte = torch.where(top.isinf(), 255.0, torch.where(top == 0, 0.0, exponent + 127.0)).to(torch.int64)
    assert torch.equal(ys.cpu().long(), byte)
    scale = torch.where((byte == 0) | (byte == 255), 0.0, torch.exp2(127.0 - byte.double())).float()
    want = (groups * scale[..., None]).view(M, n_out).to(torch.float8_e4m3fn)
    nan = want.isnan()
    assert torch.equal(got.isnan(), nan) and torch.equal(_bytes_of(got)[~nan], _bytes_of(want)[~nan])

"""GPU: products of two operands of one type, both contiguous along K (16-bit weights, fp8 x fp8), at the edges of the
kernel's tiles: row remainders (a lone row, one more than a fragment, the absorbed remainder of a 128-row block), column
remainders and K remainders, against float32 products of the same values."""
import pytest
import torch

from triton_amd.matmul import FlexCtx, InFlexData, PrecisionConfig, matmul
from triton_amd.matmul_details.opt_flags import scoped_opt_flags_constraints
from triton_amd.tensor import make_ragged_tensor_metadata

pytestmark = pytest.mark.gpu
TYPES = [torch.bfloat16, torch.float16, torch.float8_e4m3fn, torch.float8_e5m2]


def operands(shape_x, shape_w, dtype, device):
    x, w = torch.randn(shape_x).to(dtype), (torch.randn(shape_w) * 0.1).to(dtype)
    return x, w, x.to(device), w.to(device).transpose(-1, -2).contiguous().transpose(-1, -2)


def config(dtype, device):
    if dtype.itemsize > 1:
        return None, 1.0, 1.0
    sx, sw = torch.tensor([0.5]), torch.tensor([0.25])
    flex = FlexCtx(InFlexData(dtype, sx.to(device)), InFlexData(dtype, sw.to(device)))
    return PrecisionConfig(flex_ctx=flex, out_dtype=torch.bfloat16), 0.5, 0.25


@pytest.mark.parametrize("M,K,N", [(1, 16, 136), (33, 144, 264), (160, 1040, 520), (161, 64, 256), (300, 2064, 1000)])
@pytest.mark.parametrize("block_m", [None, 32, 64, 128])
@pytest.mark.parametrize("dtype", TYPES)
def test_dense(M, K, N, block_m, dtype, device):
    torch.manual_seed(0)
    x, w, xd, wd = operands((M, K), (K, N), dtype, device)
    bias = torch.randn(N)
    pc, sx, sw = config(dtype, device)
    with scoped_opt_flags_constraints({} if block_m is None else {"block_m": block_m}):
        y = matmul(xd, wd, bias.to(device), precision_config=pc)
    ref = (x.float() @ w.float()) * (sx * sw) + bias
    torch.testing.assert_close(y.cpu().float(), ref, rtol=1e-2, atol=2e-2)


@pytest.mark.parametrize("block_m", [16, 32, 64, 128])
@pytest.mark.parametrize("dtype", TYPES)
def test_ragged_with_gather_scatter_and_gate_weights(block_m, dtype, device):
    torch.manual_seed(1)
    K, N = 208, 264
    sizes = torch.tensor([0, 1, 16, 33, 160, 161, 300, 129], dtype=torch.int32)
    E, M = len(sizes), int(sizes.sum())
    x, w, xd, wd = operands((M, K), (E, K, N), dtype, device)
    gather, scatter = torch.randperm(M).int(), torch.randperm(M).int()
    scatter[::7] = -1
    gammas = torch.rand(M)
    pc, sx, sw = config(dtype, device)
    md = make_ragged_tensor_metadata(sizes.to(device), M)
    y = torch.zeros((M, N), dtype=torch.bfloat16 if dtype.itemsize == 1 else dtype, device=device)
    with scoped_opt_flags_constraints({"block_m": block_m}):
        matmul(xd, wd, None, md, gather_indx=gather.to(device), scatter_indx=scatter.to(device), precision_config=pc,
               gammas=gammas.to(device), c=y)
    ref = torch.zeros(M, N)
    rows, e0 = x.float()[gather.long()], 0
    for e, n in enumerate(sizes.tolist()):
        out = (rows[e0:e0 + n] @ w[e].float()) * (sx * sw) * gammas[e0:e0 + n, None]
        at = scatter[e0:e0 + n]
        ref[at[at >= 0].long()] = out[at >= 0]
        e0 += n
    torch.testing.assert_close(y.cpu().float(), ref, rtol=1e-2, atol=2e-2)


@pytest.mark.parametrize("sizes", [
    [160] * 20 + [1] * 20,            # tiles of five row fragments and of one, twenty experts each
    [0, 33, 0, 128, 96, 1, 161, 64],  # every number of fragments, an absorbed remainder and one row more than that
    [5], [129],
])
@pytest.mark.parametrize("quantised", [False, True])
def test_tiles_shared_out_by_their_time(sizes, quantised, device):
    torch.manual_seed(2)
    K, N = 64, 264
    sizes = torch.tensor(sizes, dtype=torch.int32)
    E, M = len(sizes), int(sizes.sum())
    x, w, xd, wd = operands((M, K), (E, K, N), torch.bfloat16, device)
    pc = None
    if quantised:
        from triton_amd.numerics_details.mxfp import downcast_to_mxfp, upcast_from_mxfp
        v, s = downcast_to_mxfp(wd, torch.uint8, axis=-2)
        w, wd = upcast_from_mxfp(v, s, torch.bfloat16, axis=-2).cpu(), v
        pc = PrecisionConfig(b_mx_scale=s, b_microblock_size=32)
    md = make_ragged_tensor_metadata(sizes.to(device), M)
    with scoped_opt_flags_constraints({"block_m": 128}):
        y = matmul(xd, wd, None, md, precision_config=pc)
    at, ref = 0, torch.zeros(M, N)
    for e, n in enumerate(sizes.tolist()):
        ref[at:at + n] = x.float()[at:at + n] @ w[e].float()
        at += n
    torch.testing.assert_close(y.cpu().float(), ref, rtol=1e-2, atol=2e-2)


@pytest.mark.parametrize("n_experts,most", [(1, 700), (7, 700), (64, 330), (65, 330), (200, 200), (512, 40), (513, 40)])
@pytest.mark.parametrize("kind", ["bf16", "mxfp4", "fp8 x mxfp4"])
def test_tiles_of_uneven_experts(n_experts, most, kind, device):
    """Experts of none to several row blocks, some of them absorbed, one to eight experts per lane and more than fit."""
    from triton_amd.numerics_details.mxfp import downcast_to_mxfp, upcast_from_mxfp
    g = torch.Generator().manual_seed(n_experts)
    K, N = 64, 520
    sizes = torch.randint(0, most + 1, (n_experts,), generator=g, dtype=torch.int32)
    sizes[::5] = torch.tensor([0, 128, 160, 161, 32], dtype=torch.int32).repeat(n_experts)[:len(sizes[::5])]
    M = int(sizes.sum())
    if M == 0:
        sizes[0] = M = 129
    x = torch.randn(M, K, generator=g).to(torch.float8_e4m3fn if kind[0] == "f" else torch.bfloat16)
    w = (torch.randn(n_experts, K, N, generator=g) * 0.1).to(torch.bfloat16).to(device).transpose(-1, -2).contiguous().transpose(-1, -2)
    pc = PrecisionConfig(out_dtype=torch.bfloat16)
    if kind != "bf16":
        v, s = downcast_to_mxfp(w, torch.uint8, axis=-2)
        pc.b_mx_scale, pc.b_microblock_size = s, 32
        dense, w = upcast_from_mxfp(v, s, torch.bfloat16, axis=-2), v
    else:
        dense = w
    md = make_ragged_tensor_metadata(sizes.to(device), M)
    with scoped_opt_flags_constraints({"block_m": 128}):
        y = matmul(x.to(device), w, None, md, precision_config=pc).cpu().float()
    dense, at = dense.cpu().float(), 0
    for e, n in enumerate(sizes.tolist()):
        torch.testing.assert_close(y[at:at + n], x[at:at + n].float() @ dense[e], rtol=1e-2, atol=2e-2)
        at += n


@pytest.mark.parametrize("M,K,N", [(1, 2064, 72), (8, 4112, 64), (9, 48, 328), (16, 1104, 200), (27, 2096, 136), (70, 6912, 608)])
@pytest.mark.parametrize("dtype", TYPES)
def test_few_rows(M, K, N, dtype, device):
    """Narrow tiles: 8, 16 and 32 row lines, K quarters that end early or hold nothing, a partial strip of columns."""
    torch.manual_seed(2)
    x, w, xd, wd = operands((M, K), (K, N), dtype, device)
    bias = torch.randn(N)
    pc, sx, sw = config(dtype, device)
    y = matmul(xd, wd, bias.to(device), precision_config=pc)
    ref = (x.float() @ w.float()) * (sx * sw) + bias
    torch.testing.assert_close(y.cpu().float(), ref, rtol=1e-2, atol=2e-2)


@pytest.mark.parametrize("M,K,N,ragged", [(13, 4960, 72, False), (59, 5312, 264, False), (40, 8064, 136, False), (2, 5856, 1072, False), (1613, 2336, 136, False),
                                          (6, 5184, 264, True), (40, 4256, 72, True)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_few_rows_of_mxfp4(M, K, N, ragged, dtype, device):
    """MXFP4 weights and few tiles with a K or N that the streaming kernel does not take: groups of waves share a tile."""
    from triton_amd.numerics_details.mxfp import downcast_to_mxfp, upcast_from_mxfp
    torch.manual_seed(3)
    E = 4 if ragged else 1
    x = torch.randn(M, K).to(dtype)
    codes, scales = downcast_to_mxfp((torch.randn(E, K, N, device=device) * 0.1), torch.uint8, axis=1)
    w = upcast_from_mxfp(codes, scales, torch.float32, axis=1).cpu()
    pc = PrecisionConfig(b_mx_scale=scales if ragged else scales[0], b_microblock_size=32)
    if not ragged:
        y, ref = matmul(x.to(device), codes[0], None, precision_config=pc), x.float() @ w[0]
    else:
        sizes = torch.tensor([M - 4, 0, 1, 3], dtype=torch.int32)
        md = make_ragged_tensor_metadata(sizes.to(device), M)
        y = matmul(x.to(device), codes, None, md, precision_config=pc)
        ref = torch.cat([part.float() @ w[e] for e, part in enumerate(x.split(sizes.tolist()))])
    torch.testing.assert_close(y.cpu().float(), ref, rtol=1e-2, atol=3e-2)


@pytest.mark.parametrize("M,K,N", [(64, 512, 768), (300, 8208, 264), (7, 4096, 72), (27, 2064, 136)])
@pytest.mark.parametrize("binades", [0, 6])
@pytest.mark.parametrize("dtype", [torch.float8_e4m3fn, torch.float8_e5m2])
def test_fp8_products_are_exact(M, K, N, binades, dtype, device):
    """fp8 x fp8 as precise as the product of the widened operands: exact products, float32 sums.  Each of at most K additions
    is off by at most half a unit in the last place of a partial sum, 2^-24 of it, in either direction: sqrt(K) 2^-24 of the
    result (the MFMAs that take fp8 operands drop parts of the products: 1.5e-5 and 6e-5 at every K)."""
    torch.manual_seed(4)

    def values(*shape):
        v = torch.randn(shape) * torch.exp2(torch.randint(-binades, binades + 1, shape).float())
        return (v * (torch.finfo(dtype).max / v.abs().max())).to(dtype)

    x, w = values(M, K), values(N, K)
    y = matmul(x.to(device), w.to(device).t(), None, precision_config=PrecisionConfig(out_dtype=torch.float32)).cpu().double()
    ref = x.double() @ w.double().t()
    assert float((y - ref).norm() / ref.norm()) <= K ** 0.5 * 2.0 ** -24

"""GPU: the persistent kernel for unquantised 16-bit weights at the sizes where it can go wrong: K of its fewest stages and off them, columns off strips,
tiles and lines, empty slices, slices of one row, of whole blocks, one more, and many, rows that are not there, against float32 products."""
import ctypes

import pytest
import torch

from triton_amd import _lib, _native
from triton_amd.matmul import FnSpecs, FusedActivation, PrecisionConfig, matmul
from triton_amd.matmul_details.opt_flags import scoped_opt_flags_constraints
from triton_amd.swiglu import swiglu_fn
from triton_amd.tensor import make_ragged_tensor_metadata

SWIGLU = FusedActivation(FnSpecs("swiglu", swiglu_fn, ("alpha", "limit"), reduction_n=2), (1.702, 7.0))


def ring_rows(m, n, k, e, swiglu=False, **changed):
    bag = _lib.MatmulArgBag()
    bag.x_dtype = bag.w_dtype = bag.y_dtype = _lib.BF16
    bag.M, bag.N, bag.K, bag.n_experts, bag.block_schedule = m, n, k, e, 1 << 20
    bag.activation = _lib.ACT_SWIGLU if swiglu else _lib.ACT_NONE
    bag.y, bag.y_rows, bag.y_stride_m = 1 << 20, m, n // 2 if swiglu else n
    for name, value in changed.items():
        setattr(bag, name, value)
    packed = bag.pack()
    return _native.ring_rows(ctypes.addressof(packed), 256)


def test_where_it_is_taken():
    assert ring_rows(1200, 5760, 2880, 32) == 64 and ring_rows(4084, 5760, 2880, 32, True) == 160
    assert ring_rows(4, 3904, 1760, 8) == 0
    assert all(ring_rows(sum(sizes), N, K, len(sizes)) == 64 for sizes, K, N in FEW)
    assert ring_rows(816, 1024, 5376, 8) == 0 and ring_rows(31, 2560, 5376, 8) == 0
    for changed in (dict(block_schedule=None), dict(n_experts=257), dict(y_dtype=_lib.F32), dict(y_rows=0), dict(y_rows=1 << 20), dict(K=248),
                    dict(y_expected_scale=1 << 20), dict(N=5759), dict(y=(1 << 20) + 2), dict(y_stride_m=5761), dict(x_dtype=_lib.F16), dict(force_variant=64)):
        assert ring_rows(4084, 5760, 2880, 32, **changed) == 0, changed


def test_where_blocks_of_64_are_the_slower():
    """Products timed at 1.05 to 1.3 of the kernels that take them now."""
    for m, n, k, e in ((412, 2328, 256, 8), (489, 1840, 384, 8), (987, 584, 392, 16), (802, 528, 336, 16)):
        assert ring_rows(m, n, k, e) == 0 and ring_rows(m, n, k + 408, e) == 64
    for m, n, k, e in ((992, 3048, 5608, 8), (1918, 760, 5304, 32), (548, 3064, 5712, 8), (1968, 720, 4856, 32)):
        assert ring_rows(m, n, k, e) == 160 and ring_rows(m, n, k - 3000, e) == 64


# (slice sizes, K, columns)
SIZES = [([1, 0, 31, 32, 33, 64, 65, 0, 129, 3], 256, 6200), ([2] * 70 + [0] * 30, 1096, 648), ([160, 161, 0, 320, 321, 95, 97, 700], 776, 3176),
         ([1500, 0, 40], 520, 4100), ([5000], 264, 1032)]
# fewer than a tile of 256 columns for every third CU, and just above: blocks of 64
FEW = [([100, 64, 65, 128, 129, 0, 200, 130], 1032, 1288), ([700, 0, 65, 127], 520, 2056), ([33, 40, 1, 64, 70, 10, 66, 0], 264, 1800),
       ([10, 0, 16, 3, 33, 1, 2, 3] * 2, 776, 1096), ([100] * 10 + [128, 129], 776, 1800)]


@pytest.mark.gpu
@pytest.mark.parametrize("sizes,K,N", SIZES + FEW)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("swiglu", [False, True])
@pytest.mark.parametrize("gathered", [False, True])
def test_edges(sizes, K, N, dtype, swiglu, gathered, device):
    E, M, T = len(sizes), sum(sizes), 50
    assert ring_rows(M, N, K, E, swiglu)
    torch.manual_seed(K)
    gather, scatter = torch.randint(0, T, (M,), dtype=torch.int32), torch.randperm(M, dtype=torch.int32)
    gather[M // 2], scatter[M // 3] = -1, -1
    x = torch.randn(T if gathered else M, K, device=device).to(dtype)
    w = (torch.randn(E, N, K, device=device) * 0.1).to(dtype).transpose(1, 2)
    bias, gammas = torch.randn(E, N, device=device), torch.rand(M, device=device)
    md = make_ragged_tensor_metadata(torch.tensor(sizes, dtype=torch.int32, device=device), M)
    kw = dict(gather_indx=gather.to(device)) if gathered else dict(scatter_indx=scatter.to(device), gammas=gammas)
    got = matmul(x, w, bias, md, precision_config=PrecisionConfig(), fused_activation=SWIGLU if swiglu else None, **kw)
    rows = torch.where((gather >= 0)[:, None].to(device), x.float()[gather.clamp(min=0).long().to(device)], 0.0) if gathered else x.float()
    full = torch.empty(M, N // 2 if swiglu else N, device=device)
    slack = torch.empty_like(full)
    at = 0
    for e, n in enumerate(sizes):
        r = slice(at, at + n)
        at += n
        v, mag = rows[r] @ w[e].float() + bias[e], K * 2.0 ** -23 * (rows[r].abs() @ w[e].float().abs())
        if swiglu:
            g, l = v[:, 0::2].clamp(max=7.0), v[:, 1::2].clamp(-7.0, 7.0)
            s = g * torch.sigmoid(1.702 * g)
            v, mag = s * (l + 1), 1.2 * mag[:, 0::2] * (l.abs() + 1) + s.abs() * mag[:, 1::2]   # (|d swish| <= 1.1)
        full[r], slack[r] = v, mag
    if not gathered:
        there = scatter >= 0
        full, slack, got = full[there.to(device)] * gammas[there.to(device), None], slack[there.to(device)], got[scatter[there].long().to(device)]
    # a 16-bit result (2^-8) of K float32 additions, and the hardware's exponential and reciprocal (2^-20)
    assert bool(((got.float() - full).abs() <= 2.0 ** -8 * full.abs() + slack + 1e-5).all())


# (slice sizes, K, columns, row block that the tiled kernels take it in) below the line
SUMMED = [([55, 64, 33, 70, 41, 60, 0, 66], 576, 2152, 64), ([200, 170, 190, 230], 640, 1800, 64), ([9, 14, 0, 11, 12, 16, 8, 20], 3784, 2560, 32),
          ([34, 20, 41, 0, 70, 36, 31, 25] * 2, 2768, 904, 32), ([60, 52, 71, 66, 40, 64, 63, 61], 2544, 1856, 64), ([85, 80, 64, 96, 0, 101, 120, 77], 712, 1288, 64)]


@pytest.mark.gpu
@pytest.mark.parametrize("sizes,K,N,block_m", SUMMED)
def test_sums_below_the_line(sizes, K, N, block_m, device):
    """As many float32 sums to a result as in the tiled kernels: their bits up to ten stages and where they take narrow tiles, elsewhere no more
    results that are not the rounded 64-bit sum."""
    E, M = len(sizes), sum(sizes)
    assert ring_rows(M, N, K, E) == 64
    g = torch.Generator().manual_seed(K)
    x, w = torch.randn(M, K, generator=g).half().to(device), (torch.randn(E, N, K, generator=g) * 0.05).half().to(device).transpose(1, 2)
    md = make_ragged_tensor_metadata(torch.tensor(sizes, dtype=torch.int32, device=device), M)
    got = matmul(x, w, None, md, precision_config=PrecisionConfig())
    with scoped_opt_flags_constraints({"block_m": block_m}):
        tiled = matmul(x, w, None, md, precision_config=PrecisionConfig())
    if K <= 640 or block_m < 64:
        assert torch.equal(got, tiled)
        return
    ends = torch.tensor(sizes).cumsum(0).tolist()
    rounded = torch.cat([x[b - n:b].double() @ w[e].double() for e, (n, b) in enumerate(zip(sizes, ends))]).half()
    assert int((got != rounded).sum()) <= int((tiled != rounded).sum())

"""GPU: the persistent kernel of few rows per slice (weights in 4 KB blocks and pre-shuffled scales, or both strided) at the sizes where it can go wrong: K below a stage, below the
ring and off both, columns off strips and tiles, empty slices and slices of several blocks, with gathered and scattered rows that are not
there, every kind of row and of output.  Rows of 8 and 4 bits give the bits of the tiled kernels, which strided weights with pre-shuffled scales take; 16-bit
rows are held against float32 products."""
import ctypes
import sys

import pytest
import torch

from triton_amd import _lib, _native
from triton_amd.matmul import Epilogue, FlexCtx, FnSpecs, FusedActivation, InFlexData, OutFlexData, PrecisionConfig, matmul
from triton_amd.matmul_details.opt_flags import scoped_opt_flags_constraints
from triton_amd.numerics_details.mxfp import downcast_to_mxfp, upcast_from_mxfp
from triton_amd.swiglu import swiglu_fn
from triton_amd.tensor import FP4, convert_layout, make_ragged_tensor_metadata, wrap_torch_tensor
from triton_amd.tensor_details.layout import CDNA4MXScaleLayout, CDNA4MXValueLayout

SWIGLU = FusedActivation(FnSpecs("swiglu", swiglu_fn, ("alpha", "limit"), reduction_n=2), (1.702, 7.0))
TO_MXFP8 = Epilogue(FnSpecs("QUANTIZE_MXFP8", None, (), ()), (), (), 6.0)
TYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "fp8": torch.float8_e4m3fn}


def ring_rows(m, n, k, e, kind, out="16", swiglu=False, **changed):
    bag = _lib.MatmulArgBag()
    bag.x_dtype = {"bf16": _lib.BF16, "f16": _lib.F16, "mxfp4": _lib.MXFP4}.get(kind, _lib.FP8_E4M3)
    bag.y_dtype = _lib.FP8_E4M3 if out != "16" else _lib.F16 if kind == "f16" else _lib.BF16
    bag.M, bag.N, bag.K, bag.n_experts, bag.w_dtype = m, n, k, e, _lib.MXFP4
    bag.w_layout, bag.w_mx_layout, bag.block_schedule = _lib.W_CDNA4_BLOCKS, _lib.SCALE_CDNA4, 1 << 20
    bag.activation = _lib.ACT_SWIGLU if swiglu else _lib.ACT_NONE
    bag.y, bag.y_rows, bag.y_stride_m = 1 << 20, m, n // 2 if swiglu else n
    if kind[:2] == "mx":
        bag.x_mx_scale = 1 << 20
    if out == "mx":
        bag.y_mx_scale, bag.y_mx_stride_m = 1 << 20, -(-n // 32)
    for name, value in changed.items():
        setattr(bag, name, value)
    packed = bag.pack()
    return _native.ring_rows(ctypes.addressof(packed), 256)


def test_where_it_is_taken():
    """Layers timed with both: large ones of few rows, by the block that covers their slices; not what the kernel does not cover."""
    assert ring_rows(2036, 11520, 5760, 128, "fp8") == 64 and ring_rows(512, 5760, 2880, 128, "fp8") == 32
    assert ring_rows(8192, 5760, 2880, 128, "mxfp4", swiglu=True) == 96 and ring_rows(2048, 5760, 2880, 128, "mxfp8") == 32
    for M, N, K, E, kind in ((256, 5760, 2880, 128, "bf16"), (16384, 5760, 2880, 128, "bf16"), (65536, 5760, 2880, 32, "fp8"),
                             (1, 5760, 2880, 128, "fp8"), (2048, 5760, 512, 128, "mxfp4")):
        assert ring_rows(M, N, K, E, kind) == 0
    for changed in (dict(w_layout=_lib.W_STRIDED), dict(w_mx_layout=_lib.SCALE_STRIDED), dict(block_schedule=None), dict(n_experts=257),
                    dict(x_dtype=_lib.FP8_E5M2), dict(y_dtype=_lib.F32), dict(y_dtype=_lib.F16), dict(y_rows=0), dict(y_rows=1 << 20),
                    dict(y_expected_scale=1 << 20), dict(N=5759), dict(y=(1 << 20) + 2), dict(y_stride_m=5761), dict(force_variant=32)):
        assert ring_rows(512, 5760, 2880, 128, "fp8", **changed) == 0, changed


def test_where_blocks_of_96_come_before_tiles():
    """SwiGLU products with about a hundred to a thousand rows per slice, by their rounds over the CUs; not without SwiGLU, few tiles or 16-bit rows."""
    for m, n, k, e, kind, out in ((6168, 2688, 1248, 32, "mxfp8", "mx"), (6432, 1152, 2048, 60, "fp8", "fp8"), (14760, 2240, 5312, 16, "mxfp4", "16")):
        assert ring_rows(m, n, k, e, kind, out, True) == 96
        assert ring_rows(m, n, k, e, kind) == 0
        assert ring_rows(m, n, k, e, kind, out, True, w_layout=_lib.W_STRIDED, w_mx_layout=_lib.SCALE_STRIDED) == 0
        assert ring_rows(m, n, k, e, kind, out, True, force_variant=128) == 0
    assert ring_rows(65536, 5760, 2880, 32, "fp8", "fp8", True) == 0 and ring_rows(2000, 1024, 2880, 16, "mxfp8", "mx", True) == 0
    assert ring_rows(6168, 2688, 1248, 32, "bf16", "16", True) == 0 and ring_rows(6168, 2688, 640, 32, "mxfp8", "mx", True) == 0


def test_where_one_round_of_tiles_is_full():
    """Products timed at 1.05 to 1.29 of the tiles' time: a tile of 128 for every slice, two to a CU, is one round."""
    for m, n, k, e, kind, out in ((10631, 832, 2400, 128, "mxfp8", "16"), (7960, 640, 3040, 128, "fp8", "fp8"), (10356, 896, 2720, 128, "mxfp8", "mx"),
                                  (1547, 6976, 2784, 16, "mxfp4", "16"), (10747, 1024, 1184, 128, "fp8", "fp8"), (1504, 8000, 1984, 16, "mxfp8", "16"),
                                  (4619, 1984, 2304, 60, "mxfp8", "mx"), (1966, 3904, 2240, 32, "mxfp8", "16")):
        assert ring_rows(m, n, k, e, kind, out, True) == 0
        assert ring_rows(m, n * 2, k, e, kind, out, True) == 96   # (two rounds)


def blocks(w, ws):
    return convert_layout(wrap_torch_tensor(w, dtype=FP4), CDNA4MXValueLayout()), convert_layout(wrap_torch_tensor(ws), CDNA4MXScaleLayout())


# (rows per slice, slices, K, columns): blocks of 32 alone on their CUs (K of one stage and less, of fewer stages than the ring, off the
# stages), in several rounds; of 64; of 96, also several of them to a slice
SIZES = [(9, 10, 96, 2832), (4, 12, 352, 1872), (14, 16, 736, 1296), (20, 16, 1440, 1392), (5, 128, 1056, 1184), (11, 64, 2144, 2320),
         (40, 16, 608, 2608), (30, 60, 1248, 2320), (72, 32, 1056, 4368), (14, 16, 800, 1296), (4, 12, 992, 1872), (190, 30, 1056, 2384), (420, 8, 1312, 4368)]


@pytest.mark.parametrize("layout", [dict(), dict(w_layout=_lib.W_STRIDED, w_mx_layout=_lib.SCALE_STRIDED, w_stride_k=1, w_stride_n=1440, w_mx_stride_k=1,
                                                 w_mx_stride_n=90)])
def test_fp8_rows_that_stream_stay_there(layout):
    """Row blocks of 16 that the streaming kernel covers are summed exactly by it; other blocks, longer K and rows with block scales are not its."""
    ptr = dict(w=1 << 20, w_mx_scale=1 << 20, block_offs=1 << 20, w_stride_e=2560 * 1440, w_mx_stride_e=2560 * 90, **layout)
    for m in (40, 100):
        assert ring_rows(m, 2560, 2880, 16, "fp8", block_m=16, **ptr) == 0
        assert ring_rows(m, 2560, 2880, 16, "fp8", block_m=32, **ptr) == 32
    assert ring_rows(100, 2560, 2880, 16, "mxfp8", block_m=16, **ptr) == 32


def test_where_strided_weights_take_it():
    """Where a call leaves CUs without a tile, and 16-bit rows in blocks of 64 over several rounds; not with one side in the other layout."""
    both = dict(w_layout=_lib.W_STRIDED, w_mx_layout=_lib.SCALE_STRIDED)
    assert ring_rows(60, 1696, 1440, 16, "mxfp4", **both) == 32 and ring_rows(500, 2048, 2880, 16, "mxfp4", **both) == 64
    assert ring_rows(100, 2560, 2880, 16, "fp8", **both) == 32 and ring_rows(1332, 5760, 2880, 32, "bf16", **both) == 64
    for M, N, K, E, kind in ((512, 5760, 2880, 128, "fp8"), (100, 2560, 2880, 16, "bf16"), (2048, 5760, 2880, 16, "bf16"), (8, 512, 2880, 16, "mxfp8")):
        assert ring_rows(M, N, K, E, kind, **both) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("kind,rows,E,K,N", [("mxfp4", 9, 10, 96, 2832), ("mxfp4", 4, 12, 544, 1872), ("mxfp4", 30, 8, 1440, 1394), ("mxfp8", 9, 10, 96, 2832),
                                             ("mxfp8", 9, 20, 800, 1298), ("fp8", 9, 20, 1056, 1298), ("fp8", 4, 12, 2144, 2832), ("bf16", 15, 20, 800, 1296),
                                             ("f16", 30, 20, 1312, 2328), ("bf16", 40, 60, 1056, 2322)])
@pytest.mark.parametrize("byte", [0, 1])
def test_strided_edges(kind, rows, E, K, N, byte, device):
    """The bits that the same kernel gives with blocks and pre-shuffled scales, weights and scales at addresses off 64 bytes and (byte) off four."""
    sizes = torch.randint(max(0, rows - 9), rows + 10, (E,), generator=torch.Generator().manual_seed(K), dtype=torch.int32)
    sizes[1] = 0
    M = int(sizes.sum())
    strided = dict(w_layout=_lib.W_STRIDED, w_mx_layout=_lib.SCALE_STRIDED)
    assert ring_rows(M, N, K, E, kind, block_m=32, **strided)
    torch.manual_seed(K + N)
    w, ws = downcast_to_mxfp((torch.randn(E, N, K, device=device) * torch.exp(2 * torch.randn(E, N, 1, device=device))).bfloat16(), torch.uint8, axis=-1)
    room = torch.full((16 + w.numel(),), 0x55, dtype=torch.uint8, device=device)
    w_at = room[16:].view(w.shape).copy_(w)
    ends = torch.full((byte + ws.numel() + 64,), 255, dtype=torch.uint8, device=device)   # (NaN scales around the tensor)
    ws_at = ends[byte:byte + ws.numel()].view(ws.shape).copy_(ws)
    x, opts = torch.randn(50, K, device=device), {}
    if kind[:2] == "mx":
        x, s = downcast_to_mxfp(x, torch.uint8 if kind == "mxfp4" else torch.float8_e4m3fn, axis=-1)
        opts.update(a_mx_scale=s, a_microblock_size=32)
    else:
        x = x.to(TYPES[kind])
    gather = torch.randint(-1, 50, (M,), dtype=torch.int32, device=device)
    bias, md = torch.randn(E, N, device=device), make_ragged_tensor_metadata(sizes.to(device), M)

    def run(weights, scales):
        return matmul(x, weights, bias, md, gather_indx=gather, precision_config=PrecisionConfig(
            b_mx_scale=scales, b_microblock_size=32, out_dtype=torch.float16 if kind == "f16" else torch.bfloat16, **opts))

    got = run(w_at.transpose(1, 2), ws_at.transpose(1, 2))
    if ring_rows(M, N, K, E, kind) or kind[:2] == "mx":
        assert torch.equal(got, run(*blocks(w.transpose(1, 2), ws.transpose(1, 2))))
        return
    # (blocks take a kernel with sums in another order: float32 sums, a rounding to 16 bits on either side)
    want = run(*blocks(w.transpose(1, 2), ws.transpose(1, 2))).float()
    wf = upcast_from_mxfp(w, ws, torch.float32, axis=-1).transpose(1, 2)
    mag = torch.cat([x.float().abs()[gather[a:b].clamp(min=0).long()] @ wf[e].abs() for e, (a, b) in enumerate(zip(*(lambda c: (c - sizes.long(), c))(sizes.long().cumsum(0))))])
    assert bool(((got.float() - want).abs() <= 2.0 ** -7 * want.abs() + K * 2.0 ** -22 * mag + 1e-6).all())


@pytest.mark.gpu
@pytest.mark.parametrize("rows,E,K,N", SIZES)
@pytest.mark.parametrize("kind", ["bf16", "f16", "fp8", "mxfp8", "mxfp4"])
@pytest.mark.parametrize("out", ["16", "16 swiglu", "fp8 swiglu", "mx swiglu"])
def test_edges(rows, E, K, N, kind, out, device):
    swiglu, to = out.endswith("swiglu"), out.split()[0]
    sizes = torch.randint(max(0, rows - 9), rows + 10, (E,), generator=torch.Generator().manual_seed(rows), dtype=torch.int32)
    sizes[1], sizes[E // 2] = 0, 3 * rows
    M, T = int(sizes.sum()), 50
    used = ring_rows(M, N, K, E, kind, to, swiglu, block_m=32)
    if not used:
        pytest.skip("another kernel's")
    torch.manual_seed(K)
    gather, scatter = torch.randint(0, T, (M,), dtype=torch.int32), torch.randperm(M, dtype=torch.int32)
    gather[3], scatter[5] = -1, -1
    x = torch.randn(T, K, device=device)
    w, ws = downcast_to_mxfp((torch.randn(E, N, K, device=device) * 0.1).bfloat16(), torch.uint8, axis=-1)
    w, ws = w.transpose(1, 2), ws.transpose(1, 2)
    wb, wsb = blocks(w, ws)
    bias, gammas = torch.randn(E, N, device=device), torch.rand(M, device=device)
    opts = {}
    if kind[:2] == "mx":
        a, s = downcast_to_mxfp(x, torch.uint8 if kind == "mxfp4" else torch.float8_e4m3fn, axis=-1)
        opts.update(a_mx_scale=s, a_microblock_size=32)
    else:
        a = x.to(TYPES[kind])
    scale = torch.full((1,), 0.25, device=device)
    lhs = InFlexData(a.dtype, scale) if kind == "fp8" else InFlexData()
    if to == "fp8":
        opts.update(flex_ctx=FlexCtx(lhs_data=lhs, out_data=OutFlexData(torch.float8_e4m3fn, torch.full((1,), 0.125, device=device))),
                    out_dtype=torch.float8_e4m3fn, flexpoint_saturate_inf=True)
    else:
        opts.update(flex_ctx=FlexCtx(lhs_data=lhs), out_dtype=torch.float8_e4m3fn if to == "mx" else torch.float16 if kind == "f16" else torch.bfloat16)
    md = make_ragged_tensor_metadata(sizes.to(device), M)

    def run(weights, scales):
        c = torch.zeros(M, -(-N // (64 if swiglu else 32)), dtype=torch.uint8, device=device) if to == "mx" else None
        pc = PrecisionConfig(b_mx_scale=scales, b_microblock_size=32, c_mx_scale=c, **opts)
        y = matmul(a, weights, bias, md, gather_indx=gather.to(device), scatter_indx=None if to == "mx" else scatter.to(device),
                   gammas=gammas, precision_config=pc, fused_activation=SWIGLU if swiglu else None, **({"epilogue": TO_MXFP8} if to == "mx" else {}))
        rows_of = torch.arange(M) if to == "mx" else scatter.long()
        there = torch.arange(M)[rows_of >= 0]
        return y[rows_of[there].to(device)], None if c is None else c, there

    got, got_scales, there = run(wb, wsb)
    if kind not in ("bf16", "f16"):
        ref, ref_scales, _ = run(w, wsb)
        assert torch.equal(got.view(torch.uint8), ref.view(torch.uint8))
        assert got_scales is None or torch.equal(got_scales, ref_scales)
        return
    wf = upcast_from_mxfp(w, ws, torch.float32, axis=1)
    expert = torch.repeat_interleave(torch.arange(E), sizes.long())
    xf = torch.where((gather >= 0)[:, None].to(device), a.float()[gather.clamp(min=0).long().to(device)], 0.0)
    full = torch.empty(M, N // 2 if swiglu else N, device=device)
    slack = torch.empty_like(full)
    for e in range(E):
        r = (expert == e).to(device)
        v, mag = xf[r] @ wf[e] + bias[e], K * 2.0 ** -23 * (xf[r].abs() @ wf[e].abs())
        if swiglu:
            g, l = v[:, 0::2].clamp(max=7.0), v[:, 1::2].clamp(-7.0, 7.0)
            s = g * torch.sigmoid(1.702 * g)
            v, mag = s * (l + 1), 1.2 * mag[:, 0::2] * (l.abs() + 1) + s.abs() * mag[:, 1::2]   # (|d swish| <= 1.1)
        full[r], slack[r] = v * gammas[r, None], mag
    full, slack = full[there.to(device)], slack[there.to(device)]
    # a 16-bit result (2^-8) of K float32 additions, and the hardware's exponential and reciprocal (2^-20)
    assert bool(((got.float() - full).abs() <= 2.0 ** -8 * full.abs() + slack + 1e-5).all())


@pytest.mark.gpu
@pytest.mark.parametrize("constraint", [{"block_m": 16}, {"block_m": 32}, {"block_m": 64}, {"block_m": 128}, {"is_persistent": False}])
@pytest.mark.parametrize("kind", ["mxfp4", "bf16 weights"])
def test_not_where_blocks_are_asked_for(kind, constraint, monkeypatch, device):
    """A product whose caller asks for a row block, or for no persistent kernel, runs in blocks of its schedule, with the same result."""
    torch.manual_seed(5)
    E, M, K, N = 40, 400, 1056, 2560
    md = make_ragged_tensor_metadata(torch.full((E,), M // E, dtype=torch.int32, device=device), M)
    x, w = torch.randn(M, K, device=device), (torch.randn(E, N, K, device=device) * 0.1).bfloat16()
    opts = {}
    if kind == "mxfp4":
        w, ws = downcast_to_mxfp(w, torch.uint8, axis=-1)
        x, s = downcast_to_mxfp(x, torch.uint8, axis=-1)
        w, ws = blocks(w.transpose(1, 2), ws.transpose(1, 2))
        opts = dict(a_mx_scale=s, a_microblock_size=32, b_mx_scale=ws, b_microblock_size=32, out_dtype=torch.bfloat16)
    else:
        x, w = x.bfloat16(), w.transpose(1, 2)
    seen = []
    module = sys.modules["triton_amd.matmul"]
    launch = module._launch
    monkeypatch.setattr(module, "_launch", lambda args, dev: seen.append(args) or launch(args, dev))
    y = []
    for c in ({"num_warps": 4}, constraint):   # (the first asks for nothing, through the general host path)
        with scoped_opt_flags_constraints(c):
            y.append(matmul(x, w, None, md, precision_config=PrecisionConfig(**opts)))
    free, asked = seen
    assert _native.ring_rows(ctypes.addressof(free), 256)
    assert not _native.ring_rows(ctypes.addressof(asked), 256)
    assert asked.block_m == constraint.get("block_m", asked.block_m)
    if kind == "mxfp4":
        assert torch.equal(y[0], y[1])
    else:
        # a 16-bit result (2^-8) of K float32 additions on either side
        mag = torch.cat([x[10 * e:10 * e + 10].float().abs() @ w[e].float().abs() for e in range(E)])
        assert bool(((y[0].float() - y[1].float()).abs() <= 2.0 ** -8 * y[0].float().abs() + K * 2.0 ** -22 * mag).all())


def test_where_stages_are_too_few():
    """A tile alone on its CU with a K of few stages is the tiled kernel's, unless the blocks are those that stream; so are 16-bit rows of one stage in several rounds."""
    strided = dict(w_layout=_lib.W_STRIDED, w_mx_layout=_lib.SCALE_STRIDED)
    for K, rows in ((768, 0), (800, 32)):
        assert ring_rows(400, 1296, K, 20, "bf16", block_m=32) == rows and ring_rows(400, 1296, K, 20, "f16", block_m=32, **strided) == rows
        assert ring_rows(180, 1298, K, 20, "mxfp8", block_m=32) == rows and ring_rows(180, 1298, K, 20, "mxfp8", block_m=32, **strided) == rows
    assert ring_rows(300, 768, 64, 60, "bf16", block_m=16) == 32
    for K, rows in ((256, 32), (288, 0), (512, 0), (544, 32)):
        assert ring_rows(40, 1872, K, 12, "mxfp4", block_m=32, **strided) == rows and ring_rows(40, 1872, K, 12, "mxfp4", block_m=32) == 32
    assert ring_rows(500, 2608, 512, 12, "mxfp4", block_m=64) == 0 and ring_rows(500, 2608, 544, 12, "mxfp4", block_m=64) == 64
    assert ring_rows(2400, 2322, 128, 60, "bf16", block_m=64, **strided) == 0 and ring_rows(2400, 2322, 160, 60, "bf16", block_m=64, **strided) == 64


@pytest.mark.gpu
@pytest.mark.parametrize("kind,rows,E,K,N,layout", [
    ("bf16", 40, 60, 160, 2322, "strided"), ("f16", 40, 60, 256, 2322, "strided"), ("bf16", 40, 60, 384, 2322, "strided"), ("f16", 15, 20, 800, 1296, "strided"),
    ("mxfp8", 9, 10, 96, 2832, "strided"), ("mxfp8", 9, 20, 800, 1298, "strided"), ("mxfp4", 9, 10, 256, 2832, "strided"), ("mxfp4", 4, 12, 544, 1872, "strided"),
    ("fp8", 20, 20, 224, 1298, "strided"), ("bf16", 5, 60, 64, 768, "blocks"), ("f16", 9, 60, 96, 768, "blocks"), ("bf16", 9, 60, 352, 752, "blocks"),
    ("mxfp8", 9, 20, 800, 1298, "blocks"), ("mxfp4", 9, 20, 288, 1298, "blocks"), ("fp8", 20, 20, 288, 1298, "blocks")])
def test_few_stages(kind, rows, E, K, N, layout, monkeypatch, device):
    """Fewer stages than the ring holds, one tile to a workgroup and several: as the tiled kernel has it, which blocks of 32 rows that a caller asks for take."""
    sizes = torch.randint(max(0, rows - 4), rows + 5, (E,), generator=torch.Generator().manual_seed(K), dtype=torch.int32)
    sizes[1] = 0
    M = int(sizes.sum())
    torch.manual_seed(K + N)
    # (columns of other scales; float16 results stay below 65504: 140 000 columns of up to e^4.5 times sums of 800 products of normal values, 28 x 5)
    w, ws = downcast_to_mxfp((torch.randn(E, N, K, device=device) * torch.exp(torch.randn(E, N, 1, device=device))).bfloat16(), torch.uint8, axis=-1)
    wf = upcast_from_mxfp(w, ws, torch.float32, axis=-1).transpose(1, 2)
    w, ws = w.transpose(1, 2), ws.transpose(1, 2)
    if layout == "blocks":
        w, ws = blocks(w, ws)
    x, opts = torch.randn(50, K, device=device), {}
    if kind[:2] == "mx":
        x, s = downcast_to_mxfp(x, torch.uint8 if kind == "mxfp4" else torch.float8_e4m3fn, axis=-1)
        opts.update(a_mx_scale=s, a_microblock_size=32)
    else:
        x = x.to(TYPES[kind])
    gather = torch.randint(-1, 50, (M,), dtype=torch.int32, device=device)
    bias, md = torch.randn(E, N, device=device), make_ragged_tensor_metadata(sizes.to(device), M)
    took, y = [], []
    module = sys.modules["triton_amd.matmul"]
    launch = module._launch
    monkeypatch.setattr(module, "_launch", lambda args, dev: took.append(_native.ring_rows(ctypes.addressof(args), 256)) or launch(args, dev))
    for c in ({"num_warps": 4}, {"block_m": 32}):   # (the first asks for nothing, through the general host path)
        with scoped_opt_flags_constraints(c):
            y.append(matmul(x, w, bias, md, gather_indx=gather, precision_config=PrecisionConfig(
                b_mx_scale=ws, b_microblock_size=32, out_dtype=torch.float16 if kind == "f16" else torch.bfloat16, **opts)))
    assert took[0] and not took[1]
    if kind not in ("bf16", "f16"):
        assert torch.equal(y[0], y[1])
        return
    at = [0, *sizes.cumsum(0).tolist()]
    mag = torch.cat([x.float().abs()[gather[at[e]:at[e + 1]].clamp(min=0).long()] @ wf[e].abs() for e in range(E)])
    # (float32 sums in another order, a rounding to 16 bits on either side)
    assert bool(((y[0].float() - y[1].float()).abs() <= 2.0 ** -7 * y[1].float().abs() + K * 2.0 ** -22 * mag + 1e-6).all())

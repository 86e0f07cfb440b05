"""Host-side logic that needs no GPU: storage layouts (literals of the reference's tests/test_tensor.py:32-35,
76-99), the opt-flags constraint API (matmul_details/opt_flags.py:405-455 of the reference), the block-count
bound, dataclass defaults and the errors raised before any launch."""
import threading

import pytest
import torch

from triton_amd.matmul import FnSpecs, FusedActivation, PrecisionConfig, matmul
from triton_amd.matmul_details import opt_flags as OF
from triton_amd.numerics import InFlexData
from triton_amd.tensor import FP4, UINT8, RaggedTensorMetadata, convert_layout, empty, wrap_torch_tensor
from triton_amd.tensor_details.layout import StridedLayout
from oracle import routing_ref as RR


@pytest.mark.parametrize("logical,is_fp4,layout,storage", [
    ((3, 258, 514), True, StridedLayout(-2), [3, 129, 514]),
    ((0, 64), True, StridedLayout(-2), [0, 64]),
    ((3, 258, 514), True, StridedLayout(-1), [3, 258, 257]),
    ((3, 70, 65), False, StridedLayout(-2), [3, 70, 65]),
])
def test_storage_shapes(logical, is_fp4, layout, storage):
    assert layout.storage_shape(list(logical), is_fp4) == storage
    t = empty(logical, FP4 if is_fp4 else UINT8, "meta", layout)
    assert list(t.storage.data.shape) == storage
    assert t.shape == list(logical)
    if 0 not in storage:
        assert t.storage.data.stride(layout.major_dim % len(storage)) == 1


@pytest.mark.parametrize("major_dim", [-1, -2])
def test_odd_fp4_packing_axis_rejected(major_dim):
    shape = [2, 2]
    shape[major_dim] = 1
    with pytest.raises(ValueError):
        StridedLayout(major_dim).storage_shape(shape, True)


@pytest.mark.parametrize("transpose,layout", [(False, StridedLayout(-1)), (False, StridedLayout(1)),
                                              (True, StridedLayout(-2)), (True, StridedLayout(0))])
def test_convert_layout_noop(transpose, layout):
    data = torch.randn(7, 11)
    t = wrap_torch_tensor(data.T if transpose else data)
    assert convert_layout(t, layout) is t


def test_wrap_fp4_doubles_the_packed_axis():
    t = wrap_torch_tensor(torch.zeros(4, 10, 6, dtype=torch.uint8).transpose(1, 2), dtype=FP4)
    assert t.shape == [4, 12, 10] and t.storage.layout.major_dim % 3 == 1
    t2 = wrap_torch_tensor(torch.zeros(4, 6, 10, dtype=torch.uint8), dtype=FP4)
    assert t2.shape == [4, 6, 20]


def test_convert_layout_repacks_fp4_codes():
    g = torch.Generator().manual_seed(0)
    codes = torch.randint(0, 16, (2, 8, 6), generator=g, dtype=torch.uint8)       # logical [2, 8, 6]
    along_last = codes[..., 0::2] | (codes[..., 1::2] << 4)                        # packed along axis -1
    t = wrap_torch_tensor(along_last, dtype=FP4)
    assert t.shape == [2, 8, 6]
    out = convert_layout(t, StridedLayout(-2))
    want = codes[:, 0::2, :] | (codes[:, 1::2, :] << 4)                            # packed along axis -2
    assert list(out.storage.data.shape) == [2, 4, 6] and out.storage.data.stride(1) == 1
    assert torch.equal(out.storage.data, want)


def test_n_blocks_matches_oracle_and_literal():
    assert RaggedTensorMetadata.n_blocks(128, 16384, 16) == 1144
    assert RaggedTensorMetadata.block_sizes() == [16, 32, 64, 128, 256]
    for S, R, b in [(4, 159, 16), (8, 5, 32), (128, 256, 16), (1, 0, 16), (32, 65536, 128)]:
        assert RaggedTensorMetadata.n_blocks(S, R, b) == RR.n_blocks(S, R, b)
    assert RaggedTensorMetadata.max_n_blocks(4, 159) == RR.n_blocks(4, 159, 16)


def test_opt_flags_constraints_scope_and_errors():
    OF.reset_opt_flags_constraints()
    assert OF.make_opt_flags(16384, 5760, 2880, 128, True).block_m == 128
    assert OF.make_opt_flags(256, 5760, 2880, 128, True).block_m == 16
    assert OF.make_opt_flags(256, 4096, 2048, 1, False).block_m == 128
    assert OF.make_opt_flags(1000, 64, 64, 10, True, expected_slice_size=40).block_m == 64
    # the block covers the mean slice and two standard deviations of a Poisson-like size: 16 + 8 -> 32, 64 + 16 -> 128,
    # 2 + 2.8 -> 16 (decode); fp8 rows never take the 16-row block (the streaming kernel would widen them to 16 bits)
    assert OF.make_opt_flags(2048, 5760, 2880, 128, True).block_m == 32
    assert OF.make_opt_flags(8192, 5760, 2880, 128, True).block_m == 128
    assert OF.make_opt_flags(256, 5760, 2880, 128, True, fp8_rows=True).block_m == 32
    assert OF.make_opt_flags(256, 5760, 2880, 1, False, fp8_rows=True).block_m == 128  # dense: rows as they are
    with OF.scoped_opt_flags_constraints({"block_m": 32}):
        assert OF.make_opt_flags(16384, 5760, 2880, 128, True).block_m == 32
        with OF.scoped_opt_flags_constraints({"block_m": 64}):
            assert OF.make_opt_flags(16384, 5760, 2880, 128, True).block_m == 64
        assert OF.make_opt_flags(16384, 5760, 2880, 128, True).block_m == 32
    assert OF.make_opt_flags(16384, 5760, 2880, 128, True).block_m == 128
    with OF.scoped_opt_flags_constraints({"block_m": 48}):
        with pytest.raises(OF.InapplicableConstraint):
            OF.make_opt_flags(100, 64, 64, 1, False)
    with OF.scoped_opt_flags_constraints({"split_k": 4}):
        assert OF.make_opt_flags(100, 64, 64, 1, False).split_k == 4
    assert OF.make_opt_flags(100, 64, 64, 1, False).split_k == 1
    with OF.scoped_opt_flags_constraints({"split_k": 0}):
        with pytest.raises(OF.InapplicableConstraint):
            OF.make_opt_flags(100, 64, 64, 1, False)
    with OF.scoped_opt_flags_constraints({"is_persistent": True}):
        with pytest.raises(OF.InapplicableConstraint):
            OF.make_opt_flags(100, 64, 64, 1, False)
    assert not OF.blocks_asked_for()
    for asked, c in ((True, {"block_m": 64}), (True, {"is_persistent": False}), (False, {"block_m": None, "is_persistent": None}), (False, {"split_k": 1})):
        with OF.scoped_opt_flags_constraints(c):
            assert OF.blocks_asked_for() == asked
    with OF.scoped_opt_flags(OF.OptFlags(block_m=64)):
        assert OF.blocks_asked_for()
    OF.update_opt_flags_constraints({"block_m": 16})
    assert OF.make_opt_flags(16384, 5760, 2880, 128, True).block_m == 16
    OF.reset_opt_flags_constraints()
    assert OF.make_opt_flags(16384, 5760, 2880, 128, True).block_m == 128


def test_opt_flags_constraint_keys_are_validated():
    """Unknown keys are a caller's mistake (AssertionError, matmul_details/opt_flags.py:71-73 of the reference); known
    keys must hold for the flags that come out (:46-50), so values the fixed tile cannot honour raise instead of
    being dropped."""
    OF.reset_opt_flags_constraints()
    with OF.scoped_opt_flags_constraints({"blok_m": 64}):
        with pytest.raises(AssertionError, match="unsupported constraint"):
            OF.make_opt_flags(100, 64, 64, 1, False)
    for key, bad, good in (("block_n", 128, 256), ("block_k", 64, 128), ("num_warps", 8, 4), ("epilogue_subtile", 2, 1),
                           ("idle_sms", 4, 0)):
        with OF.scoped_opt_flags_constraints({key: bad}):
            with pytest.raises(OF.InapplicableConstraint, match=key):
                OF.make_opt_flags(100, 64, 64, 1, False)
        with OF.scoped_opt_flags_constraints({key: good}):
            flags = OF.make_opt_flags(100, 64, 64, 1, False)
            assert getattr(flags, key, good) == good
        with OF.scoped_opt_flags_constraints({key: None}):
            OF.make_opt_flags(100, 64, 64, 1, False)
    with OF.scoped_opt_flags_constraints({"disable_mx4_block_swap": True, "is_persistent": False}):
        OF.make_opt_flags(100, 64, 64, 1, False)
    # max_allowable_mn switches a requested split_k off once the output is large (opt_flags.py:37-43, 114-117)
    with OF.scoped_opt_flags_constraints({"split_k": 4, "max_allowable_mn": 100 * 64}):
        assert OF.make_opt_flags(100, 64, 4096, 1, False).split_k == 1
        assert OF.make_opt_flags(99, 64, 4096, 1, False).split_k == 4


def test_opt_flags_constraints_are_per_thread():
    OF.reset_opt_flags_constraints()
    seen = {}

    def other():
        seen["block_m"] = OF.make_opt_flags(16384, 64, 64, 128, True).block_m

    with OF.scoped_opt_flags_constraints({"block_m": 16}):
        th = threading.Thread(target=other)
        th.start()
        th.join()
        assert OF.make_opt_flags(16384, 64, 64, 128, True).block_m == 16
    assert seen["block_m"] == 128


def test_dataclass_defaults_follow_the_reference():
    pc = PrecisionConfig()
    assert pc.b_mx_scale is None and pc.out_dtype is None and pc.acc_scale == 1.0 and pc.allow_tf32
    assert FnSpecs.default().name == "dflt" and FnSpecs.default().reduction_n == 1
    fa = FusedActivation(FnSpecs("swiglu", None, ("alpha", "limit"), reduction_n=2), (1.702, 7.0))
    assert fa.specs.reduction_n == 2 and fa.fn_args == (1.702, 7.0)
    assert not InFlexData().is_per_batch


def test_errors_before_launch():
    x = torch.zeros(4, 64, dtype=torch.bfloat16)
    w = torch.zeros(1, 64, 8, dtype=torch.bfloat16)
    with pytest.raises(NotImplementedError):
        matmul(x, w, None, fused_comm=object())
    with pytest.raises(NotImplementedError):
        matmul(x, w, None, c_acc_in=torch.zeros(4, 8))
    with pytest.raises(NotImplementedError):
        matmul(x, w, None, precision_config=PrecisionConfig(a_mx_scale=torch.zeros(4, 2, dtype=torch.uint8)))
    with pytest.raises(AssertionError):
        matmul(torch.zeros(2, 4, 64), torch.zeros(2, 64, 8), None, gather_indx=torch.zeros(4, dtype=torch.int32))
    with pytest.raises((RuntimeError, NotImplementedError)):
        matmul(x, w, None)  # CPU tensors: no CPU path exists


def test_build_reports_kernels_in_scratch_memory():
    # the build refuses a kernel that fell out of registers: it would still be right, and several times slower
    from triton_amd.build import _scratch_users
    remarks = """
x.h:1:1: remark: Function Name: _ZN4tamd1aEv [-Rpass-analysis=kernel-resource-usage]
x.h:1:1: remark:     VGPRs: 242 [-Rpass-analysis=kernel-resource-usage]
x.h:1:1: remark:     ScratchSize [bytes/lane]: 704 [-Rpass-analysis=kernel-resource-usage]
x.h:9:1: remark: Function Name: _ZN4tamd1bEv [-Rpass-analysis=kernel-resource-usage]
x.h:9:1: remark:     ScratchSize [bytes/lane]: 0 [-Rpass-analysis=kernel-resource-usage]
"""
    assert _scratch_users(remarks) == [("_ZN4tamd1aEv", 704)]
    assert _scratch_users("") == []


def test_turned_gate_weights_are_cached_per_tensor_and_version():
    """Weights with unit stride along N are turned once for the narrow-output kernel: the copy is reused while the
    caller's tensor is alive and unmodified, redone after an in-place write, dropped with the tensor."""
    import gc
    import torch
    from triton_amd import matmul as mm
    w = torch.randn(64, 16)
    t1 = mm._k_contiguous_cached(w)
    assert t1.stride() == (1, 64) and torch.equal(t1, w)
    assert mm._k_contiguous_cached(w) is t1
    w.mul_(2.0)
    t2 = mm._k_contiguous_cached(w)
    assert t2 is not t1 and torch.equal(t2, w)
    key = id(w)
    assert key in mm._TURNED
    del w
    gc.collect()
    assert key not in mm._TURNED


def test_native_tile_choice_follows_make_opt_flags():
    """The native host path chooses row blocks by the rule of make_opt_flags (no constraints set)."""
    from triton_amd import _native
    OF.reset_opt_flags_constraints()
    for m in (1, 15, 16, 17, 64, 65, 255, 256, 1000, 4097, 65536):
        for slices in (1, 7, 32, 128):
            for ragged, expected in ((False, None), (True, None), (True, 1), (True, 9), (True, 40), (True, 1000)):
                for fp8 in (False, True):
                    want = OF.make_opt_flags(m, 64, 64, slices, ragged, expected, fp8).block_m
                    assert _native.choose_block_m(m, slices, ragged, -1 if expected is None else expected, fp8) == want


def test_native_host_path_is_tied_to_its_torch(monkeypatch):
    """The extension reads tensors in place: one built for another torch is refused when it is loaded, not when it misreads."""
    from triton_amd import _native
    assert _native.load().built_for == str(torch.__version__)
    monkeypatch.setattr(torch, "__version__", "1.0.0")
    with pytest.raises(RuntimeError, match="was built for torch"):
        _native.load()


def test_tiles_block_m_is_one_rule():
    """The native host code and opt_flags choose the same block from the tiles; more tiles never get a smaller block."""
    from triton_amd import _native
    _native.load()
    for m in (1, 7, 64, 300, 1000, 2048, 9000):
        for slices in (1, 8, 60, 128):
            for expected in (None, 0, 9, 31, 33, 64, 65, 200):
                for fp8 in (False, True):
                    base = OF.make_opt_flags(m, 1, 1, slices, True, expected, fp8_rows=fp8).block_m
                    for k in (512, 640, 1152, 1184, 4096, 4128):
                        for mx4, mx_out in ((True, False), (True, True), (False, False)):
                            last = 0
                            for n in (16, 256, 272, 1000, 4096, 11520):
                                want = OF.tiles_block_m(base, m, n, k, slices, expected, mx4, fp8, mx_out)
                                got = _native.choose_block_m(m, slices, True, -1 if expected is None else expected, fp8, n, k, mx4, mx_out)
                                assert got == want and (want <= base or (base, want) == (16, 32))
                                if n % 16 == 0:
                                    assert want >= last
                                    last = want


def test_blocks_of_16_only_where_they_stream():
    """MXFP4 weights: the streaming kernel's conditions on the arguments, and no row block of 16 where one of them fails."""
    import ctypes
    from triton_amd import _lib, _native
    E, K, N, G = 3, 1280, 512, 40
    plain = dict(x=1 << 20, w=2 << 20, w_mx_scale=3 << 20, x_dtype=_lib.BF16, w_dtype=_lib.MXFP4, M=60, K=K, N=N, n_experts=E,
                 w_stride_e=K // 2 * N, w_stride_k=1, w_stride_n=K // 2, w_mx_stride_e=G * N, w_mx_stride_k=1, w_mx_stride_n=G,
                 block_offs=4 << 20, block_schedule=5 << 20)

    def streams(**changed):
        bag = _lib.MatmulArgBag()
        for name, value in {**plain, **changed}.items():
            setattr(bag, name, value)
        packed = bag.pack()
        return _native.blocks_of_16_stream(ctypes.addressof(packed))

    assert streams() is True
    assert streams(n_experts=1, w_stride_e=7, w_mx_stride_e=7) is True       # (the pitch of one matrix is never used)
    for changed in (dict(w_stride_n=K // 2 + 16), dict(w_mx_stride_n=G + 8), dict(w=(2 << 20) + 8), dict(w_mx_scale=(3 << 20) + 4),
                    dict(w_stride_e=K // 2 * N + 8), dict(w_mx_stride_e=G * N + 4), dict(w_stride_e=1 << 30), dict(N=N - 8),
                    dict(K=4128, w_stride_n=2064, w_mx_stride_n=129), dict(x_mx_scale=6 << 20), dict(y_mx_scale=6 << 20),
                    dict(x_dtype=_lib.MXFP4, x_mx_scale=6 << 20), dict(w_dtype=_lib.BF16)):
        assert streams(**changed) is False, changed
    assert streams(w_layout=_lib.W_CDNA4_BLOCKS, w_stride_n=0, w_mx_layout=_lib.SCALE_CDNA4, w_mx_stride_n=0, w_mx_stride_k=0) is True
    for base in (16, 32, 64, 128):
        for fp8 in (False, True):
            for m, slices in ((2, 1), (60, 3), (2000, 128)):
                for n in (16, 512, 5760):
                    assert OF.tiles_block_m(base, m, n, 1280, slices, None, True, fp8, True) >= 32
                    assert _native.choose_block_m(m, slices, True, -1, fp8, n, 1280, True, True) >= 32
    assert OF.tiles_block_m(32, 60, 512, 1280, 3, None, True, False, False) == 16


def dense_block_m(M, N, K, x, w, along_n=False, cus=256, batch=1, blocks=False):
    import ctypes
    from triton_amd import _lib, _native
    bag = _lib.MatmulArgBag()
    bag.M, bag.N, bag.K, bag.n_experts, bag.x_dtype, bag.w_dtype = M, N, K, batch, getattr(_lib, x), getattr(_lib, w)
    bag.w_stride_k, bag.w_stride_n = (N, 1) if along_n else (1, K)
    bag.w_layout = _lib.W_CDNA4_BLOCKS if blocks else _lib.W_STRIDED
    packed = bag.pack()
    return _native.dense_block_m(ctypes.addressof(packed), cus)


@pytest.mark.parametrize("M,N,K,block_m", [
    (2048, 4096, 2048, 128), (4096, 4096, 2048, 128), (3943, 7464, 6144, 128), (12572, 1024, 6688, 128),   # whole rounds of 128
    (256, 4096, 2048, 32), (64, 512, 576, 32), (5749, 512, 2432, 64), (603, 4864, 1344, 64), (5056, 280, 672, 64),
])
def test_dense_blocks_of_weights_along_n(M, N, K, block_m):
    """16-bit weights contiguous along N: the kernel for them holds one tile per CU, and a tile of few rows takes almost as long as one
    of many, so rounds count and rows hardly do (sizes timed with every block)."""
    assert dense_block_m(M, N, K, "BF16", "BF16", along_n=True) == block_m
    assert dense_block_m(M, N, K, "F16", "F16", along_n=True) == block_m


@pytest.mark.parametrize("M,N,K,rows,block_m", [
    (16384, 2880, 2880, "BF16", 128), (14716, 8144, 2080, "BF16", 128), (4096, 8192, 8192, "BF16", 64), (9960, 2784, 5984, "BF16", 64),
    (8192, 5760, 2880, "FP8_E4M3", 128), (16384, 1024, 8192, "FP8_E4M3", 128), (1486, 3064, 5376, "FP8_E4M3", 64),
    (4122, 3152, 7808, "MXFP4", 128), (9652, 1320, 2144, "MXFP4", 128), (256, 4096, 2048, "BF16", 32), (64, 512, 576, "MXFP4", 32),
])
def test_dense_blocks_of_mxfp4_weights(M, N, K, rows, block_m):
    """Products of many rounds in blocks of 128, except 16-bit rows whose scales such a block does not have in LDS (sizes timed with every
    block)."""
    assert dense_block_m(M, N, K, rows, "MXFP4") == block_m
    assert dense_block_m(M, N, K, rows, "MXFP4", blocks=True) == block_m


def test_dense_blocks_of_few_rounds_in_the_block_layout():
    assert dense_block_m(3337, 4768, 608, "BF16", "MXFP4", blocks=True) == 64
    assert dense_block_m(3337, 4768, 608, "BF16", "MXFP4") == 128


def _fake_native(monkeypatch, before_look_up):
    """`routing` without a GPU: the look-up of the native call, and what another thread does just before it."""
    import importlib

    from triton_amd import _lib, _native
    module = importlib.import_module("triton_amd.routing")

    def native(logits, k, layouts):
        before_look_up(module)
        lay = layouts.get((*logits.shape, k, _lib.dtype_code(logits.dtype)))
        return None if lay is None else (torch.empty(lay["ws"][0] + 1), lay)
    monkeypatch.setattr(_native, "routing", native)
    monkeypatch.setattr(_lib, "require_gpu", lambda t, name: None)
    module._layouts.clear()
    return module


def test_routing_while_another_thread_drops_the_layouts(monkeypatch):
    module = _fake_native(monkeypatch, lambda m: m._layouts.clear())
    r = module.routing(torch.zeros(3, 8), 2)
    assert r._lay["shape"] == (3, 2) and r._lay["dims"][0] == 8
    module._layouts.clear()


def test_routing_keeps_what_is_still_asked_for(monkeypatch):
    """Of very many shapes, one that every other call has is laid out once, however often old ones are dropped; no more than 1024 are held."""
    module = _fake_native(monkeypatch, lambda m: None)
    module._dropped.clear()
    made, lay_out = [], module._arena_layout
    monkeypatch.setattr(module, "_arena_layout", lambda *shape: made.append(shape) or lay_out(*shape))
    for T in range(2, 1800):
        module.routing(torch.zeros(1, 8), 2)
        module.routing(torch.zeros(T, 8), 2)
        assert len(module._layouts) + len(module._dropped) <= 1024
    assert sum(shape[0] == 1 for shape in made) == 1
    module._layouts.clear()
    module._dropped.clear()


def test_tables_asked_for_under_inference_mode_are_ordinary():
    """One call makes all tables: what the mode was when the first was asked for must not decide what may be done with the others."""
    import struct

    from triton_amd import _native
    base = torch.arange(64, dtype=torch.int32)
    numbers = struct.pack("10q", 0, 4, 1, -1, 0, 16, 2, 8, 5, 1)
    with torch.inference_mode():
        line, table = _native.int_views(base, numbers)
    line.add_(1)
    assert line.tolist() == [1, 2, 3, 4] and base[:4].tolist() == [1, 2, 3, 4] and table.tolist() == [list(range(16, 21)), list(range(24, 29))]
    with torch.inference_mode():
        of_inference = torch.arange(64, dtype=torch.int32)
    line, table = _native.int_views(of_inference, numbers)
    table.mul_(2)
    assert not line.is_inference() and table[0].tolist() == [32, 34, 36, 38, 40] and not torch.is_inference_mode_enabled()


def test_where_two_launches_route():
    """Not where their workgroups pass over many rows and leave the chip idle, nor where these are more than one round and a row gives few entries."""
    from triton_amd._native import routing_block_rows as rows
    assert rows(4096, 128, 4) == 32 and rows(3000, 512, 8) == 32 and rows(32768, 256, 1) == 128 and rows(65535, 8, 1) and rows(40000, 40, 1)
    assert rows(65536, 8, 1) == 0 and rows(1000, 513, 1) == 0 and rows(0, 8, 1) == 0
    assert all(rows(T, E, k) == 0 for T, E in ((5000, 257), (10000, 384), (65535, 512)) for k in (1, 4, 16))
    assert all(rows(T, E, k) == 0 for T, E in ((32769, 128), (32769, 256), (65535, 200)) for k in (1, 2, 3))
    assert all(rows(T, E, k) for T, E in ((32769, 128), (32769, 256), (65535, 200)) for k in (4, 8)) and rows(65535, 60, 40)

"""`routing(logits, k)`: the composition the reference spells out in
tests/test_distributed.py:201-208 (topk -> histogram / ordering -> ragged
metadata; gather = col_sorted // k, scatter = col_sorted).

One foreign call (`tamd_routing`: one launch at decode sizes, two up to 65535 rows of up to 512 experts where these fill
the chip, else the top-k and one to three launches for the metadata) writes into
one int32 arena that holds every output and the kernels' workspace; its layout is computed once per shape and the
tensors of the result are views of that arena, built when they are first asked for (the index arrays and ragged tables
together, in one call): at these sizes the host time of this function is what a step waits for."""
import struct
import threading

import torch

from . import _lib, _native
from .tensor import BIT, BitmatrixMetadata, RaggedTensorMetadata, SparseMatrix, wrap_torch_tensor
from .tensor_details.ragged_tensor import _PITCH
from .topk import topk_forward


class RoutingResult:
    """Unpacks like the reference helper into (ragged_metadata, gather_indx, scatter_indx, indx).

    gather_indx  int32 [T*k]: token of the i-th expert-sorted row
    scatter_indx int32 [T*k]: flat (token*k+slot) of the i-th expert-sorted row
    indx int16 [T, k], vals [T, k] gate weights (softmax over the k picked), col_sum int32 [E] tokens per expert,
    row_sorted_indx int32 [T*k] inverse of scatter_indx, sparse: the SparseMatrix a `topk` call returns."""
    __slots__ = ("_arena", "_lay", "_bits", "_indx", "_vals", "_cache")

    def __init__(self, arena, lay, bits=None, indx=None, vals=None):
        self._arena, self._lay, self._bits, self._indx, self._vals, self._cache = arena, lay, bits, indx, vals, {}

    def _tables(self):
        """The index arrays and the ragged tables, all with one call (seven calls of their own took twice as long)."""
        c = self._cache
        c["col_sum"], c["offs"], c["block_offs"], c["sched"], c["gather"], c["col_sorted"], c["row_sorted"] = \
            _native.int_views(self._arena, self._lay["tables"])
        return c

    def _view(self, name):
        v = self._cache.get(name)
        return self._tables()[name] if v is None else v

    def _view2(self, name, dtype, n0, stride0, n1, stride1=1, skip=0):
        """A two-dimensional view of part `name` of the arena in another type (sizes, strides and `skip` in its elements)."""
        off = self._lay[name][0] * 4 // dtype.itemsize + skip
        return _native.view(self._arena, dtype, off, n0, stride0, n1, stride1)

    col_sum = property(lambda self: self._view("col_sum"))
    scatter_indx = property(lambda self: self._view("col_sorted"))
    row_sorted_indx = property(lambda self: self._view("row_sorted"))
    gather_indx = property(lambda self: self._view("gather"))

    @property
    def indx(self):
        if self._indx is None:
            T, k = self._lay["shape"]
            self._indx = self._view2("indx", torch.int16, T, k, k)
        return self._indx

    @property
    def vals(self):
        if self._vals is None:
            T, k = self._lay["shape"]
            self._vals = self._view2("vals", self._lay["vals_dtype"], T, k, k)
        return self._vals

    @property
    def _mask_words(self):
        if self._bits is None:
            T, _ = self._lay["shape"]
            n_words, pad_t = self._lay["bits_shape"]
            self._bits = self._view2("bits", torch.int32, T, 1, n_words, pad_t)
        return self._bits

    @property
    def ragged_metadata(self):
        md = self._cache.get("ragged")
        if md is None:
            c = self._cache if "row_sorted" in self._cache else self._tables()   # (the last one that _tables() writes)
            # (an instance made field by field: the checks of its constructor hold by construction)
            md = c["ragged"] = RaggedTensorMetadata.__new__(RaggedTensorMetadata)
            md.__dict__.update(slice_sizes=c["col_sum"], slice_offs=c["offs"], block_offs_data=c["block_offs"],
                               block_schedule_data=c["sched"], expected_slice_size=None, slice_sizes_divisibility=None)
        return md

    @property
    def sparse(self):
        sp = self._cache.get("sparse")
        if sp is None:
            T, E = self.indx.shape[0], self._lay["dims"][0]
            sp = SparseMatrix.__new__(SparseMatrix)
            sp.indx, sp.vals = self.indx, self.vals
            sp.mask = wrap_torch_tensor(self._mask_words.view(torch.uint32), dtype=BIT, shape=[T, E], shape_max=[T, E])
            sp.mask_metadata = BitmatrixMetadata(self.col_sum, self.scatter_indx, self.row_sorted_indx)
            self._cache["sparse"] = sp
        return sp

    def __iter__(self):  # unpack like the reference helper
        yield self.ragged_metadata
        yield self.gather_indx
        yield self.scatter_indx
        yield self.indx

    @property
    def expert_sorted_gate_weights(self):
        """vals in expert-sorted row order: the `gammas` of the down projection.  A tensor of its own on every access: a caller
        may scale it in place.  The routing kernels write one copy where they place an entry (two indexing kernels and their
        launches fewer: 11 us at 256 rows, 13 at 16384); the first access hands it out if vals cannot have been written to."""
        mine = object()  # (of several threads one gets the kernels' copy)
        if "gates" in self._lay and self._vals_as_routed() and self._cache.setdefault("gates", mine) is mine:
            T, k = self._lay["shape"]
            off = self._lay["gates"][0] * 4 // self._lay["vals_dtype"].itemsize
            return _native.view(self._arena, self._lay["vals_dtype"], off, T * k, 1, -1, 0)
        return self.vals.reshape(-1)[self.scatter_indx.long()]

    def _vals_as_routed(self):
        # (inference tensors do not count their versions)
        return self._vals is None or (not self._vals.is_inference() and self._vals._version == 0)


def _int_tables(lay):
    """What `RoutingResult._tables` views: offset, size and stride of each axis (size -1: there is none)."""
    E, width, po, ps = lay["dims"]
    at = lambda name: lay[name][0]
    line = lambda name: (at(name), lay[name][1], 1, -1, 0)
    return struct.pack("35q", *line("col_sum"), at("offs"), E + 1, 1, -1, 0, at("offs") + po, 5, po, E + 1, 1, at("sched"), 5, ps, width, 1,
                       *line("gather"), *line("col_sorted"), *line("row_sorted"))


# (T, E, k, type code) -> _arena_layout: the native call looks the first up; the second holds up to 512 that the first dropped, of
# which those that are still asked for come back
_layouts, _dropped = {}, {}
_publishing = threading.Lock()


def _arena_layout(T: int, E: int, k: int, vals_dtype: torch.dtype):
    """Where every output of `tamd_routing` (and its workspace) sits in the int32 arena of one call: name -> (offset,
    length) in ints, each part 16-byte aligned.  Depends on the shapes only, so it is built once per shape."""
    n = T * k
    width = RaggedTensorMetadata.max_n_blocks(E, n)
    po = -(-(E + 1) // _PITCH) * _PITCH
    ps = -(-max(width, 1) // _PITCH) * _PITCH
    n_words, pad_t = -(-E // 32), -(-T // 32) * 32
    n_ws = _lib.lib().tamd_bitmatrix_metadata_workspace(n, E)
    per_int = 4 // vals_dtype.itemsize
    lay = {"dims": (E, width, po, ps), "shape": (T, k), "vals_dtype": vals_dtype, "bits_shape": (n_words, pad_t)}
    off = 0
    for name, size in (("col_sum", E), ("col_sorted", n), ("row_sorted", n), ("gather", n), ("offs", 6 * po), ("sched", 5 * ps),
                       ("bits", n_words * pad_t), ("vals", -(-n // per_int)), ("gates", -(-n // per_int)), ("indx", -(-n // 2)),
                       ("ws", n_ws)):
        lay[name] = (off, size)
        off += -(-size // 4) * 4
    # what the native call needs, in the order that csrc/host.cpp reads: the arena's length, the sizes of the tables, the
    # byte offset of every part
    lay["native"] = struct.pack("16q", off, width, po, ps, pad_t, *(4 * lay[name][0] for name in (
        "vals", "indx", "bits", "col_sum", "col_sorted", "row_sorted", "gather", "gates", "offs", "sched", "ws")))
    lay["tables"] = _int_tables(lay)
    return lay


def routing(logits: torch.Tensor, n_expts_act: int, y_indx=None) -> RoutingResult:
    if y_indx is None:
        done = _native.routing(logits, n_expts_act, _layouts)
        if done is None:
            done = _routing_first_call(logits, n_expts_act)
        if type(done) is tuple:
            return RoutingResult(*done)
        if type(done) is int:
            _lib.check(done, "routing")
    return _routing_two_calls(logits, n_expts_act, y_indx)


def _routing_first_call(logits, k):
    """A call of a shape that is not among `_layouts`: checks, the arena's layout, then what `_native.routing` answers; None for
    strided logits."""
    if logits.stride(1) != 1:
        return None
    _lib.require_gpu(logits, "logits")
    assert logits.ndim == 2 and logits.shape[1] < 32768
    T, E = logits.shape
    code = _lib.dtype_code(logits.dtype)  # (refuses other types before the layout divides by their size)
    key = T, E, k, code
    lay = _dropped.get(key) or _arena_layout(T, E, k, logits.dtype)
    done = _native.routing(logits, k, {key: lay})   # (handed over: another thread may clear what is published)
    assert done is not None, "k must be an int and logits of a floating type"
    if type(done) is tuple:
        with _publishing:
            if len(_layouts) >= 512:
                _dropped.clear()
                _dropped.update(list(_layouts.items())[-512:])
                _layouts.clear()
            _layouts[key] = lay
    return done


def _routing_two_calls(logits, n_expts_act, y_indx):
    """Provided indices or strided logits: the top-k wrapper, then the metadata entry point."""
    vals, indx, mask = topk_forward(logits, n_expts_act, apply_softmax=True, y_indx=y_indx)
    T, E = logits.shape
    k = n_expts_act
    n = T * k
    dev = logits.device
    L = _lib.lib()
    width = RaggedTensorMetadata.max_n_blocks(E, n)
    po = -(-(E + 1) // _PITCH) * _PITCH
    ps = -(-max(width, 1) // _PITCH) * _PITCH
    n_ws = L.tamd_bitmatrix_metadata_workspace(n, E)
    lay, off = {"dims": (E, width, po, ps)}, 0
    for name, size in (("col_sum", E), ("col_sorted", n), ("row_sorted", n), ("gather", n), ("offs", 6 * po), ("sched", 5 * ps),
                       ("ws", n_ws)):
        lay[name] = (off, size)
        off += -(-size // 4) * 4
    lay["tables"] = _int_tables(lay)
    arena = torch.empty(off, dtype=torch.int32, device=dev)
    base = arena.data_ptr()
    p = lambda name: base + 4 * lay[name][0]
    rc = L.tamd_routing_metadata(_lib.ptr(indx), 1, n, E, k, p("col_sum"), p("col_sorted"), p("row_sorted"), p("gather"),
                                 p("offs"), po, p("sched"), ps, width, p("ws"), _lib.stream_ptr(dev))
    _lib.check(rc, "routing")
    return RoutingResult(arena, lay, mask.storage.data.view(torch.int32), indx, vals)

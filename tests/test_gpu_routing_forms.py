"""GPU: the routing's launch forms around the lines between them (workgroups of 256, 512 and 1024 threads in the first of the two
launches, one launch, more than two), against the oracle."""
import pytest
import torch

from oracle import routing_ref as RR
from triton_amd import _lib
from triton_amd.routing import routing

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,E,k", [
    (160, 16, 8), (161, 16, 8), (192, 16, 6), (193, 16, 6), (256, 16, 2), (257, 16, 2), (129, 16, 8),   # one launch, then two
    (80, 128, 8), (81, 128, 8), (96, 128, 6), (97, 128, 6), (128, 128, 4), (129, 128, 4), (128, 128, 1),
    (2047, 128, 4), (2049, 128, 4), (4096, 128, 4), (4097, 128, 4),                           # 256, 512, 1024 threads
    (255, 60, 6), (300, 100, 6), (1000, 200, 6), (700, 256, 8),                               # chunks that need larger workgroups
    (1, 128, 4), (33, 8, 8), (64, 128, 16), (65, 128, 4), (128, 32, 4), (129, 33, 8), (32, 250, 8), (33, 256, 8), (16, 512, 40),   # one launch, then two
    (17, 512, 64), (4097, 8, 1), (8193, 128, 2), (40000, 16, 2), (65535, 8, 1), (65536, 8, 1),   # blocks of more passes; more rows than 16 bits count
    (16385, 16, 8), (32768, 64, 6), (20000, 60, 8), (8192, 256, 8), (300, 200, 1), (130, 8, 1)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_forms(T, E, k, dtype, device):
    torch.manual_seed(T)
    logits = (torch.randn(T, E) + 0.3 * torch.randn(E)).to(dtype)
    if T % 2:  # rows of few different values, zeros of both signs among them: ties, also among the columns of one lane
        logits[1::2] = torch.randint(-2, 3, logits[1::2].shape).to(dtype) * (-0.0 if T % 4 == 1 else 0.5)
    r, ref = routing(logits.to(device), k), RR.routing_ref(logits, k)
    assert torch.equal(r.indx.cpu().int(), ref["indx"].int()) and torch.equal(r.col_sum.cpu(), ref["col_sum"])
    assert torch.equal(r.scatter_indx.cpu(), ref["scatter_indx"]) and torch.equal(r.gather_indx.cpu(), ref["gather_indx"])
    gates = r.expert_sorted_gate_weights.cpu()
    assert torch.equal(gates, r.vals.cpu().flatten()[ref["scatter_indx"].long()])
    md = r.ragged_metadata
    assert torch.equal(md.slice_offs.cpu()[1:].int(), ref["col_sum"].cumsum(0).int())
    sizes = ref["col_sum"]
    for b in (16, 32, 64, 128):
        n = (sizes + b - 1) // b
        assert int(md.block_offs(b)[E]) == int(n.sum())
        want = torch.cat([torch.arange(int(c)) * 65536 + e for e, c in enumerate(n)])
        assert torch.equal(md.block_schedule(b)[: len(want)].cpu().long(), want.long())


@pytest.mark.parametrize("T,E,k", [(64, 128, 4), (65, 128, 4), (128, 128, 8), (256, 16, 8), (200, 40, 5), (64, 256, 32), (32, 512, 64)])
def test_without_a_workspace(T, E, k, device):
    """The C entry up to twice the rows that 1024 threads hold: what it writes with a workspace."""
    logits = torch.randn(T, E, generator=torch.Generator().manual_seed(T + E)).to(device)
    r = routing(logits, k)
    (_, width, po, ps), (n_words, pad_t) = r._lay["dims"], r._lay["bits_shape"]
    i32 = lambda *shape: torch.full(shape, -7, dtype=torch.int32, device=device)
    vals, indx, bits = torch.empty(T, k, device=device), torch.empty(T, k, dtype=torch.int16, device=device), i32(n_words, pad_t)
    col_sum, col_sorted, row_sorted, gather, offs, sched = i32(E), i32(T * k), i32(T * k), i32(T * k), i32(6, po), i32(5, ps)
    ptr = _lib.ptr
    rc = _lib.lib().tamd_routing(ptr(logits), _lib.F32, E, T, E, k, ptr(vals), ptr(indx), ptr(bits), 1, pad_t, ptr(col_sum), ptr(col_sorted),
                                 ptr(row_sorted), ptr(gather), ptr(offs), po, ptr(sched), ps, width, None, _lib.stream_ptr(device))
    assert rc == 0
    md = r.ragged_metadata
    assert torch.equal(indx, r.indx) and torch.equal(vals, r.vals) and torch.equal(bits[:, :T], r._mask_words.t()[:, :T])
    assert torch.equal(col_sum, r.col_sum) and torch.equal(col_sorted, r.scatter_indx) and torch.equal(row_sorted, r.row_sorted_indx)
    assert torch.equal(gather, r.gather_indx) and torch.equal(offs[0, :E + 1], md.slice_offs) and torch.equal(offs[1:, :E + 1], md.block_offs_data)
    assert torch.equal(sched[:, :width], md.block_schedule_data)


@pytest.mark.parametrize("E", [31, 33, 127, 384, 512])
@pytest.mark.parametrize("k", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_few_picks(E, k, dtype, device):
    """A lane sorts only as many of its keys as it can give: rows whose picks all come from one lane, equal ones among them."""
    T, L = 700, 8 if E <= 64 else 16 if E <= 128 else 64
    g = torch.Generator().manual_seed(E + k)
    logits = torch.randn(T, E, generator=g)
    lane = torch.randint(0, L, (T, 1), generator=g)
    own = torch.arange(E)[None, :] % L == lane
    logits = torch.where(own, 4 + torch.randint(0, 3, (T, E), generator=g).float(), logits).to(dtype)
    r, ref = routing(logits.to(device), k), RR.routing_ref(logits, k)
    assert torch.equal(r.indx.cpu().int(), ref["indx"].int()) and torch.equal(r.col_sum.cpu(), ref["col_sum"])
    assert torch.equal(r.scatter_indx.cpu(), ref["scatter_indx"])

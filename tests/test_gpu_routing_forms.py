"""GPU: the routing's launch forms around the lines between them (workgroups of 256, 512 and 1024 threads in the first of the two
launches, one launch, more than two), against the oracle."""
import pytest
import torch

from oracle import routing_ref as RR
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

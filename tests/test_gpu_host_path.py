"""GPU: what the routing kernels leave in expert-sorted order, on every launch form of the routing, against the oracle."""
import pytest
import torch

from oracle import routing_ref as RR
from triton_amd.routing import routing

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,E,k", [
    (1, 128, 4), (128, 128, 4), (129, 128, 4), (64, 500, 1),  # one launch, its last row count, the two launches after it
    (8192, 128, 4), (8193, 128, 4),                           # two launches, more blocks than they cover
    (300, 128, 3), (5000, 33, 3), (5, 600, 2),                # rows that make no whole chunks; columns past one launch
])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_expert_sorted_gate_weights(T, E, k, dtype, device):
    torch.manual_seed(0)
    logits = torch.randn(T, E).to(dtype)
    r = routing(logits.to(device), k)
    ref = RR.routing_ref(logits, k)
    assert torch.equal(r.scatter_indx.cpu(), ref["scatter_indx"])
    gates = r.expert_sorted_gate_weights
    assert gates.dtype == dtype and torch.equal(gates.cpu(), r.vals.cpu().flatten()[ref["scatter_indx"].long()])

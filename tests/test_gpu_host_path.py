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


@pytest.mark.parametrize("inference", [False, True])
def test_gate_weights_are_the_callers_own(inference, device):
    """Scaling the gate weights in place changes neither later accesses nor vals; scaling vals changes later accesses."""
    with torch.inference_mode(inference):
        torch.manual_seed(3)
        logits = torch.randn(65, 32, device=device)
        r = routing(logits, 4)
        want = r.vals.clone().reshape(-1)[r.scatter_indx.long()]
        first = routing(logits, 4).expert_sorted_gate_weights   # (vals not touched before: the kernel's own copy)
        assert torch.equal(first, want)
        g = r.expert_sorted_gate_weights
        g.mul_(3.0)
        assert torch.equal(r.expert_sorted_gate_weights, want)
        r.vals.mul_(2.0)
        assert torch.equal(r.expert_sorted_gate_weights, want * 2)
        q = routing(logits, 4)
        q.vals.mul_(2.0)
        assert torch.equal(q.expert_sorted_gate_weights, want * 2)
        q = routing(logits, 4)
        q.expert_sorted_gate_weights.zero_()
        assert torch.equal(q.expert_sorted_gate_weights, want)

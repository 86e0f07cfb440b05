"""GPU: what the routing kernels leave in expert-sorted order, on every launch form of the routing, against the oracle; what the
host code of the entry points hands out and keeps."""
import pytest
import torch

from oracle import routing_ref as RR
from triton_amd.matmul import matmul
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


def gate(device, seed):
    """A gate product whose weights have unit stride along N: they are turned, and the copy is kept."""
    g = torch.Generator().manual_seed(seed)
    x, w = torch.randn(48, 256, generator=g).bfloat16(), (torch.randn(256, 32, generator=g) * 0.1).bfloat16()
    return x.to(device), w.to(device), x.float() @ w.float()


def close(y, ref):
    torch.testing.assert_close(y.cpu().float(), ref, rtol=1e-2, atol=1e-2)


def test_turned_weights_on_another_stream(device):
    x, w, ref = gate(device, 0)
    first, second = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(first):
        torch.cuda._sleep(200_000_000)      # the copy is made about 0.1 s from now
        y1 = matmul(x, w, None)
    with torch.cuda.stream(second):
        y2 = matmul(x, w, None)
    torch.cuda.synchronize()
    close(y1, ref)
    close(y2, ref)


def test_turned_weights_in_a_graph(device):
    x, w, ref = gate(device, 1)
    warm = gate(device, 2)
    matmul(warm[0], warm[1], None)
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        y = matmul(x, w, None)              # the first call on these weights is only recorded
    close(matmul(x, w, None), ref)          # ... and leaves nothing behind
    for scale in (1.0, 2.0, 0.5):
        w.mul_(scale)
        ref = x.cpu().float() @ w.cpu().float()
        graph.replay()
        torch.cuda.synchronize()
        close(y, ref)
        close(matmul(x, w, None), ref)


def test_turned_weights_in_inference_mode(device):
    with torch.inference_mode():
        x, w, ref = gate(device, 3)
        close(matmul(x, w, None), ref)
        w.mul_(2.0)
        close(matmul(x, w, None), 2 * ref)

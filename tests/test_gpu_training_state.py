"""What a training call keeps for its backward: q, k, v, the output and the log-sum-exp as saved tensors, the rest beside them."""
import pytest
import torch

from hbsattn_amd import HBSAttention
from hbsattn_amd.workloads import make_problem

pytestmark = pytest.mark.gpu


def _problem():
    return make_problem(seed=11, q_lens=[300, 129], k_lens=[300, 129], hq=4, hk=2, d=64, qbs=64, kbs=64, keep=0.5, diag=True, causal=True,
                        scale=None)


def _args(w, metadata=True):
    args = list(w.args(with_meta=metadata))
    args[:3] = [t.detach().clone().requires_grad_(True) for t in args[:3]]
    return args


def _grads(args, dout, before_backward=lambda: None):
    out = HBSAttention(*args)
    before_backward()
    return (out.detach(),) + torch.autograd.grad(out, args[:3], dout)


@pytest.mark.parametrize("metadata", [True, False])
def test_metadata_made_in_inference_mode(metadata):
    w = _problem()
    dout = torch.randn_like(w.q)
    expected = _grads(_args(w), dout)
    args = _args(w, metadata)
    with torch.inference_mode():   # as a data loader or a scheduler makes it
        args[3:] = [a.clone() if isinstance(a, torch.Tensor) else a for a in args[3:]]
    for got, want in zip(_grads(args, dout), expected):
        assert torch.equal(got, want)


def test_metadata_buffers_written_before_backward():
    w = _problem()
    dout = torch.randn_like(w.q)
    expected = _grads(_args(w), dout)
    args = _args(w)
    buffers = [a for a in args[3:] if isinstance(a, torch.Tensor)]

    def refill():   # the same lengths again, as the next step of a loop with fixed buffers writes them
        for b in buffers:
            b.copy_(b.clone())

    for got, want in zip(_grads(args, dout, refill), expected):
        assert torch.equal(got, want)


def test_saved_tensor_hooks_see_tensors_of_the_computation_only():
    w = _problem()
    args = _args(w)
    seen = []

    def pack(t):
        seen.append((t.dtype, tuple(t.shape)))
        return t

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t):
        out = HBSAttention(*args)
    rows = (w.q.dtype, tuple(w.q.shape))
    keys = (w.k.dtype, tuple(w.k.shape))
    assert sorted(map(str, seen)) == sorted(map(str, [rows, keys, keys, rows, (torch.float32, tuple(w.q.shape[:2]))]))
    dout = torch.randn_like(w.q)
    first = torch.autograd.grad(out, args[:3], dout, retain_graph=True)
    second = torch.autograd.grad(out, args[:3], dout)
    assert all(torch.equal(a, b) for a, b in zip(first, second))
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(out, args[:3], dout)

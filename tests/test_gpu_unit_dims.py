"""Dimensions of one element, whose stride torch leaves at any number: a slice of one token, a single head."""
import pytest
import torch

import hbsattn_amd.interface as interface
from hbsattn_amd import HBSAttention
from hbsattn_amd.interface import hbsa_prepare, hbsa_run
from hbsattn_amd.workloads import make_problem
from helpers import assert_close_to_oracle, oracle_for

pytestmark = pytest.mark.gpu


def _restride(t, tok, head):
    """The same values with these strides in the dimensions of one element."""
    strides = (tok if t.shape[0] == 1 else t.stride(0), head if t.shape[1] == 1 else t.stride(1), 1)
    return torch.as_strided(t, t.shape, strides)


@pytest.fixture
def one_launch_only(monkeypatch):
    def refuse(*a, **k):
        raise AssertionError("the call left the compiled host path")

    monkeypatch.setattr(interface, "hbsa_forward", refuse)


@pytest.mark.parametrize("q_len,k_len,hq,hk", [(1, 1, 4, 2), (1, 40, 4, 4), (5, 1, 1, 1), (7, 40, 2, 1), (1, 1, 1, 1)])
@pytest.mark.parametrize("tok,head", [(772, 7), ((1 << 25) + 8, 8), (1 << 40, 1 << 40)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_strides_of_unit_dimensions(one_launch_only, q_len, k_len, hq, hk, tok, head, dtype):
    w = make_problem(seed=5, q_lens=[q_len], k_lens=[k_len], hq=hq, hk=hk, d=64, qbs=16, kbs=16, keep=1.0, diag=True, causal=False,
                     scale=None, dtype=dtype)
    args = list(w.args())
    plain = HBSAttention(*args)
    args[:3] = [_restride(t, tok, head) for t in args[:3]]
    assert any(t.stride()[:2] != u.stride()[:2] for t, u in zip(args[:3], (w.q, w.k, w.v)))
    assert torch.equal(HBSAttention(*args), plain)
    assert_close_to_oracle(plain, oracle_for(w), "unit dimensions")
    meta = (w.q_meta[0], w.q_meta[2], w.q_meta[3], w.k_meta[0], w.k_meta[3])
    prepared = hbsa_prepare(w.cu_q_seqlens, w.cu_k_seqlens, w.block_mask, 16, 16, False, *meta)
    assert_close_to_oracle(hbsa_run(*args[:3], prepared, None), oracle_for(w), "prepared")


def test_a_token_of_a_wider_buffer(one_launch_only):
    buffer = torch.randn(8, 772, device="cuda").to(torch.bfloat16)
    q = buffer[:, :256].view(8, 4, 64)[4:5]   # contiguous to torch, token stride 772: not a multiple of eight
    assert q.is_contiguous() and q.stride(0) == 772
    w = make_problem(seed=5, q_lens=[1], k_lens=[40], hq=4, hk=2, d=64, qbs=16, kbs=16, keep=1.0, diag=True, causal=True, scale=None)
    args = list(w.args())
    args[0] = q
    got = HBSAttention(*args)
    args[0] = q.reshape(256).clone().view(1, 4, 64)
    assert torch.equal(got, HBSAttention(*args))


@pytest.mark.parametrize("q_len,k_len,hq,hk", [(1, 40, 4, 2), (5, 1, 1, 1), (20, 20, 1, 1)])
def test_gradients(q_len, k_len, hq, hk):
    w = make_problem(seed=6, q_lens=[q_len], k_lens=[k_len], hq=hq, hk=hk, d=64, qbs=16, kbs=16, keep=1.0, diag=True, causal=False,
                     scale=None)
    dout = torch.randn_like(w.q)
    results = []
    for change in (lambda t: t, lambda t: _restride(t, 772, 7)):
        args = list(w.args())
        args[:3] = [change(t).detach().requires_grad_(True) for t in args[:3]]
        results.append(torch.autograd.grad(HBSAttention(*args), args[:3], change(dout)))
    for got, want in zip(results[1], results[0]):
        assert torch.equal(got, want)


def test_a_mask_of_one_k_block_with_any_stride(one_launch_only):
    w = make_problem(seed=7, q_lens=[50], k_lens=[16], hq=2, hk=2, d=96, qbs=16, kbs=16, keep=0.6, diag=True, causal=False, scale=None)
    args = list(w.args())
    plain = HBSAttention(*args)
    mask = args[5]
    args[5] = torch.as_strided(mask, mask.shape, (mask.stride(0), mask.stride(1), 3))
    assert torch.equal(HBSAttention(*args), plain)

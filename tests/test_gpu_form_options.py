"""What a call may ask for, in each form that a launch of few items takes: element types, strides, a negative scale, a capture, calls on two
streams at once, gradients and the log-sum-exp."""
import dataclasses

import pytest
import torch

from hbsattn_amd import HBSAttention
from hbsattn_amd.interface import hbsa_prepare, hbsa_run
from hbsattn_amd.workloads import make_problem
from helpers import assert_close_to_oracle, oracle_for
from oracle.grads import hbsa_oracle_grads
from test_gpu_launch_plan import plan_for

pytestmark = pytest.mark.gpu

# wavefronts, teams, more than one part
FORMS = {
    "sole": (dict(q_lens=[200, 90], k_lens=[300, 90], hq=4, hk=2, d=64, qbs=64, kbs=64, keep=0.6), (4, 1, False)),
    "sole 80": (dict(q_lens=[200, 90], k_lens=[300, 90], hq=4, hk=2, d=80, qbs=48, kbs=64, keep=0.6), (4, 1, False)),
    "teams": (dict(q_lens=[1000], k_lens=[1000], hq=4, hk=2, d=64, qbs=64, kbs=64, keep=0.6), (4, 2, False)),
    "teams 128": (dict(q_lens=[1000], k_lens=[1200], hq=2, hk=2, d=128, qbs=48, kbs=48, keep=0.6), (4, 2, False)),
    "teams 96": (dict(q_lens=[1300], k_lens=[1300], hq=2, hk=1, d=96, qbs=64, kbs=64, keep=0.4), (4, 2, False)),
    "split": (dict(q_lens=[70, 4], k_lens=[6000, 5000], hq=4, hk=2, d=64, qbs=64, kbs=64, keep=0.3), (4, 1, True)),
    "split 128": (dict(q_lens=[70, 4], k_lens=[6000, 5000], hq=8, hk=2, d=128, qbs=128, kbs=64, keep=0.3), (8, 1, True)),
    "split packed": (dict(q_lens=[70, 4], k_lens=[6000, 5000], hq=8, hk=1, d=64, qbs=48, kbs=64, keep=0.3), (4, 1, True)),
    "teams packed": (dict(q_lens=[700, 300], k_lens=[700, 300], hq=8, hk=1, d=128, qbs=16, kbs=48, keep=0.6), (4, 2, False)),
    "split 80": (dict(q_lens=[70, 4], k_lens=[6000, 5000], hq=4, hk=2, d=80, qbs=64, kbs=48, keep=0.3), (4, 1, True)),
    "split 256": (dict(q_lens=[70, 4], k_lens=[6000, 5000], hq=4, hk=2, d=256, qbs=64, kbs=64, keep=0.3), (4, 1, True)),
}
ALL = pytest.mark.parametrize("form", list(FORMS))


def _problem(form, seed=101, **over):
    size, (nw, teams, cut) = FORMS[form]
    w = make_problem(seed=seed, **dict(dict(size, diag=True, causal=True, scale=None), **over))
    got = plan_for(w)
    assert got[:2] == (nw, teams) and (got[2] > 1) == cut
    print(f"{form} {over}", flush=True)
    return w


@ALL
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("causal,scale", [(True, -0.1), (False, None), (False, -0.2)])
def test_options(form, dtype, causal, scale):
    w = _problem(form, dtype=dtype, causal=causal, scale=scale)
    out = HBSAttention(*w.args())
    assert_close_to_oracle(out, oracle_for(w), form)
    # rows, heads and elements apart by more than the shape says; the same bits
    def spread(t):
        x = torch.zeros(t.shape[0], t.shape[1] + 3, t.shape[2] + 24, dtype=t.dtype, device=t.device)
        x[:, 1:1 + t.shape[1], 8:8 + t.shape[2]] = t
        return x[:, 1:1 + t.shape[1], 8:8 + t.shape[2]]
    apart = dataclasses.replace(w, q=spread(w.q), k=spread(w.k), v=spread(w.v))
    assert not apart.q.is_contiguous()
    assert torch.equal(HBSAttention(*apart.args()), out)


@ALL
def test_captured(form):
    w = _problem(form)
    args = list(w.args())
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        HBSAttention(*args)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = HBSAttention(*args)
    for step in range(4):   # every replay is checked, with eager work between
        if step:
            w.q.copy_(torch.randn_like(w.q))
            w.v.mul_(-0.5)
            w.block_mask.copy_(torch.rand(w.block_mask.shape, device="cuda") < 0.5)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(captured, HBSAttention(*args)), f"replay {step}"
        torch.cuda.synchronize()


@ALL
def test_two_streams_at_once(form):
    problems = [_problem(form, seed=101 + i) for i in range(2)]
    want = [HBSAttention(*w.args()) for w in problems]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in problems]
    outs = [[], []]
    for _ in range(8):
        for i, w in enumerate(problems):
            with torch.cuda.stream(streams[i]):
                outs[i].append(HBSAttention(*w.args()))
    torch.cuda.synchronize()
    assert all(torch.equal(o, want[i]) for i in range(2) for o in outs[i])


@pytest.mark.parametrize("form", ["sole", "teams", "teams 128", "teams packed", "split", "split 128", "split packed"])
def test_gradients(form):
    w = _problem(form)
    plain = HBSAttention(*w.args())
    dout = torch.randn(w.q.shape, generator=torch.Generator().manual_seed(5)).to(w.q.dtype).cuda()
    leaves = [t.detach().clone().requires_grad_(True) for t in (w.q, w.k, w.v)]
    out = HBSAttention(*leaves, *w.args()[3:])
    assert torch.equal(out.detach(), plain)
    grads = torch.autograd.grad(out, leaves, dout)
    want = hbsa_oracle_grads(w.q.cpu(), w.k.cpu(), w.v.cpu(), dout.cpu(), w.cu_q, w.cu_k, w.block_mask.cpu(), w.q_block_size, w.k_block_size, True, None)
    for name, got, ref in zip("qkv", grads, want):   # (bf16 operands against fp32: as in the other tests of the gradients)
        err = (got.float().cpu() - ref).abs()
        assert err.max() <= 1e-2 * max(1.0, ref.abs().max().item()), (name, err.max())
        assert err.mean() <= max(2e-3, 1e-2 * ref.abs().mean().item()), (name, err.mean())


@pytest.mark.parametrize("form", ["sole", "teams", "teams 128", "teams packed", "split", "split 128", "split 256", "split packed"])
def test_log_sum_exp(form):
    w = _problem(form, causal=False)
    w.block_mask[0, -1] = False   # rows that see no key
    a = w.args()
    nq, _, q2b, cu_nq, nk, _, _, cu_nk = a[11:19]
    prepared = hbsa_prepare(*a[3:9], nq, q2b, cu_nq, nk, cu_nk, run_shape=(w.q.dtype, w.q.shape[0], w.k.shape[0], w.q.shape[1], w.q.shape[2]))
    out, lse = hbsa_run(w.q, w.k, w.v, prepared, None, return_lse=True)
    assert torch.equal(out, HBSAttention(*a))
    ratio = w.q.shape[1] // w.k.shape[1]
    g = kb = 0
    for b in range(len(w.cu_q) - 1):
        rows, keys = slice(w.cu_q[b], w.cu_q[b + 1]), slice(w.cu_k[b], w.cu_k[b + 1])
        n, m = rows.stop - rows.start, keys.stop - keys.start
        qb, nb = -(-n // w.q_block_size), -(-m // w.k_block_size)
        for h in range(w.q.shape[1]):
            seen = w.block_mask[h // ratio, g:g + qb, kb:kb + nb].cpu().repeat_interleave(w.q_block_size, 0)[:n].repeat_interleave(w.k_block_size, 1)[:, :m]
            s = (w.q[rows, h].double().cpu() @ w.k[keys, h // ratio].double().cpu().T) * w.q.shape[2] ** -0.5
            ref = torch.logsumexp(s.masked_fill(~seen, float("-inf")), 1)
            got = lse[rows, h].double().cpu()
            assert torch.equal(torch.isneginf(got), torch.isneginf(ref))
            fine = torch.isfinite(ref)
            assert ((got - ref)[fine].abs() < 1e-4).all()   # exact products, fp32 sums of up to 6000 terms in a logarithm: 6000 * 2^-24 at most
        g, kb = g + qb, kb + nb

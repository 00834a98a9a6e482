"""The fp32 kernel forms its products from three bf16 parts of every operand.  Elements that have no such parts (infinities, and
floats that round to an infinite bf16) send a wavefront's rows through the fp32 matrix instructions: its results are those of fp32
arithmetic.  Compared with a dense float64 product of the same operands, whose infinities and NaNs are where fp32's are."""
import pytest
import torch

from hbsattn_amd.workloads import make_problem

pytestmark = pytest.mark.gpu

INF, NAN = float("inf"), float("nan")
MOST = torch.finfo(torch.float32).max   # rounds to an infinite bf16


def _run(w):
    from hbsattn_amd import HBSAttention
    return HBSAttention(*w.args()).cpu().double()


def _dense(w, d, hq, hk, n, causal):
    """Everything kept, one sequence of n tokens."""
    q, k, v = w.q.cpu().double(), w.k.cpu().double(), w.v.cpu().double()
    out = torch.zeros_like(q)
    for h in range(hq):
        s = (q[:, h, :, None] * k[:, h * hk // hq].T[None]).sum(1) * d ** -0.5   # (sums, so that an infinity meets every factor)
        if causal:
            s = s.masked_fill(torch.arange(n)[None] > torch.arange(n)[:, None], -INF)
        p = torch.exp(s - s.amax(1, keepdim=True))
        out[:, h] = (p[:, :, None] * v[None, :, h * hk // hq]).sum(1) / p.sum(1, keepdim=True)
    return out


def _compare(got, want):
    want = torch.where(want.abs() > MOST, want.float().double(), want)
    for f in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(f(got), f(want)), (f.__name__, int(f(got).sum()), int(f(want).sum()))
    fine = torch.isfinite(want)
    # fp32 sums of up to 80 terms: 80 * 2^-24 of the largest term
    assert ((got - want)[fine].abs() <= 5e-6 * want[fine].abs().clamp(min=1.0)).all()


@pytest.mark.parametrize("d", [32, 64, 128, 256])
@pytest.mark.parametrize("where,value", [("v", INF), ("v", -INF), ("v", MOST), ("k", INF), ("k", NAN), ("q", INF), ("v", NAN)])
def test_values_without_finite_parts(d, where, value):
    n, hq, hk = 80, 2, 1
    w = make_problem(seed=d, q_lens=[n], k_lens=[n], hq=hq, hk=hk, d=d, qbs=16, kbs=16, keep=1.0, diag=True, causal=True,
                     scale=None, dtype=torch.float32)
    t = getattr(w, where)
    t[50, 0, 3] = value
    got, want = _run(w), _dense(w, d, hq, hk, n, True)
    assert torch.isfinite(got[:48]).all()   # rows whose q blocks do not reach key 50 (the dense product has 0 * inf there)
    _compare(got[48:], want[48:])


def test_a_key_of_negative_infinity_drops_out():
    """-inf times positive queries: the key's weight is zero, the others' results are what they are without it."""
    n, d = 64, 64
    w = make_problem(seed=3, q_lens=[n], k_lens=[n], hq=1, hk=1, d=d, qbs=64, kbs=64, keep=1.0, diag=True, causal=False,
                     scale=None, dtype=torch.float32)
    w.q.abs_()
    w.k[10, 0, :] = 0.0
    w.k[10, 0, 5] = -INF
    got, want = _run(w), _dense(w, d, 1, 1, n, False)
    assert torch.isfinite(want).all()
    _compare(got, want)

"""Calls without block metadata whose one launch counts the blocks itself: batches around a wavefront's 64 lanes, either side given, empty
sequences, head dims of every kernel, masks that do not fit, calls that take another route."""
import pytest
import torch

from hbsattn_amd import HBSAttention, _lib, calculate_blocks
from hbsattn_amd.workloads import make_problem
from helpers import assert_close_to_oracle, oracle_for

pytestmark = pytest.mark.gpu


def _call(args):
    return _lib.host().call(*args, _lib.DTYPE_F32)


@pytest.mark.parametrize("batch", [1, 2, 63, 64, 65, 126, 127, 128])   # 128: two launches
@pytest.mark.parametrize("d,qbs,kbs", [(32, 16, 48), (128, 64, 32)])
def test_either_side_counted(batch, d, qbs, kbs):
    q_lens, k_lens = [(7 * i) % 50 for i in range(batch)], [1 + (11 * i) % 70 for i in range(batch)]
    q_lens[batch // 2] = 33
    w = make_problem(seed=batch, q_lens=q_lens, k_lens=k_lens, hq=4, hk=2, d=d, qbs=qbs, kbs=kbs, keep=0.7, diag=True, causal=True, scale=None)
    full, none = w.args(), w.args(with_meta=False)
    print(f"counted {batch} {d}", flush=True)
    out = HBSAttention(*full)
    assert_close_to_oracle(out, oracle_for(w), f"{batch} sequences")
    for args in (none, full[:15] + (None,) * 4, full[:11] + (None,) * 4 + full[15:]):
        args = tuple(args) + (None,) * (19 - len(args))
        if args[10] is None:
            args = args[:10] + ("auto",) + args[11:]
        got = _call(args)
        assert got is not None and torch.equal(got, out)


@pytest.mark.parametrize("d", [40, 64, 96, 160, 192, 256])
def test_every_kernel(d):
    w = make_problem(seed=d, q_lens=[33, 100], k_lens=[60, 100], hq=4, hk=2, d=d, qbs=48, kbs=16, keep=0.6, diag=True, causal=False, scale=None)
    assert torch.equal(HBSAttention(*w.args(with_meta=False)), HBSAttention(*w.args()))


def test_a_mask_that_does_not_fit_is_reported():
    w = make_problem(seed=5, q_lens=[100, 70], k_lens=[100, 70], hq=2, hk=2, d=64, qbs=32, kbs=32, keep=0.6, diag=True, causal=True, scale=None)
    args = list(w.args(with_meta=False))
    for shape in ((2, 8, 7), (2, 7, 8), (2, 6, 7), (2, 7, 6)):
        args[5] = torch.ones(shape, dtype=torch.bool, device="cuda")
        with pytest.raises(AssertionError):
            HBSAttention(*args)
    args[5] = w.block_mask
    assert_close_to_oracle(HBSAttention(*args), oracle_for(w), "after refused ones")


@pytest.mark.parametrize("kw", [dict(q_lens=[1, 1], k_lens=[900, 500], hq=8, hk=2, d=128, qbs=16, kbs=64),     # few queries a block
                                dict(q_lens=[60], k_lens=[9000], hq=4, hk=2, d=64, qbs=64, kbs=64),            # split
                                dict(q_lens=[60], k_lens=[90], hq=4, hk=2, d=64, qbs=64, kbs=64, dtype=torch.float32)])
def test_other_routes(kw):
    w = make_problem(seed=7, keep=0.6, diag=True, causal=True, scale=None, **kw)
    assert torch.equal(HBSAttention(*w.args(with_meta=False)), HBSAttention(*w.args()))

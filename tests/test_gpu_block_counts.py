"""Block geometry on the device (``hbsa_block_counts``, ``hbsa_block_arrays``) and calls that leave it to the operator,
at batch sizes around one wavefront, one workgroup and several passes of it."""
import pytest
import torch

from hbsattn_amd import HBSAttention, calculate_blocks
from hbsattn_amd.workloads import make_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [1, 2, 63, 64, 65, 255, 256, 257, 700])
@pytest.mark.parametrize("block_size", [16, 80, 4096])
def test_device_arrays_equal_the_host_ones(batch, block_size):
    lens = torch.randint(0, 300, (batch,), generator=torch.Generator().manual_seed(batch))   # empty sequences among them
    lens[-1] = 0 if batch > 2 else 7
    cu = torch.cat([torch.zeros(1, dtype=torch.int64), lens.cumsum(0)]).to(torch.int32)
    host, dev = calculate_blocks(cu, block_size), calculate_blocks(cu.cuda(), block_size)
    assert host[0] == dev[0]
    for a, b in zip(host[1:], dev[1:]):
        assert b.is_cuda and a.dtype == b.dtype and torch.equal(a, b.cpu())


@pytest.mark.parametrize("given", ["none", "queries", "keys"])
@pytest.mark.parametrize("n_seq", [3, 130])   # one launch, and two (more sequences than that form holds)
def test_calls_without_metadata_equal_calls_with_it(given, n_seq):
    w = make_problem(seed=5, q_lens=[40] * n_seq, k_lens=[70] * n_seq, hq=4, hk=2, d=64, qbs=32, kbs=48, keep=0.6, diag=True,
                     causal=True, scale=None)
    base, none = w.args(with_meta=False), (None,) * 4
    meta = {"none": (), "queries": ("auto",) + tuple(w.q_meta) + none, "keys": ("auto",) + none + tuple(w.k_meta)}[given]
    assert torch.equal(HBSAttention(*base, *meta), HBSAttention(*w.args()))


def test_a_mask_that_does_not_fit_the_counts_is_reported():
    w = make_problem(seed=6, q_lens=[100, 30], k_lens=[100, 30], hq=2, hk=2, d=32, qbs=32, kbs=32, keep=0.6, diag=True, causal=True,
                     scale=None)
    args = list(w.args(with_meta=False))
    args[5] = w.block_mask[:, :, :-1].contiguous()
    with pytest.raises(AssertionError, match=r"\(nheads_k, num_q_block, num_k_block\) = \(2, 5, 5\)"):
        HBSAttention(*args)
    args[5] = w.block_mask
    assert torch.equal(HBSAttention(*args), HBSAttention(*w.args()))

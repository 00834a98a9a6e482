"""The decode kernel where items have more than 16 entries: several groups of 16 in a wavefront, their parts combined by a
launch of its own."""
import pytest
import torch

from hbsattn_amd import HBSAttention, _lib
from hbsattn_amd.interface import hbsa_prepare, hbsa_run
from hbsattn_amd.workloads import make_problem
from helpers import assert_close_to_oracle, oracle_for
from oracle.dense import hbsa_oracle

pytestmark = pytest.mark.gpu


def _problem(d, q_lens, k_lens, hq, hk, kbs, causal=True, dtype=torch.bfloat16, seed=0, **kw):
    w = make_problem(seed=seed + d + kbs, q_lens=q_lens, k_lens=k_lens, hq=hq, hk=hk, d=d, qbs=16, kbs=kbs, keep=0.5, diag=True,
                     causal=causal, scale=None, dtype=dtype, **kw)
    code = _lib.DTYPE_F16 if dtype == torch.float16 else _lib.DTYPE_BF16
    assert _lib.load().hbsa_fwd_decodes(code, w.q.shape[0], hq, hk, w.q_meta[0], w.k_meta[0], 16, kbs) == 1
    return w


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [32, 64, 128, 256])
@pytest.mark.parametrize("q_lens,k_lens,hq,hk,kbs,causal", [
    ([1] * 9 + [16], [200] * 9 + [5000], 8, 2, 64, True),            # 64 entries: four groups, or two walks of two
    ([1] * 9 + [16], [200] * 9 + [5000], 2, 1, 16, False),           # 32
    ([1, 1, 1, 13, 1, 1], [70, 900, 3000, 2500, 1, 16], 3, 1, 48, True),   # 39: the last group with seven
    ([1] * 12 + [40], [64] * 12 + [3000], 4, 1, 32, True),           # blocks of 16, 16 and 8 rows in one sequence
    ([2, 1, 5, 1, 1, 1], [40, 2, 17, 1, 300, 8], 4, 2, 16, True),    # one part each, rows before the first key
    ([1] * 70 + [11], [64] * 71, 4, 1, 64, False),                   # more sequences than a wavefront has lanes
])
def test_groups_match_the_oracle(dtype, d, q_lens, k_lens, hq, hk, kbs, causal):
    w = _problem(d, q_lens, k_lens, hq, hk, kbs, causal, dtype)
    out = HBSAttention(*w.args())
    assert_close_to_oracle(out, oracle_for(w), "groups")
    for _ in range(2):
        assert torch.equal(HBSAttention(*w.args()), out)
    meta = (w.q_meta[0], w.q_meta[2], w.q_meta[3], w.k_meta[0], w.k_meta[3])
    prepared = hbsa_prepare(w.cu_q_seqlens, w.cu_k_seqlens, w.block_mask, 16, kbs, causal, *meta,
                            run_shape=(w.q.dtype, w.q.shape[0], w.k.shape[0], hq, d))
    got, lse = hbsa_run(w.q, w.k, w.v, prepared, None, return_lse=True)
    assert torch.equal(got, out)
    _, ref_lse = hbsa_oracle(w.q.cpu(), w.k.cpu(), w.v.cpu(), w.cu_q, w.cu_k, w.block_mask.cpu(), 16, kbs, causal, None, return_lse=True)
    seen = torch.isfinite(ref_lse)
    assert torch.equal(torch.isfinite(lse.cpu()), seen) and (lse.cpu()[seen] - ref_lse[seen]).abs().max().item() <= 2e-3


def test_groups_can_be_captured_and_replayed():
    w = _problem(128, [1] * 6 + [9], [4000, 700, 9000, 50, 64, 1, 6000], 8, 2, 64)
    args = w.args()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        HBSAttention(*args)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = HBSAttention(*args)
    for step in range(4):
        w.q.mul_(-0.5)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(captured, HBSAttention(*args)), f"replay {step}"
        torch.cuda.synchronize()


@pytest.mark.parametrize("q_lens,hq", [([1, 1, 1], 2), ([1] * 9 + [16], 8)])
def test_an_infinite_value_stays_infinite(q_lens, hq):
    """Parts that are combined sixteen at a time: what fills the last sixteen up is not multiplied in."""
    w = _problem(64, q_lens, [5000] * len(q_lens), hq, 2, 64, causal=False)
    w.block_mask.fill_(True)
    token = w.cu_k[-1] - 2   # in the last part of the last sequence, inside a whole tile
    w.v[token, :, 5] = float("inf")
    out = HBSAttention(*w.args()).float()
    last = w.cu_q[-2]
    assert torch.isinf(out[last:, :, 5]).all()
    out[last:, :, 5] = 0.0
    assert torch.isfinite(out).all()


@pytest.mark.parametrize("blocks_each", [1, 6, 40])
def test_parts_follow_the_mean_length(blocks_each):
    """64 single queries, 32 / 8 heads of 128: no more room, and so no more workgroups, for parts than items of six times
    the mean number of k blocks (eight times with less than two items a compute unit) can have."""
    part_bytes = 64 * 32 * (128 + 2) * 4
    room = _lib.load().hbsa_fwd_parts_bytes(_lib.DTYPE_BF16, 64, 32, 8, 128, 64, 64 * blocks_each, 16)
    assert part_bytes < room <= min(32, 8 * blocks_each) * part_bytes + 8192

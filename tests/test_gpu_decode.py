"""The decode kernel (few queries per kv head and q block): tiles of two 16-key groups, parts, several passes of 16 entries."""
import pytest
import torch

from hbsattn_amd import HBSAttention
from hbsattn_amd.interface import hbsa_prepare, hbsa_run
from hbsattn_amd.workloads import make_problem
from helpers import assert_close_to_oracle, oracle_for
from oracle.dense import hbsa_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [32, 64, 128, 256])
@pytest.mark.parametrize("q_lens,k_lens,hq,hk,kbs,causal", [
    ([1], [1], 1, 1, 16, True),                                   # one key
    ([1, 1, 1], [17, 40, 3000], 4, 1, 16, True),                  # odd groups, items of one part and of many
    ([2, 5, 1], [100, 2000, 31], 8, 2, 48, True),                 # up to 20 entries: a second pass
    ([16, 1, 1, 1], [900, 70, 5000, 8], 4, 4, 128, False),        # 16 rows in one block, one in others
    ([1, 3], [40, 2], 2, 1, 32, True),                            # queries before the first key: rows without keys
    ([1] * 70, [64] * 70, 2, 2, 64, True),                        # more sequences than a wavefront has lanes
])
def test_decode_matches_the_oracle(dtype, d, q_lens, k_lens, hq, hk, kbs, causal):
    w = make_problem(seed=d + kbs, q_lens=q_lens, k_lens=k_lens, hq=hq, hk=hk, d=d, qbs=16, kbs=kbs, keep=0.5, diag=True, causal=causal,
                     scale=None, dtype=dtype)
    out = HBSAttention(*w.args())
    assert_close_to_oracle(out, oracle_for(w), "decode")
    for _ in range(3):   # whoever arrives last combines in the same order
        assert torch.equal(HBSAttention(*w.args()), out)
    meta = (w.q_meta[0], w.q_meta[2], w.q_meta[3], w.k_meta[0], w.k_meta[3])
    prepared = hbsa_prepare(w.cu_q_seqlens, w.cu_k_seqlens, w.block_mask, 16, kbs, causal, *meta,
                            run_shape=(w.q.dtype, w.q.shape[0], w.k.shape[0], hq, d))
    got, lse = hbsa_run(w.q, w.k, w.v, prepared, None, return_lse=True)
    assert torch.equal(got, out)
    _, ref_lse = hbsa_oracle(w.q.cpu(), w.k.cpu(), w.v.cpu(), w.cu_q, w.cu_k, w.block_mask.cpu(), 16, kbs, causal, None, return_lse=True)
    seen = torch.isfinite(ref_lse)
    assert torch.equal(torch.isfinite(lse.cpu()), seen) and (lse.cpu()[seen] - ref_lse[seen]).abs().max().item() <= 2e-3


def test_decode_can_be_captured_and_replayed():
    w = make_problem(seed=3, q_lens=[1, 2, 1, 1], k_lens=[4000, 700, 9000, 50], hq=8, hk=2, d=128, qbs=16, kbs=64, keep=0.5, diag=True,
                     causal=True, scale=None)
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

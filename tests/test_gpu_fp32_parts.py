"""The fp32 kernel where its items are cut into parts and combined, and at the edges of its 16-key groups and tiles."""
import pytest
import torch

from hbsattn_amd import HBSAttention
from hbsattn_amd.interface import hbsa_prepare, hbsa_run
from hbsattn_amd.workloads import make_problem
from helpers import assert_close_to_oracle, oracle_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [32, 64, 128, 256])
@pytest.mark.parametrize("q_lens,k_lens,hq,hk,qbs,kbs,causal", [
    ([1], [1], 1, 1, 16, 16, True),                       # one entry, one key
    ([33, 5], [257, 700], 4, 2, 16, 16, False),           # 16-key blocks, a last group of one key
    ([100, 290], [1000, 333], 6, 2, 80, 48, True),        # packed slots, 48-key blocks, q longer than its visible keys
    ([700], [2500], 2, 1, 128, 128, False),               # parts of several windows' blocks
    ([40], [5000], 8, 8, 32, 16, True),                   # 313 blocks: the second window of 64 and later ones
    ([900, 700], [900, 700], 12, 12, 16, 64, True),       # more than two items per CU: whole items
])
def test_items_in_parts_match_the_oracle(d, q_lens, k_lens, hq, hk, qbs, kbs, causal):
    w = make_problem(seed=d + qbs, q_lens=q_lens, k_lens=k_lens, hq=hq, hk=hk, d=d, qbs=qbs, kbs=kbs, keep=0.5, diag=True,
                     causal=causal, scale=None, dtype=torch.float32)
    out = HBSAttention(*w.args())
    assert_close_to_oracle(out, oracle_for(w), "fp32")
    for _ in range(3):   # whoever arrives last combines in the same order
        assert torch.equal(HBSAttention(*w.args()), out)
    # the prepared form walks the same parts
    meta = (w.q_meta[0], w.q_meta[2], w.q_meta[3], w.k_meta[0], w.k_meta[3])
    prepared = hbsa_prepare(w.cu_q_seqlens, w.cu_k_seqlens, w.block_mask, qbs, kbs, causal, *meta,
                            run_shape=(w.q.dtype, w.q.shape[0], w.k.shape[0], hq, d))
    assert torch.equal(hbsa_run(w.q, w.k, w.v, prepared, None), out)

"""Partial results of a forward split over key blocks, put together: parts around the numbers that are asked for at once, rows that
see keys in some parts only or in none, the log-sum-exp."""
import pytest
import torch

from hbsattn_amd import HBSAttention, _lib
from hbsattn_amd.interface import hbsa_prepare, hbsa_run
from hbsattn_amd.workloads import make_problem
from helpers import assert_close_to_oracle, oracle_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [32, 64, 128, 256])
@pytest.mark.parametrize("k_blocks", [64, 96, 200, 256, 272, 288, 512, 544, 1100])   # from few parts to the most
def test_merged_parts(k_blocks, d):
    w = make_problem(seed=41 + k_blocks, q_lens=[40, 3], k_lens=[k_blocks * 64 - 5, 700], hq=4, hk=2, d=d, qbs=64, kbs=64, keep=0.1,
                     diag=False, causal=False, scale=None)
    w.block_mask[0, 0, : k_blocks - 1] = False   # one head: the first sequence sees its last block only, the other sequence nothing
    w.block_mask[0, 0, k_blocks - 1] = True
    w.block_mask[0, 1] = False
    print(f"merge {k_blocks} {d}", flush=True)
    a = w.args()
    cq, ck, mask, qbs, kbs, causal = a[3:9]
    nq, _, q2b, cu_nq, nk, _, _, cu_nk = a[11:19]
    prepared = hbsa_prepare(cq, ck, mask, qbs, kbs, causal, nq, q2b, cu_nq, nk, cu_nk, run_shape=(w.q.dtype, *w.q.shape[:1], w.k.shape[0],
                                                                                                  w.q.shape[1], d))
    out, lse = hbsa_run(w.q, w.k, w.v, prepared, None, return_lse=True)
    assert_close_to_oracle(out, oracle_for(w), f"{k_blocks} key blocks")
    assert out[40:, :2].abs().max() == 0 and torch.isinf(lse[40:, :2]).all() and torch.isfinite(lse[:40]).all()
    # the prepared form and the one-launch form cut the items by themselves, and make the same parts
    assert _lib.load().hbsa_fwd_launches(_lib.DTYPE_BF16, 2, w.k.shape[0], 4, 2, d, int(nq), int(nk), 64, 64, 0, None) > 1
    assert torch.equal(HBSAttention(*a), out)
    again, lse2 = hbsa_run(w.q, w.k, w.v, prepared, None, return_lse=True)
    assert torch.equal(out, again) and torch.equal(lse, lse2)
    scores = torch.einsum("qhd,khd->hqk", w.q[:40].double().cpu()[:, 2:], w.k[: k_blocks * 64 - 5].double().cpu()[:, 1:].expand(-1, 2, -1)) * d ** -0.5
    seen = mask[1, 0, :k_blocks].cpu().repeat_interleave(64)[: k_blocks * 64 - 5]
    ref = torch.logsumexp(scores.masked_fill(~seen, float("-inf")), dim=-1).T
    assert (lse[:40, 2:].double().cpu() - ref).abs().max() < 1e-3   # bf16 products are exact in fp32; 70000 fp32 terms

"""The forms of the dK/dV kernel at head dim 128: the rule's two sides, 32-row tiles with odd ends, blocks of more than 64 keys over several
workgroups, few items in parts and whole, tile lists of several chunks, sequences that do not fit the tensors."""
import pytest
import torch

from hbsattn_amd.interface import hbsa_backward, hbsa_run
from oracle.grads import hbsa_oracle_grads
from test_gpu_backward import _check, _problem
from test_gpu_backward_tile_list import _prepare, _whole

pytestmark = pytest.mark.gpu

CASES = [
    # q_lens, k_lens, hq, hk, qbs, kbs, keep, causal
    ([130, 65, 200], [700, 300, 1100], 32, 32, 64, 64, 0.6, True),      # 1088 items of 64 keys: four wavefronts each
    ([90, 33], [410, 100], 64, 64, 48, 16, 0.5, False),                 # 2112 items of 16 keys
    ([130, 65, 200], [700, 300, 1000], 30, 30, 64, 64, 0.6, True),      # 960: eight
    ([333, 100], [200, 500], 4, 2, 80, 128, 0.7, True),                 # blocks of 128 keys, two workgroups each, in parts
    ([333, 100], [200, 500], 2, 1, 16, 160, 0.7, False),                # three workgroups a block, the last of 32 keys
    ([97, 500], [97, 500], 8, 8, 32, 96, 0.9, True),
    ([12900], [130], 4, 1, 16, 128, 1.1, False),                        # 3228 tiles of 16 rows: thirteen chunks
    ([300, 65], [300, 65], 12, 12, 208, 80, 0.8, True),
]


@pytest.mark.parametrize("case", CASES, ids=[f"case{i}" for i in range(len(CASES))])
def test_gradients_of_every_form(case):
    q_lens, k_lens, hq, hk, qbs, kbs, keep, causal = case
    q, k, v, do, cu_q, cu_k, cq, ck, mask = _problem(23, q_lens, k_lens, hq, hk, 128, qbs, kbs, keep, torch.bfloat16)
    print(f"form {case}", flush=True)
    qd, kd, vd, dod = (t.cuda().contiguous() for t in (q, k, v, do))
    prepared, nq, nk = _prepare(cq, ck, mask, qbs, kbs, causal)
    out, lse = hbsa_run(qd, kd, vd, prepared, None, return_lse=True)
    refs = hbsa_oracle_grads(q, k, v, do, cu_q, cu_k, mask, qbs, kbs, causal, None)
    for got in (_whole(qd, kd, vd, out, dod, lse, ck, prepared, nq, nk, qbs, kbs, causal),
                hbsa_backward(qd, kd, vd, out, dod, lse, prepared, None)):
        for x, ref, name in zip(got, refs, ("dq", "dk", "dv")):
            _check(x, ref, name)


@pytest.mark.parametrize("hk,qbs,kbs", [(32, 64, 64), (2, 80, 128), (2, 64, 64), (2, 64, 128)])
def test_keys_of_sequences_that_do_not_fit_get_zeros(hk, qbs, kbs):
    # the second sequence's queries end beyond q: it is skipped as a whole, and every element of its dk and dv is written
    k_lens = [1100, 1000]
    q, k, v, do, cu_q, cu_k, cq, ck, mask = _problem(29, [200, 150], k_lens, hk, hk, 128, qbs, kbs, 1.1, torch.bfloat16)
    from hbsattn_amd import calculate_blocks
    from hbsattn_amd.interface import hbsa_prepare
    (nq, _, q2b, cu_nq), (nk, _, _, cu_nk) = calculate_blocks(cq, qbs), calculate_blocks(ck, kbs)
    rows = 300
    qd, dod = q[:rows].cuda().contiguous(), do[:rows].cuda().contiguous()
    kd, vd = k.cuda(), v.cuda()
    prepared = hbsa_prepare(cq, ck, mask.cuda(), qbs, kbs, False, nq, q2b, cu_nq, nk, cu_nk,
                            run_shape=(q.dtype, rows, kd.shape[0], hk, 128))
    assert prepared.skipped_q_blocks() > 0
    out, lse = hbsa_run(qd, kd, vd, prepared, None, return_lse=True)
    junk = torch.full((4, *kd.shape), 7.0, device="cuda")   # what the allocator hands out next is not zero
    del junk
    _, dk, dv = hbsa_backward(qd, kd, vd, out, dod, lse, prepared, None)
    assert dk[1100:].abs().max() == 0 and dv[1100:].abs().max() == 0 and dk[:1100].abs().max() > 0

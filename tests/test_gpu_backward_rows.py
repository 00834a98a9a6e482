"""Rows that the backward reads and writes sixteen to an instruction: blocks and sequences whose 32-row slots end in the first or
second sixteen rows, token and head strides of every tensor, rows beyond a block's end left as they were."""
import pytest
import torch

from hbsattn_amd import calculate_blocks
from hbsattn_amd.interface import hbsa_backward, hbsa_prepare, hbsa_run
from oracle.grads import hbsa_oracle_grads
from test_gpu_backward import _check, _problem

pytestmark = pytest.mark.gpu


def _strided(t, pad):
    """The same rows in a tensor with other token and head strides."""
    room = torch.full((t.shape[0], t.shape[1] + pad, t.shape[2] + 8 * pad), 9.0, dtype=t.dtype, device="cuda")
    view = room[:, :t.shape[1], :t.shape[2]]
    view.copy_(t)
    return view


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("lens,qbs,kbs", [(([1, 15, 16], [16, 17, 1]), 16, 16), (([17, 31, 47], [33, 48, 49]), 48, 48),
                                          (([129, 80], [97, 145]), 80, 96), (([64, 200], [130, 191]), 128, 128)])
def test_rows_at_the_edges_of_a_slot(lens, qbs, kbs, d):
    q, k, v, do, cu_q, cu_k, cq, ck, mask = _problem(17, lens[0], lens[1], 4, 2, d, qbs, kbs, 0.8, torch.float16)
    print(f"rows {lens} {qbs} {kbs} {d}", flush=True)
    (nq, _, q2b, cu_nq), (nk, _, _, cu_nk) = calculate_blocks(cq, qbs), calculate_blocks(ck, kbs)
    prepared = hbsa_prepare(cq, ck, mask.cuda(), qbs, kbs, True, nq, q2b, cu_nq, nk, cu_nk)
    qd, kd, vd, dod = _strided(q, 1), _strided(k, 2), _strided(v, 3), _strided(do, 1)
    out, lse = hbsa_run(qd, kd, vd, prepared, None, return_lse=True)
    refs = hbsa_oracle_grads(q, k, v, do, cu_q, cu_k, mask, qbs, kbs, True, None)
    got = hbsa_backward(qd, kd, vd, _strided(out, 2), dod, lse, prepared, None)
    for x, ref, name in zip(got, refs, ("dq", "dk", "dv")):
        _check(x, ref, name)

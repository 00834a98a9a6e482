"""Gradients of keys and queries that nothing reaches: they are written as zeros, whatever the buffers held."""
import pytest
import torch

from hbsattn_amd import calculate_blocks
from hbsattn_amd.interface import hbsa_backward, hbsa_prepare, hbsa_run
from oracle.grads import hbsa_oracle_grads
from test_gpu_backward import _check, _problem

pytestmark = pytest.mark.gpu


@pytest.fixture
def filled(monkeypatch):
    """Buffers the backward is to write hold sevens before it does."""
    monkeypatch.setattr(torch, "empty_like", lambda t: torch.full_like(t, 7.0))


# the last sequences have keys and no queries; items cut into parts (few heads) and whole; wavefronts that share a key slot or not
@pytest.mark.parametrize("hq,hk", [(2, 1), (64, 64)], ids=["few", "many"])
@pytest.mark.parametrize("d,kbs", [(32, 32), (64, 64), (64, 96), (128, 64), (128, 160)])
def test_keys_of_last_sequences_without_queries_get_zeros(d, kbs, hq, hk, filled):
    q_lens, k_lens = [130, 0, 70, 0, 0], [700, 90, 333, 400, 65]
    q, k, v, do, cu_q, cu_k, cq, ck, mask = _problem(21, q_lens, k_lens, hq, hk, d, 64, kbs, 0.6, torch.bfloat16)
    print(f"backward, last sequences without queries, d={d} kbs={kbs} heads {hq}/{hk}", flush=True)
    qd, kd, vd, dod = (t.cuda() for t in (q, k, v, do))
    (nq, _, q2b, cu_nq), (nk, _, _, cu_nk) = calculate_blocks(cq, 64), calculate_blocks(ck, kbs)
    prepared = hbsa_prepare(cq, ck, mask.cuda(), 64, kbs, True, nq, q2b, cu_nq, nk, cu_nk)
    out, lse = hbsa_run(qd, kd, vd, prepared, None, return_lse=True)
    got = hbsa_backward(qd, kd, vd, out, dod, lse, prepared, None)
    for t in got[1:]:
        assert torch.count_nonzero(t[cu_k[3]:]) == 0 and torch.count_nonzero(t[cu_k[1]:cu_k[2]]) == 0
    for x, ref, name in zip(got, hbsa_oracle_grads(q, k, v, do, cu_q, cu_k, mask, 64, kbs, True, None), ("dq", "dk", "dv")):
        _check(x, ref, name)

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


def _grads(q, k, v, do, cq, ck, mask, kbs, nq, q2b, cu_nq):
    nk, _, _, cu_nk = calculate_blocks(ck, kbs)
    prepared = hbsa_prepare(cq, ck, mask, 64, kbs, True, nq, q2b, cu_nq, nk, cu_nk, run_shape=(q.dtype, q.shape[0], k.shape[0], q.shape[1], q.shape[2]))
    out, lse = hbsa_run(q, k, v, prepared, None, return_lse=True)
    return hbsa_backward(q, k, v, out, do, lse, prepared, None)


@pytest.mark.parametrize("heads", [2, 64], ids=["parts", "whole"])
@pytest.mark.parametrize("d,kbs", [(64, 96), (128, 64)])
def test_q_blocks_beyond_a_sequence_or_the_mask_take_no_part(d, kbs, heads, filled, monkeypatch):
    # block metadata that promises more q blocks than there are rows for: what no kernel has written (the bit rows of such
    # blocks, here all ones) is not taken for a mask, and nothing outside of the tensors and the workspace is looked at
    empty = torch.empty
    monkeypatch.setattr(torch, "empty", lambda *a, **kw: empty(*a, **kw).fill_(255) if kw.get("dtype") == torch.uint8 else empty(*a, **kw))
    q, k, v, do, cu_q, cu_k, cq, ck, mask = _problem(22, [300, 130], [333, 400], heads, heads, d, 64, kbs, 0.6, torch.bfloat16)
    print(f"backward, too many q blocks, d={d} kbs={kbs} heads {heads}", flush=True)
    qd, kd, vd, dod, maskd = (t.cuda() for t in (q, k, v, do, mask))
    nq, _, q2b, cu_nq = calculate_blocks(cq, 64)   # 5 and 3
    want = _grads(qd, kd, vd, dod, cq, ck, maskd, kbs, nq, q2b, cu_nq)
    # sequence 0 has 9 blocks, for 5 blocks' rows
    more_b = torch.tensor([0] * 9 + [1] * 3, dtype=torch.int32, device="cuda")
    more_cu = torch.tensor([0, 9, 12], dtype=torch.int32, device="cuda")
    more_mask = torch.cat([maskd[:, :5], torch.ones_like(maskd[:, :4]), maskd[:, 5:]], dim=1)
    assert all(torch.equal(a, b) for a, b in zip(want, _grads(qd, kd, vd, dod, cq, ck, more_mask, kbs, 12, more_b, more_cu)))
    # the last sequence's blocks end far beyond the mask's
    beyond = cu_nq.clone()
    beyond[-1] += 1000
    assert all(torch.equal(a, b) for a, b in zip(want, _grads(qd, kd, vd, dod, cq, ck, maskd, kbs, nq, q2b, beyond)))
    # ... of a sequence that does not fit k and v, too
    short = 333 + 350
    got = _grads(qd, kd[:short], vd[:short], dod, cq, ck, maskd, kbs, nq, q2b, beyond)
    assert torch.equal(got[0][:300], want[0][:300]) and torch.count_nonzero(got[0][300:]) == 0
    for a, b in zip(got[1:], want[1:]):
        assert torch.equal(a[:333], b[:333]) and torch.count_nonzero(a[333:]) == 0

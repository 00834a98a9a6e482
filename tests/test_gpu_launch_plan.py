"""Wavefronts, teams and parts of the attention launch: a form without kernels of two teams keeps the workgroups that suit it."""
import ctypes

import pytest
import torch

from hbsattn_amd import _lib

pytestmark = pytest.mark.gpu


def plan_of(prepared, dtype=_lib.DTYPE_BF16, *, batch, total_q, total_k, hq, hk, d, nqb, nkb, qbs, kbs):
    """(wavefronts of a team, teams, parts, items)"""
    sizes = (ctypes.c_int32 * 12)(dtype, batch, total_q, total_k, hq, hk, d, nqb, nkb, qbs, kbs, 1)
    plan = (ctypes.c_int32 * 4)()
    lib = _lib.load()
    assert lib.hbsa_fwd_plan(ctypes.addressof(sizes), int(prepared), ctypes.addressof(plan)) == 0, _lib.last_error()
    return tuple(plan)


def plan_for(w, prepared=False):
    code = {torch.bfloat16: _lib.DTYPE_BF16, torch.float16: _lib.DTYPE_F16}[w.q.dtype]
    return plan_of(prepared, code, batch=len(w.cu_q) - 1, total_q=w.q.shape[0], total_k=w.k.shape[0], hq=w.q.shape[1], hk=w.k.shape[1], d=w.q.shape[2],
                   nqb=w.q_meta[0], nkb=w.k_meta[0], qbs=w.q_block_size, kbs=w.k_block_size)


def test_forms_without_teams_keep_their_wavefronts():
    # eight q heads on one, 48-row blocks of 20 rows: 16 plain slots, twos of eight wavefronts; 12 packed ones, threes of four
    size = dict(batch=40, total_q=800, total_k=1600, hq=8, hk=1, d=128, nqb=40, nkb=40, qbs=48, kbs=64)
    lib = _lib.load()
    assert plan_of(True, **size) == (4, 2, 1, 120)
    assert plan_of(True, _lib.DTYPE_F32_STAGED16, **size) == (8, 1, 1, 80)
    deterministic, least = lib.hbsa_set_deterministic(0), lib.hbsa_set_walk_min_bytes(0)
    try:
        assert plan_of(True, **size) == (8, 1, 1, 80)   # the clocked walk
    finally:
        lib.hbsa_set_deterministic(deterministic)
        lib.hbsa_set_walk_min_bytes(least)
    # sequences of one block each: one launch leaves them to one team of packed slots
    assert plan_of(False, **size) == (4, 1, 1, 120)


@pytest.mark.parametrize("batch,q,k,hq,hk,qbs,kbs,plan", [
    (8, 342, 2919, 32, 2, 80, 16, (4, 1, 1, 800)),      # plain slots are too many to be cut, and the sequences too short for packed eights to be
    (9, 21, 856, 32, 2, 176, 48, (8, 1, 1, 198)),
    (4, 15, 1097, 64, 4, 48, 64, (4, 1, 4, 96)),        # ... which are cut as fours
    (3, 130, 2843, 64, 4, 16, 48, (4, 2, 1, 216)),      # many rows on short sequences
    (13, 9, 4407, 32, 2, 112, 64, (8, 1, 4, 182)),      # long ones
])
def test_packed_eights_are_cut_where_sequences_are_long(batch, q, k, hq, hk, qbs, kbs, plan):
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the numbers of items are for 256 compute units")
    size = dict(batch=batch, total_q=batch * q, total_k=batch * k, hq=hq, hk=hk, d=128, nqb=batch * -(-q // qbs), nkb=batch * -(-k // kbs), qbs=qbs, kbs=kbs)
    assert plan_of(False, **size) == plan
    assert plan_of(True, **size)[1:3] == plan[1:3]


@pytest.mark.parametrize("nqb,total_q,total_k,nkb,cut", [
    (16, 1016, 10264, 168, False),    # 8 x 127 queries on 1283 keys: 320 workgroups of four
    (16, 1016, 28160, 440, True),     # 88 keys to one of them
    (16, 1016, 28096, 439, False),
    (8, 243, 9728, 152, True),        # 0.8 rows of all heads to a key
    (8, 244, 9728, 152, False),
    (6, 381, 4200, 66, False),        # 120 workgroups
    (5, 381, 4200, 66, True),
])
@pytest.mark.parametrize("prepared", [False, True])
def test_many_rows_on_short_sequences_are_left_whole(nqb, total_q, total_k, nkb, cut, prepared):
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the numbers of items are for 256 compute units")
    plan = plan_of(prepared, batch=3, total_q=total_q, total_k=total_k, hq=32, hk=4, d=64, nqb=nqb, nkb=nkb, qbs=80, kbs=64)
    assert (plan[2] > 1) == cut

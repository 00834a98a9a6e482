"""Launches whose plan is cut over key blocks, in one launch and on a prepared mask: the plan is asserted, and both make the same bits."""
import dataclasses

import pytest
import torch

from hbsattn_amd import HBSAttention, _lib
from hbsattn_amd.workloads import make_problem
from helpers import assert_close_to_oracle, oracle_for
from test_gpu_launch_plan import plan_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("q_lens,k_lens,hq,hk,d,qbs,kbs,keep", [
    ([70, 4], [6000, 5000], 8, 2, 128, 128, 64, 0.4),       # workgroups of eight; slots packed over the heads, none left for some
    ([40, 3], [4091, 700], 4, 2, 64, 64, 64, 0.03),         # some items of fewer keys than a part, some of none
    ([130], [9000], 2, 1, 256, 64, 128, 0.5),
    ([129], [8200], 8, 1, 32, 80, 48, 0.9),                 # tiles of 16-key groups
    ([100], [150000], 2, 2, 32, 128, 64, 0.3),              # a row of more blocks than a window of mask bytes: cut by position
    ([60], [40000], 2, 1, 64, 64, 16, 0.3),                 # ... of groups
    ([512], [70000], 16, 16, 32, 32, 48, 1.0),              # parts of more groups than a list holds
    ([1300, 5], [5000, 40], 1, 1, 80, 64, 16, 0.5),         # head dims without a kernel of their own
    ([90, 128], [9000, 7000], 4, 2, 96, 128, 64, 0.3),
    ([90, 128], [9000, 7000], 4, 2, 192, 128, 96, 0.3),
    ([50], [12000], 8, 2, 160, 128, 32, 0.3),
    ([50], [6000], 2, 2, 24, 64, 64, 0.3),
    ([50], [6000], 2, 2, 208, 64, 64, 0.3),
])
def test_one_launch_and_prepared(q_lens, k_lens, hq, hk, d, qbs, kbs, keep):
    w = make_problem(seed=61, q_lens=q_lens, k_lens=k_lens, hq=hq, hk=hk, d=d, qbs=qbs, kbs=kbs, keep=keep, diag=False, causal=True,
                     scale=None)
    print(f"split {q_lens} {k_lens} {hq} {hk} {d} {qbs} {kbs}", flush=True)
    assert plan_for(w)[2] > 1
    lib = _lib.load()
    out = HBSAttention(*w.args())
    assert torch.equal(HBSAttention(*w.args()), out)
    before = lib.hbsa_set_onepass(0)
    try:
        prepared = HBSAttention(*w.args())
    finally:
        lib.hbsa_set_onepass(before)
    assert torch.equal(out, prepared)
    if hq > 8:   # one head is enough
        w = dataclasses.replace(w, q=w.q[:, :1], k=w.k[:, :1], v=w.v[:, :1], block_mask=w.block_mask[:1])
        out = out[:, :1]
    assert_close_to_oracle(out, oracle_for(w), "split")

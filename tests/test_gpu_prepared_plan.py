"""A prepared mask's launch of packed slots is the one that was planned: as many workgroups as the one-launch form, and its bits, where it is cut, has
teams, or would be cut with plain slots only."""
import pytest
import torch

from hbsattn_amd import HBSAttention, set_onepass
from hbsattn_amd.workloads import make_problem
from helpers import assert_close_to_oracle, oracle_for
from test_gpu_launch_plan import plan_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("q_lens,k_lens,hq,hk,d,qbs,kbs,plan", [
    ([4] * 7, [5365] * 7, 16, 2, 128, 80, 80, (4, 1, 7, 70)),         # cut: five fours, and not three eights of plain slots
    ([200, 90], [9000, 3000], 8, 1, 64, 48, 16, None),                 # ... tiles of 16-key groups; sequences of their own lengths
    ([30, 1, 99], [20000, 64, 9000], 16, 1, 128, 80, 48, None),        # ... of eights, some workgroups without rows
    ([60], [5000], 8, 1, 256, 48, 64, None),
    ([60], [5000], 8, 1, 32, 48, 64, None),
    ([980, 300], [980, 300], 8, 1, 128, 16, 48, None),                 # two teams
    ([900], [900], 16, 2, 64, 16, 128, (4, 2, 1, 114)),
    ([2] * 9, [2879] * 9, 128, 8, 128, 48, 80, (8, 1, 1, 216)),         # plain slots would be cut, packed ones are not
    ([21] * 9, [856] * 9, 32, 2, 128, 176, 48, (8, 1, 1, 198)),         # packed eights, not cut
    ([15] * 4, [1097] * 4, 64, 4, 128, 48, 64, (4, 1, 4, 96)),          # ... cut as fours
    ([130] * 3, [2843] * 3, 64, 4, 128, 16, 48, (4, 2, 1, 216)),        # many rows on short sequences: whole
    ([127] * 8, [1283] * 8, 32, 4, 64, 80, 64, (4, 1, 1, 320)),
    ([9] * 13, [4407] * 13, 32, 2, 128, 112, 64, (8, 1, 4, 182)),       # ... cut
])
@pytest.mark.parametrize("causal", [True, False])
def test_prepared_and_one_launch(q_lens, k_lens, hq, hk, d, qbs, kbs, plan, causal):
    w = make_problem(seed=111, q_lens=q_lens, k_lens=k_lens, hq=hq, hk=hk, d=d, qbs=qbs, kbs=kbs, keep=0.4, diag=False, causal=causal, scale=None)
    print(f"prepared plan {q_lens} {k_lens} {hq} {hk} {d} {qbs} {kbs} {plan_for(w)}", flush=True)
    assert plan_for(w, prepared=True)[1:3] == plan_for(w)[1:3]
    assert plan is None or plan_for(w) == plan
    out = HBSAttention(*w.args())
    previous = set_onepass(False)
    try:
        prepared = HBSAttention(*w.args())
        again = HBSAttention(*w.args())
    finally:
        set_onepass(previous)
    assert torch.equal(prepared, out) and torch.equal(again, out)
    assert_close_to_oracle(out, oracle_for(w, q_heads=[0, hq - 1]), "prepared")

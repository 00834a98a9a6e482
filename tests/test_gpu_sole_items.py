"""Launches of at most one item a workgroup, around the number of workgroups that fit the device at once, against the oracle and bit
for bit what the prepared form computes; rows of more tiles than a list holds, items without keys, block sizes that pack."""
import pytest
import torch

from hbsattn_amd import HBSAttention, set_onepass
from hbsattn_amd.workloads import make_problem
from helpers import assert_close_to_oracle, oracle_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("q_lens,k_lens,hq,hk,d,qbs,kbs,keep", [
    ([20], [20], 1, 1, 32, 16, 16, 1.0),
    ([30, 1, 90], [40, 300, 3], 4, 2, 64, 48, 32, 0.4),             # packed slots, 16-key groups, items without keys
    ([511 * 16], [700], 1, 1, 128, 16, 64, 0.5),                    # 511, 512 and 513 items: two workgroups a CU
    ([512 * 16], [700], 1, 1, 128, 16, 64, 0.5),
    ([513 * 16], [700], 1, 1, 128, 16, 64, 0.5),
    ([767 * 16], [200], 1, 1, 64, 16, 64, 0.5),                     # three a CU
    ([769 * 16], [200], 1, 1, 64, 16, 64, 0.5),
    ([100, 200], [150, 260], 4, 4, 256, 64, 64, 0.6),
    ([4200 * 16], [70000], 1, 1, 32, 256 * 16, 64, 1.0),            # more tiles than a list holds, not split: few rows see them all
    ([60, 200], [60, 200], 4, 2, 80, 64, 64, 0.6),                  # a head dim without a kernel of its own
])
@pytest.mark.parametrize("meta", [True, False])
def test_one_item_a_workgroup(q_lens, k_lens, hq, hk, d, qbs, kbs, keep, meta):
    w = make_problem(seed=71, q_lens=q_lens, k_lens=k_lens, hq=hq, hk=hk, d=d, qbs=qbs, kbs=kbs, keep=keep, diag=False, causal=True,
                     scale=None)
    print(f"sole {q_lens} {k_lens} {d} {qbs} {kbs} {meta}", flush=True)
    out = HBSAttention(*w.args(with_meta=meta))
    previous = set_onepass(False)
    try:
        assert torch.equal(out, HBSAttention(*w.args()))
    finally:
        set_onepass(previous)
    if meta:
        rows = None if sum(q_lens) < 2000 else sorted({0, 1, sum(q_lens) // 2, sum(q_lens) - 200, sum(q_lens) - 1})
        assert_close_to_oracle(out, oracle_for(w, q_rows=rows), "one item a workgroup")

"""Launches of at most one item a workgroup, around the number that is resident at head dims 32, 64 and 128: the plan is asserted, and the bits are the prepared form's."""
import pytest
import torch

from hbsattn_amd import HBSAttention, _lib, set_onepass
from hbsattn_amd.workloads import make_problem
from helpers import assert_close_to_oracle, oracle_for
from test_gpu_launch_plan import plan_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("q_lens,k_lens,hq,hk,d,qbs,kbs,keep", [
    ([20], [20], 1, 1, 32, 32, 16, 1.0),
    ([30, 1, 90], [40, 300, 3], 4, 2, 64, 48, 32, 0.4),             # packed slots, 16-key groups, items without keys
    ([511 * 16], [700], 1, 1, 128, 16, 64, 0.5),                    # 511, 512 and 513 items: two workgroups a CU
    ([512 * 16], [700], 1, 1, 128, 16, 64, 0.5),
    ([513 * 16], [700], 1, 1, 128, 16, 64, 0.5),
    ([767 * 32], [200], 1, 1, 64, 32, 64, 0.5),                     # three a CU
    ([768 * 32], [200], 1, 1, 64, 32, 64, 0.5),
    ([769 * 32], [200], 1, 1, 64, 32, 64, 0.5),
    ([1023 * 32], [100], 1, 1, 32, 32, 64, 0.5),                    # four
    ([1024 * 32], [100], 1, 1, 32, 32, 64, 0.5),
    ([1025 * 32], [100], 1, 1, 32, 32, 64, 0.5),
    ([100, 200], [150, 260], 4, 4, 256, 64, 64, 0.6),
    ([4200 * 16], [70000], 1, 1, 32, 256 * 16, 64, 1.0),            # more tiles than a list holds, not split: few rows see them all
    ([60, 200], [60, 200], 4, 2, 80, 64, 64, 0.6),                  # a head dim without a kernel of its own
])
@pytest.mark.parametrize("meta", [True, False])
def test_one_item_a_workgroup(q_lens, k_lens, hq, hk, d, qbs, kbs, keep, meta):
    w = make_problem(seed=71, q_lens=q_lens, k_lens=k_lens, hq=hq, hk=hk, d=d, qbs=qbs, kbs=kbs, keep=keep, diag=False, causal=True,
                     scale=None)
    print(f"sole {q_lens} {k_lens} {d} {qbs} {kbs} {meta}", flush=True)
    assert _lib.load().hbsa_fwd_decodes(_lib.DTYPE_BF16, sum(q_lens), hq, hk, w.q_meta[0], w.k_meta[0], qbs, kbs) == 0
    assert plan_for(w)[:3] == (4, 1, 1)
    out = HBSAttention(*w.args(with_meta=meta))
    previous = set_onepass(False)
    try:
        assert torch.equal(out, HBSAttention(*w.args()))
    finally:
        set_onepass(previous)
    if meta:
        rows = None if sum(q_lens) < 2000 else sorted({0, 1, sum(q_lens) // 2, sum(q_lens) - 200, sum(q_lens) - 1})
        assert_close_to_oracle(out, oracle_for(w, q_rows=rows), "one item a workgroup")

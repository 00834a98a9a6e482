"""One launch of workgroups of eight wavefronts whose slots are packed: five to eight of them in use, ragged q blocks, both kinds of tiles."""
import pytest
import torch

from hbsattn_amd import HBSAttention, _lib
from hbsattn_amd.workloads import make_problem
from helpers import assert_close_to_oracle, oracle_for
from test_gpu_launch_plan import plan_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hq,hk,qbs,q_lens", [
    (32, 16, 80, [1201, 65, 1200]),     # five slots, 32 q blocks
    (32, 8, 48, [1537, 1, 1440]),       # six, 64
    (32, 16, 112, [1905, 1399, 112]),   # seven, 32
    (32, 2, 16, [2033, 2047]),          # eight, 256
])
@pytest.mark.parametrize("kbs,dtype", [(64, torch.bfloat16), (48, torch.float16)], ids=["tiles", "groups"])
def test_packed_eights_are_the_prepared_form_bit_for_bit(hq, hk, qbs, q_lens, kbs, dtype):
    w = make_problem(seed=7, q_lens=q_lens, k_lens=q_lens, hq=hq, hk=hk, d=128, qbs=qbs, kbs=kbs, keep=0.3, diag=True, causal=True, scale=None, dtype=dtype)
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert plan_for(w)[:3] == (8, 1, 1)
    out = HBSAttention(*w.args())
    lib = _lib.load()
    was = lib.hbsa_set_onepass(0)
    try:
        assert torch.equal(HBSAttention(*w.args()), out)
    finally:
        lib.hbsa_set_onepass(was)
    total = sum(q_lens)
    assert_close_to_oracle(out, oracle_for(w, q_rows=sorted({0, 1, qbs - 1, qbs, q_lens[0] - 1, q_lens[0], total - 1})), f"{hq} / {hk} heads, {qbs}")

"""The one-launch forward's first round: a workgroup's second list of tiles is built before it has waited for any tile."""
import pytest
import torch

from hbsattn_amd import HBSAttention, _lib, set_onepass
from hbsattn_amd.workloads import make_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,dtype", [(128, torch.bfloat16), (64, torch.float16), (32, torch.bfloat16), (256, torch.bfloat16), (96, torch.bfloat16)])
@pytest.mark.parametrize("causal", [True, False])
def test_first_items_without_rows_for_the_scheduling_wavefront(d, dtype, causal):
    """4 q heads per kv head in blocks of 112 rows are 14 wave slots, four workgroups an item; a q block of one row fills
    an eighth of the first of them, so the other three have tiles but no rows.  The last 16 q blocks, which every
    workgroup begins with, are of that kind."""
    w = make_problem(seed=21, q_lens=[448] * 8 + [1] * 16, k_lens=[900] * 8 + [700] * 16, hq=32, hk=8, d=d, qbs=112, kbs=16, keep=0.5,
                     diag=True, causal=causal, scale=None, dtype=dtype)
    code = _lib.DTYPE_F16 if dtype == torch.float16 else _lib.DTYPE_BF16
    if d != 96:
        assert _lib.load().hbsa_fwd_launches(code, 24, w.k.shape[0], 32, 8, d, w.q_meta[0], w.k_meta[0], 112, 16, 1, None) == 1
    args = w.args()
    previous = set_onepass(False)
    try:
        expected = HBSAttention(*args)   # lists from a pre-pass
    finally:
        set_onepass(previous)
    other = torch.empty(1 << 30, dtype=torch.uint8, device="cuda")
    for i in range(40):
        other.fill_(i)   # (the mask is in no cache)
        got = HBSAttention(*args)
        if d == 96:      # (the pre-pass form runs on padded copies: another order of the sums)
            assert (got.float() - expected.float()).abs().max().item() <= 2e-2, f"call {i}"
        else:
            assert torch.equal(got, expected), f"call {i}"

"""Head dims that are no kernel's own: rows end inside the kernel's columns, at every kernel's edges, in one launch."""
import pytest
import torch

from hbsattn_amd import HBSAttention, _lib
from hbsattn_amd.workloads import make_problem
from helpers import assert_close_to_oracle, oracle_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [8, 24, 40, 56, 72, 96, 104, 120, 136, 160, 168, 192, 200, 248])
@pytest.mark.parametrize("qbs,kbs,causal,hq,hk", [(128, 128, True, 2, 2), (80, 48, False, 6, 2), (16, 64, True, 4, 1)])
def test_columns_past_the_head_dim_take_no_part(d, dtype, qbs, kbs, causal, hq, hk):
    w = make_problem(seed=d, q_lens=[3, 170, 65], k_lens=[20, 170, 333], hq=hq, hk=hk, d=d, qbs=qbs, kbs=kbs, keep=0.6, diag=True,
                     causal=causal, scale=None, dtype=dtype)
    out = HBSAttention(*w.args())
    assert_close_to_oracle(out, oracle_for(w), f"head dim {d}")
    # rows in wider storage: what lies beyond the head dim belongs to somebody else and must not be read or written
    pad = lambda t: torch.cat([t, torch.full_like(t[:, :, :8], float("nan"))], dim=2)[:, :, :d]
    args = list(w.args())
    args[:3] = [pad(t) for t in args[:3]]
    assert torch.equal(HBSAttention(*args), out)
    # what the compiled path takes it takes as one launch
    assert _lib.host().call(*w.args(), _lib.DTYPE_F32) is not None

"""The forward at both sides of the rules that choose workgroups of four or eight wavefronts and the split over key blocks."""
import pytest
import torch

from hbsattn_amd import HBSAttention
from hbsattn_amd.workloads import make_problem
from helpers import assert_close_to_oracle, oracle_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spec", [
    dict(q_lens=[512] * 8, k_lens=[512] * 8, hq=32, hk=8, d=128, qbs=128, kbs=128),            # two whole rounds of eights
    dict(q_lens=[512] * 8 + [1], k_lens=[512] * 8 + [1], hq=32, hk=8, d=128, qbs=128, kbs=128),   # one item more
    dict(q_lens=[70, 513, 333], k_lens=[70, 513, 333], hq=32, hk=8, d=128, qbs=64, kbs=64),    # a fraction of a round
    dict(q_lens=[70, 513, 333], k_lens=[70, 513, 333], hq=32, hk=8, d=64, qbs=64, kbs=48),     # head dim 64, eight slots
    dict(q_lens=[300, 412], k_lens=[9000, 2300], hq=32, hk=8, d=128, qbs=128, kbs=128),        # a chunk: split, eights
    dict(q_lens=[700, 900], k_lens=[6000, 17000], hq=32, hk=8, d=128, qbs=64, kbs=64),         # ... of somewhat more items
    dict(q_lens=[130, 60], k_lens=[5000, 6100], hq=16, hk=4, d=64, qbs=64, kbs=64),            # ... of fours
    dict(q_lens=[4000], k_lens=[15999], hq=2, hk=1, d=128, qbs=128, kbs=128),                  # one key short of a chunk, to a block
    dict(q_lens=[4000], k_lens=[16384], hq=2, hk=1, d=128, qbs=128, kbs=128),
], ids=lambda s: "q" + "-".join(map(str, s["q_lens"][:3])) + f"-d{s['d']}")
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_forward_on_both_sides_of_the_shape_rules(spec, dtype):
    w = make_problem(seed=5, keep=0.4, diag=True, causal=True, scale=None, dtype=dtype, **spec)
    out = HBSAttention(*w.args())
    total = w.q.shape[0]
    rows = sorted(set(torch.randint(0, total, (40,), generator=torch.Generator().manual_seed(1)).tolist() + [0, w.cu_q[1] - 1, total - 1]))
    assert_close_to_oracle(out, oracle_for(w, q_rows=rows), str(spec))
    assert torch.equal(HBSAttention(*w.args()), out)

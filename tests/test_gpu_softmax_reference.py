"""The reference a row's exponentials are formed against: it moves only when a sum of exponentials says that it lags too far."""
import pytest
import torch

from hbsattn_amd import HBSAttention
from hbsattn_amd.workloads import make_problem
from helpers import assert_close_to_oracle, oracle_for

pytestmark = pytest.mark.gpu


def rising(w, per_key):
    """Keys and queries whose scores rise by per_key (natural-log units) from one key to the next, the same for every query."""
    d = w.q.shape[2]
    scale = d ** -0.5
    w.q[:] = 0.
    w.q[:, :, 0] = 4.
    w.k *= 0.05
    for b in range(len(w.cu_k) - 1):
        a, z = int(w.cu_k[b]), int(w.cu_k[b + 1])
        ramp = torch.arange(z - a, device=w.k.device, dtype=torch.float32) * (per_key / (4. * scale))
        w.k[a:z, :, 0] = ramp[:, None].to(w.k.dtype)
    return w


@pytest.mark.parametrize("d", [32, 64, 96, 128, 192, 256])
@pytest.mark.parametrize("per_key", [0.01, 0.2, 1.5, -0.5], ids=lambda x: f"step{x}")
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_scores_that_rise_or_fall_along_the_keys(d, per_key, dtype):
    # steps of 1.5 move the reference in every half tile, 0.2 in some, the others never; every tile edge has its remainder
    w = rising(make_problem(seed=3, q_lens=[65, 33, 130], k_lens=[65, 97, 200], hq=4, hk=2, d=d, qbs=64, kbs=48, keep=0.8, diag=True,
                            causal=True, scale=None, dtype=dtype), per_key)
    # The largest |v| is about 4; p and the output carry 8 significant bits (2^-9 of it each, and p's is not averaged out when two
    # or three keys hold all the weight): 4 * 2 * 2^-9 = 1.6e-2, inside the usual tolerance.
    assert_close_to_oracle(HBSAttention(*w.args()), oracle_for(w), f"d={d} step {per_key}")


@pytest.mark.parametrize("d", [64, 128])
def test_rows_whose_first_tiles_are_hidden(d):
    # keys longer and shorter than the queries: rows without any key, and rows whose first visible key is far into the row's tiles
    w = make_problem(seed=4, q_lens=[150, 70], k_lens=[100, 300], hq=2, hk=1, d=d, qbs=80, kbs=16, keep=0.5, diag=False, causal=True, scale=None)
    out = HBSAttention(*w.args())
    assert_close_to_oracle(out, oracle_for(w), f"d={d}")
    assert (out[:50] == 0).all()   # q_len - k_len rows that see nothing

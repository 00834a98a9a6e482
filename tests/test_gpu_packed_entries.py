"""Packed slots number the (q head, row) entries of a q block, and the kernel divides by the rows in floating point: exact as far as the one-launch
form takes such blocks, and larger ones go to the prepared form."""
import numpy as np
import pytest
import torch

from hbsattn_amd import HBSAttention, _lib
from hbsattn_amd.workloads import make_problem
from helpers import assert_close_to_oracle, oracle_for
from test_gpu_fwd_any import _call

LIMIT = 1 << 20


def test_the_division_is_exact_below_the_limit():
    f = np.float32
    rng = np.random.default_rng(0)
    b = np.concatenate([np.arange(1, 5000), np.exp(rng.uniform(0, np.log(LIMIT), 20000)).astype(np.int64), [LIMIT - 1, LIMIT // 2, LIMIT // 3]])
    for _ in range(20):
        h = rng.integers(1, LIMIT // b + 1)
        for a in (h * b - 1, np.minimum(h * b, LIMIT - 1), LIMIT - 1 + 0 * b):   # the numbers next to a multiple
            for toward in (0.0, None, np.inf):   # a reciprocal one ulp low, rounded, one ulp high
                r = f(1) / b.astype(f)
                if toward is not None:
                    r = np.nextafter(r, f(toward), dtype=f)
                assert np.array_equal(((a.astype(f) + f(0.5)) * r).astype(np.int64), a // b)


@pytest.mark.gpu
@pytest.mark.parametrize("d,rows,rc", [(40, LIMIT // 2, 0), (40, LIMIT // 2 + 16, _lib.ERR_WORKSPACE_TOO_SMALL), (32, LIMIT // 2 - 16, 0),
                                       (32, LIMIT // 2 + 16, _lib.ERR_WORKSPACE_TOO_SMALL)])
def test_blocks_around_the_limit(d, rows, rc):
    # (the blocks of head dim 32 are no whole number of slots, which is what packs them there)
    w = make_problem(seed=97, q_lens=[rows], k_lens=[100], hq=2, hk=1, d=d, qbs=rows, kbs=64, keep=1.0, diag=True, causal=False, scale=None, gen_device="device")
    print(f"packed {d} {rows}", flush=True)
    out = torch.full_like(w.q, 9.0)
    assert _call(w, out, None, 0, one=True) == rc
    if rc != 0:
        assert bool((out == 9.0).all())
        out = HBSAttention(*w.args())
    assert_close_to_oracle(out, oracle_for(w, q_rows=[0, 1, rows // 2, rows - 17, rows - 2, rows - 1]), "packed")

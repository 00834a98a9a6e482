"""Items whose tiles two teams of wavefronts share: lists around what is shared, ragged last tiles, rows of more tiles than a list holds,
rows without keys, growing logits and NaN, every form that has to compute the same bits."""
import dataclasses

import pytest
import torch

from hbsattn_amd import HBSAttention, set_onepass
from hbsattn_amd.workloads import make_problem
from helpers import assert_close_to_oracle, oracle_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("q_lens,k_lens,hq,hk,d,qbs,kbs,keep", [
    ([1000], [1000], 2, 2, 64, 64, 64, 0.2),                        # three to five tiles an item, among them
    ([300, 1030, 7], [300, 1030, 900], 4, 2, 128, 48, 64, 0.5),     # packed slots, ragged tiles
    ([700], [1500], 1, 1, 32, 128, 16, 0.4),                        # 16-key groups
    ([2000], [2000], 1, 1, 128, 128, 80, 0.5),
    ([16 * 200], [90000], 1, 1, 32, 16 * 25, 64, 1.0),              # more tiles than a list holds
    ([900], [900], 2, 1, 80, 64, 64, 0.6),                          # head dims without a kernel of their own
    ([900], [900], 2, 1, 96, 64, 48, 0.6),
    ([900, 40], [900, 800], 2, 2, 24, 64, 64, 0.6),
    ([900], [900], 2, 2, 40, 128, 128, 0.6),
])
@pytest.mark.parametrize("meta", [True, False])
def test_shared_tiles(q_lens, k_lens, hq, hk, d, qbs, kbs, keep, meta):
    w = make_problem(seed=81, q_lens=q_lens, k_lens=k_lens, hq=hq, hk=hk, d=d, qbs=qbs, kbs=kbs, keep=keep, diag=False, causal=True,
                     scale=None)
    w.block_mask[0, 0] = False   # an item without keys
    print(f"teams {q_lens} {k_lens} {d} {qbs} {kbs} {meta}", flush=True)
    out = HBSAttention(*w.args(with_meta=meta))
    assert torch.equal(out, HBSAttention(*w.args(with_meta=meta)))
    previous = set_onepass(False)
    try:
        assert torch.equal(out, HBSAttention(*w.args()))
    finally:
        set_onepass(previous)
    if meta:
        rows = None if sum(q_lens) < 2500 else sorted({0, 1, sum(q_lens) // 2, sum(q_lens) - 200, sum(q_lens) - 1})
        assert_close_to_oracle(out, oracle_for(w, q_rows=rows), "two teams")


@pytest.mark.parametrize("d", [32, 64, 128])
def test_logits_that_grow_and_fall(d):
    # the teams end with references far apart
    for grow in (1, -1):
        w = make_problem(seed=82, q_lens=[600], k_lens=[1500], hq=1, hk=1, d=d, qbs=64, kbs=64, keep=1.0, diag=True, causal=False, scale=0.3)
        ramp = torch.linspace(0.0, 1.0, 1500, device="cuda")[:, None, None]
        k = (w.k.float() * (ramp if grow > 0 else 1.0 - ramp)).to(w.k.dtype)
        k[1440:] *= 3.0 if grow > 0 else 0.0   # the last tile is the second team's
        w = dataclasses.replace(w, k=k)
        print(f"teams, logits {grow} {d}", flush=True)
        # (a softmax this sharp is a few keys: their bf16 weights' 2^-9 of values up to 4)
        assert_close_to_oracle(HBSAttention(*w.args()), oracle_for(w), "references apart", max_abs=4e-2)


def test_a_nan_stays_in_its_rows():
    w = make_problem(seed=83, q_lens=[600], k_lens=[1500], hq=2, hk=2, d=64, qbs=64, kbs=64, keep=0.7, diag=True, causal=False, scale=None)
    clean = HBSAttention(*w.args())
    q = w.q.clone()
    q[70, 1, 3] = float("nan")
    out = HBSAttention(*dataclasses.replace(w, q=q).args())
    assert torch.isnan(out[70, 1]).all()
    out[70, 1] = clean[70, 1]
    assert torch.equal(out, clean)

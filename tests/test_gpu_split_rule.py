"""When the forward splits its items over key blocks: tiles are counted, not keys, against the places of the device."""
import pytest
import torch

from hbsattn_amd import HBSAttention, _lib
from hbsattn_amd.workloads import make_problem
from helpers import assert_close_to_oracle, oracle_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("q_lens,k_lens,hq,hk,d,qbs,kbs,launches", [
    ([3318], [3318], 4, 4, 128, 64, 16, 2),      # 208 items of 208 tiles: a k block of 16 is a tile of its own
    ([3318], [3318], 4, 4, 128, 64, 64, 1),      # ... of 52
    ([270] * 3, [20000] * 3, 32, 32, 256, 128, 128, 1),   # 288 items, 160 of them are the most that 256 places split
    ([270] * 3, [20000] * 3, 16, 16, 256, 128, 128, 2),   # 144
])
def test_split_or_one_launch(q_lens, k_lens, hq, hk, d, qbs, kbs, launches):
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the numbers of items are for 256 compute units")
    nq, nk = sum(-(-n // qbs) for n in q_lens), sum(-(-n // kbs) for n in k_lens)
    lib = _lib.load()
    assert lib.hbsa_fwd_launches(_lib.DTYPE_BF16, len(q_lens), sum(k_lens), hq, hk, d, nq, nk, qbs, kbs, 1, None) == launches


@pytest.mark.parametrize("q_lens,k_lens,hq,hk,d,qbs,kbs", [
    ([1300], [1300], 2, 2, 128, 64, 16),                  # split by tiles
    ([100, 90], [6000, 5000], 8, 2, 128, 128, 64),        # eights, two rounds of parts
    ([1] * 20 + [128], [500] * 20 + [3000], 8, 2, 128, 128, 64),   # blocks of one row and one full block: eights
])
def test_against_the_oracle(q_lens, k_lens, hq, hk, d, qbs, kbs):
    w = make_problem(seed=31, q_lens=q_lens, k_lens=k_lens, hq=hq, hk=hk, d=d, qbs=qbs, kbs=kbs, keep=0.4, diag=True,
                     causal=True, scale=None)
    out = HBSAttention(*w.args())
    assert_close_to_oracle(out, oracle_for(w), "split")
    assert torch.equal(HBSAttention(*w.args()), out)

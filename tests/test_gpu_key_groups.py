"""Key block sizes that are no multiple of the forward kernel's tile: tiles made of 16-key groups of any kept blocks."""
import pytest
import torch

from hbsattn_amd import HBSAttention, set_onepass
from hbsattn_amd.workloads import make_problem
from helpers import assert_close_to_oracle, oracle_for

pytestmark = pytest.mark.gpu


def check(w, what, same_bits=True):
    """Against the oracle, in the one-launch form and in the prepared form, which compute the same bits."""
    ref, outs = oracle_for(w), []
    for one in (True, False):
        previous = set_onepass(one)
        try:
            outs.append(HBSAttention(*w.args()))
        finally:
            set_onepass(previous)
        assert_close_to_oracle(outs[-1], ref, f"{what} one={one}")
    assert not same_bits or torch.equal(*outs)


@pytest.mark.parametrize("kbs", [16, 48, 80, 240, 272])   # 240 and more keep to runs of consecutive keys, 80 does above head dim 64
@pytest.mark.parametrize("d", [32, 40, 64, 96, 128, 160, 192, 224, 256])
def test_blocks_and_tails_of_every_remainder(d, kbs):
    # key lengths of 1, 15, 16, 17, 63, 64, 65 past whole blocks, more and fewer keys than queries, whole and missing last groups;
    # the last sequence is long, since groups are for sequences of several blocks
    for causal, gqa, k_lens in ((True, 1, [kbs + 1, 2 * kbs + 15, 3 * kbs + 16, 60 * kbs + 700]), (False, 4, [17, 4 * kbs + 63, 64, 65 + 60 * kbs])):
        w = make_problem(seed=kbs + d, q_lens=[130, 77, 300, 64], k_lens=k_lens, hq=4, hk=4 // gqa, d=d, qbs=64, kbs=kbs, keep=0.6,
                         diag=True, causal=causal, scale=None)
        check(w, f"d={d} kbs={kbs} causal={causal}")


@pytest.mark.parametrize("d", [64, 96, 192, 256])
def test_items_longer_than_a_list(d):
    # about 38000 kept keys an item, a list holds 32768; more items than are split over their key blocks
    w = make_problem(seed=5, q_lens=[350], k_lens=[40003], hq=16, hk=16, d=d, qbs=16, kbs=48, keep=0.95, diag=False, causal=False, scale=None)
    check(w, f"d={d}", same_bits=d in (64, 256))   # (padded head dims may be cut into parts differently)


@pytest.mark.parametrize("k_lens", [[16 * 48 + 1], [16 * 48 - 48 + 1], [48] * 17, [49] * 8], ids=str)
def test_sequences_on_both_sides_of_the_line(k_lens):
    # 17 blocks that can be one sequence's save more than four tiles, 16 do not; sequences that end in part of a block count as such
    w = make_problem(seed=7, q_lens=[40] * len(k_lens), k_lens=k_lens, hq=4, hk=2, d=64, qbs=32, kbs=48, keep=0.7, diag=True, causal=True, scale=None)
    check(w, str(k_lens))


@pytest.mark.parametrize("blocks", [65535, 65536], ids=lambda n: f"{n}blocks")
def test_the_last_group_that_can_be_numbered(blocks):
    # a group's number has 16 bits: one key block more and the kernel for runs is taken
    w = make_problem(seed=6, q_lens=[64], k_lens=[16 * blocks - 3], hq=1, hk=1, d=32, qbs=64, kbs=16, keep=0.01, diag=False, causal=False, scale=None)
    w.block_mask[..., -40:] = True   # (half of the kept keys' weight is where numbers are largest)
    check(w, f"{blocks} blocks")


@pytest.mark.parametrize("kbs", [32, 112, 144, 160, 176, 208])   # the largest that make groups at head dims up to 64, and one between that does not
@pytest.mark.parametrize("d", [32, 64])
def test_larger_blocks_at_small_head_dims(d, kbs):
    w = make_problem(seed=kbs + d, q_lens=[130, 77, 300, 64], k_lens=[kbs + 1, 2 * kbs + 15, 3 * kbs + 16, 60 * kbs + 700], hq=4, hk=4, d=d, qbs=64, kbs=kbs,
                     keep=0.6, diag=True, causal=True, scale=None)
    check(w, f"d={d} kbs={kbs}")


@pytest.mark.parametrize("qbs", [128, 48])   # fewer (q block, kv head) pairs than CUs, and more
@pytest.mark.parametrize("d,kbs", [(128, 80), (128, 96), (96, 80), (128, 112), (160, 32), (192, 80), (256, 80)])
def test_blocks_at_the_line_of_larger_head_dims(d, kbs, qbs):
    w = make_problem(seed=kbs + d, q_lens=[930, 1100, 1444], k_lens=[40 * kbs + 1, 1100, 70 * kbs + 15], hq=4, hk=4, d=d, qbs=qbs, kbs=kbs, keep=0.5,
                     diag=True, causal=True, scale=None)
    check(w, f"d={d} kbs={kbs} qbs={qbs}")


# Blocks whose tiles are full with 32 keys, blocks that lie in one run: groups save nothing there and cost a tenth and more.  With all
# blocks kept the work is that of blocks of whole tiles; groups took 1.22, 1.12, 1.18 and 1.24 times as long.  The least of ten runs, in turn.
@pytest.mark.parametrize("d,kbs", [(192, 96), (128, 208), (256, 144), (96, 160)])
def test_blocks_in_one_run_take_no_longer_than_whole_tiles(d, kbs):
    make = lambda n: make_problem(seed=9, q_lens=[1920] * 4, k_lens=[1920] * 4, hq=8, hk=8, d=d, qbs=64, kbs=n, keep=1.0, diag=True, causal=False,
                                  scale=None, gen_device="device").args()
    calls, times = [make(128), make(kbs)], [[], []]
    for _ in range(10):
        for i, args in enumerate(calls):
            HBSAttention(*args)
            a, z = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(10):
                HBSAttention(*args)
            z.record()
            z.synchronize()
            times[i].append(a.elapsed_time(z))
    print(f"us {min(times[0]) * 100:.1f} {min(times[1]) * 100:.1f}")
    assert min(times[1]) <= 1.09 * min(times[0]), f"{min(times[1]) * 100:.1f} us against {min(times[0]) * 100:.1f}"

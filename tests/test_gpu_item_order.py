"""Items sorted by weight in the prepared form of the forward: heaviest first, with the same results as in any other order."""
import pytest
import torch

from hbsattn_amd import HBSAttention, _lib, set_onepass
from hbsattn_amd.interface import hbsa_prepare
from hbsattn_amd.workloads import make_problem

pytestmark = pytest.mark.gpu


@pytest.fixture
def two_launches():
    previous = set_onepass(False)
    yield
    set_onepass(previous)


# (q block, kv head) pairs: under one workgroup place each, several, the most that an order is kept of (4096) and one q block more;
# batches with empty sequences, a mask without any block (all weights equal), weights beyond the last bin.  The last four are sorted.
SPECS = [
    dict(q_lens=[300, 2025, 0, 498, 3205], k_lens=[300, 2025, 77, 498, 3205], hq=16, hk=4, d=64, qbs=64, kbs=64, keep=0.4, causal=True),
    dict(q_lens=[513, 64, 2049], k_lens=[700, 64, 1500], hq=24, hk=12, d=32, qbs=32, kbs=48, keep=0.7, causal=False),
    dict(q_lens=[2048, 2048], k_lens=[2048, 2048], hq=16, hk=16, d=64, qbs=16, kbs=128, keep=0.3, causal=True),          # 4096 pairs
    dict(q_lens=[2048, 2049], k_lens=[2048, 2049], hq=16, hk=16, d=64, qbs=16, kbs=128, keep=0.3, causal=True),          # 4112
    dict(q_lens=[900, 1300], k_lens=[900, 1300], hq=16, hk=16, d=128, qbs=64, kbs=64, keep=0.0, causal=True),
    dict(q_lens=[3000], k_lens=[90000], hq=16, hk=16, d=64, qbs=64, kbs=64, keep=0.9, causal=False),
    dict(q_lens=[3300, 2025, 0, 498, 3205], k_lens=[3300, 2025, 77, 498, 3205], hq=16, hk=4, d=64, qbs=64, kbs=64, keep=0.4, causal=True),
    dict(q_lens=[2513, 64, 4049], k_lens=[2700, 64, 3500], hq=14, hk=7, d=32, qbs=32, kbs=48, keep=0.7, causal=False),
]


@pytest.mark.parametrize("spec", SPECS, ids=lambda s: f"{len(s['q_lens'])}x{s['q_lens'][0]}-h{s['hk']}-d{s['d']}-q{s['qbs']}")
def test_sorted_items_give_the_results_of_the_one_launch_form(spec, two_launches):
    w = make_problem(seed=31, diag=spec["keep"] > 0, scale=None, **spec)
    prepared = HBSAttention(*w.args())
    set_onepass(True)
    assert torch.equal(HBSAttention(*w.args()), prepared)


def test_a_captured_preparation_takes_the_order_without_weights_and_can_be_replayed(two_launches):
    w = make_problem(seed=32, diag=True, scale=None, **SPECS[6])
    eager = HBSAttention(*w.args())
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        HBSAttention(*w.args())
        with torch.cuda.graph(graph, stream=stream):
            out = HBSAttention(*w.args())
    for _ in range(3):
        out.zero_()
        graph.replay()
        assert torch.equal(HBSAttention(*w.args()), eager)   # eager work between the replays
        torch.cuda.synchronize()
        assert torch.equal(out, eager)


def test_two_streams_prepare_at_once(two_launches):
    a, b = (make_problem(seed=33 + i, diag=True, scale=None, **SPECS[i]) for i in (6, 7))   # both weighed, several rounds of items
    want = [HBSAttention(*a.args()), HBSAttention(*b.args())]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    got = [[], []]
    for _ in range(4):
        for i, w in enumerate((a, b)):
            with torch.cuda.stream(streams[i]):
                got[i].append(HBSAttention(*w.args()))
    torch.cuda.synchronize()
    assert all(torch.equal(o, want[i]) for i in range(2) for o in got[i])


def _orders(w):
    """The two orders hbsa_prepare leaves at the end of its workspace: (q block << 16 | kv head) of every item, k block numbers."""
    (nq, _, q2b, cu_nq), (nk, _, _, cu_nk) = w.q_meta, w.k_meta
    prepared = hbsa_prepare(w.cu_q_seqlens, w.cu_k_seqlens, w.block_mask, w.q_block_size, w.k_block_size, w.causal, int(nq), q2b, cu_nq, int(nk),
                            cu_nk, run_shape=(w.q.dtype, w.q.shape[0], w.k.shape[0], w.q.shape[1], w.q.shape[2]))
    up = lambda x: -(-x // 256) * 256
    pairs = w.block_mask.shape[0] * int(nq)
    words = up(4 * pairs) // 4
    at = _lib.load().hbsa_fwd_workspace_bytes(w.block_mask.shape[0], int(nq), int(nk)) - up(4 * pairs) - up(4 * int(nk))
    ints = prepared.workspace[at:at + up(4 * pairs) + up(4 * int(nk))].view(torch.int32).cpu()
    return ints[:pairs], ints[words:words + int(nk)]


def _weights(w):
    """Kept keys of every (q block, kv head), whole blocks, and the query rows that see a key of every k block."""
    items, rows, qb, kb = {}, [], 0, 0
    mask, shift = w.block_mask.cpu(), 4
    while shift < 16 and (int(w.k_meta[0]) * w.k_block_size) >> shift >= 512:   # weights are told apart in units of 2^shift keys, 512 of them
        shift += 1
    for b in range(len(w.cu_q) - 1):
        nq, nk = int(w.cu_q[b + 1] - w.cu_q[b]), int(w.cu_k[b + 1] - w.cu_k[b])
        q_blocks, k_blocks = -(-nq // w.q_block_size), -(-nk // w.k_block_size)
        for i in range(q_blocks):
            sees = min(nk, min(nq, (i + 1) * w.q_block_size) + nk - nq) if w.causal else nk   # keys before this one
            blocks = -(-max(0, sees) // w.k_block_size)
            for h in range(mask.shape[0]):
                kept = int(mask[h, qb + i, kb:kb + blocks].sum()) * w.k_block_size
                items[(qb + i) << 16 | h] = min(511, (kept + (1 << shift) - 1) >> shift)
        rows += [min(nq, nk - j * w.k_block_size) if w.causal else nq for j in range(k_blocks)]
        qb, kb = qb + q_blocks, kb + k_blocks
    return items, rows


MANY = dict(hq=4, hk=4, d=64, qbs=16, kbs=16, keep=0.5)
SIXTEEN = dict(hq=16, hk=16, d=64, qbs=64, kbs=64, keep=0.5, causal=True)
# (problem, whether its items are sorted: on both sides of every line of the rule, on 256 CUs)
ORDERED = [(SPECS[i], i >= 4) for i in (0, 1, 2, 4, 5, 6, 7)] + [
    (dict(q_lens=[40 * (i % 3) for i in range(n)], k_lens=[keys + i % 50 for i in range(n)], causal=causal, **MANY), weighed)
    for n, keys, causal, weighed in ((63, 768, True, True), (64, 768, False, True), (65, 700, True, False), (127, 768, True, True), (128, 768, True, False),
                                     (256, 300, True, False))] + [
    (dict(q_lens=[n * 64, 1024], k_lens=[n * 64, 1024], **SIXTEEN), weighed) for n, weighed in ((15, False), (16, True), (80, True), (81, False))] + [
    (dict(SIXTEEN, q_lens=[1024, 1024], k_lens=[1024, 1024], hk=17, hq=17), False)]


@pytest.mark.parametrize("spec,weighed", ORDERED, ids=lambda s: f"{len(s['q_lens'])}x{s['q_lens'][0]}-h{s['hk']}-q{s['qbs']}" if isinstance(s, dict) else str(s))
def test_items_and_k_blocks_come_heaviest_first(spec, weighed):
    w = make_problem(seed=35, diag=spec["keep"] > 0, scale=None, **spec)
    order, order_k = _orders(w)
    items, rows = _weights(w)
    assert sorted(order.tolist()) == sorted(items)
    if weighed:
        weights = [items[x] for x in order.tolist()]
        assert weights == sorted(weights, reverse=True)
        assert len(set(weights)) > 1 or spec["keep"] == 0.0
    else:   # the last q block first, its kv heads in their order
        assert order.tolist() == sorted(items, key=lambda x: (-(x >> 16), x & 0xffff))
    assert order_k.tolist() == sorted(range(len(rows)), key=lambda kb: -rows[kb])   # equals in their own order


def test_k_blocks_of_more_sequences_than_are_ordered_keep_their_order():
    n = 257
    w = make_problem(seed=36, q_lens=[30] * n, k_lens=[384] * n, hq=2, hk=2, d=64, qbs=16, kbs=16, keep=0.5, diag=True, causal=True, scale=None)
    assert _orders(w)[1].tolist() == list(range(w.block_mask.shape[2]))


@pytest.mark.parametrize("k_blocks", [32, 33])
def test_k_blocks_are_ordered_by_enough_wavefronts_alone(k_blocks):
    # two q blocks and one head are one workgroup of four wavefronts, of at most eight k blocks each: more would be put in their
    # places one after the other for longer than it gives (285 for each wavefront took 109 us of the pre-pass, which takes 4)
    w = make_problem(seed=37, q_lens=[16, 64], k_lens=[16 * 16, 16 * (k_blocks - 16)], hq=1, hk=1, d=64, qbs=64, kbs=16, keep=0.5, diag=True,
                     causal=False, scale=None)
    own = list(range(k_blocks))
    assert _orders(w)[1].tolist() == (own[16:] + own[:16] if k_blocks == 32 else own)

"""Items sorted by weight in the prepared form of the forward: the same results as in any other order."""
import pytest
import torch

from hbsattn_amd import HBSAttention, set_onepass
from hbsattn_amd.workloads import make_problem

pytestmark = pytest.mark.gpu


@pytest.fixture
def two_launches():
    previous = set_onepass(False)
    yield
    set_onepass(previous)


# (q block, kv head) pairs: under one workgroup place each, several, the most that are sorted (4096) and one q block more;
# batches with empty sequences, a mask without any block (all weights equal), weights beyond the last bin
SPECS = [
    dict(q_lens=[300, 2025, 0, 498, 3205], k_lens=[300, 2025, 77, 498, 3205], hq=16, hk=4, d=64, qbs=64, kbs=64, keep=0.4, causal=True),
    dict(q_lens=[513, 64, 2049], k_lens=[700, 64, 1500], hq=24, hk=12, d=32, qbs=32, kbs=48, keep=0.7, causal=False),
    dict(q_lens=[2048, 2048], k_lens=[2048, 2048], hq=16, hk=16, d=64, qbs=16, kbs=128, keep=0.3, causal=True),          # 4096 pairs
    dict(q_lens=[2048, 2049], k_lens=[2048, 2049], hq=16, hk=16, d=64, qbs=16, kbs=128, keep=0.3, causal=True),          # 4112
    dict(q_lens=[900, 1300], k_lens=[900, 1300], hq=16, hk=16, d=128, qbs=64, kbs=64, keep=0.0, causal=True),
    dict(q_lens=[3000], k_lens=[90000], hq=16, hk=16, d=64, qbs=64, kbs=64, keep=0.9, causal=False),
    dict(q_lens=[3300, 2025, 0, 498, 3205], k_lens=[3300, 2025, 77, 498, 3205], hq=16, hk=4, d=64, qbs=64, kbs=64, keep=0.4, causal=True),
]


@pytest.mark.parametrize("spec", SPECS, ids=lambda s: f"{len(s['q_lens'])}x{s['q_lens'][0]}-h{s['hk']}-d{s['d']}-q{s['qbs']}")
def test_sorted_items_give_the_results_of_the_one_launch_form(spec, two_launches):
    w = make_problem(seed=31, diag=spec["keep"] > 0, scale=None, **spec)
    prepared = HBSAttention(*w.args())
    set_onepass(True)
    assert torch.equal(HBSAttention(*w.args()), prepared)


def test_a_captured_preparation_takes_the_order_without_weights_and_can_be_replayed(two_launches):
    w = make_problem(seed=32, diag=True, scale=None, **SPECS[0])
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
    a, b = (make_problem(seed=33 + i, diag=True, scale=None, **SPECS[i]) for i in (2, 6))   # both weighed, several rounds of items
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

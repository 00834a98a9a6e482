"""dK/dV items taken in the order of the rows that can see them, and the form of the head dim 64 kernel for many of them."""
import ctypes

import pytest
import torch

from hbsattn_amd import _lib, calculate_blocks
from hbsattn_amd.interface import PreparedMask, hbsa_backward, hbsa_prepare, hbsa_run
from oracle.grads import hbsa_oracle_grads
from test_gpu_backward import _check, _gpu_grads, _problem

pytestmark = pytest.mark.gpu

# items of one to two rounds on 256 CUs, none cut into parts but in the last five; k blocks of one and two key slots, of a slot and a half
CASES = [
    # q_lens, k_lens, hq, hk, d, qbs, kbs, causal
    ([70, 513, 0, 300], [70, 513, 90, 300], 32, 32, 64, 64, 32, True),      # an empty sequence; 31 blocks a head
    ([40, 700, 130], [900, 200, 130], 36, 36, 64, 48, 48, True),            # keys seen by all rows, rows that see none
    ([200, 333], [1000, 333], 32, 32, 64, 128, 96, False),
    ([90, 260], [260, 90], 36, 36, 32, 16, 16, True),
    ([129, 400, 64], [129, 400, 64], 16, 8, 128, 64, 64, True),
    # sequences of one, two and more rounds of a wavefront's lanes, the last of those that are ordered (256), one more; empty ones among them
    ([i % 40 for i in range(63)], [i % 50 for i in range(63)], 4, 4, 64, 16, 16, True),
    ([i % 40 for i in range(64)], [1 + i % 50 for i in range(64)], 4, 4, 64, 16, 16, False),
    ([i % 40 for i in range(65)], [i % 50 for i in range(65)], 4, 4, 64, 16, 16, True),
    ([i % 23 for i in range(256)], [i % 37 for i in range(256)], 4, 2, 32, 16, 16, True),
    ([1 + i % 23 for i in range(257)], [1 + i % 37 for i in range(257)], 2, 2, 32, 16, 16, False),
]


@pytest.mark.parametrize("case", CASES, ids=[f"case{i}" for i in range(len(CASES))])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_gradients_in_the_order_of_the_weights(case, dtype):
    q_lens, k_lens, hq, hk, d, qbs, kbs, causal = case
    q, k, v, do, cu_q, cu_k, cq, ck, mask = _problem(11, q_lens, k_lens, hq, hk, d, qbs, kbs, 0.5, dtype)
    print(f"backward by weight {case} {dtype}", flush=True)
    qd, kd, vd, dod = (t.cuda() for t in (q, k, v, do))
    (nq, _, q2b, cu_nq), (nk, _, _, cu_nk) = calculate_blocks(cq, qbs), calculate_blocks(ck, kbs)
    prepared = hbsa_prepare(cq, ck, mask.cuda(), qbs, kbs, causal, nq, q2b, cu_nq, nk, cu_nk)
    out, lse = hbsa_run(qd, kd, vd, prepared, None, return_lse=True)
    got = hbsa_backward(qd, kd, vd, out, dod, lse, prepared, None)
    for x, ref, name in zip(got, hbsa_oracle_grads(q, k, v, do, cu_q, cu_k, mask, qbs, kbs, causal, None), ("dq", "dk", "dv")):
        _check(x, ref, name)
    # prepared under capture: the forward's items come unsorted, and nothing else changes
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    maskd = mask.cuda()
    with torch.cuda.stream(stream), torch.cuda.graph(graph, stream=stream):
        again = hbsa_prepare(cq, ck, maskd, qbs, kbs, causal, nq, q2b, cu_nq, nk, cu_nk)
        out2, lse2 = hbsa_run(qd, kd, vd, again, None, return_lse=True)
        grads = hbsa_backward(qd, kd, vd, out2, dod, lse2, again, None)
    for _ in range(2):
        for t in grads:
            t.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out2, out) and all(torch.equal(a, b) for a, b in zip(got, grads))


def test_gradients_on_the_workspace_of_a_forward_split_over_key_blocks():
    # such a forward takes its items in no order of weights; the backward's order of the k blocks has to be there all the same
    q_lens, k_lens, hq, hk, d, qbs, kbs, causal = [200, 130], [9000, 7001], 4, 4, 64, 64, 64, True
    q, k, v, do, cu_q, cu_k, cq, ck, mask = _problem(12, q_lens, k_lens, hq, hk, d, qbs, kbs, 0.5, torch.bfloat16)
    print("backward on a split forward's workspace", flush=True)
    lib = _lib.load()
    qd, kd, vd, dod, maskd = (t.cuda() for t in (q, k, v, do, mask))
    (nq, _, q2b, cu_nq), (nk, _, _, cu_nk) = calculate_blocks(cq, qbs), calculate_blocks(ck, kbs)
    need = lib.hbsa_fwd_workspace_bytes(hk, nq, nk)
    split = lib.hbsa_fwd_split_workspace_bytes(q.shape[0], hq, hk, d, nq, nk, qbs)
    assert split > 0
    ws = torch.zeros(need + split, dtype=torch.uint8, device="cuda")
    out = torch.empty_like(qd)
    meta = [t.to(torch.int32).contiguous() for t in (q2b, cu_nq, cu_nk)]
    strides = (ctypes.c_int64 * 11)(*(n for t in (qd, kd, vd, out) for n in t.stride()[:2]), *maskd.stride())
    rc = lib.hbsa_fwd(qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), out.data_ptr(), cq.data_ptr(), ck.data_ptr(), maskd.data_ptr(),
                      *(t.data_ptr() for t in meta), ws.data_ptr(), ws.numel(), _lib.DTYPE_BF16, len(q_lens), q.shape[0], k.shape[0],
                      hq, hk, d, nq, nk, qbs, kbs, int(causal), d ** -0.5, strides, torch.cuda.current_stream().cuda_stream)
    assert rc == 0, _lib.last_error()
    prepared = PreparedMask(ws, hk, nq, nk, qbs, kbs, causal, ck, meta[1], meta[2])
    out, lse = hbsa_run(qd, kd, vd, prepared, None, return_lse=True)
    got = hbsa_backward(qd, kd, vd, out, dod, lse, prepared, None)
    for x, ref, name in zip(got, hbsa_oracle_grads(q, k, v, do, cu_q, cu_k, mask, qbs, kbs, causal, None), ("dq", "dk", "dv")):
        _check(x, ref, name)


def test_a_backward_takes_no_longer_for_being_of_many_sequences():
    # equal work in 60 sequences of 256 tokens and in 240 of 64: what a dK/dV workgroup does to find its sequence must not show
    # (one sequence after the other, behind the order of the k blocks: 67 and 101 us; 64 at a time 67 and 70)
    times = []
    for n, length in ((60, 256), (240, 64)):
        q, k, v, do, cu_q, cu_k, cq, ck, mask = _problem(14, [length] * n, [length] * n, 4, 4, 128, 64, 64, 0.0, torch.bfloat16)
        for i in range(mask.shape[1]):
            mask[:, i, i] = True
        qd, kd, vd, dod = (t.cuda() for t in (q, k, v, do))
        (nq, _, q2b, cu_nq), (nk, _, _, cu_nk) = calculate_blocks(cq, 64), calculate_blocks(ck, 64)
        prepared = hbsa_prepare(cq, ck, mask.cuda(), 64, 64, True, nq, q2b, cu_nq, nk, cu_nk)
        out, lse = hbsa_run(qd, kd, vd, prepared, None, return_lse=True)
        graph = torch.cuda.CUDAGraph()
        hbsa_backward(qd, kd, vd, out, dod, lse, prepared, None)
        with torch.cuda.graph(graph):
            hbsa_backward(qd, kd, vd, out, dod, lse, prepared, None)
        best = float("inf")
        for _ in range(10):
            a, z = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(10):
                graph.replay()
            z.record()
            z.synchronize()
            best = min(best, a.elapsed_time(z) * 100)
        times.append(best)
    print("us of 60 and of 240 sequences", times)
    assert times[1] <= 1.3 * times[0], times


# The form for many items: more than 4.5 a CU at head dim 64, any number at 32.  Key blocks of up to four slots, a wavefront each: both
# halves of a tile are one wavefront's.  Sequences with fewer and more queries than keys, last blocks of a few keys, several tiles of rows.
MANY = [
    ([300, 150, 700], [1400, 1300, 1390], 40, 40, 64, 64, 128, True),
    ([300, 150, 700], [1400, 1300, 1390], 40, 40, 64, 128, 128, False),
    ([200, 0, 900], [1000, 85, 1700], 36, 36, 64, 48, 80, True),
    ([130, 333], [1601, 1630], 72, 36, 64, 80, 96, False),
    ([90, 260, 500], [1600, 1600, 500], 40, 40, 64, 64, 64, True),
    ([300, 150, 700], [1400, 1300, 1390], 40, 40, 32, 64, 128, True),
    ([130, 333], [1601, 1630], 72, 36, 32, 80, 80, False),
]


@pytest.mark.parametrize("case", MANY, ids=[f"case{i}" for i in range(len(MANY))])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_gradients_of_many_items(case, dtype):
    q_lens, k_lens, hq, hk, d, qbs, kbs, causal = case
    q, k, v, do, cu_q, cu_k, cq, ck, mask = _problem(13, q_lens, k_lens, hq, hk, d, qbs, kbs, 0.4, dtype)
    assert 2 * mask.shape[2] * hk > 9 * torch.cuda.get_device_properties(0).multi_processor_count   # the rule for head dim 64
    print(f"backward of many items {case} {dtype}", flush=True)
    _, *got = _gpu_grads(q, k, v, do, cq, ck, mask, qbs, kbs, causal, None)
    for x, ref, name in zip(got, hbsa_oracle_grads(q, k, v, do, cu_q, cu_k, mask, qbs, kbs, causal, None), ("dq", "dk", "dv")):
        _check(x, ref, name)

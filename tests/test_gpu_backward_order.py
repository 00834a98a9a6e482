"""dK/dV items taken in the order of the rows that can see them, and the form of the kernel for many of them."""
import pytest
import torch

from hbsattn_amd import calculate_blocks
from hbsattn_amd.interface import hbsa_backward, hbsa_prepare, hbsa_run
from oracle.grads import hbsa_oracle_grads
from test_gpu_backward import _check, _problem

pytestmark = pytest.mark.gpu

# 512 items of two rounds and more on 256 CUs: 32 heads x 18 .. 40 k blocks; k blocks of one and two key slots, of a slot and a half
CASES = [
    # q_lens, k_lens, hq, hk, d, qbs, kbs, causal
    ([70, 513, 0, 300], [70, 513, 90, 300], 32, 32, 64, 64, 32, True),      # an empty sequence; 31 blocks a head
    ([40, 700, 130], [900, 200, 130], 36, 36, 64, 48, 48, True),            # keys seen by all rows, rows that see none
    ([200, 333], [1000, 333], 32, 32, 64, 128, 96, False),
    ([90, 260], [260, 90], 36, 36, 32, 16, 16, True),
    ([129, 400, 64], [129, 400, 64], 16, 8, 128, 64, 64, True),
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

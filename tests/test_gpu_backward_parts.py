"""The backward kernels where their items are cut into parts: few heads or blocks, cuts inside a GQA group, inside a 32-block
word of the bit row and beyond its first 64 words, parts without a kept block; and the whole form next to it."""
import ctypes

import pytest
import torch

from hbsattn_amd import _lib, calculate_blocks
from hbsattn_amd.interface import hbsa_backward, hbsa_prepare, hbsa_run
from oracle.grads import hbsa_oracle_grads
from test_gpu_backward import _check, _problem

pytestmark = pytest.mark.gpu

CASES = [
    # q_lens, k_lens, hq, hk, d, qbs, kbs, keep, causal
    ([1], [1], 1, 1, 32, 16, 16, 1.1, True),
    ([2000], [2000], 1, 1, 128, 64, 64, 0.3, True),
    ([1500, 70], [1500, 400], 6, 1, 64, 80, 48, 0.4, False),      # cuts inside the group of six, tiles of 16 rows
    ([900, 0, 333], [700, 100, 2100], 4, 2, 128, 128, 128, 0.3, True),
    ([1100], [2100], 8, 1, 32, 128, 256, 0.5, True),              # two workgroups per k block
    ([160], [36000], 2, 1, 64, 80, 16, 0.05, False),              # 2250 k blocks: the second window of 64 words
    ([4000], [900], 2, 2, 64, 16, 128, 0.02, False),              # most parts of a k block keep nothing
]


def _prepare(cq, ck, mask, qbs, kbs, causal):
    (nq, _, q2b, cu_nq), (nk, _, _, cu_nk) = calculate_blocks(cq, qbs), calculate_blocks(ck, kbs)
    return hbsa_prepare(cq, ck, mask.cuda(), qbs, kbs, causal, nq, q2b, cu_nq, nk, cu_nk)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("case", CASES, ids=[f"case{i}" for i in range(len(CASES))])
def test_parts_match_the_oracle_and_do_not_depend_on_arrival(case, dtype):
    q_lens, k_lens, hq, hk, d, qbs, kbs, keep, causal = case
    q, k, v, do, cu_q, cu_k, cq, ck, mask = _problem(7, q_lens, k_lens, hq, hk, d, qbs, kbs, keep, dtype)
    print(f"backward in parts {case} {dtype}", flush=True)
    qd, kd, vd, dod = (t.cuda() for t in (q, k, v, do))
    prepared = _prepare(cq, ck, mask, qbs, kbs, causal)
    out, lse = hbsa_run(qd, kd, vd, prepared, None, return_lse=True)
    got = hbsa_backward(qd, kd, vd, out, dod, lse, prepared, None)
    for x, ref, name in zip(got, hbsa_oracle_grads(q, k, v, do, cu_q, cu_k, mask, qbs, kbs, causal, None), ("dq", "dk", "dv")):
        _check(x, ref, name)
    for _ in range(3):
        assert all(torch.equal(a, b) for a, b in zip(got, hbsa_backward(qd, kd, vd, out, dod, lse, prepared, None)))
    # captured: the launch may be replayed anywhere, so its counters lie in its own workspace
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = hbsa_backward(qd, kd, vd, out, dod, lse, prepared, None)
    for _ in range(3):
        for t in captured:
            t.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, captured))


def test_a_workspace_without_room_for_parts_is_served_whole():
    lib = _lib.load()
    sizes = (2000, 4, 2, 128, 32, 32, 64, 64)   # total_q, nhead_q, nhead_k, headdim, num_q_block, num_k_block, block sizes
    base, parts = lib.hbsa_bwd_workspace_bytes(2000, 4), lib.hbsa_bwd_workspace_bytes_parts(*sizes)
    assert parts > base
    assert lib.hbsa_bwd_workspace_bytes_parts(2000, 64, 64, *sizes[3:]) == lib.hbsa_bwd_workspace_bytes(2000, 64)   # 2048 items
    q, k, v, do, cu_q, cu_k, cq, ck, mask = _problem(9, [2000], [2000], 4, 2, 128, 64, 64, 0.3, torch.bfloat16)
    qd, kd, vd, dod = (t.cuda() for t in (q, k, v, do))
    prepared = _prepare(cq, ck, mask, 64, 64, True)
    out, lse = hbsa_run(qd, kd, vd, prepared, None, return_lse=True)
    lse = lse.contiguous()
    strides = (ctypes.c_int64 * 16)(*([4 * 128, 128] + [2 * 128, 128] * 2 + [4 * 128, 128] * 3 + [2 * 128, 128] * 2))
    results = []
    for nbytes in (base, parts):
        ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
        dq, dk, dv = torch.empty_like(qd), torch.empty_like(kd), torch.empty_like(vd)
        rc = lib.hbsa_bwd(qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), out.data_ptr(), dod.data_ptr(), lse.data_ptr(), dq.data_ptr(),
                          dk.data_ptr(), dv.data_ptr(), ck.data_ptr(), prepared.cu_num_q_block.data_ptr(),
                          prepared.cu_num_k_block.data_ptr(), prepared.workspace.data_ptr(), prepared.workspace.numel(),
                          ws.data_ptr(), nbytes, 0, 1, 2000, 2000, 4, 2, 128, 32, 32, 64, 64, 1, 128 ** -0.5, strides,
                          torch.cuda.current_stream().cuda_stream)
        assert rc == 0
        results.append((dq, dk, dv))
    refs = hbsa_oracle_grads(q, k, v, do, cu_q, cu_k, mask, 64, 64, True, None)
    for got in results:
        for x, ref, name in zip(got, refs, ("dq", "dk", "dv")):
            _check(x, ref, name)


@pytest.mark.parametrize("kbs", [16, 32, 48, 64, 80])
@pytest.mark.parametrize("hq,hk", [(16, 16), (2, 1)], ids=["whole", "parts"])
def test_key_blocks_of_up_to_64_keys_at_head_dim_128(kbs, hq, hk):
    """Two pairs of wavefronts share 32 keys there (up to 80: the size above); ragged tiles, a last block of one key."""
    q, k, v, do, cu_q, cu_k, cq, ck, mask = _problem(kbs, [333, 97], [321, 129], hq, hk, 128, 80, kbs, 0.6, torch.bfloat16)
    qd, kd, vd, dod = (t.cuda() for t in (q, k, v, do))
    prepared = _prepare(cq, ck, mask, 80, kbs, True)
    out, lse = hbsa_run(qd, kd, vd, prepared, None, return_lse=True)
    got = hbsa_backward(qd, kd, vd, out, dod, lse, prepared, None)
    for x, ref, name in zip(got, hbsa_oracle_grads(q, k, v, do, cu_q, cu_k, mask, 80, kbs, True, None), ("dq", "dk", "dv")):
        _check(x, ref, name)
    assert all(torch.equal(a, b) for a, b in zip(got, hbsa_backward(qd, kd, vd, out, dod, lse, prepared, None)))

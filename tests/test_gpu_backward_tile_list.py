"""The tile list of the dK/dV kernels: lists longer than a chunk of 256 tiles, odd numbers of tiles where
two wavefronts take every other one (head dims up to 64, key blocks of up to 64 keys), tiles of fewer than 64 rows, key blocks whose last part is narrow."""
import ctypes

import pytest
import torch

from hbsattn_amd import _lib, calculate_blocks
from hbsattn_amd.interface import hbsa_backward, hbsa_prepare, hbsa_run
from oracle.grads import hbsa_oracle_grads
from test_gpu_backward import _check, _problem

pytestmark = pytest.mark.gpu


def _prepare(cq, ck, mask, qbs, kbs, causal):
    (nq, _, q2b, cu_nq), (nk, _, _, cu_nk) = calculate_blocks(cq, qbs), calculate_blocks(ck, kbs)
    return hbsa_prepare(cq, ck, mask.cuda(), qbs, kbs, causal, nq, q2b, cu_nq, nk, cu_nk), nq, nk


def _whole(q, k, v, out, do, lse, ck, prepared, nq, nk, qbs, kbs, causal):
    """The gradients without room for parts: one workgroup per item."""
    lib = _lib.load()
    (tq, hq, d), (tk, hk, _) = q.shape, k.shape
    strides = (ctypes.c_int64 * 16)(*([hq * d, d] + [hk * d, d] * 2 + [hq * d, d] * 3 + [hk * d, d] * 2))
    lse = lse.contiguous()
    ws = torch.empty(lib.hbsa_bwd_workspace_bytes(tq, hq), dtype=torch.uint8, device="cuda")
    dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
    rc = lib.hbsa_bwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), do.data_ptr(), lse.data_ptr(), dq.data_ptr(),
                      dk.data_ptr(), dv.data_ptr(), ck.data_ptr(), prepared.cu_num_q_block.data_ptr(), prepared.cu_num_k_block.data_ptr(),
                      prepared.workspace.data_ptr(), prepared.workspace.numel(), ws.data_ptr(), ws.numel(), 0, len(ck) - 1, tq, tk, hq,
                      hk, d, nq, nk, qbs, kbs, int(causal), d ** -0.5, strides, torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    return dq, dk, dv


CASES = [
    # q_lens, k_lens, hq, hk, qbs, kbs, keep, causal
    ([2100], [100], 16, 1, 64, 48, 1.1, False),          # 528 tiles a key block: three chunks; tiles of 64 and of 52 rows
    ([2100], [2100], 9, 1, 80, 64, 0.9, True),           # 80-row blocks, two tiles each, an odd number of heads
    ([1030, 65], [900, 300], 3, 3, 16, 64, 0.7, True),   # tiles of 16 rows; odd numbers of them
    ([64], [64], 1, 1, 64, 64, 1.1, False),              # one tile: nothing for half of the wavefronts
    ([300], [500], 5, 1, 128, 160, 0.8, True),           # 160-key blocks: the last 32 keys are a workgroup of their own
    ([257], [257], 2, 1, 128, 80, 0.8, False),           # 80-key blocks: three slots
]


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("case", CASES, ids=[f"case{i}" for i in range(len(CASES))])
def test_gradients_from_the_tile_list(case, d):
    q_lens, k_lens, hq, hk, qbs, kbs, keep, causal = case
    q, k, v, do, cu_q, cu_k, cq, ck, mask = _problem(11, q_lens, k_lens, hq, hk, d, qbs, kbs, keep, torch.bfloat16)
    qd, kd, vd, dod = (t.cuda().contiguous() for t in (q, k, v, do))
    prepared, nq, nk = _prepare(cq, ck, mask, qbs, kbs, causal)
    out, lse = hbsa_run(qd, kd, vd, prepared, None, return_lse=True)
    refs = hbsa_oracle_grads(q, k, v, do, cu_q, cu_k, mask, qbs, kbs, causal, None)
    for got in (_whole(qd, kd, vd, out, dod, lse, ck, prepared, nq, nk, qbs, kbs, causal),
                hbsa_backward(qd, kd, vd, out, dod, lse, prepared, None)):
        for x, ref, name in zip(got, refs, ("dq", "dk", "dv")):
            _check(x, ref, name)

"""hipStreamPerThread is one handle for every host thread's own stream: calls of two threads on it may overlap."""
import ctypes
import threading

import pytest
import torch

from hbsattn_amd import HBSAttention, _lib
from hbsattn_amd.workloads import make_problem

pytestmark = pytest.mark.gpu

PER_THREAD = ctypes.c_void_p(2)   # hipStreamPerThread


def _call(w, out, ws):
    lib = _lib.load()
    nqb, _, qb2b, cu_nqb = w.q_meta
    nkb, _, _, cu_nkb = w.k_meta
    strides = (ctypes.c_int64 * 11)(*(n for t in (w.q, w.k, w.v, out) for n in t.stride()[:2]), *w.block_mask.stride())
    return lib.hbsa_fwd(w.q.data_ptr(), w.k.data_ptr(), w.v.data_ptr(), out.data_ptr(), w.cu_q_seqlens.data_ptr(), w.cu_k_seqlens.data_ptr(),
                        w.block_mask.data_ptr(), qb2b.data_ptr(), cu_nqb.data_ptr(), cu_nkb.data_ptr(), ws.data_ptr(), ws.numel(),
                        _lib.DTYPE_BF16, len(w.cu_q) - 1, w.q.shape[0], w.k.shape[0], w.q.shape[1], w.k.shape[1], w.q.shape[2], int(nqb),
                        int(nkb), w.q_block_size, w.k_block_size, int(w.causal), w.q.shape[2] ** -0.5, strides, PER_THREAD)


def test_calls_of_two_threads_on_their_own_streams():
    # more items than are handed out without the launch record's queues (8 for each of 768 workgroups); one launch a call
    lib = _lib.load()
    problems = [make_problem(seed=41 + i, q_lens=[4096 - i], k_lens=[4096 - i], hq=32, hk=32, d=64, qbs=16, kbs=64, keep=0.3, diag=True,
                             causal=True, scale=None) for i in range(2)]
    want = [HBSAttention(*w.args()) for w in problems]
    for w in problems:
        for m in (w.q_meta, w.k_meta):
            assert all(t.dtype == torch.int32 and t.is_contiguous() for t in m[2:])
    nqb, nkb = int(problems[0].q_meta[0]), int(problems[0].k_meta[0])
    assert lib.hbsa_fwd_launches(_lib.DTYPE_BF16, 1, 4096, 32, 32, 64, nqb, nkb, 16, 64, 1, PER_THREAD) == 1
    outs = [[torch.zeros_like(w.q) for _ in range(4)] for w in problems]
    ws = [torch.zeros(int(lib.hbsa_fwd_workspace_bytes(32, nqb, nkb)), dtype=torch.uint8, device="cuda") for _ in problems]
    torch.cuda.synchronize()
    codes, start = [], threading.Barrier(2)

    def work(i):
        start.wait()
        for out in outs[i]:
            codes.append(_call(problems[i], out, ws[i]))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert codes == [0] * 8
    assert all(torch.equal(o, want[i]) for i in range(2) for o in outs[i])

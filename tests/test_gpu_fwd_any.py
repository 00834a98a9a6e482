"""hbsa_fwd_any and hbsa_fwd_one through the C interface: exactly the workspace that a split needs, a byte less, one that is not aligned, none;
nothing is written behind it."""
import ctypes

import pytest
import torch

from hbsattn_amd import HBSAttention, _lib
from hbsattn_amd.workloads import make_problem
from helpers import assert_close_to_oracle, oracle_for
from test_gpu_launch_plan import plan_of

pytestmark = pytest.mark.gpu

FILL = 0x5a


def _call(w, out, ws_ptr, n, one=False):
    lib = _lib.load()
    hq, hk, d = w.q.shape[1], w.k.shape[1], w.q.shape[2]
    strides = (ctypes.c_int64 * 11)(hq * d, d, hk * d, d, hk * d, d, hq * d, d, *w.block_mask.stride())
    ptrs = (ctypes.c_void_p * 11)(w.q.data_ptr(), w.k.data_ptr(), w.v.data_ptr(), out.data_ptr(), w.cu_q_seqlens.data_ptr(), w.cu_k_seqlens.data_ptr(),
                                  w.block_mask.data_ptr(), None, w.q_meta[3].data_ptr(), w.k_meta[3].data_ptr(), ws_ptr)
    sizes = (ctypes.c_int32 * 12)(_lib.DTYPE_BF16, len(w.cu_q) - 1, w.q.shape[0], w.k.shape[0], hq, hk, d, w.q_meta[0], w.k_meta[0], w.q_block_size,
                                  w.k_block_size, int(w.causal))
    a, st = ctypes.addressof, torch.cuda.current_stream().cuda_stream
    if one:
        return lib.hbsa_fwd_one(a(ptrs), a(sizes), d ** -0.5, a(strides), st)
    return lib.hbsa_fwd_any(a(ptrs), n, a(sizes), d ** -0.5, a(strides), st)


@pytest.mark.parametrize("d", [64, 80])
def test_workspace_of_a_split(d):
    w = make_problem(seed=95, q_lens=[70, 5], k_lens=[6000, 5000], hq=4, hk=2, d=d, qbs=64, kbs=64, keep=0.4, diag=False, causal=True, scale=None)
    nqb, nkb, rows = w.q_meta[0], w.k_meta[0], 75 * 4
    _, teams, parts, _ = plan_of(False, batch=2, total_q=75, total_k=11000, hq=4, hk=2, d=d, nqb=nqb, nkb=nkb, qbs=64, kbs=64)
    assert teams == 1 and parts > 1
    up = lambda n: (n + 255) // 256 * 256
    need = _lib.load().hbsa_fwd_workspace_bytes_dtype(_lib.DTYPE_BF16, 75, 11000, 4, 2, d, nqb, nkb)
    enough = need + up(parts * rows * d * 4) + up((parts + 1) * rows * 4)
    print(f"any {d} parts {parts}", flush=True)
    ws = torch.full((enough + 4096,), FILL, dtype=torch.uint8, device="cuda")
    out = torch.full_like(w.q, 9.0)
    assert _call(w, out, ws.data_ptr(), enough) == 0
    assert bool((ws[enough:] == FILL).all())
    assert torch.equal(out, HBSAttention(*w.args()))
    assert_close_to_oracle(out, oracle_for(w), "split")
    ws.fill_(FILL)
    out.fill_(9.0)
    rc = _call(w, out, ws.data_ptr(), enough - 1)
    if d == 80:   # such rows have no uncut form of so much work
        assert rc == _lib.ERR_WORKSPACE_TOO_SMALL and bool((out == 9.0).all()) and bool((ws == FILL).all())
        assert _call(w, out, None, 0) == _lib.ERR_WORKSPACE_TOO_SMALL
    else:
        assert rc == 0 and bool((ws[need:] == FILL).all())
        assert_close_to_oracle(out, oracle_for(w), "uncut")
        assert _call(w, out, ws.data_ptr(), need - 1) == _lib.ERR_WORKSPACE_TOO_SMALL
    out.fill_(9.0)
    assert _call(w, out, ws.data_ptr() + 16, enough) == -1 and "aligned" in _lib.last_error()
    assert _call(w, out, None, 0, one=True) == _lib.ERR_WORKSPACE_TOO_SMALL
    assert bool((out == 9.0).all())


@pytest.mark.parametrize("d", [8, 32, 80, 128, 248])
def test_without_a_workspace(d):
    w = make_problem(seed=96, q_lens=[130, 40], k_lens=[200, 90], hq=4, hk=2, d=d, qbs=64, kbs=64, keep=0.6, diag=True, causal=True, scale=None)
    print(f"one {d}", flush=True)
    want = HBSAttention(*w.args())
    for one in (False, True):
        out = torch.full_like(w.q, 9.0)
        assert _call(w, out, None, 0, one) == 0
        assert torch.equal(out, want)
    assert_close_to_oracle(want, oracle_for(w), "one launch")

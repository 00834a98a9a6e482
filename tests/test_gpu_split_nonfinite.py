"""Work cut over its key blocks keeps what is not finite: a row is NaN where its query or a key that it sees is, whichever part that
key falls to and whichever form computes it, and every other row has the bits it has without."""
import pytest
import torch

from hbsattn_amd import HBSAttention, _lib, set_onepass
from hbsattn_amd.workloads import make_problem

pytestmark = pytest.mark.gpu

INF, NAN = float("inf"), float("nan")


def _run(w, form):
    if form == "train":
        q = w.q.detach().requires_grad_(True)
        try:
            return HBSAttention(q, *w.args()[1:]).detach()
        finally:
            w.q.requires_grad_(False)
    previous = set_onepass(form != "prepared")
    try:
        return HBSAttention(*w.args())
    finally:
        set_onepass(previous)


@pytest.mark.parametrize("d,form", [(32, "one"), (64, "one"), (80, "one"), (128, "one"), (256, "one"), (64, "prepared"), (128, "prepared"),
                                    (64, "train"), (128, "train")])
@pytest.mark.parametrize("where,value", [("q", NAN), ("k", NAN), ("k", INF), ("v", NAN)])
@pytest.mark.parametrize("token", [0, 3000, 5999])   # a key of the first part, of one between, of the last
def test_what_is_not_finite_stays(d, form, where, value, token):
    w = make_problem(seed=91, q_lens=[40, 3], k_lens=[6000, 900], hq=4, hk=2, d=d, qbs=64, kbs=64, keep=0.5, diag=True, causal=False,
                     scale=None)
    w.block_mask[1, 0, token // 64] = True
    assert _lib.load().hbsa_fwd_parts_bytes(_lib.DTYPE_BF16, 43, 4, 2, d, w.block_mask.shape[1], w.block_mask.shape[2], 64) > 0
    print(f"not finite {d} {form} {where} {value} {token}", flush=True)
    clean = _run(w, form)
    bad = torch.zeros_like(clean, dtype=torch.bool)
    if where == "q":
        w.q[token % 40, 2, 3] = value
        bad[token % 40, 2] = True
    elif where == "k":
        w.k[token, 1, 3] = value
        bad[:40, 2:] = True
        if value == INF:   # a query whose score is -inf does not see that key
            gone = (w.q[:40, 2:, 3] <= 0)
            bad[:40, 2:][gone] = False
    else:
        w.v[token, 1, 3] = value
        bad[:40, 2:, 3] = True
    out = _run(w, form)
    assert torch.equal(torch.isnan(out), bad)
    if where == "k" and value == INF:   # (their other keys' results are what they are without it, up to the reference they are formed against)
        assert (out.float() - clean.float()).abs()[~bad].max() < 0.1
    else:
        assert torch.equal(out[~bad], clean[~bad])


def test_a_part_of_nan_in_the_log_sum_exp():
    """A row that is NaN has the log-sum-exp -inf, cut or not."""
    import ctypes
    lib = _lib.load()
    w = make_problem(seed=92, q_lens=[40], k_lens=[6000], hq=2, hk=2, d=64, qbs=64, kbs=64, keep=0.5, diag=True, causal=False, scale=None)
    w.q[7, 1, 3] = NAN
    n0 = lib.hbsa_fwd_workspace_bytes_dtype(_lib.DTYPE_BF16, 40, 6000, 2, 2, 64, w.block_mask.shape[1], w.block_mask.shape[2])
    n1 = lib.hbsa_fwd_parts_bytes(_lib.DTYPE_BF16, 40, 2, 2, 64, w.block_mask.shape[1], w.block_mask.shape[2], 64)
    assert n1 > 0
    got = []
    for n in (n0, n0 + n1):   # whole, and cut
        ws = torch.empty(n, dtype=torch.uint8, device="cuda")
        out, lse = torch.empty_like(w.q), torch.empty(40, 2, dtype=torch.float32, device="cuda")
        st = torch.cuda.current_stream().cuda_stream
        ms = (ctypes.c_int64 * 3)(*w.block_mask.stride())
        assert lib.hbsa_fwd_prepare(w.cu_q_seqlens.data_ptr(), w.cu_k_seqlens.data_ptr(), w.block_mask.data_ptr(), None, w.q_meta[3].data_ptr(),
                                    w.k_meta[3].data_ptr(), ws.data_ptr(), n, 1, 2, w.q_meta[0], w.k_meta[0], 64, 64, 0, 40, 6000, ms, st) == 0
        strides = (ctypes.c_int64 * 8)(*([128, 64] * 4))
        assert lib.hbsa_fwd_run_lse(w.q.data_ptr(), w.k.data_ptr(), w.v.data_ptr(), out.data_ptr(), lse.data_ptr(), (ctypes.c_int64 * 2)(2, 1),
                                    ws.data_ptr(), n, _lib.DTYPE_BF16, 40, 6000, 2, 2, 64, w.q_meta[0], w.k_meta[0], 64, 64, 0, 0.125, strides, st) == 0
        got.append((out, lse))
    (whole, lse_whole), (cut, lse_cut) = got
    for t in (whole, cut):
        assert torch.isnan(t[7, 1]).all() and int(torch.isnan(t).sum()) == 64
    assert lse_whole[7, 1] == -INF and lse_cut[7, 1] == -INF
    fine = torch.isfinite(lse_whole)
    assert int(fine.sum()) == 79
    # both are fp32 sums of up to 6000 terms, in another order: 1e-5 of values below 16
    assert (lse_whole - lse_cut)[fine].abs().max() < 2e-4

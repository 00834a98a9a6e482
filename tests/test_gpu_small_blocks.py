"""Prefill and training in 16-row q blocks, one q head per kv head: whole items of the decode kernel, or the other kernel."""
import pytest
import torch

from hbsattn_amd import HBSAttention, _lib
from hbsattn_amd.workloads import make_problem
from helpers import assert_close_to_oracle, oracle_for
from oracle.grads import hbsa_oracle_grads

pytestmark = pytest.mark.gpu


def _problem(d, q_lens, k_lens, heads, kbs, causal, dtype, decodes):
    w = make_problem(seed=d + kbs, q_lens=q_lens, k_lens=k_lens or q_lens, hq=heads, hk=heads, d=d, qbs=16, kbs=kbs, keep=0.5, diag=True,
                     causal=causal, scale=None, dtype=dtype)
    code = _lib.DTYPE_F16 if dtype == torch.float16 else _lib.DTYPE_BF16
    assert _lib.load().hbsa_fwd_decodes(code, w.q.shape[0], heads, heads, w.q_meta[0], w.k_meta[0], 16, kbs) == decodes
    return w


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [32, 64, 128, 256])
@pytest.mark.parametrize("q_lens,k_lens,heads,kbs,causal,decodes", [
    ([100, 37, 16, 1, 15], None, 2, 64, True, 1),        # short, ragged
    ([500], None, 2, 48, False, 1),                      # k blocks smaller than a tile
    ([33, 18], [90, 700], 52, 16, True, 1),              # ... chunks, many items
    ([700, 420], None, 30, 128, True, 1),                # many items
    ([700, 420], None, 3, 128, True, 0),                 # few
    ([64, 48], [3000, 5000], 4, 64, True, 0),            # chunks
])
def test_forward_matches_the_oracle(dtype, d, q_lens, k_lens, heads, kbs, causal, decodes):
    w = _problem(d, q_lens, k_lens, heads, kbs, causal, dtype, decodes)
    out = HBSAttention(*w.args())
    assert_close_to_oracle(out, oracle_for(w), "16-row blocks")
    assert torch.equal(HBSAttention(*w.args()), out)


@pytest.mark.parametrize("decodes,heads", [(1, 2), (0, 3)])
def test_gradients_match_the_oracle(decodes, heads):
    w = _problem(64, [120, 75] if decodes else [700, 420], None, heads, 64, True, torch.bfloat16, decodes)
    args = list(w.args())
    args[:3] = [t.detach().clone().requires_grad_(True) for t in args[:3]]
    dout = torch.randn(w.q.shape, generator=torch.Generator().manual_seed(3)).to(w.q.dtype)
    got = torch.autograd.grad(HBSAttention(*args), args[:3], dout.cuda())
    refs = hbsa_oracle_grads(w.q.cpu(), w.k.cpu(), w.v.cpu(), dout, w.cu_q, w.cu_k, w.block_mask.cpu(), 16, 64, True, None)
    for g, ref in zip(got, refs):
        err = (g.float().cpu() - ref).abs()
        assert err.max().item() <= 1e-2 * max(1.0, ref.abs().max().item()) and err.mean().item() <= 2e-3

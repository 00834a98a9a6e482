"""The public operator: same call as the reference's ``hbsattn.HBSAttention``.

Mirrors reference ``hbsattn/hbsa_interface.py:6-35`` (a ``torch.autograd.Function``
used through ``.apply``, positional arguments, no backward) and the host-side checks
of its two launchers (reference ``hbsattn/fwd_triton_auto_tile_size.py:254-281``,
``hbsattn/fwd_triton_fix_tile_size.py:216-242``).  Both ``tile_mode`` values run the
one HIP kernel family; ``'fix'`` keeps the reference's power-of-two assertion so code
that relies on it behaves the same.
"""
from __future__ import annotations

import collections
import ctypes
import os
import weakref
from typing import Optional

import torch

from . import _lib
from .utils import calculate_blocks

_NATIVE_HEADDIMS = (32, 64, 128, 256)      # head dims every form of the forward has kernels for; others run zero-padded here
_BWD_MAX_HEADDIM = 128                      # the backward kernels stop here
_DTYPE_CODES = {torch.bfloat16: _lib.DTYPE_BF16, torch.float16: _lib.DTYPE_F16, torch.float32: _lib.DTYPE_F32}

# How fp32 q/k/v are multiplied: "exact" = unrounded operands, the arithmetic of the reference's
# fp32 path (``tl.dot(..., allow_tf32=False)``, reference hbsattn/fwd_triton_auto_tile_size.py:205,225);
# "fast" = scaled fp16 staging copies and the 16-bit kernel (11-bit operand significands, several
# times faster).  The environment variable HBSATTN_AMD_FP32_MODE sets the initial mode.
_fp32_mode = os.environ.get("HBSATTN_AMD_FP32_MODE", "exact")
if _fp32_mode not in ("exact", "fast"):
    raise ValueError(f"HBSATTN_AMD_FP32_MODE must be 'exact' or 'fast', not {_fp32_mode!r}")


def set_fp32_mode(mode: str) -> str:
    """Selects how fp32 inputs are multiplied ("exact" or "fast"); returns the previous mode."""
    global _fp32_mode
    if mode not in ("exact", "fast"):
        raise ValueError(f"fp32 mode must be 'exact' or 'fast', not {mode!r}")
    previous, _fp32_mode = _fp32_mode, mode
    return previous


def set_deterministic(on: bool) -> bool:
    """Deterministic mode of the library (``hbsa_set_deterministic``), on by default: every query block
    walks its key tiles in ascending order and results are bitwise reproducible at every size, like the
    reference's kernels.  Switched off (here, or with HBSATTN_AMD_DETERMINISTIC=0 in the environment when
    the library is loaded), very large problems order the walk by a clock shared between workgroups,
    which saves HBM traffic and lets the last bits of the result depend on timing.  Returns the previous
    setting."""
    return bool(_lib.load().hbsa_set_deterministic(1 if on else 0))


def _dtype_code(dtype: torch.dtype) -> int:
    if dtype == torch.float32 and _fp32_mode == "fast":
        return _lib.DTYPE_F32_STAGED16
    return _DTYPE_CODES[dtype]


def _as_int32(t: torch.Tensor) -> torch.Tensor:
    if t.dtype != torch.int32:
        t = t.to(torch.int32)
    return t if t.is_contiguous() else t.contiguous()


def _row_strides(t: torch.Tensor):
    """Token and head stride of ``[tokens, heads, headdim]``.  The stride of a dimension of one element means nothing
    (torch leaves any number there, in a tensor it calls contiguous too): the shape's stands in for it."""
    return (t.shape[1] * t.shape[2] if t.shape[0] == 1 else t.stride(0), t.shape[2] if t.shape[1] == 1 else t.stride(1))


def _rows_ok(t: torch.Tensor) -> bool:
    """16-byte aligned rows with a unit head-dim stride are what the kernels load."""
    unit = 16 // t.element_size()
    tok, head = _row_strides(t)
    return t.stride(2) == 1 and tok % unit == 0 and head % unit == 0 and t.data_ptr() % 16 == 0 and 0 <= tok <= 1 << 24


def _pad_headdim(t: torch.Tensor, d_pad: int) -> torch.Tensor:
    out = t.new_zeros((t.shape[0], t.shape[1], d_pad))
    out[:, :, : t.shape[2]] = t
    return out


class PreparedMask:
    """Result of the pre-pass for one (block_mask, sequence boundaries, block sizes, causal)
    combination: the device scratch the attention kernel reads.  Reusable across calls that
    share those, e.g. the layers of a model that share one sparsity pattern, as long as those calls
    are ordered on ONE stream: the scratch also holds per-launch state (work-queue counters, softmax
    constants, staging copies and split partials), so two ``hbsa_run`` calls on one ``PreparedMask``
    that overlap on different streams corrupt each other."""

    def __init__(self, workspace, nhead_k, num_q_block, num_k_block, q_block_size, k_block_size, causal,
                 cu_k_seqlens=None, cu_num_q_block=None, cu_num_k_block=None):
        self.workspace = workspace
        # int32 device tensors the backward reads besides the workspace
        self.cu_k_seqlens = cu_k_seqlens
        self.cu_num_q_block = cu_num_q_block
        self.cu_num_k_block = cu_num_k_block
        self.nhead_k = nhead_k
        self.num_q_block = num_q_block
        self.num_k_block = num_k_block
        self.q_block_size = q_block_size
        self.k_block_size = k_block_size
        self.causal = bool(causal)

    def skipped_q_blocks(self) -> int:
        """Number of q blocks whose sequence did not fit the tensors it was prepared for (boundaries beyond
        the token counts of q or k/v, inconsistent block metadata).  Such sequences get no keys: their
        output rows and gradients are zeros.  Reads device memory (synchronises): for diagnostics, not
        for the hot path."""
        records = self.workspace[: self.num_q_block * 48].view(torch.int32).view(self.num_q_block, 12)
        return int(records[:, 9].ne(0).sum())


def _check_on_device(dev, **tensors):
    """The kernels dereference these pointers on ``dev``: a host tensor, or one on another GPU, would be
    a memory fault there, not an exception."""
    for name, t in tensors.items():
        if not isinstance(t, torch.Tensor) or t.device != dev:
            where = t.device if isinstance(t, torch.Tensor) else type(t).__name__
            raise RuntimeError(f"{name} must be a tensor on {dev} (the device of block_mask), not on {where}")


def _check_block_sizes(q_block_size, k_block_size):
    assert q_block_size > 0 and k_block_size > 0 and q_block_size % 16 == 0 and k_block_size % 16 == 0, \
        "q_block_size and k_block_size must be integer multiples of 16."


_ws_bytes_cache = {}


def _run_workspace_bytes(lib, device, code, total_q, total_k, nhead_q, nhead_k, headdim, num_q_block, num_k_block,
                         q_block_size) -> int:
    """Bytes ``hbsa_fwd_run`` can use for one call: the work description, fp16 staging copies (fast
    fp32 mode) and room for the split over key blocks the library uses when the work items cannot
    fill the device.  Pure functions of the shape and the device, so the answers are kept."""
    key = (device.index, code, total_q, total_k, nhead_q, nhead_k, headdim, num_q_block, num_k_block, q_block_size)
    need = _ws_bytes_cache.get(key)
    if need is None:
        need = int(lib.hbsa_fwd_workspace_bytes_dtype(code, total_q, total_k, nhead_q, nhead_k, headdim, num_q_block,
                                                      num_k_block))
        with torch.cuda.device(device):
            need += int(lib.hbsa_fwd_parts_bytes(code, total_q, nhead_q, nhead_k, headdim, num_q_block, num_k_block,
                                                 q_block_size))
        if len(_ws_bytes_cache) > 4096:
            _ws_bytes_cache.clear()
        _ws_bytes_cache[key] = need
    return need


def hbsa_prepare(cu_q_seqlens, cu_k_seqlens, block_mask, q_block_size, k_block_size, causal, num_q_block,
                 q_block_to_batch, cu_num_q_block, num_k_block, cu_num_k_block, run_shape=None) -> PreparedMask:
    """Runs the pre-pass kernel (``hbsa_fwd_prepare``) on the current stream.  ``run_shape`` =
    ``(dtype, total_q, total_k, nhead_q, headdim)`` of the q/k/v the mask will be used with sizes the
    workspace for them at once (``hbsa_run`` grows it otherwise) and gives the pre-pass the token counts it
    checks the sequence boundaries against: a sequence that does not fit the tensors is skipped as a
    whole instead of being read and written out of bounds (without ``run_shape`` nothing is checked)."""
    if not block_mask.is_cuda:
        raise RuntimeError("hbsattn_amd runs on MI355X only: block_mask must be a CUDA(HIP) tensor; there is no CPU path")
    _check_block_sizes(q_block_size, k_block_size)
    if block_mask.dtype != torch.bool:
        raise TypeError(f"block_mask must be a boolean tensor, not {block_mask.dtype}")
    if block_mask.dim() != 3 or tuple(block_mask.shape[1:]) != (int(num_q_block), int(num_k_block)):
        raise ValueError("block_mask must have shape (nheads_k, num_q_block, num_k_block) = "
                         f"(*, {int(num_q_block)}, {int(num_k_block)}), not {tuple(block_mask.shape)}")
    dev = block_mask.device
    _check_on_device(dev, cu_q_seqlens=cu_q_seqlens, cu_k_seqlens=cu_k_seqlens, q_block_to_batch=q_block_to_batch,
                     cu_num_q_block=cu_num_q_block, cu_num_k_block=cu_num_k_block)
    if cu_q_seqlens.numel() != cu_k_seqlens.numel() or cu_num_q_block.numel() != cu_q_seqlens.numel() \
            or cu_num_k_block.numel() != cu_q_seqlens.numel() or q_block_to_batch.numel() != int(num_q_block):
        raise ValueError("sequence boundaries and block metadata disagree in length (batch + 1 entries each, "
                         "num_q_block entries in q_block_to_batch)")
    lib = _lib.load()
    nhead_k = block_mask.shape[0]
    ws_bytes = int(lib.hbsa_fwd_workspace_bytes(nhead_k, num_q_block, num_k_block))
    bound_q = bound_k = 2 ** 31 - 1
    if run_shape is not None:
        dtype, total_q, total_k, nhead_q, headdim = run_shape
        bound_q, bound_k = int(total_q), int(total_k)
        d_run = next((d for d in _NATIVE_HEADDIMS if d >= headdim), headdim)
        if dtype in _DTYPE_CODES and total_q > 0 and nhead_q > 0:
            ws_bytes = max(ws_bytes, _run_workspace_bytes(lib, dev, _dtype_code(dtype), total_q, total_k, nhead_q, nhead_k,
                                                          d_run, num_q_block, num_k_block, q_block_size))
    workspace = torch.empty(ws_bytes, dtype=torch.uint8, device=dev)
    cu_q, cu_k = _as_int32(cu_q_seqlens), _as_int32(cu_k_seqlens)
    qb2b, cu_nqb, cu_nkb = _as_int32(q_block_to_batch), _as_int32(cu_num_q_block), _as_int32(cu_num_k_block)
    mstr = (ctypes.c_int64 * 3)(*block_mask.stride())
    with torch.cuda.device(dev):
        rc = lib.hbsa_fwd_prepare(cu_q.data_ptr(), cu_k.data_ptr(), block_mask.data_ptr(), qb2b.data_ptr(),
                                  cu_nqb.data_ptr(), cu_nkb.data_ptr(), workspace.data_ptr(), ws_bytes, cu_q.numel() - 1,
                                  nhead_k, num_q_block, num_k_block, q_block_size, k_block_size, int(bool(causal)),
                                  bound_q, bound_k, mstr, torch.cuda.current_stream().cuda_stream)
    if rc != 0:
        raise RuntimeError(f"hbsa_fwd_prepare failed (code {rc}): {_lib.last_error()}")
    return PreparedMask(workspace, nhead_k, num_q_block, num_k_block, q_block_size, k_block_size, causal, cu_k, cu_nqb,
                        cu_nkb)


def hbsa_run(q, k, v, prepared: PreparedMask, softmax_scale, return_lse: bool = False):
    """Runs the attention kernel (``hbsa_fwd_run`` / ``hbsa_fwd_run_lse``) on the current stream from a
    prepared mask (calls that share a ``PreparedMask`` must be ordered on one stream; a call may
    replace ``prepared.workspace`` by a larger one).  With ``return_lse`` the result is ``(out, lse)``, ``lse`` a float32
    ``[total_q, nhead_q]`` tensor: log of the sum over a row's visible keys of exp(scale * q.k)."""
    if not q.is_cuda:
        raise RuntimeError("hbsattn_amd runs on MI355X only: q/k/v must be CUDA(HIP) tensors; there is no CPU path")
    if not (k.device == q.device and v.device == q.device and prepared.workspace.device == q.device):
        raise RuntimeError("q, k, v and block_mask must live on the same device")
    if q.dim() != 3 or k.dim() != 3 or v.dim() != 3:
        raise ValueError("q, k, v must have shape (total_tokens, nheads, headdim)")
    if not (k.dtype == q.dtype and v.dtype == q.dtype):
        raise TypeError("q, k and v must share one dtype")
    if q.dtype not in _DTYPE_CODES:
        raise TypeError(f"hbsattn_amd: dtype {q.dtype} is not supported (bfloat16, float16 and float32 are)")
    total_q, nhead_q, headdim = q.shape
    total_k, nhead_k = k.shape[0], k.shape[1]
    if k.shape[2] != headdim or v.shape != k.shape:
        raise ValueError("k and v must have shape (total_k, nhead_k, headdim) with q's headdim")
    if nhead_k != prepared.nhead_k:
        raise ValueError("k has a different number of heads than the prepared block_mask")
    assert nhead_q % nhead_k == 0, "nhead_q must be divisible by nhead_k (for GQA)"
    if headdim > _NATIVE_HEADDIMS[-1]:
        raise NotImplementedError(f"hbsattn_amd: headdim {headdim} > {_NATIVE_HEADDIMS[-1]} is not supported")
    scale = float(softmax_scale) if softmax_scale is not None else headdim ** -0.5

    lib = _lib.load()
    out = torch.empty((total_q, nhead_q, headdim), dtype=q.dtype, device=q.device)
    lse = torch.empty((total_q, nhead_q), dtype=torch.float32, device=q.device) if return_lse else None
    if total_q == 0:
        return (out, lse) if return_lse else out
    d_run = next(d for d in _NATIVE_HEADDIMS if d >= headdim)
    if d_run != headdim:  # zero columns add nothing to q.k and give zero output columns
        q, k, v = _pad_headdim(q, d_run), _pad_headdim(k, d_run), _pad_headdim(v, d_run)
        out_run = torch.empty((total_q, nhead_q, d_run), dtype=q.dtype, device=q.device)
    else:
        q = q if _rows_ok(q) else q.contiguous()
        k = k if _rows_ok(k) else k.contiguous()
        v = v if _rows_ok(v) else v.contiguous()
        out_run = out
    strides = (ctypes.c_int64 * 8)(*(n for t in (q, k, v, out_run) for n in _row_strides(t)))
    ws = prepared.workspace
    code = _dtype_code(q.dtype)
    need = _run_workspace_bytes(lib, q.device, code, total_q, total_k, nhead_q, nhead_k, d_run, prepared.num_q_block,
                                prepared.num_k_block, prepared.q_block_size)
    if ws.numel() < need:
        grown = torch.empty(need, dtype=torch.uint8, device=ws.device)
        grown[: ws.numel()].copy_(ws)
        prepared.workspace = ws = grown
    with torch.cuda.device(q.device):
        lse_strides = (ctypes.c_int64 * 2)(*lse.stride()) if return_lse else None
        rc = lib.hbsa_fwd_run_lse(q.data_ptr(), k.data_ptr(), v.data_ptr(), out_run.data_ptr(),
                                  lse.data_ptr() if return_lse else None, lse_strides, ws.data_ptr(), ws.numel(),
                                  code, total_q, total_k, nhead_q, nhead_k, d_run, prepared.num_q_block,
                                  prepared.num_k_block, prepared.q_block_size, prepared.k_block_size,
                                  int(prepared.causal), scale, strides, torch.cuda.current_stream().cuda_stream)
    if rc != 0:
        raise RuntimeError(f"hbsa_fwd_run failed (code {rc}): {_lib.last_error()}")
    # The launch is queued on the current stream; torch's caching allocator keeps padded copies
    # alive until work queued on that stream before their release has run.
    if out_run is not out:
        out.copy_(out_run[:, :, :headdim])
    return (out, lse) if return_lse else out


def backward_supported(q: torch.Tensor) -> bool:
    """The backward kernels take bf16 / fp16 tensors; head dims up to 128 (others than 32, 64, 128 run
    zero-padded, like the forward).  fp32 tensors get their gradients from the bf16 kernels on rounded
    copies (``hbsa_backward``).  The forward alone goes up to head dim 256."""
    return q.dtype in _DTYPE_CODES and q.dim() == 3 and 0 < q.shape[2] <= _BWD_MAX_HEADDIM


def hbsa_backward(q, k, v, out, dout, lse, prepared: PreparedMask, softmax_scale):
    """``(dq, dk, dv)`` through ``hbsa_bwd`` on the current stream.  ``out`` and ``lse`` are what
    ``hbsa_run(..., return_lse=True)`` returned for the same q, k, v, prepared mask and scale."""
    if not backward_supported(q):
        raise NotImplementedError("hbsattn_amd: the backward takes bfloat16 / float16 / float32 tensors with headdim <= 128")
    if q.dtype == torch.float32:
        # There are no fp32 backward kernels (the fp32 matrix rate is a sixteenth of the 16-bit one, and the
        # backward is 2.5 forwards).  The gradients are those of the bf16 computation on rounded copies of q, k, v
        # (bf16 keeps fp32's range, so no scaling is involved; 8-bit operand significands, fp32 accumulation): its
        # forward is run again for the output and log-sum-exp that belong to the rounded operands (the
        # probabilities the backward forms from them then sum to one), and the gradients are returned as fp32.
        lo = torch.bfloat16
        q16, k16, v16 = q.to(lo), k.to(lo), v.to(lo)
        out16, lse16 = hbsa_run(q16, k16, v16, prepared, softmax_scale, return_lse=True)
        dq, dk, dv = hbsa_backward(q16, k16, v16, out16, dout.to(lo), lse16, prepared, softmax_scale)
        return dq.float(), dk.float(), dv.float()
    if prepared.cu_k_seqlens is None:
        raise ValueError("this PreparedMask was built without the sequence boundaries the backward needs")
    _check_on_device(prepared.workspace.device, q=q, k=k, v=v, out=out, dout=dout, lse=lse)
    lib = _lib.load()
    total_q, nhead_q, headdim = q.shape
    total_k, nhead_k = k.shape[0], k.shape[1]
    scale = float(softmax_scale) if softmax_scale is not None else headdim ** -0.5
    if total_q == 0 or total_k == 0:
        return torch.zeros_like(q), torch.zeros_like(k), torch.zeros_like(v)
    d_run = next(d for d in _NATIVE_HEADDIMS if d >= headdim)
    if d_run != headdim:  # zero columns change neither q.k nor rowsum(dout * out) and get zero gradients
        q, k, v, out, dout = (_pad_headdim(t, d_run) for t in (q, k, v, out, dout))
    else:
        q = q if _rows_ok(q) else q.contiguous()
        k = k if _rows_ok(k) else k.contiguous()
        v = v if _rows_ok(v) else v.contiguous()
        out = out if _rows_ok(out) else out.contiguous()
        dout = dout if _rows_ok(dout) else dout.contiguous()
    lse = lse.contiguous()
    dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
    bws_bytes = int(lib.hbsa_bwd_workspace_bytes_parts(total_q, nhead_q, nhead_k, d_run, prepared.num_q_block, prepared.num_k_block,
                                                       prepared.q_block_size, prepared.k_block_size))
    bws = torch.empty(bws_bytes, dtype=torch.uint8, device=q.device)
    strides = (ctypes.c_int64 * 16)(*(n for t in (q, k, v, out, dout, dq, dk, dv) for n in _row_strides(t)))
    ws = prepared.workspace
    with torch.cuda.device(q.device):
        rc = lib.hbsa_bwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), dout.data_ptr(), lse.data_ptr(),
                          dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), prepared.cu_k_seqlens.data_ptr(),
                          prepared.cu_num_q_block.data_ptr(), prepared.cu_num_k_block.data_ptr(), ws.data_ptr(), ws.numel(),
                          bws.data_ptr(), bws_bytes, _dtype_code(q.dtype), prepared.cu_k_seqlens.numel() - 1, total_q,
                          total_k, nhead_q, nhead_k, d_run, prepared.num_q_block, prepared.num_k_block,
                          prepared.q_block_size, prepared.k_block_size, int(prepared.causal), scale, strides,
                          torch.cuda.current_stream().cuda_stream)
    if rc != 0:
        raise RuntimeError(f"hbsa_bwd failed (code {rc}): {_lib.last_error()}")
    if d_run != headdim:
        dq, dk, dv = (t[:, :, :headdim].contiguous() for t in (dq, dk, dv))
    return dq, dk, dv


# Prepared masks of recent calls (opt-in: set_prepared_cache_size(n) or HBSATTN_AMD_PREPARED_CACHE=n).  A
# model applies one sparsity pattern in many layers and steps, and the reference's own sweep calls the
# operator many times on one mask (reference test/test_speedup.py:101-152); the pre-pass result depends only
# on (block_mask, sequence boundaries, block sizes, causal), so a call that repeats those launches the
# attention kernel alone.  An entry is reused only for the SAME tensor objects (held weakly) at the same
# version counters, and only on the stream it was made on (its workspace also holds per-launch state).
# Off by default because torch's version counters do not see writes made behind its back: a mask buffer
# that a custom kernel (or ``mask.data``) rewrites in place would be served from a stale entry.
_prepared_cache = collections.OrderedDict()
_prepared_cache_size = max(0, int(os.environ.get("HBSATTN_AMD_PREPARED_CACHE", "0")))


def set_prepared_cache_size(n: int) -> int:
    """Number of prepared masks kept for reuse (0 switches the reuse off); returns the previous value."""
    global _prepared_cache_size
    previous, _prepared_cache_size = _prepared_cache_size, max(0, int(n))
    while len(_prepared_cache) > _prepared_cache_size:
        _prepared_cache.popitem(last=False)
    return previous


def clear_prepared_cache() -> None:
    _prepared_cache.clear()


def _cached_prepare(cu_q_seqlens, cu_k_seqlens, block_mask, q_block_size, k_block_size, causal, num_q_block,
                    q_block_to_batch, cu_num_q_block, num_k_block, cu_num_k_block, run_shape) -> PreparedMask:
    # everything the pre-pass reads or bakes in: the mask, the boundaries, the block metadata, and the
    # token counts the boundaries were checked against
    tensors = (block_mask, cu_q_seqlens, cu_k_seqlens, q_block_to_batch, cu_num_q_block, cu_num_k_block)
    key = None
    if _prepared_cache_size > 0 and all(isinstance(t, torch.Tensor) for t in tensors) and block_mask.is_cuda:
        try:
            key = tuple((id(t), t._version, t.data_ptr(), tuple(t.shape), tuple(t.stride())) for t in tensors) + (
                int(q_block_size), int(k_block_size), bool(causal), int(num_q_block), int(num_k_block),
                None if run_shape is None else (int(run_shape[1]), int(run_shape[2])),
                block_mask.device.index, torch.cuda.current_stream(block_mask.device).cuda_stream)
        except RuntimeError:   # tensors without a version counter (inference mode): no reuse
            key = None
    if key is not None:
        hit = _prepared_cache.get(key)
        if hit is not None:
            prepared, refs = hit
            if all(r() is t for r, t in zip(refs, tensors)):
                _prepared_cache.move_to_end(key)
                return prepared
            del _prepared_cache[key]   # an address and id reused by other tensors
    prepared = hbsa_prepare(cu_q_seqlens, cu_k_seqlens, block_mask, q_block_size, k_block_size, causal, num_q_block,
                            q_block_to_batch, cu_num_q_block, num_k_block, cu_num_k_block, run_shape)
    if key is not None:
        _prepared_cache[key] = (prepared, tuple(weakref.ref(t) for t in tensors))
        while len(_prepared_cache) > _prepared_cache_size:
            _prepared_cache.popitem(last=False)
    return prepared


# The one-launch form is also a switch of the compiled host path: with it off, calls take the general path below.
_onepass = os.environ.get("HBSATTN_AMD_ONEPASS", "1") != "0"


def set_onepass(on: bool) -> bool:
    """The library's one-launch form of the forward (``hbsa_set_onepass``), on by default; returns the
    previous setting."""
    global _onepass
    _onepass = bool(on)
    return bool(_lib.load().hbsa_set_onepass(1 if on else 0))


def hbsa_forward(q, k, v, cu_q_seqlens, cu_k_seqlens, block_mask, q_block_size, k_block_size, causal, softmax_scale,
                 num_q_block, q_block_to_batch, cu_num_q_block, num_k_block, cu_num_k_block, ctx=None) -> torch.Tensor:
    """Host launcher of the calls the compiled host path leaves alone: checks, scratch allocation, pre-pass (skipped when
    the same mask and sequence boundaries were prepared by a recent call) and attention kernel.
    No device synchronisation happens here."""
    if not q.is_cuda:
        raise RuntimeError("hbsattn_amd runs on MI355X only: q/k/v must be CUDA(HIP) tensors; there is no CPU path")
    if block_mask.device != q.device:
        raise RuntimeError("q, k, v and block_mask must live on the same device")
    assert q.shape[1] % k.shape[1] == 0, "nhead_q must be divisible by nhead_k (for GQA)"
    wants_grad = ctx is not None and any(ctx.needs_input_grad[:3]) and backward_supported(q)
    run_shape = (q.dtype, q.shape[0], k.shape[0], q.shape[1], q.shape[2]) if q.dim() == 3 and k.dim() == 3 else None
    prepared = _cached_prepare(cu_q_seqlens, cu_k_seqlens, block_mask, q_block_size, k_block_size, causal, num_q_block,
                               q_block_to_batch, cu_num_q_block, num_k_block, cu_num_k_block, run_shape)
    if wants_grad:
        # keep what the backward needs: the log-sum-exp, the output and the prepared mask
        out, lse = hbsa_run(q, k, v, prepared, softmax_scale, return_lse=True)
        ctx.save_for_backward(q, k, v, out, lse)
        ctx.prepared = prepared
        ctx.softmax_scale = softmax_scale
        return out
    return hbsa_run(q, k, v, prepared, softmax_scale)


class _HBSAttentionFunction(torch.autograd.Function):
    """Positional signature identical to reference ``hbsattn/hbsa_interface.py:9``."""

    @staticmethod
    def forward(ctx, q, k, v, cu_q_seqlens, cu_k_seqlens, block_mask, q_block_size, k_block_size, causal,
                softmax_scale, tile_mode="auto", num_q_block=None, cu_q_block=None, q_block_to_batch=None,
                cu_num_q_block=None, num_k_block=None, cu_k_block=None, k_block_to_batch=None, cu_num_k_block=None):
        # Block metadata is all-or-recompute per side (reference hbsa_interface.py:14-17).
        if num_q_block is None or cu_q_block is None or q_block_to_batch is None or cu_num_q_block is None:
            num_q_block, cu_q_block, q_block_to_batch, cu_num_q_block = calculate_blocks(cu_q_seqlens, q_block_size)
        if num_k_block is None or cu_k_block is None or k_block_to_batch is None or cu_num_k_block is None:
            num_k_block, cu_k_block, k_block_to_batch, cu_num_k_block = calculate_blocks(cu_k_seqlens, k_block_size)

        assert block_mask.dtype == torch.bool, "block_mask must be a boolean tensor"
        assert block_mask.shape == (k.shape[1], num_q_block, num_k_block), (
            "block_mask must be a boolean tensor of shape (nheads_k, num_q_block, num_k_block) = "
            f"({k.shape[1]}, {num_q_block}, {num_k_block})")

        if tile_mode == "auto":
            pass
        elif tile_mode == "fix":
            assert (q_block_size & (q_block_size - 1) == 0) and (k_block_size & (k_block_size - 1) == 0), \
                "q_block_size and k_block_size must be powers of 2"
        else:
            raise ValueError(f"Invalid tile mode: {tile_mode}")
        return hbsa_forward(q, k, v, cu_q_seqlens, cu_k_seqlens, block_mask, q_block_size, k_block_size, causal,
                            softmax_scale, int(num_q_block), q_block_to_batch, cu_num_q_block, int(num_k_block),
                            cu_num_k_block, ctx=ctx)

    @staticmethod
    def backward(ctx, do):
        # The reference stops here (reference hbsattn/hbsa_interface.py:31-32 raises NotImplementedError);
        # head dims up to 128 get their gradients, anything else still raises.
        if getattr(ctx, "prepared", None) is None:
            raise NotImplementedError("It does not support gradient propagation yet for this dtype / headdim")
        q, k, v, out, lse = ctx.saved_tensors
        dq, dk, dv = hbsa_backward(q, k, v, out, do, lse, ctx.prepared, ctx.softmax_scale)
        return (dq, dk, dv) + (None,) * 16


_host_call = None


def _load_host_call():
    global _host_call
    _host_call = _lib.host().call
    return _host_call


def HBSAttention(q, k, v, cu_q_seqlens, cu_k_seqlens, block_mask, q_block_size, k_block_size, causal, softmax_scale,
                 tile_mode="auto", num_q_block=None, cu_q_block=None, q_block_to_batch=None, cu_num_q_block=None,
                 num_k_block=None, cu_k_block=None, k_block_to_batch=None, cu_num_k_block=None):
    """Same call as the reference's ``HBSAttention`` (``_HBSAttentionFunction.apply``, reference
    ``hbsattn/hbsa_interface.py:35``).  The ordinary call, with or without gradients and block metadata, runs in the
    compiled host path (``csrc/torch_host.cpp``); what that leaves alone (it returns ``None``) runs, and is reported, here."""
    if _prepared_cache_size == 0 and _onepass and isinstance(q, torch.Tensor) and q.is_cuda:
        out = (_host_call or _load_host_call())(
            q, k, v, cu_q_seqlens, cu_k_seqlens, block_mask, q_block_size, k_block_size, causal, softmax_scale, tile_mode,
            num_q_block, cu_q_block, q_block_to_batch, cu_num_q_block, num_k_block, cu_k_block, k_block_to_batch,
            cu_num_k_block, _lib.DTYPE_F32 if _fp32_mode == "exact" else _lib.DTYPE_F32_STAGED16)
        if out is not None:
            return out
    if torch.is_grad_enabled() and (q.requires_grad or k.requires_grad or v.requires_grad):
        return _HBSAttentionFunction.apply(q, k, v, cu_q_seqlens, cu_k_seqlens, block_mask, q_block_size, k_block_size,
                                           causal, softmax_scale, tile_mode, num_q_block, cu_q_block, q_block_to_batch,
                                           cu_num_q_block, num_k_block, cu_k_block, k_block_to_batch, cu_num_k_block)
    return _HBSAttentionFunction.forward(None, q, k, v, cu_q_seqlens, cu_k_seqlens, block_mask, q_block_size, k_block_size,
                                         causal, softmax_scale, tile_mode, num_q_block, cu_q_block, q_block_to_batch,
                                         cu_num_q_block, num_k_block, cu_k_block, k_block_to_batch, cu_num_k_block)

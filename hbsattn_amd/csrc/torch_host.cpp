// Host path of hbsattn_amd.HBSAttention: argument checks, allocations, launches and autograd in C++ over the C ABI of
// libhbsattn_amd.so (include/hbsattn_amd.h).  At the sizes where a call's kernels take tens of microseconds the
// Python statements around them are most of a call: 8 us for a plain call, 38 with a workspace, 200 for a call with
// gradients (two trips of the interpreter lock between the caller's thread and autograd's), 330 when the block metadata
// was left to the call (about forty small torch launches and two waits for the device).  Measured with this path: 5, 14,
// 74 and 12 us.
//
// `call` takes the ordinary case of every argument and returns None for anything else (CPU tensors, wrong types or
// shapes, head dims and strides that need copies, tensor subclasses), which hbsattn_amd/interface.py then handles, and
// reports, in Python.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/core/grad_mode.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>

#include <atomic>
#include <cmath>

#include "count_slots.h"
#include "hbsattn_amd.h"

namespace {

// The current device is `index` inside the scope.
struct OnDevice {
  int before;
  explicit OnDevice(int index) : before(c10::hip::current_device()) {
    if (index != before) c10::hip::set_device((c10::DeviceIndex)index);
    else before = -1;
  }
  ~OnDevice() {
    if (before >= 0) c10::hip::set_device((c10::DeviceIndex)before);
  }
};

// ---- Pinned slots the device writes block counts to (count_slots.h).  A call that finds none free goes the long way round.
hbsa_host::CountSlots g_slots;
std::atomic<int32_t> g_ticket{0};

int32_t *count_page() {
  void *p = nullptr;
  constexpr size_t n = hbsa_host::kSlots * hbsa_host::kSlotInts;
  if (hipHostMalloc(&p, n * sizeof(int32_t), hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess) {
    (void)hipGetLastError();
    return nullptr;
  }
  for (size_t i = 0; i < n; ++i) ((int32_t *)p)[i] = 0;
  return (int32_t *)p;
}

struct StateOf {
  hipStream_t stream;
  hbsa_host::StreamState operator()() const {
    const hipError_t e = hipStreamQuery(stream);
    if (e == hipErrorNotReady) return hbsa_host::StreamState::kBusy;
    if (e == hipSuccess) return hbsa_host::StreamState::kIdle;
    (void)hipGetLastError();
    return hbsa_host::StreamState::kUnknown;
  }
};
using CountTicket = hbsa_host::CountTicket<StateOf>;

struct Problem {
  at::Tensor q, k, v, mask;
  at::Tensor cu_q, cu_k, qb2b, cu_nqb, cu_nkb;   // int32, contiguous, on q's device
  int64_t qbs, kbs, nqb, nkb;
  bool causal;
  double scale;
  int dtype;   // HBSA_DTYPE_*
};

bool int32_on(const at::Tensor &t, int index, int64_t n) {
  return t.scalar_type() == at::kInt && t.is_cuda() && t.get_device() == index && t.numel() == n && t.is_contiguous();
}

// Token and head stride of [tokens, heads, head dim].  The stride of a dimension of one element means nothing (torch leaves
// any number there, in a tensor it calls contiguous too): the shape's stands in for it.
int64_t tok_stride(const at::Tensor &t) { return t.size(0) == 1 ? t.size(1) * t.size(2) : t.stride(0); }
int64_t head_stride(const at::Tensor &t) { return t.size(1) == 1 ? t.size(2) : t.stride(1); }

// 16-byte rows with a unit head-dim stride, and token strides the kernels' 32-bit tile offsets can hold
bool rows_ok(const at::Tensor &t) {
  const int64_t unit = 16 / t.element_size(), tok = tok_stride(t);
  return t.stride(2) == 1 && tok % unit == 0 && head_stride(t) % unit == 0 && (uintptr_t)t.const_data_ptr() % 16 == 0 && tok >= 0 &&
         tok <= (1 << 24);
}

[[noreturn]] void raise(const char *what, int rc) {
  TORCH_CHECK(false, what, " failed (code ", rc, "): ", hbsa_last_error());
  __builtin_unreachable();
}

// Room for partial results of work that is cut over its key blocks (0: it is not), and the whole workspace
size_t parts_bytes(const Problem &p) {
  return hbsa_fwd_parts_bytes(p.dtype, (int)p.q.size(0), (int)p.q.size(1), (int)p.k.size(1), (int)p.q.size(2), (int)p.nqb, (int)p.nkb,
                              (int)p.qbs);
}
size_t workspace_bytes(const Problem &p) {
  return hbsa_fwd_workspace_bytes_dtype(p.dtype, (int)p.q.size(0), (int)p.k.size(0), (int)p.q.size(1), (int)p.k.size(1),
                                        (int)p.q.size(2), (int)p.nqb, (int)p.nkb) + parts_bytes(p);
}

at::Tensor bytes_like(const at::Tensor &t, size_t n) { return at::empty({(int64_t)n}, t.options().dtype(at::kByte)); }

bool native_dim(int64_t d) { return d == 32 || d == 64 || d == 128 || d == 256; }

// Computes `out` (like q).  False when the head dim has to be padded first, or (with a ticket for the block counts) when the call is not
// one launch that counts the blocks itself; nothing has been launched then.
bool plain_forward(const Problem &p, hipStream_t stream, at::Tensor &out, CountTicket *counts = nullptr) {
  const int64_t strides[11] = {tok_stride(p.q), head_stride(p.q), tok_stride(p.k), head_stride(p.k), tok_stride(p.v), head_stride(p.v),
                               tok_stride(out), head_stride(out), p.mask.stride(0), p.mask.stride(1),
                               p.mask.size(2) == 1 ? 1 : p.mask.stride(2)};
  const int32_t sizes[12] = {p.dtype, (int32_t)(p.cu_q.numel() - 1), (int32_t)p.q.size(0), (int32_t)p.k.size(0),
                             (int32_t)p.q.size(1), (int32_t)p.k.size(1), (int32_t)p.q.size(2), (int32_t)p.nqb, (int32_t)p.nkb,
                             (int32_t)p.qbs, (int32_t)p.kbs, p.causal ? 1 : 0};
  const void *ptrs[11] = {p.q.const_data_ptr(), p.k.const_data_ptr(), p.v.const_data_ptr(), out.mutable_data_ptr(),
                          p.cu_q.const_data_ptr(), p.cu_k.const_data_ptr(), p.mask.const_data_ptr(),
                          p.qb2b.defined() ? p.qb2b.const_data_ptr() : nullptr, p.cu_nqb.defined() ? p.cu_nqb.const_data_ptr() : nullptr,
                          p.cu_nkb.defined() ? p.cu_nkb.const_data_ptr() : nullptr, nullptr};
  if (counts != nullptr) {
    const int rc = hbsa_fwd_counted(ptrs, sizes, (float)p.scale, strides, counts->slot, counts->ticket, stream);
    counts->launched = rc >= 0;   // (negative codes: refused, nothing will write the ticket)
    if (rc == HBSA_ERR_WORKSPACE_TOO_SMALL) return false;
    if (rc != 0) raise("hbsa_fwd_counted", rc);
    return true;
  }
  if (!native_dim(p.q.size(2))) {
    const size_t n = parts_bytes(p) == 0 ? 0 : workspace_bytes(p);
    at::Tensor ws;
    if (n != 0) {
      ws = bytes_like(p.q, n);
      ptrs[10] = ws.mutable_data_ptr();
    }
    const int rc = hbsa_fwd_any(ptrs, n, sizes, (float)p.scale, strides, stream);
    if (rc == HBSA_ERR_WORKSPACE_TOO_SMALL) return false;   // neither form that reads such rows: the caller pads
    if (rc != 0) raise("hbsa_fwd_any", rc);
    return true;
  }
  int rc = HBSA_ERR_WORKSPACE_TOO_SMALL;
  if (p.dtype < HBSA_DTYPE_F32 && parts_bytes(p) == 0) rc = hbsa_fwd_v(ptrs, 0, sizes, (float)p.scale, strides, stream);
  if (rc == HBSA_ERR_WORKSPACE_TOO_SMALL) {   // nothing was launched: this call needs a workspace
    const size_t n = workspace_bytes(p);
    at::Tensor ws = bytes_like(p.q, n);
    ptrs[10] = ws.mutable_data_ptr();
    rc = hbsa_fwd_any(ptrs, n, sizes, (float)p.scale, strides, stream);
  }
  if (rc != 0) raise("hbsa_fwd", rc);
  return true;
}

// ---- the call with gradients
struct Attention : public torch::autograd::Function<Attention> {
  static at::Tensor forward(torch::autograd::AutogradContext *ctx, const at::Tensor &q, const at::Tensor &k, const at::Tensor &v,
                            const Problem &p) {
    at::AutoDispatchBelowADInplaceOrView guard;
    const OnDevice on(q.get_device());
    const hipStream_t stream = c10::hip::getCurrentHIPStream((c10::DeviceIndex)q.get_device()).stream();
    const int batch = (int)p.cu_q.numel() - 1, tq = (int)q.size(0), tk = (int)k.size(0), hq = (int)q.size(1), hk = (int)k.size(1),
              d = (int)q.size(2), nqb = (int)p.nqb, nkb = (int)p.nkb;
    const size_t n = workspace_bytes(p);
    at::Tensor ws = bytes_like(q, n);
    const int64_t mask_strides[3] = {p.mask.stride(0), p.mask.stride(1), p.mask.stride(2)};
    int rc = hbsa_fwd_prepare(p.cu_q.const_data_ptr<int32_t>(), p.cu_k.const_data_ptr<int32_t>(), (const uint8_t *)p.mask.const_data_ptr(),
                              p.qb2b.defined() ? p.qb2b.const_data_ptr<int32_t>() : nullptr, p.cu_nqb.const_data_ptr<int32_t>(),
                              p.cu_nkb.const_data_ptr<int32_t>(), ws.mutable_data_ptr(), n, batch, hk, nqb, nkb, (int)p.qbs,
                              (int)p.kbs, p.causal ? 1 : 0, tq, tk, mask_strides, stream);
    if (rc != 0) raise("hbsa_fwd_prepare", rc);
    at::Tensor out = at::empty(q.sizes(), q.options());
    at::Tensor lse = at::empty({q.size(0), q.size(1)}, q.options().dtype(at::kFloat));
    const int64_t strides[8] = {tok_stride(q), head_stride(q), tok_stride(k), head_stride(k), tok_stride(v), head_stride(v),
                                tok_stride(out), head_stride(out)};
    const int64_t lse_strides[2] = {lse.stride(0), lse.stride(1)};
    rc = hbsa_fwd_run_lse(q.const_data_ptr(), k.const_data_ptr(), v.const_data_ptr(), out.mutable_data_ptr(), lse.mutable_data_ptr<float>(),
                          lse_strides, ws.mutable_data_ptr(), n, p.dtype, tq, tk, hq, hk, d, nqb, nkb, (int)p.qbs, (int)p.kbs,
                          p.causal ? 1 : 0, (float)p.scale, strides, stream);
    if (rc != 0) raise("hbsa_fwd_run_lse", rc);
    ctx->save_for_backward({q, k, v, out, lse});
    // The work description and the boundaries go beside the saved tensors: they may be inference tensors (made by a data
    // loader or scheduler), their versions are the caller's business, and they are nothing for saved-tensor hooks.
    ctx->saved_data["workspace"] = ws;
    ctx->saved_data["cu_k"] = p.cu_k;
    ctx->saved_data["cu_num_q_block"] = p.cu_nqb;
    ctx->saved_data["cu_num_k_block"] = p.cu_nkb;
    ctx->saved_data["shape"] = std::vector<int64_t>{p.nqb, p.nkb, p.qbs, p.kbs, p.causal ? 1 : 0, p.dtype};
    ctx->saved_data["scale"] = p.scale;
    return out;
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext *ctx, torch::autograd::variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const at::Tensor &q = saved[0], &k = saved[1], &v = saved[2], &out = saved[3], &lse = saved[4];
    const at::Tensor ws = ctx->saved_data["workspace"].toTensor(), cu_k = ctx->saved_data["cu_k"].toTensor();
    const at::Tensor cu_nqb = ctx->saved_data["cu_num_q_block"].toTensor(), cu_nkb = ctx->saved_data["cu_num_k_block"].toTensor();
    const auto shape = ctx->saved_data["shape"].toIntVector();
    const float scale = (float)ctx->saved_data["scale"].toDouble();
    at::NoGradGuard no_grad;
    at::Tensor dout = grads[0];
    if (!dout.defined()) return {at::Tensor(), at::Tensor(), at::Tensor(), at::Tensor()};
    if (!rows_ok(dout)) dout = dout.contiguous();
    const OnDevice on(q.get_device());
    const hipStream_t stream = c10::hip::getCurrentHIPStream((c10::DeviceIndex)q.get_device()).stream();
    at::Tensor dq = at::empty(q.sizes(), q.options()), dk = at::empty(k.sizes(), k.options()), dv = at::empty(v.sizes(), v.options());
    const int tq = (int)q.size(0), tk = (int)k.size(0), hq = (int)q.size(1), hk = (int)k.size(1), d = (int)q.size(2);
    const size_t n = hbsa_bwd_workspace_bytes_parts(tq, hq, hk, d, (int)shape[0], (int)shape[1], (int)shape[2], (int)shape[3]);
    at::Tensor bws = bytes_like(q, n);
    const int64_t strides[16] = {tok_stride(q), head_stride(q), tok_stride(k), head_stride(k), tok_stride(v), head_stride(v),
                                 tok_stride(out), head_stride(out), tok_stride(dout), head_stride(dout), tok_stride(dq), head_stride(dq),
                                 tok_stride(dk), head_stride(dk), tok_stride(dv), head_stride(dv)};
    const int rc = hbsa_bwd(q.const_data_ptr(), k.const_data_ptr(), v.const_data_ptr(), out.const_data_ptr(), dout.const_data_ptr(),
                            lse.const_data_ptr<float>(), dq.mutable_data_ptr(), dk.mutable_data_ptr(), dv.mutable_data_ptr(),
                            cu_k.const_data_ptr<int32_t>(), cu_nqb.const_data_ptr<int32_t>(), cu_nkb.const_data_ptr<int32_t>(),
                            ws.const_data_ptr(), (size_t)ws.numel(), bws.mutable_data_ptr(), n, (int)shape[5],
                            (int)cu_k.numel() - 1, tq, tk, hq, hk, d, (int)shape[0], (int)shape[1], (int)shape[2], (int)shape[3],
                            (int)shape[4], scale, strides, stream);
    if (rc != 0) raise("hbsa_bwd", rc);
    return {dq, dk, dv, at::Tensor()};
  }
};

// ---- arguments
bool to_int(PyObject *o, int64_t &v) {
  if (!PyLong_Check(o)) return false;
  v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}
bool plain_tensor(PyObject *o) {   // no subclass with a dispatch of its own, no functorch wrapper
  if (!THPVariable_Check(o)) return false;
  const auto keys = THPVariable_Unpack(o).unsafeGetTensorImpl()->key_set();
  return !keys.has(c10::DispatchKey::Python) && !keys.has(c10::DispatchKey::FuncTorchGradWrapper) &&
         !keys.has(c10::DispatchKey::FuncTorchBatched) && !keys.has(c10::DispatchKey::Functionalize);
}

enum { A_Q, A_K, A_V, A_CUQ, A_CUK, A_MASK, A_QBS, A_KBS, A_CAUSAL, A_SCALE, A_MODE, A_NQB, A_CUQB, A_QB2B, A_CUNQB, A_NKB, A_CUKB,
       A_KB2B, A_CUNKB, A_F32, A_COUNT };

// HBSAttention's 19 arguments in their order, and the dtype code for fp32 tensors.
PyObject *call(PyObject *, PyObject *const *a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != A_COUNT) Py_RETURN_NONE;
  for (int i : {A_Q, A_K, A_V, A_CUQ, A_CUK, A_MASK})
    if (!plain_tensor(a[i])) Py_RETURN_NONE;
  Problem p;
  p.q = THPVariable_Unpack(a[A_Q]);
  if (!p.q.is_cuda()) Py_RETURN_NONE;
  p.k = THPVariable_Unpack(a[A_K]);
  p.v = THPVariable_Unpack(a[A_V]);
  p.mask = THPVariable_Unpack(a[A_MASK]);
  p.cu_q = THPVariable_Unpack(a[A_CUQ]);
  p.cu_k = THPVariable_Unpack(a[A_CUK]);
  const int index = p.q.get_device();
  if (!p.k.is_cuda() || !p.v.is_cuda() || !p.mask.is_cuda() || p.k.get_device() != index || p.v.get_device() != index ||
      p.mask.get_device() != index)
    Py_RETURN_NONE;
  const auto st = p.q.scalar_type();
  int64_t f32_code = HBSA_DTYPE_F32;
  if (st == at::kBFloat16) p.dtype = HBSA_DTYPE_BF16;
  else if (st == at::kHalf) p.dtype = HBSA_DTYPE_F16;
  else if (st == at::kFloat && to_int(a[A_F32], f32_code)) p.dtype = (int)f32_code;
  else Py_RETURN_NONE;
  if (p.k.scalar_type() != st || p.v.scalar_type() != st || p.mask.scalar_type() != at::kBool) Py_RETURN_NONE;
  if (p.q.dim() != 3 || p.k.dim() != 3 || p.v.dim() != 3 || p.mask.dim() != 3 || p.cu_q.dim() != 1) Py_RETURN_NONE;
  const int64_t tq = p.q.size(0), tk = p.k.size(0), hq = p.q.size(1), hk = p.k.size(1), d = p.q.size(2);
  if (tq <= 0 || tk <= 0 || tq > 0x7fffffff || tk > 0x7fffffff || hq <= 0 || hk <= 0 || hq % hk != 0) Py_RETURN_NONE;
  if (d <= 0 || d > 256 || (!native_dim(d) && (d % 8 != 0 || st == at::kFloat))) Py_RETURN_NONE;
  if (p.k.size(2) != d || p.v.sizes() != p.k.sizes()) Py_RETURN_NONE;
  if (!rows_ok(p.q) || !rows_ok(p.k) || !rows_ok(p.v)) Py_RETURN_NONE;
  if (!to_int(a[A_QBS], p.qbs) || !to_int(a[A_KBS], p.kbs) || p.qbs <= 0 || p.kbs <= 0 || p.qbs % 16 || p.kbs % 16 ||
      p.qbs > (1 << 24) || p.kbs > (1 << 24))
    Py_RETURN_NONE;
  if (!PyBool_Check(a[A_CAUSAL])) Py_RETURN_NONE;
  p.causal = a[A_CAUSAL] == Py_True;
  if (a[A_SCALE] == Py_None) p.scale = std::pow((double)d, -0.5);
  else if (PyFloat_Check(a[A_SCALE])) p.scale = PyFloat_AS_DOUBLE(a[A_SCALE]);
  else Py_RETURN_NONE;
  if (!PyUnicode_Check(a[A_MODE])) Py_RETURN_NONE;
  if (PyUnicode_CompareWithASCIIString(a[A_MODE], "auto") != 0 &&
      !(PyUnicode_CompareWithASCIIString(a[A_MODE], "fix") == 0 && (p.qbs & (p.qbs - 1)) == 0 && (p.kbs & (p.kbs - 1)) == 0))
    Py_RETURN_NONE;
  const int64_t n_seq = p.cu_q.numel();
  if (n_seq < 2 || !int32_on(p.cu_q, index, n_seq) || !int32_on(p.cu_k, index, n_seq)) Py_RETURN_NONE;
  if (p.mask.size(0) != hk || p.mask.size(1) <= 0 || p.mask.size(2) <= 0 || p.mask.size(1) > 0x7fffffff || p.mask.size(2) > 0x7fffffff)
    Py_RETURN_NONE;

  const bool wants_grad = at::GradMode::is_enabled() && (p.q.requires_grad() || p.k.requires_grad() || p.v.requires_grad());
  if (wants_grad && (st == at::kFloat || d > 128 || !native_dim(d))) Py_RETURN_NONE;

  // Block metadata is all-or-recompute per side.
  const bool q_given = a[A_NQB] != Py_None && a[A_CUQB] != Py_None && a[A_QB2B] != Py_None && a[A_CUNQB] != Py_None;
  const bool k_given = a[A_NKB] != Py_None && a[A_CUKB] != Py_None && a[A_KB2B] != Py_None && a[A_CUNKB] != Py_None;
  if (q_given) {
    if (!to_int(a[A_NQB], p.nqb) || p.nqb != p.mask.size(1) || !plain_tensor(a[A_QB2B]) || !plain_tensor(a[A_CUNQB])) Py_RETURN_NONE;
    p.qb2b = THPVariable_Unpack(a[A_QB2B]);
    p.cu_nqb = THPVariable_Unpack(a[A_CUNQB]);
    if (!int32_on(p.qb2b, index, p.nqb) || !int32_on(p.cu_nqb, index, n_seq)) Py_RETURN_NONE;
  }
  if (k_given) {
    if (!to_int(a[A_NKB], p.nkb) || p.nkb != p.mask.size(2) || !plain_tensor(a[A_CUNKB])) Py_RETURN_NONE;
    p.cu_nkb = THPVariable_Unpack(a[A_CUNKB]);
    if (!int32_on(p.cu_nkb, index, n_seq)) Py_RETURN_NONE;
  }

  const OnDevice on(index);
  const hipStream_t stream = c10::hip::getCurrentHIPStream((c10::DeviceIndex)index).stream();
  const bool counting = !q_given || !k_given;
  if (counting) {
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &capturing) != hipSuccess || capturing != hipStreamCaptureStatusNone) {
      (void)hipGetLastError();
      Py_RETURN_NONE;
    }
  }
  CountTicket counts(g_slots, counting ? g_slots.take(count_page) : nullptr, StateOf{stream});
  at::Tensor out;
  if (!wants_grad) out = at::empty(p.q.sizes(), p.q.options());
  bool done = false;
  if (counting) {
    // One launch that counts the blocks itself, or counts and first blocks of the sequences in one small launch.  The device checks the counts against the mask's
    // shape and leaves empty sequences when they differ, so the attention launch can follow at once; the host reads
    // the counts while it runs, and a call whose mask does not fit is reported by the caller.
    if (counts.slot == nullptr) Py_RETURN_NONE;
    counts.ticket = g_ticket.fetch_add(1, std::memory_order_relaxed) + 1;
    p.nqb = p.mask.size(1);
    p.nkb = p.mask.size(2);
    if (!wants_grad && st != at::kFloat) done = plain_forward(p, stream, out, &counts);
  }
  if (counting && !done) {
    at::Tensor firsts = at::empty({2, n_seq}, p.cu_q.options());
    int32_t *first = firsts.mutable_data_ptr<int32_t>();
    counts.launched = true;
    const int rc = hbsa_block_counts(q_given ? nullptr : p.cu_q.const_data_ptr<int32_t>(), (int)p.qbs, (int)p.mask.size(1), first,
                                     k_given ? nullptr : p.cu_k.const_data_ptr<int32_t>(), (int)p.kbs, (int)p.mask.size(2),
                                     first + n_seq, (int)n_seq - 1, counts.slot, counts.ticket, stream);
    if (rc != 0) Py_RETURN_NONE;
    if (!q_given) p.cu_nqb = firsts.select(0, 0);
    if (!k_given) p.cu_nkb = firsts.select(0, 1);
  }

  if (wants_grad) {
    out = Attention::apply(p.q, p.k, p.v, p);
    done = true;
  } else if (!done) {
    done = plain_forward(p, stream, out);
  }
  bool counts_fit = true;
  if (counting) {
    Py_BEGIN_ALLOW_THREADS
    counts_fit = counts.wait() && counts.slot[2] == 1;
    Py_END_ALLOW_THREADS
  }
  if (!counts_fit || !done) Py_RETURN_NONE;
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// calculate_blocks for an int32 tensor on the device: (num_block, cu_block, block_to_batch, cu_num_block), or None.
PyObject *blocks(PyObject *, PyObject *const *a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  int64_t block_size = 0;
  if (n_args != 2 || !plain_tensor(a[0]) || !to_int(a[1], block_size) || block_size <= 0 || block_size > 0x7fffffff) Py_RETURN_NONE;
  const at::Tensor &cu = THPVariable_Unpack(a[0]);
  if (!cu.is_cuda() || cu.dim() != 1 || cu.numel() < 2 || !int32_on(cu, cu.get_device(), cu.numel())) Py_RETURN_NONE;
  const OnDevice on(cu.get_device());
  const hipStream_t stream = c10::hip::getCurrentHIPStream((c10::DeviceIndex)cu.get_device()).stream();
  hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &capturing) != hipSuccess || capturing != hipStreamCaptureStatusNone) {
    (void)hipGetLastError();
    Py_RETURN_NONE;
  }
  CountTicket counts(g_slots, g_slots.take(count_page), StateOf{stream});
  if (counts.slot == nullptr) Py_RETURN_NONE;
  counts.ticket = g_ticket.fetch_add(1, std::memory_order_relaxed) + 1;
  at::Tensor first = at::empty({cu.numel()}, cu.options());
  const int batch = (int)cu.numel() - 1;
  counts.launched = true;
  if (hbsa_block_counts(cu.const_data_ptr<int32_t>(), (int)block_size, -1, first.mutable_data_ptr<int32_t>(), nullptr, 1, -1, nullptr,
                        batch, counts.slot, counts.ticket, stream) != 0)
    Py_RETURN_NONE;
  bool good;
  Py_BEGIN_ALLOW_THREADS
  good = counts.wait() && counts.slot[2] == 1;
  Py_END_ALLOW_THREADS
  if (!good) Py_RETURN_NONE;
  const int64_t num = counts.slot[0];
  at::Tensor cu_block = at::empty({num + 1}, cu.options()), to_batch = at::empty({num}, cu.options());
  const int rc2 = hbsa_block_arrays(cu.const_data_ptr<int32_t>(), first.const_data_ptr<int32_t>(), batch, (int)block_size, (int)num,
                                    cu_block.mutable_data_ptr<int32_t>(), to_batch.mutable_data_ptr<int32_t>(), stream);
  if (rc2 != 0) Py_RETURN_NONE;
  PyObject *r = PyTuple_New(4);
  if (r == nullptr) return nullptr;
  PyTuple_SET_ITEM(r, 0, PyLong_FromLongLong(num));
  PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(std::move(cu_block)));
  PyTuple_SET_ITEM(r, 2, THPVariable_Wrap(std::move(to_batch)));
  PyTuple_SET_ITEM(r, 3, THPVariable_Wrap(std::move(first)));
  return r;
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"call", (PyCFunction)(void (*)(void))call, METH_FASTCALL, "one HBSAttention call, or None when the general path has to take it"},
    {"blocks", (PyCFunction)(void (*)(void))blocks, METH_FASTCALL, "calculate_blocks on the device, or None"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_torch_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__torch_host(void) { return PyModule_Create(&module_def); }

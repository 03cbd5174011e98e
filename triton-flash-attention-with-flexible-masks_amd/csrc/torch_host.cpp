// The operator's host path in native code: checks, allocation, launches and the autograd node of one call.
//
// A call of a few microseconds of GPU work is bound by what the host does around it.  Through Python
// (autograd.Function, ctypes, one attribute at a time into fa_params) that was 27 us for a forward, 44 with ids and
// 80 - 104 for forward and backward; here it is 6 - 9 and 24 - 28 (tiny shapes, calls back to back).
//
// Every function takes the usual calls and returns None for anything else -- an argument it would have to convert,
// copy or refuse -- so that flash_mi355/api.py, which handles all of that, has the checks and their messages in one
// place.  Nothing is launched before it is clear that the call is taken.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <cmath>
#include <limits>

#include "../../include/flash_mi355.h"

namespace {

using at::Tensor;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

constexpr double kLn2 = 0.69314718055994530942;

void check(int rc, const char* what) {
  TORCH_CHECK(rc == FA_OK, what, ": ", fa_error_string(rc), " [code ", rc, ", hipError ", fa_last_hip_error(), "]");
}

// One call's problem: everything fa_params needs besides the results.
struct Problem {
  Tensor q, k, v, eq, ek, qpos;   // [B, H, M, D] ..., or [tokens, heads, D] when packed
  int mode = 0, window = 0, prefix = 0, nseq = 0;
  bool causal = false, packed = false;
  double scale = 0;
  int B, H, Hk, M, N, D;
  int64_t id_strides[2][3] = {};   // of eq, ek: the plan's layout follows them, and what saved-tensor hooks hand back may lie otherwise
};

int elem_type(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kBFloat16: return FA_DTYPE_BF16;
    case at::kHalf: return FA_DTYPE_FP16;
    case at::kFloat: return FA_DTYPE_FP32;
    default: return -1;
  }
}

// innermost stride 1, 16-byte aligned base and outer strides
bool laid_out(const Tensor& t) {
  const int64_t per16 = 16 / t.element_size();
  if (reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 != 0 || t.stride(-1) != 1) return false;
  for (int64_t i = 0; i + 1 < t.dim(); ++i)
    if (t.stride(i) % per16 != 0) return false;
  return true;
}
Tensor laid_out_or_copy(const Tensor& t) { return laid_out(t) ? t : t.contiguous(); }

// strides of a [B, heads, rows, D] operand; a packed [rows, heads, D] one is batch 0 of it
void set_strides(int64_t (&dst)[4], const Tensor& t) {
  if (t.dim() == 4) {
    for (int i = 0; i < 4; ++i) dst[i] = t.stride(i);
  } else {
    dst[0] = 0; dst[1] = t.stride(1); dst[2] = t.stride(0); dst[3] = t.stride(2);
  }
}

void set_block_map(fa_params& p, const Tensor& map) {
  p.eq = map.data_ptr();
  p.eq_stride[0] = map.size(0) == 1 ? 0 : map.stride(0);
  p.eq_stride[1] = map.size(1) == 1 ? 0 : map.stride(1);
  p.eq_stride[2] = map.size(2) == 1 ? map.size(3) : map.stride(2);
}

fa_params params_of(const Problem& x) {
  fa_params p = {};
  p.q = x.q.data_ptr(); p.k = x.k.data_ptr(); p.v = x.v.data_ptr();
  set_strides(p.q_stride, x.q); set_strides(p.k_stride, x.k); set_strides(p.v_stride, x.v);
  p.B = x.B; p.H = x.H; p.Hk = x.Hk; p.M = x.M; p.N = x.N; p.D = x.D;
  p.causal = x.causal; p.score_mode = x.mode; p.dtype = elem_type(x.q); p.sm_scale = (float)x.scale;
  p.window = x.window; p.prefix = x.prefix;
  p.flags = x.mode == FA_SCORE_MODE0_NOPE ? FA_FLAG_SPLIT_KEYS : 0;
  if (x.mode == FA_SCORE_MODE1_DOC) {
    p.eq = x.eq.data_ptr(); p.ek = x.ek.data_ptr();
    for (int i = 0; i < 3; ++i) { p.eq_stride[i] = x.id_strides[0][i]; p.ek_stride[i] = x.id_strides[1][i]; }
    p.id_dtype = x.eq.scalar_type() == at::kInt ? FA_IDTYPE_I32 : FA_IDTYPE_I64;
  } else if (x.mode == FA_SCORE_MODE2_BLOCK) {
    set_block_map(p, x.eq);
  } else if (x.mode == FA_SCORE_MODE3_PACKED) {
    p.nseq = x.nseq;
    if (x.eq.defined()) {   // the forward (see backward())
      p.eq = x.eq.data_ptr(); p.ek = x.ek.data_ptr();
      p.id_dtype = x.eq.scalar_type() == at::kInt ? FA_IDTYPE_I32 : FA_IDTYPE_I64;
    }
  }
  if (x.qpos.defined()) {
    p.qpos = x.qpos.const_data_ptr<int32_t>();
    p.qpos_stride = x.qpos.size(0) > 1 ? x.qpos.stride(0) : 0;
  }
  return p;
}

Tensor bytes_on(const Tensor& like, uint64_t n) { return at::empty({(int64_t)n}, like.options().dtype(at::kByte)); }

// The workspace: the plan, which the backward uses again, and the scratch of split key ranges, which lives for the call.
// plan undefined: a new one (the caller enqueues fa_mask_plan).
Tensor set_workspace(fa_params& p, const Tensor& like, Tensor& plan) {
  Tensor scratch;
  const uint64_t np = plan.defined() ? (uint64_t)plan.numel() : fa_workspace_plan_bytes(&p);
  if (np == 0) return scratch;
  if (!plan.defined()) plan = bytes_on(like, np);
  const uint64_t ns = fa_workspace_scratch_bytes(&p);
  p.workspace = plan.data_ptr(); p.workspace_bytes = np;
  if (ns > 0) {
    scratch = bytes_on(like, ns);
    p.split_scratch = scratch.data_ptr(); p.split_scratch_bytes = ns;
  }
  return scratch;
}

// gradients of k and v: as the operand lies when it is dense, head by head otherwise
Tensor grad_like(const Tensor& t, bool packed) { return packed ? at::empty_like(t, at::MemoryFormat::Contiguous) : at::empty(t.sizes(), t.options()); }

variable_list backward(const Problem& x, const Tensor& o, const Tensor& lse, Tensor plan, Tensor dout, const Tensor& dlse) {
  const c10::DeviceGuard guard(x.q.device());
  void* stream = c10::hip::getCurrentHIPStream(x.q.device().index()).stream();
  if (!dout.defined()) dout = at::zeros_like(o);   // only LSE was used
  dout = laid_out_or_copy(dout);
  TORCH_CHECK(dout.device() == x.q.device() && dout.scalar_type() == x.q.scalar_type(), "the gradient must share q's device and type");
  fa_params p = params_of(x);
  // The boundaries of packed sequences are read by the plan kernel alone and not kept (a caller may refill their buffer
  // while the backward is outstanding); the plan stands in for the pointers that the C ABI wants set.
  if (x.packed) p.eq = p.ek = plan.data_ptr();
  Tensor scratch;
  if (plan.defined()) scratch = set_workspace(p, x.q, plan);
  Tensor delta = at::empty_like(lse), dq = at::empty_like(x.q), dk = grad_like(x.k, x.packed), dv = grad_like(x.v, x.packed);
  p.o = o.data_ptr(); p.lse = lse.data_ptr<float>(); p.dout = dout.data_ptr(); p.delta = delta.data_ptr<float>();
  p.dq = dq.data_ptr(); p.dk = dk.data_ptr(); p.dv = dv.data_ptr();
  set_strides(p.o_stride, o); set_strides(p.do_stride, dout);
  set_strides(p.dq_stride, dq); set_strides(p.dk_stride, dk); set_strides(p.dv_stride, dv);
  if (!dlse.defined()) {
    check(fa_bwd(&p, stream), "fa_bwd");
  } else {
    check(fa_bwd_delta(&p, stream), "fa_bwd_delta");
    // dS = P * (dP - delta) + dLSE * P: a gradient arriving at LSE only shifts delta
    delta.sub_(at::where(at::isinf(lse), at::zeros_like(lse), dlse.to(at::kFloat)));
    check(fa_bwd_dkdv(&p, stream), "fa_bwd_dkdv");
    check(fa_bwd_dq(&p, stream), "fa_bwd_dq");
  }
  return {dq, dk, dv};
}

struct AttentionBackward : public torch::autograd::Node {
  Problem x;   // its q, k, v, eq, ek, qpos are empty: the tensors are the saved ones below
  SavedVariable q, k, v, o, lse, eq, ek, plan, qpos;
  variable_list apply(variable_list&& grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    auto self = shared_from_this();
    Problem y = x;
    y.q = q.unpack(); y.k = k.unpack(); y.v = v.unpack(); y.eq = eq.unpack(); y.ek = ek.unpack(); y.qpos = qpos.unpack();
    const Tensor o_ = o.unpack(self), lse_ = lse.unpack(), plan_ = plan.unpack();
    at::NoGradGuard no_grad;
    return backward(y, o_, lse_, plan_, grads[0], grads.size() > 1 ? grads[1] : Tensor());
  }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    for (SavedVariable* s : {&q, &k, &v, &o, &lse, &eq, &ek, &plan, &qpos}) s->reset_data();
  }
  std::string name() const override { return "FlashAttentionBackward"; }
};

// O and, when want_lse, LSE in natural-log units
std::pair<Tensor, Tensor> run(const Problem& x, fa_params& p, bool want_lse) {
  const bool grad = at::GradMode::is_enabled() && (x.q.requires_grad() || x.k.requires_grad() || x.v.requires_grad());
  Tensor o, lse, lse_e, plan, eq = x.eq;
  {
    const at::NoGradGuard no_grad;
    const c10::DeviceGuard guard(x.q.device());
    void* stream = c10::hip::getCurrentHIPStream(x.q.device().index()).stream();
    if (grad && x.mode == FA_SCORE_MODE2_BLOCK) {   // the backward reads the map again: it keeps one that nobody else writes
      eq = at::ne(x.eq, 0).contiguous();
      set_block_map(p, eq);
    }
    o = at::empty_like(x.q);
    lse = at::empty({x.B, x.H, x.M}, x.q.options().dtype(at::kFloat));
    p.o = o.data_ptr(); p.lse = lse.data_ptr<float>();
    set_strides(p.o_stride, o);
    const Tensor scratch = set_workspace(p, x.q, plan);
    if (plan.defined()) check(fa_mask_plan(&p, stream), "fa_mask_plan");
    check(fa_fwd(&p, stream), "fa_fwd");
    if (want_lse) lse_e = lse * kLn2;
  }
  if (grad) {
    auto node = std::shared_ptr<AttentionBackward>(new AttentionBackward(), torch::autograd::deleteNode);
    node->set_next_edges(torch::autograd::collect_next_edges(x.q, x.k, x.v));
    node->x = x;
    for (Tensor* t : {&node->x.q, &node->x.k, &node->x.v, &node->x.eq, &node->x.ek, &node->x.qpos}) *t = Tensor();
    node->q = SavedVariable(x.q, false); node->k = SavedVariable(x.k, false); node->v = SavedVariable(x.v, false);
    if (!x.packed) { node->eq = SavedVariable(eq, false); node->ek = SavedVariable(x.ek, false); }
    node->qpos = SavedVariable(x.qpos, false);
    node->lse = SavedVariable(lse, false); node->plan = SavedVariable(plan, false);
    torch::autograd::set_history(o, node);
    if (want_lse) torch::autograd::set_history(lse_e, node);
    node->o = SavedVariable(o, true);
  }
  return {o, lse_e};
}

// -- arguments ----------------------------------------------------------------------------------------------------------
// A tensor the kernels may read as it is.  Subclasses and dual tensors (the node has no forward-mode rule) are for the
// Python classes, which serve them or refuse them.
bool tensor_arg(PyObject* a, Tensor& t) {
  if (!THPVariable_CheckExact(a)) return false;
  t = THPVariable_Unpack(a);
  return t.defined() && t.has_storage() && !t.unsafeGetTensorImpl()->is_python_dispatch() && !t._fw_grad(0).defined();
}
// ... and so is every call under a tracer, which would record the allocations and not the launches, or a function
// transform (vmap, grad, jvp of torch.func), whose tensors are wrappers without memory.
bool plain_call() {
  return !torch::jit::tracer::isTracing() && !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode);
}
bool int_arg(PyObject* a, int& v) {
  if (a == Py_None) { v = 0; return true; }
  if (!PyLong_Check(a)) return false;
  int overflow = 0;
  const long long x = PyLong_AsLongLongAndOverflow(a, &overflow);
  if (overflow != 0 || x < 0 || x > 0x7fffffff) return false;
  v = (int)x;
  return true;
}
bool scale_arg(PyObject* a, int D, double& v) {
  if (a == Py_None) { v = 1.0 / std::sqrt((double)D); return true; }
  if (PyFloat_Check(a)) { v = PyFloat_AS_DOUBLE(a); return true; }
  return false;
}
bool operands_ok(const Problem& x) {
  if (!x.q.is_cuda() || x.k.device() != x.q.device() || x.v.device() != x.q.device()) return false;
  const int ty = elem_type(x.q);
  if (ty < 0 || x.k.scalar_type() != x.q.scalar_type() || x.v.scalar_type() != x.q.scalar_type()) return false;
  return x.q.numel() > 0 && x.k.numel() > 0 && laid_out(x.q) && laid_out(x.k) && laid_out(x.v);
}
bool id_type(const Tensor& t) { return t.scalar_type() == at::kInt || t.scalar_type() == at::kLong; }
bool fits(int64_t v) { return v <= std::numeric_limits<int32_t>::max(); }

PyObject* finish(const Problem& x, bool want_lse) {
  fa_params p = params_of(x);
  // what the library would refuse is left to the Python path and its messages
  fa_params probe = p;
  probe.o = const_cast<void*>(p.q); set_strides(probe.o_stride, x.q);
  probe.lse = reinterpret_cast<float*>(probe.o);
  if (fa_workspace_bytes(&p) > 0) {
    probe.workspace = reinterpret_cast<void*>(uintptr_t(256)); probe.workspace_bytes = ~uint64_t(0);
    probe.split_scratch = nullptr;
  }
  if (fa_validate(&probe, 0) != FA_OK) Py_RETURN_NONE;
  std::pair<Tensor, Tensor> r;
  {
    pybind11::gil_scoped_release no_gil;
    r = run(x, p, want_lse);
  }
  if (!want_lse) return THPVariable_Wrap(std::move(r.first));
  PyObject* t = PyTuple_New(2);
  PyTuple_SET_ITEM(t, 0, THPVariable_Wrap(std::move(r.first)));
  PyTuple_SET_ITEM(t, 1, THPVariable_Wrap(std::move(r.second)));
  return t;
}

// attention(q, k, v, causal, sm_scale, eq, ek, score_func_mode, window, prefix, qpos, want_lse)
PyObject* attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Problem x;
  if (n != 12 || !plain_call() || !tensor_arg(a[0], x.q) || !tensor_arg(a[1], x.k) || !tensor_arg(a[2], x.v)) Py_RETURN_NONE;
  if (x.q.dim() != 4 || x.k.dim() != 4 || x.v.dim() != 4) Py_RETURN_NONE;
  const auto qs = x.q.sizes(), ks = x.k.sizes();
  if (ks != x.v.sizes() || qs[3] != ks[3] || qs[0] != ks[0] || !fits(qs[0] * qs[1]) || !fits(qs[2]) || !fits(ks[2])) Py_RETURN_NONE;
  x.B = (int)qs[0]; x.H = (int)qs[1]; x.M = (int)qs[2]; x.D = (int)qs[3]; x.Hk = (int)ks[1]; x.N = (int)ks[2];
  if (!operands_ok(x) || x.H % x.Hk != 0) Py_RETURN_NONE;
  if (!int_arg(a[7], x.mode) || !int_arg(a[8], x.window) || !int_arg(a[9], x.prefix) || !scale_arg(a[4], x.D, x.scale)) Py_RETURN_NONE;
  const int causal = PyObject_IsTrue(a[3]), want_lse = PyObject_IsTrue(a[11]);
  if (causal < 0 || want_lse < 0) { PyErr_Clear(); Py_RETURN_NONE; }
  x.causal = causal != 0;
  const bool has_pos = a[10] != Py_None;
  if (x.causal && x.N < x.M && !has_pos) Py_RETURN_NONE;
  if (has_pos) {
    if (!tensor_arg(a[10], x.qpos) || !x.causal || x.mode != FA_SCORE_MODE1_DOC || x.prefix != 0) Py_RETURN_NONE;
    if (x.qpos.dim() != 2 || x.qpos.scalar_type() != at::kInt || x.qpos.device() != x.q.device() || !x.qpos.is_contiguous() ||
        x.qpos.size(1) != x.M || (x.qpos.size(0) != 1 && x.qpos.size(0) != x.B)) Py_RETURN_NONE;
  }
  if (x.mode == FA_SCORE_MODE0_NOPE) {
    if (a[5] != Py_None || a[6] != Py_None) {   // ids are checked and then not used in this mode
      Py_RETURN_NONE;
    }
  } else if (x.mode == FA_SCORE_MODE1_DOC) {
    if (!tensor_arg(a[5], x.eq) || !tensor_arg(a[6], x.ek) || !id_type(x.eq) || x.ek.scalar_type() != x.eq.scalar_type()) Py_RETURN_NONE;
    if (x.eq.device() != x.q.device() || x.ek.device() != x.q.device()) Py_RETURN_NONE;
    if (x.eq.sizes() != at::IntArrayRef({x.B, x.H, x.M}) || x.ek.sizes() != at::IntArrayRef({x.B, x.H, x.N})) Py_RETURN_NONE;
    for (int i = 0; i < 3; ++i) { x.id_strides[0][i] = x.eq.stride(i); x.id_strides[1][i] = x.ek.stride(i); }
  } else if (x.mode == FA_SCORE_MODE2_BLOCK) {
    // bytes that are zero or not are what the kernels read: a bool map is used as it is (a copy of it with a gradient, see run())
    if (!tensor_arg(a[5], x.eq) || x.eq.dim() != 4 || x.eq.device() != x.q.device()) Py_RETURN_NONE;
    if (x.eq.scalar_type() != at::kBool && x.eq.scalar_type() != at::kByte) Py_RETURN_NONE;
    const auto es = x.eq.sizes();
    if ((es[0] != 1 && es[0] != x.B) || (es[1] != 1 && es[1] != x.H) || es[2] != (x.M + FA_MASK_BLOCK - 1) / FA_MASK_BLOCK ||
        es[3] != (x.N + FA_MASK_BLOCK - 1) / FA_MASK_BLOCK || (x.eq.stride(3) != 1 && es[3] != 1)) Py_RETURN_NONE;
  } else {
    Py_RETURN_NONE;
  }
  return finish(x, want_lse != 0);
  END_HANDLE_TH_ERRORS
}

// Whether a packed batch goes to the kernels as a document mask.  With tile tables every sequence has tiles of its own,
// which very short ones leave nearly empty, while the tiles of a document mask hold many of them; the ids (and, with two
// vectors of boundaries, the positions) take some kernels and 30 (100) us on the host, which only a launch of many tiles
// is worth.  Below 112 / (G + 2) tokens on average (G heads to a key head), forward and backward, tables : mask, us:
//   20000 tokens, D = 128: G = 1, 8 heads, average 8 701 : 202, 24 264 : 205, 32 212 : 202, 44 179 : 204; G = 4, 32 heads, 8 1184 :
//   567, 16 773 : 568, 24 493 : 567; G = 8, 8 1021 : 584, 12 656 : 588, 16 557 : 589; D = 64, G = 1, 32 heads, 16 963 : 421, 32 543 : 422,
//   44 452 : 428.  From 4096 sequences x key heads (D = 128), more of the shorter tiles of a smaller D: 5000 tokens, G = 1, 8
//   heads, average 4 (9900) 351 : 196, 8 (4980) 186 : 163, 12 (3340) 135 : 162; D = 64, 32 heads, 12 (13300) 300 : 172, 24 (6660) 169 : 189.
// Two vectors: 20000 tokens, G = 1, average 4 1355 : 292, 16 372 : 289, 32 213 : 288.  (Different totals: queries on a cache of
// keys, where the tables are 3 - 20 times faster.)
bool as_documents(int64_t Tq, int64_t Tk, int64_t nseq, int64_t H, int64_t Hk, int64_t D, bool same) {
  if (Tq != Tk || Hk <= 0) return false;
  const int64_t more = same ? 1 : 2;
  return Tq * (H / Hk + 2) * more < 112 * nseq && nseq * Hk * D >= 4096 * 128 * more;
}
// varlen_as_documents(Tq, Tk, nseq, H, Hk, D, same): the rule, for the Python path
PyObject* varlen_as_documents(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n == 7, "varlen_as_documents takes seven numbers");
  int64_t v[7];
  for (int i = 0; i < 7; ++i) {
    v[i] = PyLong_AsLongLong(a[i]);
    if (v[i] == -1 && PyErr_Occurred()) return nullptr;
  }
  if (as_documents(v[0], v[1], v[2], v[3], v[4], v[5], v[6] != 0)) Py_RETURN_TRUE;
  Py_RETURN_FALSE;
  END_HANDLE_TH_ERRORS
}

// attention_varlen(q, k, v, cu_seqlens_q, cu_seqlens_k, causal, sm_scale, window)
PyObject* attention_varlen(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Problem x;
  if (n != 8 || !plain_call() || !tensor_arg(a[0], x.q) || !tensor_arg(a[1], x.k) || !tensor_arg(a[2], x.v) || !tensor_arg(a[3], x.eq)) Py_RETURN_NONE;
  const bool same = a[4] == Py_None || a[4] == a[3];
  if (same) x.ek = x.eq;
  else if (!tensor_arg(a[4], x.ek)) Py_RETURN_NONE;
  if (x.q.dim() != 3 || x.k.dim() != 3 || x.v.dim() != 3 || x.eq.dim() != 1 || x.eq.sizes() != x.ek.sizes()) Py_RETURN_NONE;
  const auto qs = x.q.sizes(), ks = x.k.sizes();
  if (ks != x.v.sizes() || qs[2] != ks[2] || !fits(qs[0]) || !fits(ks[0]) || !fits(qs[1]) || !fits(x.eq.numel()) || (same && qs[0] != ks[0])) Py_RETURN_NONE;
  x.B = 1; x.M = (int)qs[0]; x.H = (int)qs[1]; x.D = (int)qs[2]; x.N = (int)ks[0]; x.Hk = (int)ks[1];
  if (!operands_ok(x) || x.H % x.Hk != 0 || x.q.scalar_type() == at::kFloat) Py_RETURN_NONE;
  if (!id_type(x.eq) || x.ek.scalar_type() != x.eq.scalar_type() || x.eq.device() != x.q.device() || x.ek.device() != x.q.device() ||
      !x.eq.is_contiguous() || !x.ek.is_contiguous() || x.eq.numel() < 2) Py_RETURN_NONE;
  if (as_documents(x.M, x.N, x.eq.numel() - 1, x.H, x.Hk, x.D, same)) Py_RETURN_NONE;
  const int causal = PyObject_IsTrue(a[5]);
  if (causal < 0) { PyErr_Clear(); Py_RETURN_NONE; }
  if (!scale_arg(a[6], x.D, x.scale) || !int_arg(a[7], x.window)) Py_RETURN_NONE;
  x.causal = causal != 0;
  x.mode = FA_SCORE_MODE3_PACKED;
  x.packed = true;
  x.nseq = (int)x.eq.numel() - 1;
  return finish(x, false);
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"attention", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&attention)), METH_FASTCALL, nullptr},
    {"attention_varlen", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&attention_varlen)), METH_FASTCALL, nullptr},
    {"varlen_as_documents", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&varlen_as_documents)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native() {
  if (fa_version() != FA_ABI_VERSION || fa_params_size() != sizeof(fa_params)) {
    PyErr_SetString(PyExc_ImportError, "libflash_mi355.so does not match _native.so: build both again");
    return nullptr;
  }
  return PyModule_Create(&module);
}

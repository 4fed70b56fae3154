// Native host path of the package's public calls (module prefixlm._torch_calls).
//
// A plain eager call of the Python operators spends most of its time on the host: the
// dispatcher's Python kernels, argument structs filled through ctypes and, in a backward,
// Python running on the autograd engine's thread. For small batches and single-token decode
// that is several times the GPU's work. Here the same checks, allocations and C entry
// points run in C++, forward and backward, as C++ autograd functions: 700 tokens x 8 heads x
// d64, forward + backward 271 -> 102 us a pass (then the kernels in a row), one decode step 34 ->
// 9.6 us, the recurrent stack over 1100 tokens 1.90 -> 1.33 ms.
//
// Each function takes the Python call's own arguments and returns None when the call is not
// a plain one, and the caller then takes its Python path, which serves every case: tensor
// subclasses, modes and transforms (torch.compile, make_fx, FakeTensor, functorch, forward
// mode AD), operands that need a copy first, and whatever has to be refused with a message.
// A backward that is itself recorded (create_graph), batched or fed an unusual gradient goes
// through the registered custom op as before.
#include <ATen/ATen.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/InferenceMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/PythonDispatcherTLS.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/record_function.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/utils/pybind.h>

#include <atomic>
#include <cmath>
#include <cstdlib>
#include <functional>
#include <optional>

#include "prefixlm.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// ---- the library's entry points (the handle ctypes loaded) ---------------------------
struct Lib {
  decltype(&prefixlm_fwd) fwd;
  decltype(&prefixlm_bwd) bwd;
  decltype(&prefixlm_fwd_q_amax_count) q_amax_count;
  decltype(&prefixlm_fwd_workspace_size) fwd_ws;
  decltype(&prefixlm_bwd_workspace_size) bwd_ws;
  decltype(&prefixlm_bwd_ds_bytes) ds_bytes;
  decltype(&prefixlm_bwd_ds_bytes_blocks) ds_bytes_blocks;
  decltype(&prefixlm_rope) rope;
  decltype(&prefixlm_swiglu_fwd) swiglu_fwd;
  decltype(&prefixlm_swiglu_bwd) swiglu_bwd;
  decltype(&prefixlm_rmsnorm_fwd) rmsnorm_fwd;
  decltype(&prefixlm_rmsnorm_bwd) rmsnorm_bwd;
  decltype(&prefixlm_add_rmsnorm) add_rmsnorm;
  decltype(&prefixlm_proj_gemm) proj_gemm;
  decltype(&prefixlm_proj_gemm_scaled) proj_gemm_scaled;
  decltype(&prefixlm_kvcache_workspace_size) kv_ws;
  decltype(&prefixlm_kvcache_fwd) kv_fwd;
  decltype(&prefixlm_last_error) last_error;
} lib{};
std::vector<int64_t> g_ds_cap;            // per device: an eighth of its memory
std::atomic<void*> g_timer{nullptr};      // the active Timer's handle (_capi.Timer)
PyObject* g_parameter = nullptr;          // torch.nn.Parameter

void check(int rc, const char* what) {
  if (rc != 0) throw std::runtime_error(std::string(what) + " failed (status " + std::to_string(rc) + "): " + lib.last_error());
}
void* stream_of(const Tensor& t) {
  return at::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream();
}
Tensor empty_like_on(const Tensor& t, at::IntArrayRef sizes, at::ScalarType dt) {
  return at::empty(sizes, t.options().dtype(dt).requires_grad(false));
}
int i32(bool b) { return b ? 1 : 0; }
// The calls do not pass the dispatcher, which would show them to torch.profiler: each records the
// name of the custom op that it stands for, with its tensors, for as long as this object lives.
struct Recorded {
  at::RecordFunction fn{at::RecordScope::FUNCTION};
  Recorded(const char* op, std::initializer_list<std::reference_wrapper<const Tensor>> tensors) {
    if (!fn.isActive()) return;
    if (fn.needsInputs()) {
      const std::vector<c10::IValue> in(tensors.begin(), tensors.end());
      fn.before(op, c10::ArrayRef<const c10::IValue>(in.data(), in.size()));
    } else {
      fn.before(op);
    }
  }
};

// ---- what counts as a plain call --------------------------------------------------------
// No mode, transform or tracer that would want to see the operators.
bool plain_state() {
  using c10::DispatchKey;
  const auto tls = c10::impl::tls_local_dispatch_key_set();
  return !c10::impl::TorchDispatchModeTLS::any_modes_set() && at::impl::PythonTorchFunctionTLS::stack_len() == 0 &&
         !c10::impl::PythonDispatcherTLS::get_state() && !torch::jit::tracer::isTracing() &&
         !tls.included_.has(DispatchKey::FuncTorchDynamicLayerFrontMode) && !tls.included_.has(DispatchKey::Python) &&
         !tls.included_.has(DispatchKey::Functionalize) && !tls.included_.has(DispatchKey::PreDispatch);
}
// A dense GPU tensor without wrappers, lazy bits or a tangent.
bool plain_tensor(const Tensor& t, bool gpu = true) {
  using c10::DispatchKey;
  static const c10::DispatchKeySet odd({DispatchKey::Python, DispatchKey::PythonTLSSnapshot, DispatchKey::Functionalize,
                                        DispatchKey::FuncTorchBatched, DispatchKey::FuncTorchGradWrapper,
                                        DispatchKey::Batched, DispatchKey::Conjugate, DispatchKey::Negative,
                                        DispatchKey::ZeroTensor});
  return t.defined() && t.layout() == at::kStrided && (gpu ? t.is_cuda() : t.device().is_cpu()) &&
         !t.key_set().has_any(odd) && !t.is_inference() && !t._fw_grad(0).defined();
}
// An object that is exactly a Tensor or Parameter, as a plain tensor
bool get_tensor(PyObject* o, Tensor* t) {
  if (!(THPVariable_CheckExact(o) || reinterpret_cast<PyObject*>(Py_TYPE(o)) == g_parameter)) return false;
  *t = THPVariable_Unpack(o);
  return plain_tensor(*t);
}
// A host scalar: an int, or a one-element integer CPU tensor (kept, to be saved with the call)
struct Scalar {
  int64_t v = 0;
  Tensor t;
};
bool get_scalar(PyObject* o, Scalar* s) {
  if (PyLong_CheckExact(o)) {
    s->v = PyLong_AsLongLong(o);
    if (s->v == -1 && PyErr_Occurred()) {
      PyErr_Clear();
      return false;
    }
  } else {
    if (!THPVariable_CheckExact(o)) return false;
    s->t = THPVariable_Unpack(o);
    if (!plain_tensor(s->t, false) || s->t.numel() != 1) return false;
    if (s->t.scalar_type() == at::kLong)
      s->v = *s->t.const_data_ptr<int64_t>();
    else if (s->t.scalar_type() == at::kInt)
      s->v = *s->t.const_data_ptr<int32_t>();
    else
      return false;
  }
  return s->v >= INT32_MIN && s->v <= INT32_MAX;
}
bool get_bool(PyObject* o, bool* b) {
  if (!PyBool_Check(o)) return false;
  *b = o == Py_True;
  return true;
}
bool get_double(PyObject* o, double* d) {
  if (!PyFloat_CheckExact(o)) return false;
  *d = PyFloat_AS_DOUBLE(o);
  return true;
}
bool aligned(const Tensor& t, uintptr_t a) { return reinterpret_cast<uintptr_t>(t.const_data_ptr()) % a == 0; }
// what the attention kernels read in place: bf16 [T, H, D], 16-byte rows
bool operand_layout(const Tensor& x) {
  return x.stride(2) == 1 && x.stride(0) % 8 == 0 && x.stride(1) % 8 == 0 && x.stride(0) >= x.size(2) && aligned(x, 16);
}
bool operand(const Tensor& x) { return x.scalar_type() == at::kBFloat16 && x.dim() == 3 && operand_layout(x); }
Tensor as_operand(const Tensor& x) { return operand_layout(x) ? x : x.contiguous(); }
bool meta(const Tensor& x, const Tensor& like) {
  return x.scalar_type() == at::kInt && x.device() == like.device() && x.is_contiguous();
}
bool wants_grad(const Tensor& t) { return at::GradMode::is_enabled() && t.requires_grad(); }

// ---- the metadata of a packed batch ------------------------------------------------------
struct Batch {
  Tensor pre, cau, cu, plan;      // plan: undefined without one
  Scalar total, nseq, mp, mc, ma, dsb;
  bool has_dsb = false, causal = false;
  double scale = 0.0;

  // args: is_causal, prefix_lens, causal_lens, cu_seqlens, the five scalars, softmax_scale
  // (float or None), plan, plan_ds_blocks
  bool parse(PyObject* const* a, const Tensor& like, int64_t head_dim) {
    if (!get_bool(a[0], &causal)) return false;
    if (!get_tensor(a[1], &pre) || !get_tensor(a[2], &cau) || !get_tensor(a[3], &cu)) return false;
    if (!meta(pre, like) || !meta(cau, like) || !meta(cu, like)) return false;
    Scalar* s[] = {&total, &nseq, &mp, &mc, &ma};
    for (int i = 0; i < 5; ++i)
      if (!get_scalar(a[4 + i], s[i])) return false;
    if (a[9] == Py_None)
      scale = 1.0 / std::sqrt((double)head_dim);
    else if (!get_double(a[9], &scale))
      return false;
    if (a[10] != Py_None) {
      if (!get_tensor(a[10], &plan) || !meta(plan, like) || plan.dim() != 1 || !aligned(plan, 256)) return false;
    }
    if (a[11] != Py_None) {
      if (!get_scalar(a[11], &dsb) || dsb.v < 0) return false;
      has_dsb = true;
    }
    return true;
  }
  int64_t meta_len() const { return std::min({pre.numel(), cau.numel(), cu.numel()}); }
  template <class Args>
  void fill(Args& a, const Tensor& pl) const {
    a.struct_size = sizeof(Args);
    a.prefix_lens = pre.const_data_ptr<int32_t>();
    a.causal_lens = cau.const_data_ptr<int32_t>();
    a.cu_seqlens = cu.const_data_ptr<int32_t>();
    a.meta_len = meta_len();
    a.total_seqlen = (int32_t)total.v;
    a.numseqs = (int32_t)nseq.v;
    a.max_seqlen_prefix = (int32_t)mp.v;
    a.max_seqlen_causal = (int32_t)mc.v;
    a.max_seqlen_all = (int32_t)ma.v;
    a.is_causal = i32(causal);
    a.softmax_scale = (float)scale;
    if (pl.defined()) {
      a.plan = pl.const_data_ptr();
      a.plan_bytes = (size_t)pl.numel() * 4;
    }
    a.timer = g_timer.load();
  }
  // whether the metadata that a backward got back is what parse accepted
  bool restored(const Tensor& like) const {
    if (!meta(pre, like) || !meta(cau, like) || !meta(cu, like)) return false;
    if (plan.defined() && (!meta(plan, like) || plan.dim() != 1 || !aligned(plan, 256))) return false;
    for (const Scalar* s : {&total, &nseq, &mp, &mc, &ma, &dsb}) {
      if (s == &dsb && !has_dsb) continue;
      const Tensor& t = s->t;
      if (!t.defined() || !t.device().is_cpu() || t.numel() != 1) return false;
      const bool same = t.scalar_type() == at::kLong  ? *t.const_data_ptr<int64_t>() == s->v
                        : t.scalar_type() == at::kInt ? *t.const_data_ptr<int32_t>() == s->v
                                                      : false;
      if (!same) return false;
    }
    return true;
  }
  static Tensor scalar(const Scalar& s) { return s.t.defined() ? s.t : at::scalar_tensor(s.v, at::kLong); }
  // saved with the call: the tensors that the Python function saves, in its order (an in-place
  // change is noticed, and a recomputation may take either path), and the values
  void save(variable_list& to, AutogradContext* ctx) const {
    for (const Tensor& t : {pre, cau, cu, scalar(total), scalar(nseq), scalar(mp), scalar(mc), scalar(ma), plan})
      to.push_back(t);
    to.push_back(has_dsb ? scalar(dsb) : Tensor());
    ctx->saved_data["ints"] = std::vector<int64_t>{total.v, nseq.v, mp.v, mc.v, ma.v, dsb.v, has_dsb, causal};
    ctx->saved_data["scale"] = scale;
  }
  static Batch restore(const variable_list& from, size_t at, AutogradContext* ctx) {
    Batch b;
    const auto v = ctx->saved_data["ints"].toIntVector();
    b.pre = from[at];
    b.cau = from[at + 1];
    b.cu = from[at + 2];
    b.plan = from[at + 8];
    Scalar* s[] = {&b.total, &b.nseq, &b.mp, &b.mc, &b.ma, &b.dsb};
    for (int i = 0; i < 6; ++i) {
      s[i]->v = v[i];
      s[i]->t = from[at + (i < 5 ? 3 + i : 9)];
    }
    b.has_dsb = v[6];
    b.causal = v[7];
    b.scale = ctx->saved_data["scale"].toDouble();
    return b;
  }
  // the trailing arguments of the custom ops' schemas
  void push(torch::jit::Stack& st, bool with_dsb) const {
    for (const Tensor& t : {pre, cau, cu}) st.emplace_back(t);
    for (const Scalar* s : {&total, &nseq, &mp, &mc, &ma}) st.emplace_back(scalar(*s));
    st.emplace_back(scale);
    st.emplace_back(plan.defined() ? c10::IValue(plan) : c10::IValue());
    if (with_dsb) st.emplace_back(has_dsb ? c10::IValue(scalar(dsb)) : c10::IValue());
  }
};

variable_list call_op(const char* name, torch::jit::Stack stack) {
  const auto op = c10::Dispatcher::singleton().findSchemaOrThrow(name, "");
  op.callBoxed(stack);
  variable_list out;
  for (auto& v : stack) out.push_back(v.toTensor());
  return out;
}

// The dS buffer of a backward (see the Python op's _ds_arg): exact with a plan's block
// count, else the scalars' bound; none past the cap or when its allocation fails.
bool ds_cap(const Tensor& like, int64_t* cap) {
  const char* env = std::getenv("PREFIXLM_DS_MAX_BYTES");
  if (!env) {
    *cap = g_ds_cap.at(like.device().index());
    return true;
  }
  char* end = nullptr;
  *cap = std::strtoll(env, &end, 10);
  return end != env && *end == 0;
}
Tensor ds_buffer(const Tensor& like, int64_t T, int64_t H, const Batch& b, int64_t blocks, int64_t cap) {
  const int64_t n = blocks > 0 ? (b.ma.v <= 32768 ? (int64_t)lib.ds_bytes_blocks(T, H, b.nseq.v, blocks) : 0)
                               : (int64_t)lib.ds_bytes(T, H, b.nseq.v, b.ma.v);
  if (n <= 0 || n > cap) return Tensor();
  try {
    return empty_like_on(like, {n}, at::kByte);
  } catch (const c10::OutOfMemoryError&) {
    return Tensor();
  }
}

// ---- the attention calls -------------------------------------------------------------------
struct FwdOut {
  Tensor out, lse, out_lo, q_amax, y;
};
FwdOut attn_forward(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& gate, const Batch& b) {
  const int64_t T = q.size(0), H = q.size(1), D = q.size(2);
  FwdOut r;
  r.out = empty_like_on(q, {T, H, D}, at::kBFloat16);
  r.out_lo = empty_like_on(q, {T, H, D}, at::kChar);
  r.lse = empty_like_on(q, {H, T}, at::kFloat);
  r.q_amax = empty_like_on(q, {(int64_t)lib.q_amax_count(T, H)}, at::kFloat);
  Tensor ws;
  prefixlm_fwd_args a{};
  b.fill(a, b.plan);
  a.num_tokens = (int32_t)T;
  a.num_heads = (int32_t)H;
  a.head_dim = (int32_t)D;
  a.q = q.const_data_ptr();
  a.k = k.const_data_ptr();
  a.v = v.const_data_ptr();
  a.out = r.out.data_ptr();
  a.out_lo = r.out_lo.data_ptr();
  a.lse = r.lse.data_ptr<float>();
  a.q_amax = r.q_amax.data_ptr<float>();
  a.q_stride_t = q.stride(0), a.q_stride_h = q.stride(1);
  a.k_stride_t = k.stride(0), a.k_stride_h = k.stride(1);
  a.v_stride_t = v.stride(0), a.v_stride_h = v.stride(1);
  a.out_stride_t = a.out_lo_stride_t = H * D;
  a.out_stride_h = a.out_lo_stride_h = D;
  if (gate.defined()) {
    r.y = empty_like_on(q, {T, H, D}, at::kBFloat16);
    a.gate = gate.const_data_ptr();
    a.out_gated = r.y.data_ptr();
    a.gate_stride_t = gate.stride(0), a.gate_stride_h = gate.stride(1);
    a.out_gated_stride_t = H * D, a.out_gated_stride_h = D;
  }
  if (!b.plan.defined()) {
    a.workspace_bytes = lib.fwd_ws(T, H, D, b.total.v, b.nseq.v);
    ws = empty_like_on(q, {(int64_t)a.workspace_bytes}, at::kByte);
    a.workspace = ws.data_ptr();
  }
  check(lib.fwd(&a, stream_of(q)), gate.defined() ? "prefixlm_fwd (gated)" : "prefixlm_fwd");
  return r;
}

// dq, dk, dv: [T, H, D] views the gradients go to; gated: dgate as well, dout is dy
void attn_backward(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& out, const Tensor& lse,
                   const Tensor& out_lo, const Tensor& q_amax, const Tensor& dout, const Tensor& dq, const Tensor& dk,
                   const Tensor& dv, const Tensor& gate, const Tensor& dgate, const Batch& b, int64_t cap) {
  const int64_t T = q.size(0), H = q.size(1), D = q.size(2);
  prefixlm_bwd_args a{};
  b.fill(a, b.plan);
  a.num_tokens = (int32_t)T;
  a.num_heads = (int32_t)H;
  a.head_dim = (int32_t)D;
  a.q = q.const_data_ptr();
  a.k = k.const_data_ptr();
  a.v = v.const_data_ptr();
  a.out = out.const_data_ptr();
  a.out_lo = out_lo.const_data_ptr();
  a.dout = dout.const_data_ptr();
  a.lse = lse.const_data_ptr<float>();
  a.q_amax = q_amax.const_data_ptr<float>();
  a.dq = dq.data_ptr();
  a.dk = dk.data_ptr();
  a.dv = dv.data_ptr();
  a.q_stride_t = q.stride(0), a.q_stride_h = q.stride(1);
  a.k_stride_t = k.stride(0), a.k_stride_h = k.stride(1);
  a.v_stride_t = v.stride(0), a.v_stride_h = v.stride(1);
  a.out_stride_t = out.stride(0), a.out_stride_h = out.stride(1);
  a.out_lo_stride_t = out_lo.stride(0), a.out_lo_stride_h = out_lo.stride(1);
  a.dout_stride_t = dout.stride(0), a.dout_stride_h = dout.stride(1);
  a.dq_stride_t = dq.stride(0), a.dq_stride_h = dq.stride(1);
  a.dk_stride_t = dk.stride(0), a.dk_stride_h = dk.stride(1);
  a.dv_stride_t = dv.stride(0), a.dv_stride_h = dv.stride(1);
  Tensor dout_attn;
  if (gate.defined()) {
    dout_attn = empty_like_on(q, {T, H, D}, at::kBFloat16);
    a.gate = gate.const_data_ptr();
    a.dgate = dgate.data_ptr();
    a.dout_attn = dout_attn.data_ptr();
    a.gate_stride_t = gate.stride(0), a.gate_stride_h = gate.stride(1);
    a.dgate_stride_t = dgate.stride(0), a.dgate_stride_h = dgate.stride(1);
    a.dout_attn_stride_t = H * D, a.dout_attn_stride_h = D;
  }
  a.workspace_bytes = lib.bwd_ws(T, H, D, b.total.v, b.nseq.v);
  const Tensor ws = empty_like_on(q, {(int64_t)a.workspace_bytes}, at::kByte);
  a.workspace = ws.data_ptr();
  const int64_t blocks = b.plan.defined() && b.has_dsb ? b.dsb.v : 0;
  const Tensor ds = ds_buffer(q, T, H, b, blocks, cap);
  if (ds.defined()) {
    a.ds_buf = ds.data_ptr();
    a.ds_buf_bytes = (size_t)ds.numel();
    a.ds_blocks = blocks;
  }
  check(lib.bwd(&a, stream_of(q)), gate.defined() ? "prefixlm_bwd (gated)" : "prefixlm_bwd");
}

// A backward runs the kernels directly on plain tensors; one that is recorded itself, or
// under a mode or a batched gradient, is the custom op's. So is one whose saved tensors are not
// those the forward saved: a saved-tensors hook may give back another dtype, shape, layout or
// device, and the kernels get raw pointers. The custom op copies or refuses such operands.
bool direct_backward(const variable_list& saved, const Tensor& grad, const Tensor& like, int64_t* cap) {
  if (at::GradMode::is_enabled() || !plain_state() || !ds_cap(like, cap)) return false;
  for (const Tensor& t : saved)
    if (t.defined() && !plain_tensor(t, !t.device().is_cpu())) return false;
  return plain_tensor(grad) && grad.scalar_type() == at::kBFloat16 && plain_tensor(like) &&
         grad.device() == like.device();
}
bool is_array(const Tensor& x, at::ScalarType dt, at::IntArrayRef sizes, const Tensor& like) {
  return x.defined() && x.scalar_type() == dt && x.sizes() == sizes && x.device() == like.device();
}
// out, lse, out_lo and q_amax as attn_forward makes them for the [T, H, D] of `sizes`
bool attn_saved(const Tensor& out, const Tensor& lse, const Tensor& out_lo, const Tensor& q_amax, at::IntArrayRef sizes,
                const Tensor& like) {
  return is_array(out, at::kBFloat16, sizes, like) && operand_layout(out) &&
         is_array(lse, at::kFloat, {sizes[1], sizes[0]}, like) && lse.is_contiguous() &&
         is_array(out_lo, at::kChar, sizes, like) && out_lo.stride(2) == 1 && out_lo.stride(0) % 16 == 0 &&
         out_lo.stride(1) % 16 == 0 && aligned(out_lo, 16) &&
         is_array(q_amax, at::kFloat, {(int64_t)lib.q_amax_count(sizes[0], sizes[1])}, like) && q_amax.is_contiguous();
}
// what the fused layer reads of cos and sin [T, 128]
bool rope_tables(const Tensor& cos, const Tensor& sin, int64_t T, const Tensor& like) {
  for (const Tensor& c : {cos, sin})
    if (!is_array(c, at::kFloat, {T, 128}, like) || c.stride(1) != 1 || c.stride(0) % 4 ||
        c.stride(0) != cos.stride(0) || !aligned(c, 16))
      return false;
  return true;
}

FwdOut varlen_forward(const Tensor& q, const Tensor& k, const Tensor& v, const Batch& b) {
  const Recorded call("prefixlm::varlen_fwd", {q, k, v});
  return attn_forward(q, k, v, Tensor(), b);
}

struct Varlen : torch::autograd::Function<Varlen> {
  static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const Batch& b) {
    FwdOut r = varlen_forward(q, k, v, b);
    variable_list s{q, k, v, r.out, r.lse, r.out_lo, r.q_amax};
    b.save(s, ctx);
    ctx->save_for_backward(std::move(s));
    return r.out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const Batch b = Batch::restore(s, 7, ctx);
    int64_t cap = 0;
    variable_list g;
    bool direct = direct_backward(s, grads[0], s[0], &cap) &&
                  attn_saved(s[3], s[4], s[5], s[6], grads[0].sizes(), s[0]) && b.restored(s[0]);
    for (int i = 0; i < 3 && direct; ++i)
      direct = is_array(s[i], at::kBFloat16, grads[0].sizes(), s[0]) && operand_layout(s[i]);
    if (direct) {
      const Recorded call("prefixlm::varlen_bwd", {s[0], s[1], s[2], grads[0]});
      const c10::DeviceGuard guard(s[0].device());
      const Tensor dout = as_operand(grads[0]);
      for (int i = 0; i < 3; ++i) g.push_back(empty_like_on(s[0], s[0].sizes(), at::kBFloat16));
      attn_backward(s[0], s[1], s[2], s[3], s[4], s[5], s[6], dout, g[0], g[1], g[2], Tensor(), Tensor(), b, cap);
    } else {
      torch::jit::Stack st{s[0], s[1], s[2], b.causal, grads[0], s[3], s[4], s[5], s[6]};
      b.push(st, true);
      g = call_op("prefixlm::varlen_bwd", std::move(st));
    }
    g.emplace_back();
    return g;
  }
};

void rope(const Tensor& x, const Tensor& y, const Tensor& cos, const Tensor& sin, bool backward) {
  prefixlm_rope_args a{};
  a.x = x.const_data_ptr();
  a.y = y.data_ptr();
  a.cos = cos.const_data_ptr<float>();
  a.sin = sin.const_data_ptr<float>();
  a.x_stride_t = x.stride(0), a.x_stride_h = x.stride(1);
  a.y_stride_t = y.stride(0), a.y_stride_h = y.stride(1);
  a.cs_stride_t = cos.stride(0);
  a.num_tokens = (int32_t)x.size(0);
  a.num_heads = (int32_t)x.size(1);
  a.head_dim = (int32_t)x.size(2);
  a.backward = i32(backward);
  check(lib.rope(&a, stream_of(x)), "prefixlm_rope");
}

struct LayerOut {
  FwdOut attn;
  Tensor qk;
};
LayerOut layer_forward(const Tensor& gqkv, const Tensor& cos, const Tensor& sin, const Batch& b) {
  const int64_t T = gqkv.size(0), H = gqkv.size(1) / 4, D = gqkv.size(2);
  const Recorded call("prefixlm::attn_layer_fwd", {gqkv, cos, sin});
  LayerOut r;
  r.qk = empty_like_on(gqkv, {T, 2 * H, D}, at::kBFloat16);
  rope(gqkv.narrow(1, H, 2 * H), r.qk, cos, sin, false);
  r.attn = attn_forward(r.qk.narrow(1, 0, H), r.qk.narrow(1, H, H), gqkv.narrow(1, 3 * H, H), gqkv.narrow(1, 0, H), b);
  return r;
}

struct Layer : torch::autograd::Function<Layer> {
  static Tensor forward(AutogradContext* ctx, const Tensor& gqkv, const Tensor& cos, const Tensor& sin, const Batch& b) {
    LayerOut r = layer_forward(gqkv, cos, sin, b);
    variable_list s{gqkv, r.qk, r.attn.out, r.attn.lse, r.attn.out_lo, r.attn.q_amax, cos, sin};
    b.save(s, ctx);
    ctx->save_for_backward(std::move(s));
    return r.attn.y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const Batch b = Batch::restore(s, 8, ctx);
    int64_t cap = 0;
    Tensor dg;
    const Tensor &gqkv = s[0], &qk = s[1];
    bool direct = direct_backward(s, grads[0], gqkv, &cap) && b.restored(gqkv);
    if (direct) {
      const int64_t T = grads[0].size(0), H = grads[0].size(1);
      direct = is_array(gqkv, at::kBFloat16, {T, 4 * H, 128}, gqkv) && gqkv.is_contiguous() && aligned(gqkv, 16) &&
               is_array(qk, at::kBFloat16, {T, 2 * H, 128}, gqkv) && qk.is_contiguous() && aligned(qk, 16) &&
               attn_saved(s[2], s[3], s[4], s[5], grads[0].sizes(), gqkv) && rope_tables(s[6], s[7], T, gqkv);
    }
    if (direct) {
      const Recorded call("prefixlm::attn_layer_bwd", {grads[0], gqkv});
      const int64_t H = grads[0].size(1);
      const c10::DeviceGuard guard(gqkv.device());
      const Tensor dy = grads[0].contiguous();
      dg = empty_like_on(gqkv, gqkv.sizes(), at::kBFloat16);
      attn_backward(qk.narrow(1, 0, H), qk.narrow(1, H, H), gqkv.narrow(1, 3 * H, H), s[2], s[3], s[4], s[5], dy,
                    dg.narrow(1, H, H), dg.narrow(1, 2 * H, H), dg.narrow(1, 3 * H, H), gqkv.narrow(1, 0, H),
                    dg.narrow(1, 0, H), b, cap);
      const Tensor dqk = dg.narrow(1, H, 2 * H);
      rope(dqk, dqk, s[6], s[7], true);
    } else {
      torch::jit::Stack st{grads[0], s[0], s[1], s[2], s[3], s[4], s[5], s[6], s[7], b.causal};
      b.push(st, true);
      dg = call_op("prefixlm::attn_layer_bwd", std::move(st))[0];
    }
    return {dg, Tensor(), Tensor(), Tensor()};
  }
};

// ---- the block's norm and activation ----------------------------------------------------------
// x as [rows, cols] with 16-byte rows, or undefined; one row repeated only with `repeated`
Tensor rows_view(const Tensor& x, bool repeated = false) {
  if (x.scalar_type() != at::kBFloat16 || x.dim() < 1 || x.size(-1) < 1 || x.numel() == 0) return Tensor();
  Tensor r;
  if (x.dim() == 2) {
    r = x;
  } else {
    if (!x.is_contiguous()) return Tensor();
    r = x.view({-1, x.size(-1)});
  }
  return r.stride(1) == 1 && r.stride(0) % 8 == 0 &&
                 (r.stride(0) >= r.size(1) || (repeated && r.stride(0) == 0)) && aligned(r, 16)
             ? r
             : Tensor();
}
Tensor rows_of(const Tensor& x) {   // a gradient: copied where its layout does not serve
  const Tensor r = rows_view(x);
  return r.defined() ? r : x.reshape({-1, x.size(-1)}).contiguous();
}

Tensor swiglu_forward(const Tensor& gu, const Tensor& g2) {
  const Recorded call("prefixlm::swiglu_fwd", {gu});
  const int64_t rows = g2.size(0), F = g2.size(1) / 2;
  auto sizes = gu.sizes().vec();
  sizes.back() = F;
  const Tensor y = empty_like_on(gu, sizes, at::kBFloat16);
  prefixlm_swiglu_args a{};
  a.gu = g2.const_data_ptr();
  a.y = y.data_ptr();
  a.gu_stride = g2.stride(0);
  a.y_stride = F;
  a.rows = rows;
  a.cols = F;
  check(lib.swiglu_fwd(&a, stream_of(gu)), "prefixlm_swiglu_fwd");
  return y;
}
struct Swiglu : torch::autograd::Function<Swiglu> {
  static Tensor forward(AutogradContext* ctx, const Tensor& gu, const Tensor& g2) {
    ctx->save_for_backward({gu});
    return swiglu_forward(gu, g2);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const Tensor& gu = s[0];
    int64_t cap = 0;
    Tensor g2;
    if (direct_backward(s, grads[0], gu, &cap) && (g2 = rows_view(gu)).defined() &&
        g2.size(1) == 2 * grads[0].size(-1) && gu.numel() == 2 * grads[0].numel()) {
      const Recorded call("prefixlm::swiglu_bwd", {gu, grads[0]});
      const c10::DeviceGuard guard(gu.device());
      const Tensor d2 = rows_of(grads[0]);
      const Tensor dgu = empty_like_on(gu, gu.sizes(), at::kBFloat16);
      prefixlm_swiglu_args a{};
      a.gu = g2.const_data_ptr();
      a.dy = d2.const_data_ptr();
      a.dgu = dgu.data_ptr();
      a.gu_stride = g2.stride(0);
      a.dy_stride = d2.stride(0);
      a.dgu_stride = g2.size(1);
      a.rows = g2.size(0);
      a.cols = g2.size(1) / 2;
      check(lib.swiglu_bwd(&a, stream_of(gu)), "prefixlm_swiglu_bwd");
      return {dgu, Tensor()};
    }
    return {call_op("prefixlm::swiglu_bwd", {gu, grads[0]})[0], Tensor()};
  }
};

Tensor rms_forward(const Tensor& x, const Tensor& x2, double eps, Tensor* rstd) {
  const Recorded call("prefixlm::rms_norm_fwd", {x});
  const Tensor y = empty_like_on(x, x.sizes(), at::kBFloat16);
  *rstd = empty_like_on(x, {x2.size(0)}, at::kFloat);
  prefixlm_rmsnorm_args a{};
  a.x = x2.const_data_ptr();
  a.y = y.data_ptr();
  a.rstd = rstd->data_ptr<float>();
  a.x_stride = x2.stride(0);
  a.y_stride = x2.size(1);
  a.rows = x2.size(0);
  a.cols = (int32_t)x2.size(1);
  a.eps = (float)eps;
  check(lib.rmsnorm_fwd(&a, stream_of(x)), "prefixlm_rmsnorm_fwd");
  return y;
}
struct RmsNorm : torch::autograd::Function<RmsNorm> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& x2, double eps) {
    Tensor rstd;
    const Tensor y = rms_forward(x, x2, eps, &rstd);
    ctx->save_for_backward({x, rstd});
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const Tensor& x = s[0];
    int64_t cap = 0;
    Tensor x2;
    if (direct_backward(s, grads[0], x, &cap) && (x2 = rows_view(x)).defined() && x.sizes() == grads[0].sizes() &&
        is_array(s[1], at::kFloat, {x2.size(0)}, x) && s[1].is_contiguous()) {
      const Recorded call("prefixlm::rms_norm_bwd", {x, grads[0]});
      const c10::DeviceGuard guard(x.device());
      const Tensor d2 = rows_of(grads[0]);
      const Tensor dx = empty_like_on(x, x.sizes(), at::kBFloat16);
      prefixlm_rmsnorm_args a{};
      a.x = x2.const_data_ptr();
      a.dy = d2.const_data_ptr();
      a.dx = dx.data_ptr();
      a.rstd = s[1].data_ptr<float>();
      a.x_stride = x2.stride(0);
      a.dy_stride = d2.stride(0);
      a.dx_stride = x2.size(1);
      a.rows = x2.size(0);
      a.cols = (int32_t)x2.size(1);
      check(lib.rmsnorm_bwd(&a, stream_of(x)), "prefixlm_rmsnorm_bwd");
      return {dx, Tensor(), Tensor()};
    }
    return {call_op("prefixlm::rms_norm_bwd", {x, s[1], grads[0]})[0], Tensor(), Tensor()};
  }
};

// ---- Python entry points ------------------------------------------------------------------------
// Each returns None for a call that is not plain. The interpreter lock is released around the
// call itself.
PyObject* none() { Py_RETURN_NONE; }
bool ready(Py_ssize_t n, Py_ssize_t want) { return lib.fwd != nullptr && n == want && plain_state(); }

PyObject* py_varlen(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor q, k, v;
  Batch b;
  if (!ready(n, 15) || c10::InferenceMode::is_enabled()) return none();
  if (!get_tensor(a[0], &q) || !get_tensor(a[1], &k) || !get_tensor(a[2], &v)) return none();
  if (!operand(q) || !operand(k) || !operand(v) || q.sizes() != k.sizes() || q.sizes() != v.sizes() ||
      k.device() != q.device() || v.device() != q.device() || q.numel() == 0)
    return none();
  if (!b.parse(a + 3, q, q.size(2))) return none();
  Tensor out;
  {
    pybind11::gil_scoped_release no_gil;
    const c10::DeviceGuard guard(q.device());
    out = wants_grad(q) || wants_grad(k) || wants_grad(v) ? Varlen::apply(q, k, v, b)
                                                          : varlen_forward(q, k, v, b).out;
  }
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

PyObject* py_layer(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor g, cos, sin;
  Batch b;
  if (!ready(n, 15) || c10::InferenceMode::is_enabled()) return none();
  if (!get_tensor(a[0], &g) || !get_tensor(a[1], &cos) || !get_tensor(a[2], &sin)) return none();
  if (g.scalar_type() != at::kBFloat16 || g.dim() != 3 || g.size(1) % 4 || g.size(2) != 128 || g.numel() == 0 ||
      !g.is_contiguous() || !aligned(g, 16))
    return none();
  if (!rope_tables(cos, sin, g.size(0), g) || wants_grad(cos) || wants_grad(sin)) return none();
  if (!b.parse(a + 3, g, g.size(2))) return none();
  Tensor y;
  {
    pybind11::gil_scoped_release no_gil;
    const c10::DeviceGuard guard(g.device());
    y = wants_grad(g) ? Layer::apply(g, cos, sin, b) : layer_forward(g, cos, sin, b).attn.y;
  }
  return THPVariable_Wrap(y);
  END_HANDLE_TH_ERRORS
}

bool cache_layout(const Tensor& x) {
  return x.scalar_type() == at::kBFloat16 && x.dim() == 4 && x.stride(3) == 1 && x.stride(0) % 8 == 0 &&
         x.stride(1) % 8 == 0 && x.stride(2) % 8 == 0 && aligned(x, 16);
}
// q, k_cache, v_cache, k, v, cache_seqlens (int or tensor), softmax_scale (float or None), causal
PyObject* py_kvcache(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor q, kc, vc, k, v, lens;
  bool causal;
  double scale;
  int64_t len = 0;
  if (!ready(n, 8) || c10::InferenceMode::is_enabled()) return none();
  if (!get_tensor(a[0], &q) || !get_tensor(a[1], &kc) || !get_tensor(a[2], &vc)) return none();
  const bool has_new = a[3] != Py_None;
  if (has_new != (a[4] != Py_None) || (has_new && (!get_tensor(a[3], &k) || !get_tensor(a[4], &v)))) return none();
  for (const Tensor* t : {&q, &kc, &vc, &k, &v})
    if (t->defined() && (!cache_layout(*t) || t->device() != q.device() || t->numel() == 0 || wants_grad(*t))) return none();
  const int64_t B = q.size(0), S = q.size(1), H = q.size(2), D = q.size(3), Smax = kc.size(1);
  if (kc.sizes() != vc.sizes() || kc.size(0) != B || kc.size(2) != H || kc.size(3) != D) return none();
  if (has_new && (k.sizes() != q.sizes() || v.sizes() != q.sizes())) return none();
  if (PyLong_CheckExact(a[5])) {
    Scalar s;
    if (!get_scalar(a[5], &s)) return none();
    len = s.v;
  } else if (!get_tensor(a[5], &lens) || !meta(lens, q) || lens.numel() != B) {
    return none();
  }
  if (a[6] == Py_None)
    scale = 1.0 / std::sqrt((double)D);
  else if (!get_double(a[6], &scale))
    return none();
  if (!get_bool(a[7], &causal)) return none();
  Tensor out;
  {
    pybind11::gil_scoped_release no_gil;
    const Recorded call("prefixlm::kvcache_attn", {q, kc, vc});
    const c10::DeviceGuard guard(q.device());
    out = empty_like_on(q, {B, S, H, D}, at::kBFloat16);
    prefixlm_kvcache_args p{};
    p.workspace_bytes = lib.kv_ws(B, S, H, D, Smax);
    const Tensor ws = empty_like_on(q, {(int64_t)p.workspace_bytes}, at::kByte);
    p.workspace = ws.data_ptr();
    p.q = q.const_data_ptr();
    p.k_cache = kc.data_ptr();
    p.v_cache = vc.data_ptr();
    p.out = out.data_ptr();
    p.q_stride_b = q.stride(0), p.q_stride_s = q.stride(1), p.q_stride_h = q.stride(2);
    if (has_new) {
      p.k = k.const_data_ptr();
      p.v = v.const_data_ptr();
      p.k_stride_b = k.stride(0), p.k_stride_s = k.stride(1), p.k_stride_h = k.stride(2);
      p.v_stride_b = v.stride(0), p.v_stride_s = v.stride(1), p.v_stride_h = v.stride(2);
    }
    p.k_cache_stride_b = kc.stride(0), p.k_cache_stride_s = kc.stride(1), p.k_cache_stride_h = kc.stride(2);
    p.v_cache_stride_b = vc.stride(0), p.v_cache_stride_s = vc.stride(1), p.v_cache_stride_h = vc.stride(2);
    p.out_stride_b = S * H * D, p.out_stride_s = H * D, p.out_stride_h = D;
    p.cache_seqlens = lens.defined() ? lens.const_data_ptr<int32_t>() : nullptr;
    p.cache_seqlen = (int32_t)len;
    p.batch = (int32_t)B;
    p.seqlen_q = (int32_t)S;
    p.num_heads = (int32_t)H;
    p.head_dim = (int32_t)D;
    p.max_seqlen_cache = (int32_t)Smax;
    p.is_causal = i32(causal);
    p.softmax_scale = (float)scale;
    check(lib.kv_fwd(&p, stream_of(q)), "prefixlm_kvcache_fwd");
    // the op writes the caches in place
    kc.unsafeGetTensorImpl()->bump_version();
    vc.unsafeGetTensorImpl()->bump_version();
  }
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

PyObject* py_swiglu(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor gu;
  if (!ready(n, 1) || c10::InferenceMode::is_enabled() || !get_tensor(a[0], &gu)) return none();
  Tensor g2;
  Tensor y;
  {
    pybind11::gil_scoped_release no_gil;
    const at::NoGradGuard no_grad;
    g2 = rows_view(gu);
  }
  if (!g2.defined() || g2.size(1) % 16) return none();
  {
    pybind11::gil_scoped_release no_gil;
    const c10::DeviceGuard guard(gu.device());
    y = wants_grad(gu) ? Swiglu::apply(gu, g2.detach()) : swiglu_forward(gu, g2);
  }
  return THPVariable_Wrap(y);
  END_HANDLE_TH_ERRORS
}

PyObject* py_rms_norm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor x;
  double eps;
  if (!ready(n, 2) || c10::InferenceMode::is_enabled() || !get_tensor(a[0], &x) || !get_double(a[1], &eps)) return none();
  Tensor x2;
  Tensor y;
  {
    pybind11::gil_scoped_release no_gil;
    const at::NoGradGuard no_grad;
    x2 = rows_view(x);
  }
  if (!x2.defined() || x2.size(1) > INT32_MAX) return none();
  {
    pybind11::gil_scoped_release no_gil;
    const c10::DeviceGuard guard(x.device());
    Tensor rstd;
    y = wants_grad(x) ? RmsNorm::apply(x, x2.detach(), eps) : rms_forward(x, x2, eps, &rstd);
  }
  return THPVariable_Wrap(y);
  END_HANDLE_TH_ERRORS
}

// x, r, eps, with_y -> (x + r, its norm) or (x + r, its row scales)
PyObject* py_add_rmsnorm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor x, r;
  double eps;
  bool with_y;
  if (!ready(n, 4) || c10::InferenceMode::is_enabled()) return none();
  if (!get_tensor(a[0], &x) || !get_tensor(a[1], &r) || !get_double(a[2], &eps) || !get_bool(a[3], &with_y) ||
      wants_grad(x) || wants_grad(r) || x.sizes() != r.sizes() || x.device() != r.device())
    return none();
  Tensor s, y;
  {
    pybind11::gil_scoped_release no_gil;
    const at::NoGradGuard no_grad;
    const Tensor x2 = rows_view(x, true), r2 = rows_view(r, true);
    if (x2.defined() && r2.defined() && x2.size(1) <= INT32_MAX) {
      const Recorded call("prefixlm::add_rmsnorm", {x, r});
      const c10::DeviceGuard guard(x.device());
      s = empty_like_on(x, x.sizes(), at::kBFloat16);
      if (with_y) y = empty_like_on(x, x.sizes(), at::kBFloat16);
      const Tensor rstd = empty_like_on(x, {x2.size(0)}, at::kFloat);
      prefixlm_add_rmsnorm_args p{};
      p.x = x2.const_data_ptr();
      p.r = r2.const_data_ptr();
      p.s = s.data_ptr();
      p.y = with_y ? y.data_ptr() : nullptr;
      p.rstd = rstd.data_ptr<float>();
      p.x_stride = x2.stride(0);
      p.r_stride = r2.stride(0);
      p.s_stride = p.y_stride = x2.size(1);
      p.rows = x2.size(0);
      p.cols = (int32_t)x2.size(1);
      p.eps = (float)eps;
      check(lib.add_rmsnorm(&p, stream_of(x)), "prefixlm_add_rmsnorm");
      if (!with_y) y = rstd;
    }
  }
  if (!s.defined()) return none();
  PyObject* t = PyTuple_New(2);
  if (!t) return nullptr;
  PyTuple_SET_ITEM(t, 0, THPVariable_Wrap(s));
  PyTuple_SET_ITEM(t, 1, THPVariable_Wrap(y));
  return t;
  END_HANDLE_TH_ERRORS
}

// The projection of x by w; scales: the row scales of x, or undefined (norm says whether the
// call finds them itself). Undefined for operands that are not plain.
Tensor projection(const Tensor& x, const Tensor& w, const Tensor& scales, bool sw, bool norm, double eps) {
  const at::NoGradGuard no_grad;
  const Tensor x2 = rows_view(x);
  if (!x2.defined() || w.scalar_type() != at::kBFloat16 || w.dim() != 2 || w.device() != x.device() ||
      w.stride(1) != 1 || w.stride(0) % 8 || !aligned(w, 16) || w.size(1) != x2.size(1) || x2.size(0) > INT32_MAX ||
      w.size(0) > INT32_MAX)
    return Tensor();
  const c10::DeviceGuard guard(x.device());
  const int64_t M = x2.size(0), N = w.size(0), nout = sw ? N / 2 : N;
  auto sizes = x.sizes().vec();
  sizes.back() = nout;
  const Tensor y = empty_like_on(x, sizes, at::kBFloat16);
  Tensor rstd = scales;
  prefixlm_proj_gemm_args p{};
  if (norm && !rstd.defined()) rstd = empty_like_on(x, {M}, at::kFloat);
  if (rstd.defined()) p.rstd = rstd.data_ptr<float>();
  p.x = x2.const_data_ptr();
  p.w = w.const_data_ptr();
  p.y = y.data_ptr();
  p.x_stride = x2.stride(0);
  p.w_stride = w.stride(0);
  p.y_stride = nout;
  p.M = (int32_t)M;
  p.K = (int32_t)x2.size(1);
  p.N = (int32_t)N;
  p.swiglu = i32(sw);
  p.norm = i32(norm);
  p.eps = (float)eps;
  if (scales.defined()) {
    const Recorded call("prefixlm::proj_gemm_scaled", {x, w, scales});
    check(lib.proj_gemm_scaled(&p, stream_of(x)), "prefixlm_proj_gemm_scaled");
  } else {
    const Recorded call("prefixlm::proj_gemm", {x, w});
    check(lib.proj_gemm(&p, stream_of(x)), "prefixlm_proj_gemm");
  }
  return y;
}
// x, w, swiglu, norm, eps
PyObject* py_proj_gemm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor x, w;
  bool sw, norm;
  double eps;
  if (!ready(n, 5) || c10::InferenceMode::is_enabled()) return none();
  if (!get_tensor(a[0], &x) || !get_tensor(a[1], &w) || !get_bool(a[2], &sw) || !get_bool(a[3], &norm) ||
      !get_double(a[4], &eps) || wants_grad(x) || wants_grad(w))
    return none();
  Tensor y;
  {
    pybind11::gil_scoped_release no_gil;
    y = projection(x, w, Tensor(), sw, norm, eps);
  }
  return y.defined() ? THPVariable_Wrap(y) : none();
  END_HANDLE_TH_ERRORS
}
// x, w, rstd, swiglu, eps
PyObject* py_proj_gemm_scaled(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor x, w, rstd;
  bool sw;
  double eps;
  if (!ready(n, 5) || c10::InferenceMode::is_enabled()) return none();
  if (!get_tensor(a[0], &x) || !get_tensor(a[1], &w) || !get_tensor(a[2], &rstd) || !get_bool(a[3], &sw) ||
      !get_double(a[4], &eps) || wants_grad(x) || wants_grad(w) || wants_grad(rstd))
    return none();
  if (rstd.scalar_type() != at::kFloat || rstd.device() != x.device() || !rstd.is_contiguous() || x.dim() < 1 ||
      x.size(-1) < 1 || rstd.numel() != x.numel() / x.size(-1))
    return none();
  Tensor y;
  {
    pybind11::gil_scoped_release no_gil;
    y = projection(x, w, rstd, sw, true, eps);
  }
  return y.defined() ? THPVariable_Wrap(y) : none();
  END_HANDLE_TH_ERRORS
}

// bind(addresses in Lib's order, dS buffer cap per device, torch.nn.Parameter)
PyObject* py_bind(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  PyObject *addrs, *caps, *param;
  if (!PyArg_ParseTuple(args, "OOO", &addrs, &caps, &param)) return nullptr;
  const auto p = pybind11::cast<std::vector<uintptr_t>>(pybind11::handle(addrs));
  TORCH_CHECK(p.size() * sizeof(void*) == sizeof(Lib), "bind takes ", sizeof(Lib) / sizeof(void*), " addresses");
  g_ds_cap = pybind11::cast<std::vector<int64_t>>(pybind11::handle(caps));
  Py_INCREF(param);
  g_parameter = param;
  memcpy(&lib, p.data(), sizeof(Lib));
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}
PyObject* py_set_timer(PyObject*, PyObject* h) {
  HANDLE_TH_ERRORS
  g_timer.store(h == Py_None ? nullptr : PyLong_AsVoidPtr(h));
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

#define FAST(f) reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)), METH_FASTCALL
PyMethodDef methods[] = {
    {"bind", py_bind, METH_VARARGS, nullptr},
    {"set_timer", py_set_timer, METH_O, nullptr},
    {"varlen", FAST(py_varlen), nullptr},
    {"layer", FAST(py_layer), nullptr},
    {"kvcache", FAST(py_kvcache), nullptr},
    {"swiglu", FAST(py_swiglu), nullptr},
    {"rms_norm", FAST(py_rms_norm), nullptr},
    {"add_rmsnorm", FAST(py_add_rmsnorm), nullptr},
    {"proj_gemm", FAST(py_proj_gemm), nullptr},
    {"proj_gemm_scaled", FAST(py_proj_gemm_scaled), nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_torch_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__torch_calls() { return PyModule_Create(&module); }

// The launch path of the hot operators in native code: argument checks, output allocation, the kernel
// choice that needs a workspace, and the C-ABI call. The Python operators call these first. Each takes
// the plain case (strided GPU tensors that the kernel reads as they are) and returns None for
// anything else — another layout that needs a copy, a type to convert, an input to refuse — so that the
// Python code behind it stays the one place for conversions and error messages. Per launch the
// host takes about 7 us on this path and 20 on the Python one; a 1152-token image block (18 launches,
// 160 us of kernels) was bound by it.
//
// Tensors are read only: no autograd graph, no view. The entry points are reached through the
// addresses that the ctypes binding holds, so both bindings run the same loaded library.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/torch.h>

#include <array>
#include <cmath>
#include <unordered_map>

#include "kx355.h"

namespace {

using at::Tensor;

// ---- the library's entry points, by address --------------------------------------------------------

struct Api {
  decltype(&kx_gemm_bf16) gemm[2];  // [fp16]
  decltype(&kx_gemm_splitk_bf16) splitk[2];
  decltype(&kx_adaln_norm_bf16) adaln[2];
  decltype(&kx_modulate_bf16) modulate[2];
  decltype(&kx_rmsnorm_rope_bf16) rmsnorm[2];
  decltype(&kx_qk_rmsnorm_rope_bf16) qk128[2], qk64[2];
  decltype(&kx_attention_gqa_fwd_bf16) attention[2];
  decltype(&kx_attention_split_fwd_bf16) attention_split[2];
  decltype(&kx_attention_tail_fwd_bf16) attention_tail[2];
  decltype(&kx_gemm_columns_bf16) columns;
  decltype(&kx_table_add_f32) table_add;
  decltype(&kx_last_error) last_error;
} api;

PyObject* kernel_error = nullptr;    // the exception of a failed entry point
PyObject* gemm_plan_fn = nullptr;    // (m, n, k) -> (head rows or 0, splits)
PyObject* attn_plan_fn = nullptr;    // (batch, tq, tk, heads) -> (slices of the tail, slices)

struct Refused {};  // raised inside a function: return None to the Python caller
struct PyFailed {};  // a Python error is set

// Runs an entry point without the interpreter lock (a launch can wait for room in its stream's queue).
struct Unlocked {
  PyThreadState* state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
};
template <typename F, typename... A>
void call(const char* name, F* fn, A... args) {
  int rc;
  {
    Unlocked unlocked;
    rc = fn(args...);
  }
  if (rc == KX_OK) return;
  PyErr_Format(kernel_error, "%s failed (%d): %s", name, rc, api.last_error());
  throw PyFailed{};
}

// ---- arguments -------------------------------------------------------------------------------------

// A plain GPU tensor (not a subclass, not a wrapper without storage).
const Tensor& tensor(PyObject* o) {
  if (!THPVariable_CheckExact(o)) throw Refused{};
  const Tensor& t = THPVariable_Unpack(o);
  if (!t.is_cuda() || t.layout() != c10::kStrided || !t.has_storage()) throw Refused{};
  return t;
}
const Tensor* optional(PyObject* o) { return o == Py_None ? nullptr : &tensor(o); }
int64_t integer(PyObject* o) {
  const int64_t v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) throw PyFailed{};
  return v;
}
float real(PyObject* o) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) throw PyFailed{};
  return (float)v;
}
void need(bool ok) {
  if (!ok) throw Refused{};
}

uintptr_t address(const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()); }
void* ptr(const Tensor& t) { return t.data_ptr(); }
void* ptr(const Tensor* t) { return t ? t->data_ptr() : nullptr; }
bool at16(const Tensor& t) { return address(t) % 16 == 0; }
bool is_half(at::ScalarType s) { return s == at::kBFloat16 || s == at::kHalf; }

// (rows, width, row stride) of a tensor whose last axis is contiguous and whose leading axes
// flatten into evenly strided rows.
struct Rows {
  int64_t rows, width, ld;
};
Rows rows_of(const Tensor& t) {
  const auto sizes = t.sizes();
  const auto strides = t.strides();
  const int64_t dims = (int64_t)sizes.size();
  need(dims >= 1);
  const int64_t width = sizes[dims - 1];
  need(width > 0 && (strides[dims - 1] == 1 || width == 1));
  if (dims == 1) return {1, width, width};
  int64_t rows = 1;
  for (int64_t a = 0; a < dims - 1; ++a) rows *= sizes[a];
  const int64_t stride = strides[dims - 2];
  int64_t expected = stride;
  for (int64_t a = dims - 2; a >= 0; --a) {
    need(sizes[a] == 1 || strides[a] == expected);
    expected *= sizes[a];
  }
  return {rows, width, std::max(stride, width)};
}

// (divisor, stride) of an fp32 modulation tensor broadcast over `rows` rows.
struct Mod {
  int64_t div, stride;
};
Mod mod_of(const Tensor& t, int64_t rows, int64_t width) {
  need(t.scalar_type() == at::kFloat && t.dim() >= 1 && t.size(-1) == width && t.stride(-1) == 1 && at16(t));
  const int64_t count = t.numel() / width;
  if (count == 1) return {1, 0};
  need(count > 0 && rows % count == 0);
  const int64_t stride = t.dim() >= 2 && t.size(-2) != 1 ? t.stride(-2) : t.stride(0);
  need(stride % 4 == 0);
  return {rows / count, stride};
}

int type_code(at::ScalarType s) {
  need(s == at::kFloat || is_half(s));
  return s == at::kFloat ? KX_F32 : s == at::kBFloat16 ? KX_BF16 : KX_F16;
}
at::ScalarType type_of(int64_t code) {
  return code == KX_F32 ? at::kFloat : code == KX_BF16 ? at::kBFloat16 : at::kHalf;
}

Tensor empty_like_rows(const Tensor& t, int64_t width, at::ScalarType type) {
  c10::SmallVector<int64_t, 6> sizes(t.sizes().begin(), t.sizes().end());
  sizes.back() = width;
  return at::empty(sizes, t.options().dtype(type).requires_grad(false));
}
Tensor floats(const Tensor& like, int64_t count) {
  return at::empty({count}, like.options().dtype(at::kFloat).requires_grad(false));
}

// ---- the kernel choices that need a workspace: asked of Python once per shape --------------------

struct ShapeHash {
  size_t operator()(const std::array<int64_t, 4>& s) const {
    uint64_t h = 1469598103934665603ull;
    for (const int64_t v : s) h = (h ^ (uint64_t)v) * 1099511628211ull;
    return (size_t)h;
  }
};
using Plans = std::unordered_map<std::array<int64_t, 4>, std::array<int64_t, 2>, ShapeHash>;
constexpr size_t kMaxPlans = 4096;

std::array<int64_t, 2> plan(Plans& plans, PyObject* fn, const std::array<int64_t, 4>& shape, int arity) {
  const auto it = plans.find(shape);
  if (it != plans.end()) return it->second;
  PyObject* r = arity == 3 ? PyObject_CallFunction(fn, "LLL", shape[0], shape[1], shape[2])
                           : PyObject_CallFunction(fn, "LLLL", shape[0], shape[1], shape[2], shape[3]);
  if (!r) throw PyFailed{};
  long long a = 0, b = 0;
  const int ok = PyArg_ParseTuple(r, "LL", &a, &b);
  Py_DECREF(r);
  if (!ok) throw PyFailed{};
  if (plans.size() >= kMaxPlans) plans.clear();
  return plans[shape] = {a, b};
}
Plans gemm_plans, attn_plans;  // used under the interpreter lock only

// ---- operators -------------------------------------------------------------------------------------

// linear(value, weight, bias, flags, residual, gate, out, out_type, stream): residual + gate *
// act(value @ weight.T + bias); out_type -1: the value's.
Tensor linear(PyObject* const* a) {
  const Tensor& x = tensor(a[0]);
  const Tensor& w = tensor(a[1]);
  const Tensor *bias = optional(a[2]), *resid = optional(a[4]), *gate = optional(a[5]), *out_arg = optional(a[6]);
  int flags = (int)integer(a[3]);
  void* stream = reinterpret_cast<void*>(integer(a[8]));
  const auto type = x.scalar_type();
  need(is_half(type) && w.scalar_type() == type && w.dim() == 2 && w.stride(1) == 1 && w.stride(0) % 8 == 0 && at16(w));
  const Rows rx = rows_of(x);
  const int64_t n = w.size(0), k = w.size(1), m = rx.rows;
  const int64_t ldw = std::max(w.stride(0), k);
  need(rx.width == k && m > 0 && n > 0 && rx.ld % 8 == 0 && at16(x));
  const int64_t code = integer(a[7]);
  Tensor made;
  if (!out_arg) made = empty_like_rows(x, n, code < 0 ? type : type_of(code));
  const Tensor& out = out_arg ? *out_arg : made;
  const Rows ro = rows_of(out);
  need(ro.rows == m && ro.width == n && (out.scalar_type() == type || out.scalar_type() == at::kFloat));
  if (out.scalar_type() == at::kFloat) flags |= KX_EPI_OUT_F32;
  if (bias) {
    need(bias->scalar_type() == type && bias->dim() == 1 && bias->size(0) == n && (n == 1 || bias->stride(0) == 1));
    flags |= KX_EPI_BIAS;
  }
  Rows rr{0, 0, 0};
  Mod mod{1, 0};
  int64_t resid_size = 0;
  if (resid) {
    need(gate);
    rr = rows_of(*resid);
    need(rr.rows == m && rr.width == n && (resid->scalar_type() == type || resid->scalar_type() == at::kFloat));
    mod = mod_of(*gate, m, n);
    flags |= KX_EPI_GATED_RESIDUAL;
    if (resid->scalar_type() == at::kFloat) flags |= KX_EPI_RESID_F32;
    resid_size = resid->element_size();
  }
  const void* gp = resid ? ptr(gate) : nullptr;
  const int h = type == at::kHalf;
  const bool strides_ok = rx.ld <= (1 << 22) && ldw <= (1 << 22);
  const auto [head, splits] = plan(gemm_plans, gemm_plan_fn, {m, n, k, 0}, 3);
  if (strides_ok && head > 0 && (!resid || mod.stride == 0)) {
    // the last rows as K slices, then whole rounds of 256 x 256 tiles over the first (see tail_split)
    const int64_t tail = m - head;
    const Tensor work = floats(x, splits * tail * n);
    const char* xt = static_cast<const char*>(ptr(x)) + head * rx.ld * x.element_size();
    char* ot = static_cast<char*>(ptr(out)) + head * ro.ld * out.element_size();
    const char* rt = resid ? static_cast<const char*>(ptr(resid)) + head * rr.ld * resid_size : nullptr;
    call("kx_gemm_splitk", api.splitk[h], xt, rx.ld, ptr(w), ldw, ptr(bias), ot, ro.ld, tail, n, k, flags, rt,
         rr.ld, (const float*)gp, mod.div, mod.stride, ptr(work), work.numel() * 4, (int)splits, stream);
    call("kx_gemm", api.gemm[h], ptr(x), rx.ld, ptr(w), ldw, ptr(bias), ptr(out), ro.ld, head, n, k, flags,
         ptr(resid), rr.ld, (const float*)gp, mod.div, mod.stride, stream);
  } else if (strides_ok && head == 0 && splits > 1) {
    const Tensor work = floats(x, splits * m * n);
    call("kx_gemm_splitk", api.splitk[h], ptr(x), rx.ld, ptr(w), ldw, ptr(bias), ptr(out), ro.ld, m, n, k, flags,
         ptr(resid), rr.ld, (const float*)gp, mod.div, mod.stride, ptr(work), work.numel() * 4, (int)splits,
         stream);
  } else {
    need(head == 0);  // a tail-split shape with a gate per row or wide rows: the Python rule decides
    call("kx_gemm", api.gemm[h], ptr(x), rx.ld, ptr(w), ldw, ptr(bias), ptr(out), ro.ld, m, n, k, flags,
         ptr(resid), rr.ld, (const float*)gp, mod.div, mod.stride, stream);
  }
  return out;
}

// columns(value, weight, bias, out, q_end, k_end, head_dim, norm_q, norm_k, eps, offset, cos, sin,
//         table_ld, table_rows, table_bs, swiglu_begin, swiglu_out, stream)
Tensor columns(PyObject* const* a) {
  const Tensor& x = tensor(a[0]);
  const Tensor& w = tensor(a[1]);
  const Tensor *bias = optional(a[2]), *out = optional(a[3]), *nq = optional(a[7]), *nk = optional(a[8]);
  const Tensor *cos = optional(a[11]), *sin = optional(a[12]), *sw = optional(a[17]);
  const int64_t q_end = integer(a[4]), k_end = integer(a[5]), head_dim = integer(a[6]), begin = integer(a[16]);
  need(x.scalar_type() == at::kBFloat16 && w.scalar_type() == at::kBFloat16 && w.dim() == 2 && w.stride(1) == 1 &&
       w.stride(0) % 8 == 0 && at16(w) && at16(x));
  const Rows rx = rows_of(x);
  const int64_t n = w.size(0), k = w.size(1);
  need(rx.width == k && rx.rows > 0 && rx.ld % 8 == 0 && (out || begin == 0) && (sw || begin == n));
  if (bias)
    need(bias->scalar_type() == at::kBFloat16 && bias->dim() == 1 && bias->size(0) == n && bias->stride(0) == 1);
  Rows ro{0, 0, 0}, rs{0, 0, 0};
  if (out) {
    ro = rows_of(*out);
    need(out->scalar_type() == at::kBFloat16 && ro.rows == rx.rows && ro.width == begin);
  }
  if (sw) {
    rs = rows_of(*sw);
    need(sw->scalar_type() == at::kBFloat16 && rs.rows == rx.rows && 2 * rs.width == n - begin);
  }
  int code = KX_F32;
  if (k_end > 0) {
    need(nq && nk && cos && sin && nq->scalar_type() == nk->scalar_type() && cos->scalar_type() == at::kFloat &&
         sin->scalar_type() == at::kFloat && nq->dim() == 1 && nk->dim() == 1 && nq->size(0) == head_dim &&
         nk->size(0) == head_dim && nq->stride(0) == 1 && nk->stride(0) == 1);
    code = type_code(nq->scalar_type());
    need(code != KX_F16);
  }
  call("kx_gemm_columns_bf16", api.columns, ptr(x), rx.ld, ptr(w), std::max(w.stride(0), k), ptr(bias), ptr(out),
       ro.ld, rx.rows, n, k, q_end, k_end, head_dim, ptr(nq), ptr(nk), code, real(a[9]), real(a[10]),
       (const float*)ptr(cos), (const float*)ptr(sin), integer(a[13]), 0, integer(a[14]), integer(a[15]), begin,
       ptr(sw), rs.ld, reinterpret_cast<void*>(integer(a[18])));
  return sw ? *sw : *out;
}

// adaln(value, shift, scale, eps, kind, out_type, stream): out_type as the caller's (-1: none given)
Tensor adaln(PyObject* const* a) {
  const Tensor &x = tensor(a[0]), &shift = tensor(a[1]), &scale = tensor(a[2]);
  int kind = (int)integer(a[4]);
  const int64_t code = integer(a[5]);
  const auto type = x.scalar_type();
  at::ScalarType to = code < 0 ? (type == at::kFloat ? at::kBFloat16 : type) : type_of(code);
  need(is_half(to) && (type == to || type == at::kFloat));
  const Rows rx = rows_of(x);
  need(rx.rows > 0 && shift.sizes() == scale.sizes() && shift.strides() == scale.strides());
  const Mod mod = mod_of(shift, rx.rows, rx.width);
  need(scale.scalar_type() == at::kFloat && at16(scale));
  if (type == at::kFloat) kind |= KX_NORM_IN_F32;
  Tensor out = empty_like_rows(x, rx.width, to);
  call("kx_adaln_norm", api.adaln[to == at::kHalf], ptr(x), rx.ld, ptr(out), rx.width, rx.rows, rx.width,
       (const float*)ptr(shift), (const float*)ptr(scale), mod.div, mod.stride, real(a[3]), kind,
       reinterpret_cast<void*>(integer(a[6])));
  return out;
}

// modulate(value, shift, scale, stream)
Tensor modulate(PyObject* const* a) {
  const Tensor &x = tensor(a[0]), &shift = tensor(a[1]), &scale = tensor(a[2]);
  need(is_half(x.scalar_type()) && shift.sizes() == scale.sizes() && shift.strides() == scale.strides());
  const Rows rx = rows_of(x);
  need(rx.rows > 0);
  const Mod mod = mod_of(shift, rx.rows, rx.width);
  need(scale.scalar_type() == at::kFloat && at16(scale));
  Tensor out = empty_like_rows(x, rx.width, x.scalar_type());
  call("kx_modulate", api.modulate[x.scalar_type() == at::kHalf], ptr(x), rx.ld, ptr(out), rx.width, rx.rows,
       rx.width, (const float*)ptr(shift), (const float*)ptr(scale), mod.div, mod.stride,
       reinterpret_cast<void*>(integer(a[3])));
  return out;
}

// The token-major storage of head-major (1 | B, H, T, half) fp32 tables: their token stride, or refused.
int64_t table_ld(const Tensor& cos, const Tensor& sin, int64_t batch, int64_t heads, int64_t tokens, int64_t half) {
  need(cos.scalar_type() == at::kFloat && sin.scalar_type() == at::kFloat && cos.dim() == 4 &&
       cos.sizes() == sin.sizes() && cos.strides() == sin.strides() && (cos.size(0) == 1 || cos.size(0) == batch) &&
       cos.size(1) == heads && cos.size(2) == tokens && cos.size(3) == half);
  const int64_t ld = heads * half;
  need(cos.stride(3) == 1 && (heads == 1 || cos.stride(1) == half) && (tokens == 1 || cos.stride(2) == ld) &&
       (cos.size(0) == 1 || cos.stride(0) == tokens * ld) && at16(cos) && at16(sin));
  return ld;
}

// norm(value, weight, eps, cos, sin, heads, stream): the full-width weighted RMSNorm, with split RoPE
// where tables are given
Tensor norm(PyObject* const* a) {
  const Tensor &x = tensor(a[0]), &w = tensor(a[1]);
  const Tensor *cos = optional(a[3]), *sin = optional(a[4]);
  const int64_t heads = integer(a[5]);
  need(is_half(x.scalar_type()) && x.dim() == 3 && heads > 0);
  const Rows rx = rows_of(x);
  const int64_t dim = rx.width, tokens = x.size(1), head_dim = dim / heads;
  need(rx.rows > 0 && w.dim() == 1 && w.size(0) == dim && w.is_contiguous());
  int64_t ld = 0;
  if (cos) {
    need(sin && dim % heads == 0 && dim % 512 == 0 && head_dim >= 16 && head_dim % 16 == 0 && 512 % head_dim == 0);
    const int64_t vpl = dim / 512;
    need(vpl == 1 || vpl == 2 || vpl == 4 || vpl == 8);
    ld = table_ld(*cos, *sin, x.size(0), heads, tokens, head_dim / 2);
  }
  Tensor out = empty_like_rows(x, dim, x.scalar_type());
  need(!cos || (rx.ld % 8 == 0 && at16(x)));
  call("kx_rmsnorm_rope", api.rmsnorm[x.scalar_type() == at::kHalf], ptr(x), rx.ld, ptr(out), dim, rx.rows, dim,
       dim, ptr(w), type_code(w.scalar_type()), real(a[2]), 0.0f, cos ? KX_ROPE_SPLIT : KX_ROPE_NONE,
       (const float*)ptr(cos), (const float*)ptr(sin), ld, head_dim / 2, tokens, cos && cos->size(0) > 1,
       cos ? head_dim : 0, reinterpret_cast<void*>(integer(a[6])));
  return out;
}

// norm_qk(q, k, wq, wk, eps, cos, sin, heads, stream) -> (q, k): both norms and rotations in one pass
PyObject* norm_qk(PyObject* const* a) {
  const Tensor &q = tensor(a[0]), &k = tensor(a[1]), &wq = tensor(a[2]), &wk = tensor(a[3]);
  const Tensor &cos = tensor(a[5]), &sin = tensor(a[6]);
  const int64_t heads = integer(a[7]);
  need(is_half(q.scalar_type()) && k.scalar_type() == q.scalar_type() && q.dim() == 3 && k.sizes() == q.sizes() &&
       heads > 0);
  const Rows rq = rows_of(q), rk = rows_of(k);
  const int64_t dim = rq.width, head_dim = dim / heads, vpl = dim / 512;
  need(rq.rows > 0 && dim % heads == 0 && (head_dim == 64 || head_dim == 128) && dim % 512 == 0 &&
       (vpl == 2 || vpl == 4 || vpl == 8) && rq.ld % 8 == 0 && rk.ld % 8 == 0 && at16(q) && at16(k));
  need(wq.dim() == 1 && wk.dim() == 1 && wq.size(0) == dim && wk.size(0) == dim && wq.is_contiguous() &&
       wk.is_contiguous() && wq.scalar_type() == wk.scalar_type());
  const int64_t ld = table_ld(cos, sin, q.size(0), heads, q.size(1), head_dim / 2);
  Tensor yq = empty_like_rows(q, dim, q.scalar_type()), yk = empty_like_rows(q, dim, q.scalar_type());
  const int h = q.scalar_type() == at::kHalf;
  call("kx_qk_rmsnorm_rope", (head_dim == 64 ? api.qk64 : api.qk128)[h], ptr(q), rq.ld, ptr(k), rk.ld, ptr(yq),
       dim, ptr(yk), dim, rq.rows, dim, ptr(wq), ptr(wk), type_code(wq.scalar_type()), real(a[4]), 0.0f,
       (const float*)ptr(cos), (const float*)ptr(sin), ld, head_dim / 2, q.size(1), cos.size(0) > 1,
       reinterpret_cast<void*>(integer(a[8])));
  PyObject* pair = PyTuple_New(2);
  if (!pair) throw PyFailed{};
  PyTuple_SET_ITEM(pair, 0, THPVariable_Wrap(std::move(yq)));
  PyTuple_SET_ITEM(pair, 1, THPVariable_Wrap(std::move(yk)));
  return pair;
}

// attention(q, k, v, heads, kv_heads, gate, scale, out, stream): unmasked, (B, T, heads * dim) rows;
// scale None: dim ** -0.5
Tensor attention(PyObject* const* a) {
  const Tensor &q = tensor(a[0]), &k = tensor(a[1]), &v = tensor(a[2]);
  const Tensor *gate = optional(a[5]), *out_arg = optional(a[7]);
  const int64_t heads = integer(a[3]), kv = integer(a[4]);
  void* stream = reinterpret_cast<void*>(integer(a[8]));
  const auto type = q.scalar_type();
  need(is_half(type) && k.scalar_type() == type && v.scalar_type() == type && q.dim() == 3 && k.dim() == 3 &&
       v.sizes() == k.sizes() && q.size(0) == k.size(0) && heads > 0 && kv > 0 && heads % kv == 0);
  const int64_t batch = q.size(0), tq = q.size(1), tk = k.size(1), width = q.size(2), dim = width / heads;
  need(width == heads * dim && (dim == 64 || dim == 128) && k.size(2) == kv * dim && batch > 0 && tq > 0 && tk > 0);
  for (const Tensor* t : {&q, &k, &v})
    need(t->stride(2) == 1 && t->stride(1) % 8 == 0 && at16(*t) &&
         (batch == 1 || t->stride(0) == t->size(1) * t->stride(1)));
  const int64_t kvw = kv * dim;
  need(q.stride(1) >= width && k.stride(1) >= kvw && v.stride(1) >= kvw);
  Tensor made;
  if (!out_arg) made = at::empty({batch, tq, width}, q.options().requires_grad(false));
  const Tensor& out = out_arg ? *out_arg : made;
  need(out.scalar_type() == type && out.dim() == 3 && out.size(0) == batch && out.size(1) == tq &&
       out.size(2) == width && out.stride(2) == 1 && out.stride(1) >= width &&
       (batch == 1 || out.stride(0) == tq * out.stride(1)));
  int64_t ld_gate = 0;
  if (gate) {
    const Rows rg = rows_of(*gate);
    need(gate->scalar_type() == type && rg.rows == batch * tq && rg.width == heads);
    ld_gate = rg.ld;
  }
  const int h = type == at::kHalf;
  const float scale = a[6] == Py_None ? (float)std::pow((double)dim, -0.5) : real(a[6]);
  const auto [tail, splits] = plan(attn_plans, attn_plan_fn, {batch, tq, tk, heads}, 4);
  if (splits > 1) {
    const int64_t chunk = ((tk + splits - 1) / splits + 63) / 64 * 64, used = (tk + chunk - 1) / chunk;
    const Tensor work = floats(q, used * batch * heads * tq * (dim + 2));
    call("kx_attention_split_fwd", api.attention_split[h], ptr(q), q.stride(1), ptr(k), k.stride(1), ptr(v),
         v.stride(1), ptr(out), out.stride(1), batch, tq, tk, heads, kv, dim, scale, ptr(gate), ld_gate, nullptr,
         0, 0, 0, ptr(work), work.numel() * 4, (int)splits, stream);
  } else if (tail > 1 && dim == 128) {
    const int64_t chunk = ((tk + tail - 1) / tail + 63) / 64 * 64, used = (tk + chunk - 1) / chunk;
    const int64_t rest = (tq + 383) / 384 * heads * batch % 256;
    const Tensor work = floats(q, used * rest * 384 * (dim + 2));
    call("kx_attention_tail_fwd", api.attention_tail[h], ptr(q), q.stride(1), ptr(k), k.stride(1), ptr(v), v.stride(1),
         ptr(out), out.stride(1), batch, tq, tk, heads, kv, dim, scale, ptr(gate), ld_gate, ptr(work),
         work.numel() * 4, (int)tail, stream);
  } else {
    call("kx_attention_gqa_fwd", api.attention[h], ptr(q), q.stride(1), ptr(k), k.stride(1), ptr(v), v.stride(1),
         ptr(out), out.stride(1), batch, tq, tk, heads, kv, dim, scale, ptr(gate), ld_gate, stream);
  }
  return out;
}

// table_add(table, ts, round_code, stream): fp32(table) + fp32(ts) as (B, T, rows, D)
Tensor table_add(PyObject* const* a) {
  const Tensor& table = tensor(a[0]);
  const Tensor* ts = optional(a[1]);
  need(table.dim() == 2 && table.stride(1) == 1 && (table.size(0) <= 1 || table.stride(0) == table.size(1)));
  const int64_t rows = table.size(0), dim = table.size(1);
  int64_t batch = 1, tokens = 1, bs = 0, tstr = 0, rs = 0;
  int code = KX_F32;
  if (ts) {
    need(ts->dim() == 4 && ts->size(2) == rows && ts->size(3) == dim && ts->stride(3) == 1);
    batch = ts->size(0);
    tokens = ts->size(1);
    bs = ts->stride(0);
    tstr = ts->stride(1);
    rs = ts->stride(2);
    code = type_code(ts->scalar_type());
  }
  need(batch > 0 && tokens > 0 && rows > 0 && dim > 0);
  Tensor out = at::empty({batch, tokens, rows, dim}, table.options().dtype(at::kFloat).requires_grad(false));
  call("kx_table_add_f32", api.table_add, ptr(table), type_code(table.scalar_type()), ptr(ts), code, bs, tstr, rs,
       (float*)ptr(out), batch, tokens, rows, dim, (int)integer(a[2]), reinterpret_cast<void*>(integer(a[3])));
  return out;
}

// ---- the module ------------------------------------------------------------------------------------

PyObject* wrapped(Tensor (*f)(PyObject* const*), PyObject* const* args) { return THPVariable_Wrap(f(args)); }
PyObject* wrapped(PyObject* (*f)(PyObject* const*), PyObject* const* args) { return f(args); }

template <auto F, int N>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t count) {
  HANDLE_TH_ERRORS
  if (count != N) {
    PyErr_Format(PyExc_TypeError, "expected %d arguments, got %zd", N, count);
    return nullptr;
  }
  if (!api.last_error) {
    PyErr_SetString(PyExc_RuntimeError, "the native launch path is not bound to the library");
    return nullptr;
  }
  try {
    return wrapped(F, args);
  } catch (const Refused&) {
    Py_RETURN_NONE;
  } catch (const PyFailed&) {
    return nullptr;
  }
  END_HANDLE_TH_ERRORS
}

// bind(addresses: dict name -> int, KernelError, gemm_plan, attention_plan)
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t count) {
  if (count != 4 || !PyDict_Check(args[0])) {
    PyErr_SetString(PyExc_TypeError, "bind(addresses, error, gemm_plan, attention_plan)");
    return nullptr;
  }
  Api a{};
  bool ok = true;
  auto get = [&](auto& fn, const char* name) {
    PyObject* v = PyDict_GetItemString(args[0], name);
    const unsigned long long p = v ? PyLong_AsUnsignedLongLong(v) : 0;
    if (!p) ok = false;
    fn = reinterpret_cast<std::remove_reference_t<decltype(fn)>>(static_cast<uintptr_t>(p));
  };
  const char* suffix[2] = {"bf16", "f16"};
  for (int h = 0; h < 2; ++h) {
    auto both = [&](auto& fn, const char* base) { get(fn, (std::string(base) + suffix[h]).c_str()); };
    both(a.gemm[h], "kx_gemm_");
    both(a.splitk[h], "kx_gemm_splitk_");
    both(a.adaln[h], "kx_adaln_norm_");
    both(a.modulate[h], "kx_modulate_");
    both(a.rmsnorm[h], "kx_rmsnorm_rope_");
    both(a.qk128[h], "kx_qk_rmsnorm_rope_");
    both(a.qk64[h], "kx_qk_rmsnorm_rope_h64_");
    both(a.attention[h], "kx_attention_gqa_fwd_");
    both(a.attention_split[h], "kx_attention_split_fwd_");
    both(a.attention_tail[h], "kx_attention_tail_fwd_");
  }
  get(a.columns, "kx_gemm_columns_bf16");
  get(a.table_add, "kx_table_add_f32");
  get(a.last_error, "kx_last_error");
  if (!ok) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_KeyError, "an entry point's address is missing");
    return nullptr;
  }
  for (int i = 1; i < 4; ++i) Py_INCREF(args[i]);
  Py_XSETREF(kernel_error, args[1]);
  Py_XSETREF(gemm_plan_fn, args[2]);
  Py_XSETREF(attn_plan_fn, args[3]);
  gemm_plans.clear();
  attn_plans.clear();
  api = a;
  Py_RETURN_NONE;
}

#define KX_METHOD(f, n) {#f, (PyCFunction)(void (*)(void))entry<f, n>, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    {"bind", (PyCFunction)(void (*)(void))bind, METH_FASTCALL, nullptr},
    KX_METHOD(linear, 9),
    KX_METHOD(columns, 19),
    KX_METHOD(adaln, 7),
    KX_METHOD(modulate, 4),
    KX_METHOD(norm, 7),
    KX_METHOD(norm_qk, 9),
    KX_METHOD(attention, 9),
    KX_METHOD(table_add, 4),
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", "Native launch path of the hot operators", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__host() { return PyModule_Create(&module); }

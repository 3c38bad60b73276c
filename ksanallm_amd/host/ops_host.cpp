// The host side of ksanallm_amd/ops.py's hot calls, in C++: argument checks, output and scratch allocation, the current
// stream and the C-ABI call, on torch tensors.  What bounds a small call is this path and not its kernel: one W4A16 GEMM
// of one row (n = k = 4096, 4 us on the GPU) took 11.9 us of host time when written in Python over ctypes (2.7 us of it
// for torch.cuda.current_stream(), 1.8 us for torch.empty), and a MoE block of one token 36 us.
//
// The library is not linked: bind() takes the addresses of its entry points from the ctypes binding, so that both sides
// always call the same library.  Outputs and scratch come from torch's caching allocator, per call: nothing is shared
// between streams or threads, and nothing is kept.  A call runs on the device of its first tensor and on that device's
// current stream, whatever device is current outside: the allocator hands scratch out, and takes it back, for that stream.
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/ops/empty.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <tuple>
#include <utility>

#include "ksq.h"

namespace {

// ------------------------------------------------------------------------------------------------ the bound library
#define KSQ_FOR_EACH_FN(F) \
  F(w4a16_workspace_size) F(w4a16_gemm) F(fp8_group_quant) F(fp8_blockwise_workspace_size) F(fp8_blockwise_gemm) \
  F(w4a8_static_quant) F(w4a8_workspace_size) F(w4a8_gemm) F(moe_topk_softmax) F(moe_grouped_topk) \
  F(moe_align_capacity) F(moe_align_scratch_bytes) F(moe_align) F(moe_w4a16_row_block) F(moe_fp8_row_block) F(moe_w4a16_gemm) \
  F(moe_w4a16_gate_up_silu) F(moe_w4a16_down_sum) F(moe_fp8_blockwise_gemm) F(moe_fp8_fused_quant) F(moe_fp8_gate_up_quant) \
  F(moe_fp8_down_sum) F(moe_silu_mul) F(moe_sum)

struct Library {
#define KSQ_FN(name) decltype(&::ksq_##name) name;
  KSQ_FOR_EACH_FN(KSQ_FN)
#undef KSQ_FN
} lib;
PyObject* check_fn = nullptr;  // ksanallm_amd.lib.check: raises KsqError with the library's message

// Lets other Python threads run from the first allocation of a call on, to its end (its arguments are read before):
// allocations and the library's calls may wait for the device (an allocator that has to ask the driver, or to give memory
// back first).  One hand-over per call: with one per allocation and launch, and the device set and reset beside it, the
// smallest call took 4.46 us, 4.28 before that and 4.0 to 4.1 now.  The state is this thread's; an entry point puts an outer
// call's aside (a Python allocator or dispatch mode may call back).
thread_local PyThreadState* without_gil = nullptr;
void release_gil() {
  if (!without_gil) without_gil = PyEval_SaveThread();
}
void hold_gil() {
  if (PyThreadState* state = without_gil) {
    without_gil = nullptr;
    PyEval_RestoreThread(state);
  }
}

// A Python exception is set; unwinds to the entry point.
struct PyRaised {};

[[noreturn]] void raise(PyObject* type, const char* fmt, ...) {
  hold_gil();
  va_list ap;
  va_start(ap, fmt);
  PyErr_FormatV(type, fmt, ap);
  va_end(ap);
  throw PyRaised{};
}

template <typename F>
void call(F&& f) {
  release_gil();
  const int rc = f();
  if (rc == 0) return;
  hold_gil();
  PyObject* r = PyObject_CallFunction(check_fn, "i", rc);
  Py_XDECREF(r);
  if (!PyErr_Occurred()) PyErr_Format(PyExc_RuntimeError, "ksq status %d", rc);
  throw PyRaised{};
}

// ------------------------------------------------------------------------------------------------ arguments
struct Args {
  PyObject* const* v;
  Py_ssize_t n;
};

const at::Tensor& tensor(PyObject* o) {
  if (!THPVariable_Check(o)) raise(PyExc_TypeError, "a tensor is required, got %s", Py_TYPE(o)->tp_name);
  return THPVariable_Unpack(o);
}
const at::Tensor* tensor_or_null(PyObject* o) { return o == Py_None ? nullptr : &tensor(o); }
size_t size_arg(PyObject* o) {
  const Py_ssize_t v = PyNumber_AsSsize_t(o, PyExc_OverflowError);
  if (v == -1 && PyErr_Occurred()) throw PyRaised{};
  if (v < 0) raise(PyExc_ValueError, "a size must not be negative");
  return static_cast<size_t>(v);
}
bool bool_arg(PyObject* o) {
  const int v = PyObject_IsTrue(o);
  if (v < 0) throw PyRaised{};
  return v != 0;
}
double float_arg(PyObject* o) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) throw PyRaised{};
  return v;
}
at::ScalarType dtype_arg(PyObject* o) {
  if (!THPDtype_Check(o)) raise(PyExc_TypeError, "a torch.dtype is required, got %s", Py_TYPE(o)->tp_name);
  return reinterpret_cast<THPDtype*>(o)->scalar_type;
}

int dt(const at::Tensor& t, bool allow_f32 = false) {
  const at::ScalarType s = t.scalar_type();
  if (s == at::kHalf) return KSQ_F16;
  if (s == at::kBFloat16) return KSQ_BF16;
  if (allow_f32 && s == at::kFloat) return KSQ_F32;
  raise(PyExc_TypeError, "activation dtype must be float16 or bfloat16, got %s", at::toString(s));
}

void* ptr(const at::Tensor& t) {
  if (!t.is_cuda() || !t.is_contiguous()) raise(PyExc_AssertionError, "device-resident contiguous tensor required");
  return t.data_ptr();
}
void* ptr(const at::Tensor* t) { return t ? ptr(*t) : nullptr; }

// The C-ABI takes bare pointers: a tensor that is smaller than the layout it is declared to hold would be read past
// its end on the device, so the size is checked here.  (`nbytes` of sizes that the caller states: by product() below.)
void need_bytes(const at::Tensor& t, size_t nbytes, const char* what) {
  const size_t have = t.numel() * t.element_size();
  if (have < nbytes) raise(PyExc_ValueError, "%s: tensor holds %zu bytes, the declared layout needs %zu", what, have, nbytes);
}

// the product of sizes, or the largest size where it does not fit: a declared layout that no tensor can hold
size_t product(std::initializer_list<size_t> factors) {
  size_t p = 1;
  bool over = false, zero = false;
  for (size_t f : factors) {
    zero |= f == 0;
    over |= __builtin_mul_overflow(p, f, &p);
  }
  return zero ? 0 : over ? SIZE_MAX : p;
}

size_t rows(const at::Tensor& t) {
  if (t.dim() == 0) raise(PyExc_IndexError, "a tensor without dimensions has no rows");
  return static_cast<size_t>(t.size(0));
}
size_t dim(const at::Tensor& t, int64_t d, int64_t dims, const char* what) {
  if (t.dim() != dims) raise(PyExc_ValueError, "%s: a tensor of %d dimensions is required", what, static_cast<int>(dims));
  return static_cast<size_t>(t.size(d));
}

// ------------------------------------------------------------------------------------------------ device, allocation, stream
// Makes the tensor's device the current one for the rest of the call, where it is not that already.
struct OnDevice {
  c10::OptionalDeviceGuard guard;
  explicit OnDevice(const at::Tensor& t) {
    if (t.is_cuda() && t.device().index() != c10::hip::current_device()) guard.reset_device(t.device());
  }
};

at::Tensor empty(std::initializer_list<size_t> shape, at::ScalarType dtype, const at::Tensor& like) {
  int64_t s[4];
  int n = 0;
  for (size_t v : shape) s[n++] = static_cast<int64_t>(v);
  const at::IntArrayRef sizes(s, n);
  release_gil();
  if (!like.is_cuda()) return at::empty(sizes, like.options().dtype(dtype));
  return at::Tensor(at::detail::empty_cuda(sizes, dtype, like.device(), std::nullopt));
}

struct Scratch {  // nullptr and 0 where nothing is needed
  at::Tensor t;
  void* p = nullptr;
  size_t bytes = 0;
  Scratch(const at::Tensor* given, const at::Tensor& like, size_t need) {
    if (given) {
      p = ptr(*given);
      bytes = given->numel() * given->element_size();
    } else if (need) {
      t = empty({need}, at::kByte, like);
      p = ptr(t);
      bytes = need;
    }
  }
};

// the stream that is current on the tensor's device (without one: on the current device)
void* stream(const at::Tensor* t = nullptr) {
  return c10::hip::getCurrentHIPStream(t && t->is_cuda() ? t->device().index() : -1).stream();
}

// fp32, flat, contiguous: the tensor itself when it is that already
at::Tensor flat(const at::Tensor& t, at::ScalarType dtype) {
  if (t.scalar_type() == dtype && t.is_contiguous()) return t;
  release_gil();
  at::Tensor r = t.reshape({-1}).to(dtype).contiguous();
  hold_gil();  // further arguments are read after it
  return r;
}

// ------------------------------------------------------------------------------------------------ the calls
at::Tensor w4a16_gemm(const Args& a) {
  const at::Tensor &x = tensor(a.v[0]), &w = tensor(a.v[1]), &s = tensor(a.v[2]);
  const OnDevice on(x);
  const at::Tensor* z = tensor_or_null(a.v[3]);
  const size_t n = size_arg(a.v[4]), k = size_arg(a.v[5]), group = size_arg(a.v[6]);
  const at::Tensor *given = tensor_or_null(a.v[7]), *ws = tensor_or_null(a.v[8]);
  const size_t m = rows(x);
  if (group == 0) raise(PyExc_ZeroDivisionError, "group size 0");
  need_bytes(x, product({m, k, 2}), "w4a16_gemm: x");
  need_bytes(w, product({k, n}) / 2, "w4a16_gemm: packed weight");
  need_bytes(s, product({k / group, n, 2}), "w4a16_gemm: scales");
  if (z) need_bytes(*z, product({k / group, n}), "w4a16_gemm: zero points");
  const int d = dt(x);
  if (given) {
    if (given->scalar_type() != x.scalar_type())
      raise(PyExc_TypeError, "w4a16_gemm: out must be of x's type, got %s", at::toString(given->scalar_type()));
    need_bytes(*given, product({m, n, 2}), "w4a16_gemm: out");
  }
  at::Tensor out = given ? *given : empty({m, n}, x.scalar_type(), x);
  const Scratch scratch(ws, x, ws ? 0 : lib.w4a16_workspace_size(m, n, k, group, d));
  void *po = ptr(out), *px = ptr(x), *pw = ptr(w), *ps = ptr(s), *pz = ptr(z), *st = stream(&x);
  call([&] { return lib.w4a16_gemm(po, px, pw, ps, pz, scratch.p, scratch.bytes, m, n, k, group, d, st); });
  return out;
}

// codes and scales of per_token_group_quant_fp8
std::pair<at::Tensor, at::Tensor> group_quant(const at::Tensor& x, size_t k, size_t group, bool column_major, bool fuse,
                                              const at::Tensor* q_given, const at::Tensor* s_given) {
  const OnDevice on(x);
  const size_t m = rows(x);
  if (group == 0) raise(PyExc_ZeroDivisionError, "group size 0");
  need_bytes(x, product({m, k, static_cast<size_t>(x.element_size()), fuse ? size_t(2) : size_t(1)}), "fp8_group_quant: x");
  if (q_given) need_bytes(*q_given, product({m, k}), "fp8_group_quant: q");
  if (s_given) need_bytes(*s_given, product({m, k / group, 4}), "fp8_group_quant: s");
  at::Tensor q = q_given ? *q_given : empty({m, k}, at::kByte, x);
  at::Tensor s = s_given ? *s_given
                         : (column_major ? empty({k / group, m}, at::kFloat, x) : empty({m, k / group}, at::kFloat, x));
  const int d = dt(x, true);
  void *px = ptr(x), *pq = ptr(q), *ps = ptr(s), *st = stream(&x);
  call([&] { return lib.fp8_group_quant(px, pq, ps, m, k, group, column_major, fuse, d, st); });
  return {std::move(q), std::move(s)};
}

at::Tensor fp8_blockwise_gemm(const Args& a) {
  const at::Tensor &aq = tensor(a.v[0]), &as = tensor(a.v[1]), &b = tensor(a.v[2]), &bs = tensor(a.v[3]);
  const OnDevice on(aq);
  const at::Tensor *given = tensor_or_null(a.v[5]), *ws = tensor_or_null(a.v[6]);
  const size_t m = dim(aq, 0, 2, "fp8_blockwise_gemm: a_q"), k = aq.size(1), n = rows(b);
  need_bytes(as, product({k / 128, m, 4}), "fp8_blockwise_gemm: activation scales");
  need_bytes(b, product({n, k}), "fp8_blockwise_gemm: weight");
  need_bytes(bs, product({(n + 127) / 128, k / 128, 4}), "fp8_blockwise_gemm: weight scales");
  at::Tensor out = given ? *given : empty({m, n}, dtype_arg(a.v[4]), aq);
  const int d = dt(out, true);
  need_bytes(out, product({m, n, static_cast<size_t>(out.element_size())}), "fp8_blockwise_gemm: out");
  const Scratch scratch(ws, aq, ws ? 0 : lib.fp8_blockwise_workspace_size(m, n, k));
  void *po = ptr(out), *pa = ptr(aq), *pas = ptr(as), *pb = ptr(b), *pbs = ptr(bs), *st = stream(&aq);
  call([&] { return lib.fp8_blockwise_gemm(pa, pas, pb, pbs, po, m, n, k, d, scratch.p, scratch.bytes, st); });
  return out;
}

std::pair<at::Tensor, at::Tensor> w4a8_static_quant(const Args& a) {
  const at::Tensor &x = tensor(a.v[0]), &scale = tensor(a.v[1]);
  const OnDevice on(x);
  const bool per_channel = bool_arg(a.v[2]), per_token = bool_arg(a.v[3]);
  const size_t group = size_arg(a.v[4]);
  const size_t m = dim(x, 0, 2, "w4a8_static_quant: x"), k = x.size(1);
  if (group == 0) raise(PyExc_ZeroDivisionError, "group size 0");
  if (scale.scalar_type() != at::kFloat) raise(PyExc_ValueError, "w4a8_static_quant: scale must be fp32");
  need_bytes(scale, product({per_channel ? k : (per_token ? m : 1), 4}), "w4a8_static_quant: scale");
  at::Tensor q = empty({m, k}, at::kByte, x), xsum = empty({k / group, m}, at::kFloat, x);
  int mode = per_channel ? KSQ_W4A8_PER_CHANNEL : (per_token ? KSQ_W4A8_PER_TOKEN : KSQ_W4A8_PER_TENSOR);
  if (group == 64) mode |= KSQ_W4A8_SUMS_PER_64;
  const int d = dt(x);
  void *px = ptr(x), *psc = ptr(scale), *pq = ptr(q), *pxs = ptr(xsum), *st = stream(&x);
  call([&] { return lib.w4a8_static_quant(px, psc, pq, pxs, m, k, mode, d, st); });
  return {std::move(q), std::move(xsum)};
}

at::Tensor w4a8_gemm(const Args& a) {
  const at::Tensor &aq = tensor(a.v[0]), &xsum = tensor(a.v[1]), &w = tensor(a.v[2]), &scales = tensor(a.v[3]);
  const OnDevice on(aq);
  const double alpha = float_arg(a.v[4]);
  const size_t n = size_arg(a.v[5]);
  const at::Tensor *given = tensor_or_null(a.v[7]), *ws = tensor_or_null(a.v[8]);
  const size_t group = size_arg(a.v[9]);
  const size_t m = dim(aq, 0, 2, "w4a8_gemm: a_q"), k = aq.size(1);
  if (group == 0) raise(PyExc_ZeroDivisionError, "group size 0");
  need_bytes(xsum, product({k / group, m, 4}), "w4a8_gemm: group sums");
  need_bytes(w, product({n, k}) / 2, "w4a8_gemm: packed weight");
  need_bytes(scales, product({k / group, n, 2}), "w4a8_gemm: scales");
  if (scales.scalar_type() != at::kHalf) raise(PyExc_AssertionError, "w4a8_gemm: scales must be float16");
  at::Tensor out = given ? *given : empty({m, n}, dtype_arg(a.v[6]), aq);
  const int d = dt(out);
  need_bytes(out, product({m, n, 2}), "w4a8_gemm: out");
  const Scratch scratch(ws, aq, ws ? 0 : lib.w4a8_workspace_size(m, n, k));
  void *po = ptr(out), *pa = ptr(aq), *pxs = ptr(xsum), *pw = ptr(w), *ps = ptr(scales), *st = stream(&aq);
  call([&] {
    return lib.w4a8_gemm(pa, pxs, pw, ps, static_cast<float>(alpha), po, m, n, k, group, d, scratch.p, scratch.bytes, st);
  });
  return out;
}

std::pair<at::Tensor, at::Tensor> moe_topk_softmax(const Args& a) {
  const at::Tensor& gating = tensor(a.v[0]);
  const OnDevice on(gating);
  const size_t top_k = size_arg(a.v[1]);
  const int norm = bool_arg(a.v[2]);
  const float scaling = static_cast<float>(float_arg(a.v[3]));
  const size_t tokens = dim(gating, 0, 2, "moe_topk_softmax: gating"), E = gating.size(1);
  const int d = dt(gating, true);
  at::Tensor w = empty({tokens, top_k}, at::kFloat, gating), ids = empty({tokens, top_k}, at::kInt, gating);
  void *pg = ptr(gating), *pw = ptr(w), *pi = ptr(ids), *st = stream(&gating);
  call([&] { return lib.moe_topk_softmax(pg, pw, pi, tokens, E, top_k, norm, scaling, d, st); });
  return {std::move(w), std::move(ids)};
}

std::pair<at::Tensor, at::Tensor> moe_grouped_topk(const Args& a) {
  const at::Tensor& gating = tensor(a.v[0]);
  const OnDevice on(gating);
  const size_t top_k = size_arg(a.v[1]), groups = size_arg(a.v[2]), topk_group = size_arg(a.v[3]);
  const int sigmoid = bool_arg(a.v[4]);
  const at::Tensor* bias = tensor_or_null(a.v[5]);
  const int renormalize = bool_arg(a.v[6]);
  const float scaling = static_cast<float>(float_arg(a.v[7]));
  const size_t tokens = dim(gating, 0, 2, "moe_grouped_topk: gating"), E = gating.size(1);
  const int d = dt(gating, true);
  at::Tensor w = empty({tokens, top_k}, at::kFloat, gating), ids = empty({tokens, top_k}, at::kInt, gating);
  if (bias) {
    if (bias->scalar_type() != at::kFloat) raise(PyExc_ValueError, "e_bias must be fp32");
    need_bytes(*bias, product({E, 4}), "moe_grouped_topk: e_bias");
  }
  void *pg = ptr(gating), *pb = ptr(bias), *pw = ptr(w), *pi = ptr(ids), *st = stream(&gating);
  call([&] {
    return lib.moe_grouped_topk(pg, pb, pw, pi, tokens, E, top_k, groups, topk_group, sigmoid, renormalize, scaling, d, st);
  });
  return {std::move(w), std::move(ids)};
}

// ---- MoE blocks
struct Aligned {
  at::Tensor sorted_ids, expert_ids, num_post_pad, scratch;
};
Aligned moe_align(const at::Tensor& ids, size_t E, size_t block_m, void* st) {
  const size_t numel = ids.numel(), cap = lib.moe_align_capacity(numel, E, block_m);
  Aligned r{empty({cap}, at::kInt, ids), empty({(cap + block_m - 1) / block_m}, at::kInt, ids), empty({1}, at::kInt, ids),
            empty({lib.moe_align_scratch_bytes(numel, E)}, at::kByte, ids)};
  void *pi = ptr(ids), *ps = ptr(r.sorted_ids), *pe = ptr(r.expert_ids), *pn = ptr(r.num_post_pad), *pt = ptr(r.scratch);
  call([&] { return lib.moe_align(pi, numel, E, block_m, ps, pe, pn, pt, st); });
  return r;
}

at::Tensor top_k_sum(const at::Tensor& slots, size_t tokens, size_t top_k, size_t hidden, int d, void* st) {
  at::Tensor out = empty({tokens, hidden}, slots.scalar_type(), slots);
  void *pi = ptr(slots), *po = ptr(out);
  call([&] { return lib.moe_sum(pi, po, tokens, top_k, hidden, d, st); });
  return out;
}

struct Routed {  // the router's outputs, flat
  size_t tokens, top_k, numel;
  at::Tensor ids, w;
  Routed(const at::Tensor& topk_ids, const at::Tensor& topk_w) {
    tokens = dim(topk_ids, 0, 2, "topk_ids");
    top_k = topk_ids.size(1);
    numel = tokens * top_k;
    w = flat(topk_w, at::kFloat);
    ids = flat(topk_ids, at::kInt);
    need_bytes(w, product({numel, 4}), "topk_w");
  }
};

at::Tensor fused_moe_w4a16(const Args& a) {
  const at::Tensor &x = tensor(a.v[0]), &w13 = tensor(a.v[1]), &s13 = tensor(a.v[2]), &w2 = tensor(a.v[3]), &s2 = tensor(a.v[4]);
  const OnDevice on(x);
  const Routed r(tensor(a.v[5]), tensor(a.v[6]));
  const size_t E = size_arg(a.v[7]), hidden = size_arg(a.v[8]), inter = size_arg(a.v[9]), group = size_arg(a.v[10]);
  const bool block_given = a.v[11] != Py_None;
  size_t block_m = block_given ? size_arg(a.v[11]) : 0;
  const size_t few_tokens = size_arg(a.v[12]);
  if (group == 0) raise(PyExc_ZeroDivisionError, "group size 0");
  need_bytes(x, product({r.tokens, hidden, 2}), "fused_moe_w4a16: x");
  need_bytes(w13, product({E, hidden, inter}), "fused_moe_w4a16: packed gate / up weight");
  need_bytes(s13, product({E, hidden / group, inter, 4}), "fused_moe_w4a16: gate / up scales");
  need_bytes(w2, product({E, hidden, inter}) / 2, "fused_moe_w4a16: packed down weight");
  need_bytes(s2, product({E, inter / group, hidden, 2}), "fused_moe_w4a16: down scales");
  const int d = dt(x);
  const at::ScalarType t = x.scalar_type();
  void *st = stream(&x), *px = ptr(x), *pw13 = ptr(w13), *ps13 = ptr(s13), *pw2 = ptr(w2), *ps2 = ptr(s2), *ptw = ptr(r.w),
       *pids = ptr(r.ids);
  if (!block_given && r.tokens <= few_tokens && r.numel <= 64 && r.top_k <= 32 && (2 * inter) % 32 == 0) {
    // a few decode tokens: two launches - the first GEMM with every slot a block of its own (no aligned permutation) and
    // the activation in its epilogue, the second with the sum over top-k in it
    at::Tensor c2 = empty({r.numel, inter}, t, x), out = empty({r.tokens, hidden}, t, x);
    void *p2 = ptr(c2), *po = ptr(out);
    call([&] {
      const int rc = lib.moe_w4a16_gate_up_silu(p2, px, pw13, ps13, nullptr, nullptr, pids, nullptr, r.numel, r.top_k, E,
                                                2 * inter, hidden, group, 16, d, st);
      return rc ? rc : lib.moe_w4a16_down_sum(po, p2, pw2, ps2, ptw, pids, r.tokens, r.top_k, E, hidden, inter, group, d, st);
    });
    return out;
  }
  if (!block_given) block_m = lib.moe_w4a16_row_block(r.numel, E, hidden, inter);
  if (block_m == 0) raise(PyExc_ZeroDivisionError, "block size 0");
  const Aligned al = moe_align(r.ids, E, block_m, st);
  void *ps = ptr(al.sorted_ids), *pe = ptr(al.expert_ids), *pn = ptr(al.num_post_pad);
  at::Tensor c2 = empty({r.numel, inter}, t, x);
  void* p2 = ptr(c2);
  // the activation runs in the first GEMM's epilogue, except with 128-row blocks (a size moe_w4a16_row_block does not pick but
  // a caller may ask for), where the two launches measured faster (64 rows per expert: 1.75 against 1.87 ms)
  if (block_m != 128 && (2 * inter) % 32 == 0) {
    call([&] {
      return lib.moe_w4a16_gate_up_silu(p2, px, pw13, ps13, nullptr, ps, pe, pn, r.numel, r.top_k, E, 2 * inter, hidden, group,
                                        block_m, d, st);
    });
  } else {
    at::Tensor c1 = empty({r.numel, 2 * inter}, t, x);
    void* p1 = ptr(c1);
    call([&] {
      const int rc = lib.moe_w4a16_gemm(p1, px, pw13, ps13, nullptr, nullptr, ps, pe, pn, r.numel, r.top_k, E, 2 * inter, hidden,
                                        group, block_m, d, st);
      return rc ? rc : lib.moe_silu_mul(p1, p2, r.numel, inter, d, st);
    });
  }
  at::Tensor c3 = empty({r.numel, hidden}, t, x);
  void* p3 = ptr(c3);
  call([&] {
    return lib.moe_w4a16_gemm(p3, p2, pw2, ps2, nullptr, ptw, ps, pe, pn, r.numel, 1, E, hidden, inter, group, block_m, d, st);
  });
  return top_k_sum(c3, r.tokens, r.top_k, hidden, d, st);
}

at::Tensor fused_moe_fp8_blockwise(const Args& a) {
  const at::Tensor &x = tensor(a.v[0]), &w13 = tensor(a.v[1]), &s13 = tensor(a.v[2]), &w2 = tensor(a.v[3]), &s2 = tensor(a.v[4]);
  const OnDevice on(x);
  const Routed r(tensor(a.v[5]), tensor(a.v[6]));
  const bool block_given = a.v[7] != Py_None;
  size_t block_m = block_given ? size_arg(a.v[7]) : 0;
  const size_t few_tokens = size_arg(a.v[8]);
  const size_t E = dim(w13, 0, 3, "fused_moe_fp8_blockwise: w13"), n1 = w13.size(1), hidden = w13.size(2), inter = n1 / 2;
  need_bytes(x, product({r.tokens, hidden, static_cast<size_t>(x.element_size())}), "fused_moe_fp8_blockwise: x");
  need_bytes(w2, product({E, hidden, inter}), "fused_moe_fp8_blockwise: down weight");
  need_bytes(s13, product({E, (n1 + 127) / 128, hidden / 128, 4}), "fused_moe_fp8_blockwise: gate / up scales");
  need_bytes(s2, product({E, (hidden + 127) / 128, inter / 128, 4}), "fused_moe_fp8_blockwise: down scales");
  const int d = dt(x);
  const at::ScalarType t = x.scalar_type();
  void *st = stream(&x), *pw13 = ptr(w13), *ps13 = ptr(s13), *pw2 = ptr(w2), *ps2 = ptr(s2), *ptw = ptr(r.w), *pids = ptr(r.ids);
  const bool few = !block_given && r.tokens <= few_tokens && r.numel <= 64 && r.top_k <= 32;
  if (!block_given && !few) block_m = lib.moe_fp8_row_block(r.numel, E, hidden, inter);
  if (!few && block_m == 0) raise(PyExc_ZeroDivisionError, "block size 0");
  Aligned al;
  if (!few) al = moe_align(r.ids, E, block_m, st);
  // a few decode tokens: no aligned permutation, the sum over top-k inside the second GEMM (as fused_moe_w4a16)
  void *ps = few ? nullptr : ptr(al.sorted_ids), *pe = few ? pids : ptr(al.expert_ids), *pn = few ? nullptr : ptr(al.num_post_pad);
  if (few) block_m = 16;
  auto [q1, q1s] = group_quant(x, hidden, 128, false, false, nullptr, nullptr);
  void *pq1 = ptr(q1), *pq1s = ptr(q1s);
  at::Tensor q2, q2s;
  if (!few && lib.moe_fp8_fused_quant(r.numel, E, n1, hidden, block_m)) {
    // the activation and the second quantization run in the first GEMM's epilogue
    q2 = empty({r.numel, inter}, at::kByte, x);
    q2s = empty({r.numel, inter / 128}, at::kFloat, x);
    void *pq = ptr(q2), *pqs = ptr(q2s);
    call([&] {
      return lib.moe_fp8_gate_up_quant(pq, pqs, pq1, pq1s, 0, r.tokens, pw13, ps13, ps, pe, pn, r.numel, r.top_k, E, n1, hidden, block_m,
                                       d, st);
    });
  } else {
    at::Tensor c1 = empty({r.numel, n1}, t, x);
    void* p1 = ptr(c1);
    call([&] {
      return lib.moe_fp8_blockwise_gemm(p1, pq1, pq1s, 0, r.tokens, pw13, ps13, nullptr, ps, pe, pn, r.numel, r.top_k, E, n1, hidden,
                                        block_m, d, st);
    });
    std::tie(q2, q2s) = group_quant(c1, inter, 128, false, true, nullptr, nullptr);
  }
  void *pq2 = ptr(q2), *pq2s = ptr(q2s);
  if (few) {
    at::Tensor out = empty({r.tokens, hidden}, t, x);
    void* po = ptr(out);
    call([&] {
      return lib.moe_fp8_down_sum(po, pq2, pq2s, pw2, ps2, ptw, pids, r.tokens, r.top_k, E, hidden, inter, d, st);
    });
    return out;
  }
  at::Tensor c3 = empty({r.numel, hidden}, t, x);
  void* p3 = ptr(c3);
  call([&] {
    return lib.moe_fp8_blockwise_gemm(p3, pq2, pq2s, 0, r.numel, pw2, ps2, ptw, ps, pe, pn, r.numel, 1, E, hidden, inter, block_m,
                                      d, st);
  });
  return top_k_sum(c3, r.tokens, r.top_k, hidden, d, st);
}

std::pair<at::Tensor, at::Tensor> per_token_group_quant_fp8(const Args& a) {
  return group_quant(tensor(a.v[0]), size_arg(a.v[1]), size_arg(a.v[2]), bool_arg(a.v[3]), bool_arg(a.v[4]),
                     tensor_or_null(a.v[5]), tensor_or_null(a.v[6]));
}

// ------------------------------------------------------------------------------------------------ the Python module
PyObject* wrap(at::Tensor&& t) { return THPVariable_Wrap(std::move(t)); }
PyObject* wrap(std::pair<at::Tensor, at::Tensor>&& p) {
  PyObject* a = THPVariable_Wrap(std::move(p.first));
  PyObject* b = a ? THPVariable_Wrap(std::move(p.second)) : nullptr;
  PyObject* r = b ? PyTuple_Pack(2, a, b) : nullptr;
  Py_XDECREF(a);
  Py_XDECREF(b);
  return r;
}

template <auto F, int N>
PyObject* entry(PyObject*, PyObject* const* v, Py_ssize_t n) {
  if (n != N) {
    PyErr_Format(PyExc_TypeError, "%d arguments are required, got %zd", N, n);
    return nullptr;
  }
  if (!check_fn) {
    PyErr_SetString(PyExc_RuntimeError, "bind() has not been called");
    return nullptr;
  }
  PyThreadState* const outer = std::exchange(without_gil, nullptr);
  PyObject* r = nullptr;
  try {
    auto result = F(Args{v, n});
    hold_gil();
    r = wrap(std::move(result));
  } catch (const PyRaised&) {  // (raise() holds the lock)
  } catch (const std::bad_alloc&) {
    hold_gil();
    PyErr_NoMemory();
  } catch (const std::exception& e) {  // out of device memory, among others: torch's own exception types
    hold_gil();
    torch::translate_exception_to_python(std::current_exception());
  }
  without_gil = outer;
  return r;
}

PyObject* current_stream(PyObject*, PyObject*) {
  try {
    return PyLong_FromVoidPtr(stream());
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

// bind({"ksq_...": address, ...}, check)
PyObject* bind(PyObject*, PyObject* args) {
  PyObject *table, *check;
  if (!PyArg_ParseTuple(args, "O!O", &PyDict_Type, &table, &check)) return nullptr;
  Library l{};
  bool ok = true;
  auto get = [&](const char* name, auto* slot) {
    PyObject* v = ok ? PyDict_GetItemString(table, name) : nullptr;
    void* p = v ? PyLong_AsVoidPtr(v) : nullptr;
    if (!p) {
      if (ok && !PyErr_Occurred()) PyErr_Format(PyExc_KeyError, "%s", name);
      ok = false;
    }
    *slot = reinterpret_cast<std::remove_pointer_t<decltype(slot)>>(p);
  };
#define KSQ_FN(name) get("ksq_" #name, &l.name);
  KSQ_FOR_EACH_FN(KSQ_FN)
#undef KSQ_FN
  if (!ok) return nullptr;
  lib = l;
  Py_INCREF(check);
  Py_XSETREF(check_fn, check);
  Py_RETURN_NONE;
}

#define KSQ_ENTRY(name, n) \
  { #name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&entry<name, n>)), METH_FASTCALL, nullptr }
PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, nullptr},
    {"current_stream", current_stream, METH_NOARGS, nullptr},
    KSQ_ENTRY(w4a16_gemm, 9),
    KSQ_ENTRY(per_token_group_quant_fp8, 7),
    KSQ_ENTRY(fp8_blockwise_gemm, 7),
    KSQ_ENTRY(w4a8_static_quant, 5),
    KSQ_ENTRY(w4a8_gemm, 10),
    KSQ_ENTRY(moe_topk_softmax, 4),
    KSQ_ENTRY(moe_grouped_topk, 8),
    KSQ_ENTRY(fused_moe_w4a16, 13),
    KSQ_ENTRY(fused_moe_fp8_blockwise, 9),
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_ops_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__ops_host() { return PyModule_Create(&module_def); }

// Native host path of the operator layer (Python extension
// tcfp_amd._tcfp_host): argument checks, output allocation and the C-ABI
// call of the ops that every layer pass makes, in one call from Python.
//
// What bounds a small layer is the host: in Python an op is 5-15 torch.empty
// calls (2-3 us each), a ctypes call of some 20 converted arguments (5-8 us)
// and its checks, so a layer's forward and backward enqueued ~150 us of
// launches that take the GPU ~100 us (4096 tokens, 256 -> 1024).  Here an
// allocation is ~0.7 us and the C ABI is called directly.
//
// The functions keep their Python predecessors' semantics: the same checks in
// the same order with the same exception types, the same outputs, the
// current stream of the tensors' device.  They run without the GIL, which
// torch.empty and a ctypes call release too: an allocation may wait for the
// GPU, a launch for room in its queue, and Python's other threads go on.  So
// nothing in them touches a Python object; results and errors become Python's
// at the boundary (Outs, Raise).  Scratch for the reductions is one buffer per
// (device, stream), as stream order makes its reuse safe; it is allocated
// once and lives as long as the process.
#include <Python.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/extension.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <optional>
#include <string>
#include <utility>
#include <vector>

#include "../../include/tcfp_hip.h"

namespace {

namespace py = pybind11;
using at::Tensor;
using OptT = std::optional<Tensor>;

// A Python exception to be raised at the boundary.
struct Raise {
  PyObject* type;
  std::string msg;
};
[[noreturn]] void raise(PyObject* type, const std::string& msg) { throw Raise{type, msg}; }
[[noreturn]] void assertion(const std::string& m) { raise(PyExc_AssertionError, m); }
[[noreturn]] void value_error(const std::string& m) { raise(PyExc_ValueError, m); }
[[noreturn]] void type_error(const std::string& m) { raise(PyExc_TypeError, m); }
[[noreturn]] void runtime_error(const std::string& m) { raise(PyExc_RuntimeError, m); }

// A tuple of tensors, None where undefined.
struct Outs {
  std::vector<Tensor> t;
};
// (takes the caller's locals: a copy is two atomic counts, and a second owner
// where Python's object is made)
template <typename... T>
Outs outs(T&... t) {
  Outs o;
  o.t.reserve(sizeof...(t));
  (o.t.push_back(std::move(t)), ...);
  return o;
}

std::string shape_str(at::IntArrayRef s) {
  std::string r = "(";
  for (size_t i = 0; i < s.size(); ++i) r += (i ? ", " : "") + std::to_string(s[i]);
  return r + (s.size() == 1 ? ",)" : ")");
}

const char* dtype_str(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return "torch.float32";
    case at::kBFloat16: return "torch.bfloat16";
    case at::kHalf: return "torch.float16";
    case at::kDouble: return "torch.float64";
    case at::kFloat8_e4m3fn: return "torch.float8_e4m3fn";
    case at::kFloat8_e5m2: return "torch.float8_e5m2";
    default: return c10::toString(t);
  }
}

// A status from the C ABI as the Python binding reports it.
void check(int status, const char* what) {
  if (status != TCFP_OK)
    runtime_error(std::string(what) + " failed: " + tcfp_status_string(status) + " (status " +
                  std::to_string(status) + ")");
}

// All tensors on one GPU.
class OnGpu {
 public:
  explicit OnGpu(std::initializer_list<const Tensor*> ts) {
    for (const Tensor* t : ts) add(*t);
    done();
  }
  OnGpu() = default;
  void add(const Tensor& t) {
    if (!t.defined()) return;
    if (!t.is_cuda())
      runtime_error("tcfp_amd ops run only on the GPU (hand-written HIP kernels); got a " +
                    t.device().str() + " tensor");
    if (!dev_) dev_ = t.device();
    else if (*dev_ != t.device())
      runtime_error("tensors on different devices: " + dev_->str() + " vs " + t.device().str());
  }
  void add(const OptT& t) {
    if (t) add(*t);
  }
  void done() const {
    if (!dev_) runtime_error("no tensor given");
  }
  at::Device device() const { return *dev_; }
  void* stream() const { return c10::hip::getCurrentHIPStream(dev_->index()).stream(); }
  Tensor empty(at::IntArrayRef shape, at::ScalarType t) const {
    return at::empty(shape, at::TensorOptions().dtype(t).device(*dev_));
  }

 private:
  std::optional<at::Device> dev_;
};

const Tensor& opt(const OptT& t) {
  static const Tensor* const none = new Tensor();
  return t ? *t : *none;
}

template <typename T = void>
T* ptr(const Tensor& t) {
  return t.defined() ? static_cast<T*>(t.data_ptr()) : nullptr;
}
uint8_t* bytes(const Tensor& t) { return ptr<uint8_t>(t); }
int8_t* exps(const Tensor& t) { return ptr<int8_t>(t); }
float* f32(const Tensor& t) { return ptr<float>(t); }

int fmt_of(at::ScalarType t) {
  if (t == at::kFloat8_e4m3fn) return TCFP_FP8_E4M3;
  if (t == at::kFloat8_e5m2) return TCFP_FP8_E5M2;
  type_error(std::string("unsupported fp8 dtype ") + dtype_str(t));
}
bool is_fp8(const Tensor& t) {
  return t.scalar_type() == at::kFloat8_e4m3fn || t.scalar_type() == at::kFloat8_e5m2;
}
int in_dtype(const Tensor& t) {
  if (t.scalar_type() == at::kFloat) return TCFP_DTYPE_F32;
  if (t.scalar_type() == at::kBFloat16) return TCFP_DTYPE_BF16;
  type_error(std::string("unsupported input dtype ") + dtype_str(t.scalar_type()) +
             ": expected float32 or bfloat16");
}
int out_dtype_of(at::ScalarType t) {
  if (t == at::kFloat) return TCFP_DTYPE_F32;
  if (t == at::kBFloat16) return TCFP_DTYPE_BF16;
  type_error(std::string("unsupported output dtype ") + dtype_str(t));
}

bool al16(const Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15u) == 0; }

// fp32, contiguous, 16-byte aligned bias of n elements.
Tensor bias_f32(const Tensor& bias, int64_t n) {
  Tensor b = bias.to(at::kFloat).contiguous();
  if (b.dim() != 1 || b.size(0) != n)
    assertion("bias shape " + shape_str(b.sizes()) + " != (" + std::to_string(n) + ",)");
  if (!al16(b)) b = b.clone();
  return b;
}

Tensor scalar(const Tensor& t, const char* name) {
  if (t.numel() != 1 || t.scalar_type() != at::kFloat)
    value_error(std::string(name) + " must be a single-element float32 tensor");
  return t.is_contiguous() ? t : t.contiguous();
}

// ---- reduction scratch: one per (device, stream) --------------------------
struct Scratch {
  std::mutex mu;
  Tensor t;
};
std::mutex g_ws_mu;  // of the maps
using WsMap = std::map<std::pair<int, void*>, Scratch>;
// (never destroyed: tensors must not outlive the allocator at exit)
WsMap& ws_map(int kind) {
  static WsMap* const m = new WsMap[2];
  return m[kind];
}

// A call's hold on its stream's scratch, to be taken after its allocations and
// kept over its launches: another thread's call on the same stream enqueues
// its own before or after all of them.  The scratch is allocated
// outside the locks, as a dispatch mode's Python code may run there.
class Workspace {
 public:
  Workspace(const OnGpu& g, void* stream, bool batch) {
    Scratch* s;
    {
      std::lock_guard<std::mutex> lk(g_ws_mu);
      s = &ws_map(batch ? 1 : 0)[{int(g.device().index()), stream}];
    }
    lock_ = std::unique_lock<std::mutex>(s->mu);
    if (!s->t.defined()) {
      lock_.unlock();
      Tensor t = g.empty({int64_t(batch ? tcfp_quantize_batch_workspace_bytes(4)
                                        : tcfp_workspace_bytes())},
                         at::kByte);
      lock_.lock();
      if (!s->t.defined()) s->t = t;
    }
    p_ = s->t.data_ptr();
    n_ = size_t(s->t.numel());
  }
  void* ptr() const { return p_; }
  size_t bytes() const { return n_; }

 private:
  std::unique_lock<std::mutex> lock_;
  void* p_;
  size_t n_;
};

struct View2d {
  Tensor t;
  int64_t rows, cols;
};
// contiguous x as [numel / last, last]
View2d as_2d(const Tensor& x) {
  View2d v{x.is_contiguous() ? x : x.contiguous(), 0, 0};
  v.cols = v.t.dim() > 0 ? v.t.size(-1) : 1;
  v.rows = v.cols ? v.t.numel() / v.cols : 0;
  return v;
}

// ---- per-tensor quantisation -------------------------------------------------

Outs quantize_per_tensor(const Tensor& x, at::ScalarType fp8, const OptT& scale,
                              bool transpose, bool return_scale) {
  OnGpu g;
  g.add(x);
  g.add(scale);
  const View2d v = as_2d(x);
  const int dt = in_dtype(v.t), fmt = fmt_of(fp8);
  Tensor q = g.empty(x.sizes(), fp8), q_t, s_out, s_in;
  if (transpose) q_t = g.empty({v.cols, v.rows}, fp8);
  Tensor inv = g.empty({1}, at::kFloat);
  if (return_scale) s_out = g.empty({1}, at::kFloat);
  void* st = g.stream();
  std::optional<Workspace> ws;
  if (scale) s_in = scalar(scale->to(at::kFloat), "scale");
  else ws.emplace(g, st, false);
  check(tcfp_quantize_per_tensor(ptr(v.t), dt, v.rows, v.cols, fmt, f32(s_in), bytes(q),
                                 bytes(q_t), f32(s_out), f32(inv), ws ? ws->ptr() : nullptr, st),
        "quantize_per_tensor");
  if (transpose && return_scale) return outs(q, inv, q_t, s_out);
  if (transpose) return outs(q, inv, q_t);
  if (return_scale) return outs(q, inv, s_out);
  return outs(q, inv);
}

Outs quantize_per_tensor_colsum(const Tensor& x, at::ScalarType fp8, bool transpose) {
  OnGpu g({&x});
  const View2d v = as_2d(x);
  if (v.cols % 8 != 0)
    value_error("column count (" + std::to_string(v.cols) + ") must be divisible by 8");
  const int dt = in_dtype(v.t), fmt = fmt_of(fp8);
  Tensor q = g.empty(x.sizes(), fp8), q_t;
  if (transpose) q_t = g.empty({v.cols, v.rows}, fp8);
  Tensor inv = g.empty({1}, at::kFloat), cs = g.empty({v.cols}, at::kFloat);
  const size_t n = tcfp_colsum_workspace_bytes(v.rows, v.cols);
  Tensor cws = g.empty({int64_t(std::max<size_t>(n, 16))}, at::kByte);
  void* st = g.stream();
  const Workspace ws(g, st, false);
  check(tcfp_quantize_per_tensor_colsum(ptr(v.t), dt, v.rows, v.cols, fmt, bytes(q), bytes(q_t),
                                        f32(inv), f32(cs), ws.ptr(), ptr(cws), n, st),
        "quantize_per_tensor_colsum");
  if (transpose) return outs(q, inv, q_t, cs);
  return outs(q, inv, cs);
}

void check_ef(const Tensor& ef, int64_t n, int64_t k) {
  if (ef.scalar_type() != at::kFloat) assertion("error_buf must be float32");
  if (ef.dim() != 2 || ef.size(0) != n || ef.size(1) != k)
    assertion("error_buf shape " + shape_str(ef.sizes()) + " != weight shape (" +
              std::to_string(n) + ", " + std::to_string(k) + ")");
  if (!ef.is_contiguous()) assertion("error_buf must be contiguous");
}

// The amax-rule dual quantisation (no NF-aware scaling).
Outs dual_quantize_per_tensor(const Tensor& weight, const OptT& error_buf, bool update_ef,
                                   bool stochastic_lo, bool transposed, uint64_t seed) {
  OnGpu g;
  g.add(weight);
  g.add(error_buf);
  if (weight.dim() != 2) assertion("weight must be 2-D (N, K)");
  const Tensor w = weight.is_contiguous() ? weight : weight.contiguous();
  const int64_t n = w.size(0), k = w.size(1);
  if (error_buf) check_ef(*error_buf, n, k);
  const int dt = in_dtype(w);
  const at::ScalarType e4 = at::kFloat8_e4m3fn;
  Tensor hi = g.empty({n, k}, e4), lo = g.empty({n, k}, e4), hi_t, lo_t;
  Tensor ih = g.empty({1}, at::kFloat), il = g.empty({1}, at::kFloat);
  if (transposed) {
    hi_t = g.empty({k, n}, e4);
    lo_t = g.empty({k, n}, e4);
  }
  void* st = g.stream();
  const Workspace ws(g, st, false);
  check(tcfp_dual_quantize_per_tensor(ptr(w), dt, n, k, f32(opt(error_buf)), update_ef ? 1 : 0,
                                      stochastic_lo ? 1 : 0, seed, 0, bytes(hi), bytes(lo),
                                      f32(ih), f32(il), bytes(hi_t), bytes(lo_t), ws.ptr(), st),
        "dual_quantize_per_tensor");
  if (transposed) return outs(hi, lo, ih, il, hi_t, lo_t);
  return outs(hi, lo, ih, il);
}

// (weight, error_buf, update_ef, transposed) and (x, fp8_dtype, transpose)
using DualIn = std::tuple<Tensor, OptT, bool, bool>;
using ActIn = std::tuple<Tensor, at::ScalarType, bool>;

// The batch itself (its caller has checked that every tensor fits).
std::pair<std::vector<Outs>, std::vector<Outs>> quantize_batch(const std::vector<DualIn>& dual,
                                             const std::vector<ActIn>& act) {
  if (dual.size() + act.size() > 4) value_error("at most four tensors in a batch");
  OnGpu g;
  for (const auto& d : dual) {
    g.add(std::get<0>(d));
    g.add(std::get<1>(d));
  }
  for (const auto& a : act) g.add(std::get<0>(a));
  g.done();
  tcfp_quant_job jobs[4] = {};
  std::vector<Tensor> held;  // contiguous copies, alive until the launch
  int nj = 0;
  std::vector<Outs> rd, ra;
  const at::ScalarType e4 = at::kFloat8_e4m3fn;
  for (const auto& d : dual) {
    Tensor w = std::get<0>(d);
    if (!w.is_contiguous()) w = w.contiguous();
    held.push_back(w);
    const int64_t n = w.size(0), k = w.size(1);
    const OptT& ef = std::get<1>(d);
    if (ef) check_ef(*ef, n, k);
    const bool t = std::get<3>(d);
    Tensor hi = g.empty({n, k}, e4), lo = g.empty({n, k}, e4), ht, lt;
    Tensor ih = g.empty({1}, at::kFloat), il = g.empty({1}, at::kFloat);
    if (t) {
      ht = g.empty({k, n}, e4);
      lt = g.empty({k, n}, e4);
    }
    tcfp_quant_job& j = jobs[nj++];
    j.kind = TCFP_JOB_DUAL;
    j.x = ptr(w);
    j.x_dtype = in_dtype(w);
    j.rows = n;
    j.cols = k;
    j.ef = f32(opt(ef));
    j.update_ef = std::get<2>(d) ? 1 : 0;
    j.q = bytes(hi);
    j.q_t = bytes(ht);
    j.inv = f32(ih);
    j.q_lo = bytes(lo);
    j.q_lo_t = bytes(lt);
    j.inv_lo = f32(il);
    if (t) rd.push_back(outs(hi, lo, ih, il, ht, lt));
    else rd.push_back(outs(hi, lo, ih, il));
  }
  for (const auto& a : act) {
    Tensor x = std::get<0>(a);
    if (!x.is_contiguous()) x = x.contiguous();
    held.push_back(x);
    const int64_t rows = x.size(0), cols = x.size(1);
    const at::ScalarType fp8 = std::get<1>(a);
    const int fmt = fmt_of(fp8);
    Tensor q = g.empty({rows, cols}, fp8), qt, inv;
    if (std::get<2>(a)) qt = g.empty({cols, rows}, fp8);
    inv = g.empty({1}, at::kFloat);
    tcfp_quant_job& j = jobs[nj++];
    j.kind = TCFP_JOB_ACT;
    j.x = ptr(x);
    j.x_dtype = in_dtype(x);
    j.rows = rows;
    j.cols = cols;
    j.fp8_fmt = fmt;
    j.q = bytes(q);
    j.q_t = bytes(qt);
    j.inv = f32(inv);
    if (std::get<2>(a)) ra.push_back(outs(q, inv, qt));
    else ra.push_back(outs(q, inv));
  }
  void* st = g.stream();
  const Workspace ws(g, st, true);
  check(tcfp_quantize_batch(nj, jobs, ws.ptr(), ws.bytes(), st), "quantize_batch");
  return {std::move(rd), std::move(ra)};
}

// ---- GEMMs ----------------------------------------------------------------------

// FP8, 2-D, rows K-contiguous on 16-byte boundaries.
Tensor gemm_operand(const Tensor& t, const char* name) {
  if (!is_fp8(t))
    type_error(std::string(name) + " must be float8_e4m3fn or float8_e5m2, got " +
               dtype_str(t.scalar_type()));
  if (t.dim() != 2) value_error(std::string(name) + " must be 2-D");
  if (t.stride(1) != 1 || t.stride(0) % 16 != 0 || !al16(t)) return t.contiguous();
  return t;
}

Tensor dual_gemm(const Tensor& a_, const Tensor& b_hi_, const OptT& b_lo_, const Tensor& s_a,
                 const Tensor& s_hi, const OptT& s_lo, const OptT& bias, at::ScalarType out_dtype) {
  OnGpu g;
  g.add(a_);
  g.add(b_hi_);
  g.add(b_lo_);
  g.add(s_a);
  g.add(s_hi);
  g.add(s_lo);
  g.add(bias);
  const Tensor a = gemm_operand(a_, "A");
  Tensor b_hi = gemm_operand(b_hi_, "B_hi"), b_lo;
  if (b_lo_) b_lo = gemm_operand(*b_lo_, "B_lo");
  const int64_t m = a.size(0), k = a.size(1), n = b_hi.size(0);
  if (k % 16 != 0) value_error("K (" + std::to_string(k) + ") must be divisible by 16");
  if (b_lo.defined() && b_hi.stride(0) != b_lo.stride(0)) {
    b_lo = b_lo.contiguous();
    b_hi = b_hi.contiguous();
  }
  Tensor out = g.empty({m, n}, out_dtype), b;
  if (bias) b = bias_f32(*bias, n);
  const Tensor sa = scalar(s_a, "scale_a"), sh = scalar(s_hi, "scale_hi");
  Tensor sl;
  if (s_lo) sl = scalar(*s_lo, "scale_lo");
  check(tcfp_dual_gemm(bytes(a), fmt_of(a.scalar_type()), a.stride(0), bytes(b_hi), bytes(b_lo),
                       fmt_of(b_hi.scalar_type()), b_hi.stride(0), m, n, k, f32(sa), f32(sh),
                       f32(sl), f32(b), ptr(out), out_dtype_of(out_dtype), n, g.stream()),
        "dual_gemm");
  return out;
}

Outs block_quantize(const Tensor& x_, int64_t bs, at::ScalarType fp8, bool f32s) {
  OnGpu g({&x_});
  if (x_.dim() != 2) value_error("expected a 2-D tensor");
  const int64_t m = x_.size(0), k = x_.size(1);
  if (bs == 0 || k % bs != 0)
    assertion("K (" + std::to_string(k) + ") must be divisible by block_size (" +
              std::to_string(bs) + ")");
  if (bs != 32 && bs != 64 && bs != 128)
    value_error("block_size must be 32, 64, or 128, got " + std::to_string(bs));
  const Tensor x = x_.is_contiguous() ? x_ : x_.contiguous();
  const int dt = in_dtype(x), fmt = fmt_of(fp8);
  Tensor q = g.empty({m, k}, fp8);
  Tensor s = g.empty({k / bs, m}, f32s ? at::kFloat : at::kChar);
  const int rc = f32s ? tcfp_block_quantize_f32s(ptr(x), dt, m, k, int(bs), fmt, bytes(q), f32(s),
                                                 g.stream())
                      : tcfp_block_quantize(ptr(x), dt, m, k, int(bs), fmt, bytes(q), exps(s),
                                            g.stream());
  check(rc, "block_quantize_fp8");
  return outs(q, s);
}

Tensor block_scales(const Tensor& e, int64_t rows, int64_t nkb, const char* name,
                    at::ScalarType t) {
  if (e.scalar_type() != t)
    type_error(std::string(name) + " must be " +
               (t == at::kChar ? "int8 power-of-two exponents" : "float32 multipliers") +
               " like the other scales, got " + dtype_str(e.scalar_type()));
  if (e.dim() != 2 || e.size(0) != nkb || e.size(1) != rows)
    value_error(std::string(name) + " must have shape (" + std::to_string(nkb) + ", " +
                std::to_string(rows) + "), got " + shape_str(e.sizes()));
  return e.is_contiguous() ? e : e.contiguous();
}

Tensor block_gemm(const Tensor& a_, const Tensor& e_a_, const Tensor& b_hi_, const OptT& b_lo_,
                  const Tensor& e_hi_, const OptT& e_lo_, int64_t bs, const OptT& bias,
                  at::ScalarType out_dtype) {
  OnGpu g;
  g.add(a_);
  g.add(e_a_);
  g.add(b_hi_);
  g.add(b_lo_);
  g.add(e_hi_);
  g.add(e_lo_);
  g.add(bias);
  const Tensor a = gemm_operand(a_, "A");
  Tensor b_hi = gemm_operand(b_hi_, "B_hi"), b_lo, e_lo;
  if (b_lo_) b_lo = gemm_operand(*b_lo_, "B_lo");
  const int64_t m = a.size(0), k = a.size(1), n = b_hi.size(0);
  if (bs == 0 || k % bs != 0)
    assertion("K (" + std::to_string(k) + ") not divisible by block_size (" + std::to_string(bs) +
              ")");
  if (bs != 32 && bs != 64 && bs != 128)
    value_error("block_size must be 32, 64, or 128, got " + std::to_string(bs));
  const int64_t nkb = k / bs;
  // int8 exponents or fp32 multipliers, not mixed
  const at::ScalarType sdt = e_a_.scalar_type() == at::kFloat ? at::kFloat : at::kChar;
  const Tensor e_a = block_scales(e_a_, m, nkb, "scales_a", sdt);
  const Tensor e_hi = block_scales(e_hi_, n, nkb, "scales_b", sdt);
  if (b_lo.defined()) {
    if (!e_lo_) type_error("scales_lo is missing");
    e_lo = block_scales(*e_lo_, n, nkb, "scales_lo", sdt);
    if (b_hi.stride(0) != b_lo.stride(0)) {
      b_hi = b_hi.contiguous();
      b_lo = b_lo.contiguous();
    }
  }
  Tensor out = g.empty({m, n}, out_dtype), b;
  if (bias) b = bias_f32(*bias, n);
  const int fa = fmt_of(a.scalar_type()), fb = fmt_of(b_hi.scalar_type());
  const int od = out_dtype_of(out_dtype);
  const int rc =
      sdt == at::kFloat
          ? tcfp_block_dual_gemm_f32s(bytes(a), fa, a.stride(0), f32(e_a), bytes(b_hi),
                                      bytes(b_lo), fb, b_hi.stride(0), f32(e_hi), f32(e_lo), m, n,
                                      k, int(bs), f32(b), ptr(out), od, n, g.stream())
          : tcfp_block_dual_gemm(bytes(a), fa, a.stride(0), exps(e_a), bytes(b_hi), bytes(b_lo),
                                 fb, b_hi.stride(0), exps(e_hi), exps(e_lo), m, n, k, int(bs),
                                 f32(b), ptr(out), od, n, g.stream());
  check(rc, "block_dual_gemm");
  return out;
}

// ---- the GELU between two per-tensor layers --------------------------------------

struct GemmOps {
  Tensor a, b_hi, b_lo;
};
GemmOps gemm_operands(const Tensor& a_, const Tensor& b_hi_, const Tensor& b_lo_) {
  GemmOps o{gemm_operand(a_, "A"), gemm_operand(b_hi_, "B_hi"), gemm_operand(b_lo_, "B_lo")};
  if (o.a.size(1) != o.b_hi.size(1) || o.b_hi.sizes() != o.b_lo.sizes())
    assertion("Shape mismatch: A" + shape_str(o.a.sizes()) + ", B_hi" + shape_str(o.b_hi.sizes()) +
              ", B_lo" + shape_str(o.b_lo.sizes()));
  if (o.a.size(1) % 16 != 0)
    value_error("K (" + std::to_string(o.a.size(1)) + ") must be divisible by 16");
  if (o.b_hi.stride(0) != o.b_lo.stride(0)) {
    o.b_hi = o.b_hi.contiguous();
    o.b_lo = o.b_lo.contiguous();
  }
  return o;
}

Outs dual_gemm_gelu_quantize(const Tensor& a_, const Tensor& b_hi_, const Tensor& b_lo_,
                                  const Tensor& s_a, const Tensor& s_hi, const Tensor& s_lo,
                                  const OptT& bias, at::ScalarType fp8, bool transpose,
                                  bool return_act, bool return_dgelu) {
  OnGpu g;
  for (const Tensor* t : {&a_, &b_hi_, &b_lo_, &s_a, &s_hi, &s_lo}) g.add(*t);
  g.add(bias);
  const GemmOps o = gemm_operands(a_, b_hi_, b_lo_);
  const int64_t m = o.a.size(0), k = o.a.size(1), n = o.b_hi.size(0);
  if (return_dgelu && n % 8 != 0)
    value_error("return_dgelu needs N divisible by 8, got " + std::to_string(n));
  Tensor h = g.empty({m, n}, at::kFloat), act, dg, q_t, b;
  // (a ragged last dim quantises gelu(h) from a stored copy)
  if (return_act || n % 8 != 0) act = g.empty({m, n}, at::kFloat);
  if (return_dgelu) dg = g.empty({m, n}, at::kFloat);
  const int fmt = fmt_of(fp8);
  Tensor q = g.empty({m, n}, fp8);
  if (transpose) q_t = g.empty({n, m}, fp8);
  Tensor inv = g.empty({1}, at::kFloat);
  if (bias) b = bias_f32(*bias, n);
  const Tensor sa = scalar(s_a, "scale_a"), sh = scalar(s_hi, "scale_hi"),
               sl = scalar(s_lo, "scale_lo");
  void* st = g.stream();
  const Workspace ws(g, st, false);
  check(tcfp_dual_gemm_gelu_quantize(
            bytes(o.a), fmt_of(o.a.scalar_type()), o.a.stride(0), bytes(o.b_hi), bytes(o.b_lo),
            fmt_of(o.b_hi.scalar_type()), o.b_hi.stride(0), m, n, k, f32(sa), f32(sh), f32(sl),
            f32(b), f32(h), f32(act), f32(dg), fmt, bytes(q), bytes(q_t), f32(inv), ws.ptr(), st),
        "dual_gemm_gelu_quantize");
  Outs r = outs(h, q, inv);
  if (transpose) r.t.push_back(std::move(q_t));
  if (return_act) r.t.push_back(std::move(act));
  if (return_dgelu) r.t.push_back(std::move(dg));
  return r;
}

Outs dual_gemm_dgelu_quantize_colsum(const Tensor& a_, const Tensor& b_hi_,
                                          const Tensor& b_lo_, const Tensor& s_a,
                                          const Tensor& s_hi, const Tensor& s_lo,
                                          const Tensor& dgelu, at::ScalarType fp8, bool transpose,
                                          bool col_sum, bool return_grad, bool codes) {
  OnGpu g;
  for (const Tensor* t : {&a_, &b_hi_, &b_lo_, &s_a, &s_hi, &s_lo, &dgelu}) g.add(*t);
  const GemmOps o = gemm_operands(a_, b_hi_, b_lo_);
  const int64_t m = o.a.size(0), k = o.a.size(1), n = o.b_hi.size(0);
  if (dgelu.scalar_type() != at::kFloat || dgelu.dim() != 2 || dgelu.size(0) != m ||
      dgelu.size(1) != n)
    assertion("dgelu must be float32 of shape (" + std::to_string(m) + ", " + std::to_string(n) +
              "), got " + dtype_str(dgelu.scalar_type()) + " " + shape_str(dgelu.sizes()));
  if (n % 8 != 0)
    value_error("column count (" + std::to_string(n) + ") must be divisible by 8");
  const Tensor dc = dgelu.is_contiguous() ? dgelu : dgelu.contiguous();
  const int fmt = fmt_of(fp8);
  Tensor gr = g.empty({m, n}, at::kFloat), q, q_t, cs, cws;
  if (codes) q = g.empty({m, n}, fp8);
  if (transpose) q_t = g.empty({n, m}, fp8);
  Tensor inv = g.empty({1}, at::kFloat);
  size_t nbytes = 0;
  if (col_sum) {
    cs = g.empty({n}, at::kFloat);
    nbytes = tcfp_colsum_workspace_bytes(m, n);
    cws = g.empty({int64_t(std::max<size_t>(nbytes, 16))}, at::kByte);
  }
  const Tensor sa = scalar(s_a, "scale_a"), sh = scalar(s_hi, "scale_hi"),
               sl = scalar(s_lo, "scale_lo");
  void* st = g.stream();
  const Workspace ws(g, st, false);
  check(tcfp_dual_gemm_dgelu_quantize_colsum(
            bytes(o.a), fmt_of(o.a.scalar_type()), o.a.stride(0), bytes(o.b_hi), bytes(o.b_lo),
            fmt_of(o.b_hi.scalar_type()), o.b_hi.stride(0), m, n, k, f32(sa), f32(sh), f32(sl),
            f32(dc), f32(gr), fmt, bytes(q), bytes(q_t), f32(inv), f32(cs), ws.ptr(), ptr(cws),
            nbytes, st),
        "dual_gemm_dgelu_quantize_colsum");
  Outs r = outs(q, inv);
  if (transpose) r.t.push_back(std::move(q_t));
  if (col_sum) r.t.push_back(std::move(cs));
  if (return_grad) r.t.push_back(std::move(gr));
  return r;
}

// ---- the block-scaled layer -------------------------------------------------------

Outs block_linear_forward(const Tensor& x2d, const Tensor& weight, const OptT& bias,
                               int64_t bs, const OptT& error_buf, bool srr, bool update_ef,
                               uint64_t seed) {
  if (bs != 32 && bs != 64 && bs != 128)
    value_error("block_size must be 32, 64, or 128, got " + std::to_string(bs));
  const int64_t M = x2d.size(0), K = x2d.size(1), N = weight.size(0);
  if (!weight.is_contiguous() || weight.size(1) != K || K % bs != 0)
    assertion("weight " + shape_str(weight.sizes()) + " vs input (" + std::to_string(M) + ", " +
              std::to_string(K) + "), block " + std::to_string(bs));
  if (srr && error_buf) value_error("stochastic_lo and error_buf are mutually exclusive");
  OnGpu g;
  g.add(x2d);
  g.add(weight);
  g.add(error_buf);
  g.add(bias);
  void* st = g.stream();
  const int64_t nkb = K / bs;
  const at::ScalarType e4 = at::kFloat8_e4m3fn;
  Tensor hi = g.empty({N, K}, e4), lo = g.empty({N, K}, e4);
  Tensor eh = g.empty({nkb, N}, at::kChar), el = g.empty({nkb, N}, at::kChar);
  check(tcfp_block_dual_quantize(ptr(weight), in_dtype(weight), N, K, int(bs),
                                 f32(opt(error_buf)), update_ef ? 1 : 0, srr ? 1 : 0, seed, 0,
                                 bytes(hi), bytes(lo), exps(eh), exps(el), st),
        "fused_dual_quantize_fp8");
  Tensor act = x2d;
  if (!act.is_contiguous() || !al16(act)) act = act.contiguous();
  Tensor b;
  if (bias) b = bias_f32(*bias, N);
  Tensor out = g.empty({M, N}, at::kFloat);
  Tensor aq = g.empty({M, K}, e4), ae = g.empty({nkb, M}, at::kChar);
  if ((N + 127) / 128 <= 4) {
    check(tcfp_act_quant_block_dual_gemm(ptr(act), in_dtype(act), K, bytes(hi), bytes(lo), K,
                                         exps(eh), exps(el), M, N, K, int(bs), f32(b), f32(out),
                                         N, bytes(aq), exps(ae), st),
          "fused_act_quant_dual_gemm_forward");
  } else {
    check(tcfp_block_quantize(ptr(act), in_dtype(act), M, K, int(bs), TCFP_FP8_E4M3, bytes(aq),
                              exps(ae), st),
          "block_quantize_fp8");
    check(tcfp_block_dual_gemm(bytes(aq), TCFP_FP8_E4M3, K, exps(ae), bytes(hi), bytes(lo),
                               TCFP_FP8_E4M3, K, exps(eh), exps(el), M, N, K, int(bs), f32(b),
                               ptr(out), TCFP_DTYPE_F32, N, st),
          "block_dual_gemm");
  }
  return outs(out, hi, lo, eh, el, aq, ae);
}

// G^T deq(X) to fp32 accuracy for any token count: per-tensor codes with their
// inverse scale, or block codes with their exponents.
Tensor wgrad_f32(const Tensor& grad, const Tensor& act, const OptT& inv, const OptT& act_e,
                 int64_t bs) {
  OnGpu g;
  g.add(grad);
  g.add(act);
  g.add(inv);
  g.add(act_e);
  if (grad.dim() != 2 || act.dim() != 2 || grad.size(0) != act.size(0))
    assertion("token mismatch: grad " + shape_str(grad.sizes()) + " vs act " +
              shape_str(act.sizes()));
  const int64_t m = grad.size(0), n = grad.size(1), k = act.size(1);
  Tensor gr = grad.to(at::kFloat).contiguous();
  if (!al16(gr)) gr = gr.clone();
  const Tensor a = act.contiguous();
  Tensor s, e;
  if (inv) s = scalar(*inv, "scale");
  if (act_e) e = block_scales(*act_e, m, bs > 0 ? k / bs : 0, "act_scales", at::kChar);
  // the GEMM's descriptors span a tile's rows of the split gradient, 6 bytes a
  // token: sums of more tokens (1.4 million with its 256-row tile) are formed
  // in runs of these and added
  constexpr int64_t kTokens = int64_t(1) << 20;
  Tensor dw;
  for (int64_t r = 0; r < std::max<int64_t>(m, 1); r += kTokens) {
    const int64_t c = std::min(kTokens, m - r);
    const size_t nb = tcfp_wgrad_f32_workspace_bytes(c, n, k);
    Tensor part = g.empty({n, k}, at::kFloat), er = e;
    Tensor ws = g.empty({int64_t(std::max<size_t>(nb, 1))}, at::kByte);
    if (e.defined() && c < m) er = e.narrow(1, r, c).contiguous();
    check(tcfp_wgrad_f32(f32(gr) + r * n, c, n, bytes(a) + r * k, fmt_of(a.scalar_type()), f32(s),
                         exps(er), k, int(bs), f32(part), ptr(ws), nb, g.stream()),
          "wgrad_f32");
    if (dw.defined()) dw.add_(part);
    else dw = part;
  }
  return dw;
}

Outs block_linear_backward(const Tensor& grad_2d, const OptT& act_fp8, const OptT& act_e,
                                const OptT& w_hi, const OptT& w_lo, const OptT& e_hi,
                                const OptT& e_lo, int64_t bs, bool need_dx, bool need_dw,
                                bool want_db, bool split_lo, at::ScalarType dx_dtype) {
  const int64_t M = grad_2d.size(0), N = grad_2d.size(1);
  const int64_t K = need_dx ? w_hi->size(1) : need_dw ? act_fp8->size(1) : 0;
  OnGpu g;
  g.add(grad_2d);
  g.add(act_fp8);
  g.add(w_hi);
  void* st = g.stream();
  auto scratch = [&](size_t n) { return g.empty({int64_t(std::max<size_t>(n, 1))}, at::kByte); };
  Tensor gr = grad_2d;
  if (gr.scalar_type() != at::kFloat || !gr.is_contiguous()) gr = gr.to(at::kFloat).contiguous();
  Tensor g_deq, g_split, db, dw, dx;
  if (need_dx) g_deq = g.empty({M, N}, at::kBFloat16);
  if (need_dw) g_split = g.empty({N, split_lo ? 2 * M : M}, at::kBFloat16);
  if (want_db) db = g.empty({N}, at::kFloat);
  {
    const size_t n = want_db ? tcfp_block_grad_prep_workspace_bytes(M, N) : 0;
    Tensor ws;
    if (want_db) ws = scratch(n);
    check(tcfp_block_grad_prep(f32(gr), M, N, int(bs), ptr<uint16_t>(g_deq),
                               ptr<uint16_t>(g_split), split_lo ? 1 : 0, f32(db), nullptr,
                               nullptr, ptr(ws), n, st),
          "block_backward_prep");
  }
  // (the gradient copy, each scratch and the split gradient are released
  // before the next allocation)
  gr.reset();
  if (need_dw) {
    dw = g.empty({N, K}, at::kFloat);
    const size_t n = tcfp_block_wgrad_presplit_workspace_bytes(M, N, K, split_lo ? 1 : 0);
    Tensor ws = scratch(n);
    check(tcfp_block_wgrad_presplit(ptr<uint16_t>(g_split), split_lo ? 1 : 0, M, N,
                                    bytes(*act_fp8), fmt_of(act_fp8->scalar_type()), exps(*act_e),
                                    K, int(bs), f32(dw), ptr(ws), n, st),
          "block_wgrad_from_prep");
  }
  g_split.reset();
  if (need_dx) {
    dx = g.empty({M, K}, dx_dtype);
    const size_t n = tcfp_block_dual_gemm_dx_bf16_workspace_bytes(N, K);
    Tensor ws = scratch(n);
    check(tcfp_block_dual_gemm_dx_bf16_to(ptr<uint16_t>(g_deq), bytes(*w_hi), bytes(opt(w_lo)),
                                          exps(*e_hi), exps(opt(e_lo)), M, N, K, int(bs), ptr(dx),
                                          out_dtype_of(dx_dtype), ptr(ws), n, st),
          "block_dgrad_from_prep");
  }
  return outs(dx, dw, db);
}

}  // namespace

namespace pybind11::detail {
template <>
struct type_caster<Outs> {
  PYBIND11_TYPE_CASTER(Outs, const_name("tuple"));
  bool load(handle, bool) { return false; }  // results only
  static handle cast(Outs&& o, return_value_policy, handle) {
    tuple r(o.t.size());
    for (size_t i = 0; i < o.t.size(); ++i) {
      PyObject* t = THPVariable_Wrap(std::move(o.t[i]));
      if (!t) throw error_already_set();
      PyTuple_SET_ITEM(r.ptr(), ssize_t(i), t);
    }
    return r.release();
  }
};
}  // namespace pybind11::detail

PYBIND11_MODULE(_tcfp_host, m) {
  m.doc() = "Native host path of tcfp_amd.kernels";
  // torch's errors as torch raises them from Python: a caller that handles
  // torch.OutOfMemoryError, or the exception that its dispatch mode raised
  // (pybind11 alone would make each a RuntimeError)
  py::register_local_exception_translator([](std::exception_ptr p) {
    try {
      if (p) std::rethrow_exception(p);
    } catch (const Raise& e) {
      PyErr_SetString(e.type, e.msg.c_str());
    } catch (python_error& e) {
      e.restore();
    } catch (const c10::Error&) {
      torch::translate_exception_to_python(p);
    }
  });
  // (results are converted after the guard has taken the GIL back)
  using NoGil = py::call_guard<py::gil_scoped_release>;
  m.def("quantize_per_tensor", &quantize_per_tensor, NoGil());
  m.def("quantize_per_tensor_colsum", &quantize_per_tensor_colsum, NoGil());
  m.def("dual_quantize_per_tensor", &dual_quantize_per_tensor, NoGil());
  m.def("quantize_batch", &quantize_batch, NoGil());
  m.def("dual_gemm", &dual_gemm, NoGil());
  m.def("block_quantize", &block_quantize, NoGil());
  m.def("block_gemm", &block_gemm, NoGil());
  m.def("dual_gemm_gelu_quantize", &dual_gemm_gelu_quantize, NoGil());
  m.def("dual_gemm_dgelu_quantize_colsum", &dual_gemm_dgelu_quantize_colsum, NoGil());
  m.def("wgrad_f32", &wgrad_f32, NoGil());
  m.def("block_linear_forward", &block_linear_forward, NoGil());
  m.def("block_linear_backward", &block_linear_backward, NoGil());
}

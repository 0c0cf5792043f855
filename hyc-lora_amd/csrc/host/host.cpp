// The host side of a calibrated operator's call in native code: checks, output allocation, descriptors and launches of one
// step of kernels.py / operators / decoder_layer.py, without the interpreter in between.
//
// A short call is bound by its host work (rms norm of 45 x 4096, forward and backward: the kernels take 18 us of 70 to 150), and most
// of that is a few dozen interpreted steps around each launch.  Every function here covers the plain case only - dense bf16
// tensors on the GPU of the expected layout, a plan that matches - and returns None for everything else, before anything is
// allocated or launched; the caller then goes through the interpreted form, which handles the rest and raises the errors.  A
// kernel's entry may still refuse behind these checks (a size or an alignment that is its own to judge): what the call has launched by then
// wrote results only, and the interpreted form writes them again before it raises.  What is launched, and with what, is the
// same in both.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/autocast_mode.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_cpp_function.h>
#include <torch/csrc/autograd/python_variable.h>

#include <atomic>
#include <cstring>
#include <string>
#include <vector>

#include "../../../include/hyc_abi.h"

namespace {

using at::Tensor;
constexpr auto BF16 = at::kBFloat16;

// torch.nn.Parameter, kernels.ChannelCompressed, ChannelPlan, ThresholdCompressed, SparseRows
PyObject *t_parameter, *t_compressed, *t_plan, *t_threshold, *t_sparse, *t_namespace /* types.SimpleNamespace */;
PyObject *s_H, *s_M, *s_S, *s_k, *s_idx, *s_plan, *s_scale_rule, *s_stored, *s_vals, *s_scales, *s_bits, *s_group, *s_row_ptr, *s_cols, *s_threshold,
    *s_scale, *s_L, *s_R;

struct Ref {                                                           // an owned reference
  PyObject* p;
  explicit Ref(PyObject* o) : p(o) {}
  Ref(const Ref&) = delete;
  ~Ref() { Py_XDECREF(p); }
};

void* stream() { return c10::hip::getCurrentHIPStream().stream(); }

// f() without the interpreter's lock: allocations, launches and library products may wait for the device or for a lock of the runtime,
// and other threads go on meanwhile.  Nothing in f touches an object of the interpreter; the arguments' tensors are held by the call.
template <class F>
auto unlocked(F&& f) {
  struct Release {
    PyThreadState* state = PyEval_SaveThread();
    ~Release() { PyEval_RestoreThread(state); }
  } release;
  return f();
}

// a dense GPU tensor of the exact type (a subclass may do anything on access, a functorch wrapper has no memory of its own)
bool dense_gpu(const Tensor& t) { return t.defined() && t.is_cuda() && t.layout() == at::kStrided && t.has_storage() && !t.is_conj() && !t.is_neg(); }
const Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o) && (PyObject*)Py_TYPE(o) != t_parameter) return nullptr;
  const Tensor& t = THPVariable_Unpack(o);
  return dense_gpu(t) ? &t : nullptr;
}
const Tensor* bf16(PyObject* o) {
  const Tensor* t = plain(o);
  return t && t->scalar_type() == BF16 ? t : nullptr;
}
bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

// [..., H] contiguous -> M rows
bool rows_of(const Tensor& t, int64_t* M, int64_t* H) {
  if (t.dim() < 1 || !t.is_contiguous()) return false;
  *H = t.size(-1);
  if (*H <= 0) return false;
  *M = t.numel() / *H;
  return true;
}
// [..., H] with contiguous, evenly spaced rows -> M rows `pitch` elements apart: the forms t.view(-1, H) takes
bool spaced_rows(const Tensor& t, int64_t* M, int64_t* H, int64_t* pitch) {
  const int64_t d = t.dim();
  if (d < 2 || t.size(-1) <= 0 || t.numel() == 0 || t.stride(-1) != 1) return false;
  *H = t.size(-1);
  *M = 1;
  *pitch = *H;
  for (int64_t i = d - 2; i >= 0; --i) {                               // innermost first; the stride of a dimension of 1 says nothing
    if (t.size(i) == 1) continue;
    if (*M == 1) *pitch = t.stride(i);
    else if (t.stride(i) != *M * *pitch) return false;
    *M *= t.size(i);
  }
  return true;
}
// the same as the fused kernels read it in place
bool kernel_rows(const Tensor& t, int64_t* M, int64_t* H, int64_t* pitch) {
  return spaced_rows(t, M, H, pitch) && aligned16(t.data_ptr()) && *pitch % 8 == 0 && *pitch >= *H;
}

int64_t attr_i64(PyObject* o, PyObject* name, bool* ok) {
  Ref v(PyObject_GetAttr(o, name));
  if (!v.p || !PyLong_CheckExact(v.p)) { PyErr_Clear(); *ok = false; return 0; }
  return PyLong_AsLongLong(v.p);
}

struct Plan {
  int64_t H = 0, k = 0;
  Tensor idx, plan;
  int rule = 0;
  void describe(int64_t bits, int64_t group, hyc_desc* d) const {
    std::memset(d, 0, sizeof *d);
    d->mode = HYC_MODE_CHANNEL;
    d->bits = (int32_t)bits;
    d->group = (int32_t)group;
    d->k = (int32_t)k;
    d->chan_plan = (decltype(d->chan_plan))plan.data_ptr();
    d->chan_idx = k ? (decltype(d->chan_idx))idx.data_ptr() : nullptr;
    d->scale_rule = rule;
  }
  // what kernels._check_plan asks of a plan, for an activation of n channels on `device`
  bool usable(int64_t n, c10::Device device) const {
    return H == n && k >= 0 && dense_gpu(idx) && dense_gpu(plan) && idx.scalar_type() == at::kInt && plan.scalar_type() == at::kInt &&
           idx.is_contiguous() && plan.is_contiguous() && idx.numel() == k && plan.numel() == H / 8 && idx.device() == device && plan.device() == device;
  }
};
bool get_plan(PyObject* o, int64_t H, c10::Device device, Plan* p) {
  if ((PyObject*)Py_TYPE(o) != t_plan) return false;
  bool ok = true;
  p->H = attr_i64(o, s_H, &ok);
  p->k = attr_i64(o, s_k, &ok);
  if (!ok) return false;
  Ref idx(PyObject_GetAttr(o, s_idx)), plan(PyObject_GetAttr(o, s_plan)), rule(PyObject_GetAttr(o, s_scale_rule));
  if (!idx.p || !plan.p || !rule.p) { PyErr_Clear(); return false; }
  const Tensor *ti = plain(idx.p), *tp = plain(plan.p);
  if (!ti || !tp || !PyUnicode_Check(rule.p)) return false;
  if (PyUnicode_CompareWithASCIIString(rule.p, "absmax") == 0) p->rule = HYC_SCALE_ABSMAX;
  else if (PyUnicode_CompareWithASCIIString(rule.p, "range") == 0) p->rule = HYC_SCALE_RANGE;
  else return false;
  p->idx = *ti;
  p->plan = *tp;
  return p->usable(H, device);
}

// the threshold scheme's descriptor: a static scale read through two strides, a base of rank 0 or more
struct Threshold {
  hyc_desc d;
  static bool readable(const Tensor* t) { return t && dense_gpu(*t) && t->scalar_type() == BF16 && t->is_contiguous(); }
  bool init(double threshold, PyObject* scale, int64_t bits, int64_t S, int64_t H, PyObject* L, PyObject* R) {
    const Tensor *l = L != Py_None ? bf16(L) : nullptr, *r = L != Py_None ? bf16(R) : nullptr;
    return (L == Py_None || (l && r)) && init(threshold, bf16(scale), bits, S, H, l, r);
  }
  bool init(double threshold, const Tensor* sc, int64_t bits, int64_t S, int64_t H, const Tensor* l, const Tensor* r) {
    if (!readable(sc)) return false;
    std::memset(&d, 0, sizeof d);
    d.mode = HYC_MODE_THRESHOLD;
    d.bits = (int32_t)bits;
    d.threshold = (float)threshold;
    d.scale = (decltype(d.scale))sc->data_ptr();
    const int64_t n = sc->numel();
    if (n == 1) { d.scale_stride_token = 0; d.scale_stride_channel = 0; }
    else if (sc->dim() >= 2 && sc->size(-1) == H && n == H) { d.scale_stride_token = 0; d.scale_stride_channel = 1; }
    else if (sc->dim() >= 2 && sc->size(-1) == 1 && n == S) { d.scale_stride_token = 1; d.scale_stride_channel = 0; }
    else return false;
    d.S = S;
    if (l) {
      if (!readable(l) || !readable(r) || l->dim() != 2 || r->dim() != 2 || l->size(0) < S || l->size(1) != r->size(0) || r->size(1) != H)
        return false;                                                  // (fewer rows than S: padded by the general form)
      d.rank = (int32_t)l->size(1);
      if (d.rank) { d.L = (decltype(d.L))l->data_ptr(); d.R = (decltype(d.R))r->data_ptr(); }
    }
    return true;
  }
};
bool vec(const Tensor& t, at::ScalarType type) { return dense_gpu(t) && t.scalar_type() == type && t.is_contiguous(); }
const Tensor* attr_vec(const Ref& v, at::ScalarType type) {
  const Tensor* t = v.p ? plain(v.p) : nullptr;
  if (!v.p) PyErr_Clear();
  return t && vec(*t, type) ? t : nullptr;
}
Tensor empty_like_on(const Tensor& t, at::IntArrayRef sizes, at::ScalarType type) { return at::empty(sizes, at::TensorOptions().device(t.device()).dtype(type)); }

// a compressed activation: of the channel scheme as it is read, of the threshold scheme restored first (ready()).  A value: a node of the graph
// keeps one, and each pass over it works on a copy whose descriptor is made anew (a tensor may have been given other memory since).
struct Saved {
  Tensor stored, vals, scales, row_ptr, cols, scale, L, R;
  Plan p;
  hyc_desc d;
  int64_t M = 0, H = 0, S = 0, bits = 0, group = 0;
  double threshold = 0.0;
  bool restore_first = false;
  // the descriptor, from where the tensors lie now; false: not as the kernels read them
  bool describe() {
    if (!dense_gpu(stored) || !dense_gpu(vals)) return false;
    if (!restore_first) {
      if (!dense_gpu(scales) || !p.usable(H, stored.device())) return false;
      p.describe(bits, group, &d);
      return true;
    }
    Threshold t;
    if (!vec(row_ptr, at::kInt) || !vec(cols, at::kInt) ||
        !t.init(threshold, &scale, bits, S, H, L.defined() ? &L : nullptr, R.defined() ? &R : nullptr))
      return false;
    d = t.d;
    d.csr_row_ptr = (decltype(d.csr_row_ptr))row_ptr.data_ptr();
    d.csr_cols = cols.numel() ? (decltype(d.csr_cols))cols.data_ptr() : nullptr;
    d.csr_vals = vals.numel() ? (decltype(d.csr_vals))vals.data_ptr() : nullptr;
    return true;
  }
  const void* codes() const { return stored.data_ptr(); }
  const void* values() const { return vals.defined() ? vals.data_ptr() : nullptr; }
  const void* group_scales() const { return scales.defined() ? scales.data_ptr() : nullptr; }
  // the dense x_hat [M, H]
  bool restore(Tensor* x) const {
    *x = empty_like_on(stored, {M, H}, BF16);
    const bool thr = restore_first;
    return hyc_decompress(stored.data_ptr(), thr ? nullptr : values(), thr ? nullptr : group_scales(), M, H, &d, x->data_ptr(), stream()) == 0;
  }
  // from here on `stored` is the restored matrix itself
  bool make_dense() {
    Tensor x;
    if (!restore(&x)) return false;
    stored = x;
    vals = Tensor();
    scales = Tensor();
    std::memset(&d, 0, sizeof d);
    d.mode = HYC_MODE_DENSE;
    d.bits = 4;
    restore_first = false;
    return true;
  }
  // what a consumer kernel reads: the last thing before its launch
  bool ready() { return !restore_first || make_dense(); }
  PyObject* wrap(PyObject* plan) const;                                // kernels.ChannelCompressed / ThresholdCompressed; plan: its plan, or null
};
struct In : Saved {
  bool init(PyObject* c) {
    const bool thr = (PyObject*)Py_TYPE(c) == t_threshold;
    if (!thr && (PyObject*)Py_TYPE(c) != t_compressed) return false;
    bool ok = true;
    M = attr_i64(c, s_M, &ok);
    H = attr_i64(c, s_H, &ok);
    bits = attr_i64(c, s_bits, &ok);
    Ref st(PyObject_GetAttr(c, s_stored)), va(PyObject_GetAttr(c, s_vals));
    const Tensor *ts = st.p ? plain(st.p) : nullptr, *tv = va.p ? plain(va.p) : nullptr;
    if (!ok || !ts || !tv) { PyErr_Clear(); return false; }
    stored = *ts; vals = *tv;
    if (thr) {
      S = attr_i64(c, s_S, &ok);
      Ref rp(PyObject_GetAttr(c, s_row_ptr)), co(PyObject_GetAttr(c, s_cols)), th(PyObject_GetAttr(c, s_threshold)), sc(PyObject_GetAttr(c, s_scale)),
          l(PyObject_GetAttr(c, s_L)), r(PyObject_GetAttr(c, s_R));
      const Tensor *tr = attr_vec(rp, at::kInt), *tc = attr_vec(co, at::kInt), *ts = sc.p ? plain(sc.p) : nullptr,
                   *tl = l.p && l.p != Py_None ? plain(l.p) : nullptr, *tR = r.p && r.p != Py_None ? plain(r.p) : nullptr;
      if (!ok || !tr || !tc || !ts || !th.p || !l.p || !r.p || !PyFloat_CheckExact(th.p) || (l.p != Py_None && (!tl || !tR))) {
        PyErr_Clear();
        return false;
      }
      row_ptr = *tr; cols = *tc; scale = *ts;
      if (tl) L = *tl;
      if (tR) R = *tR;
      threshold = PyFloat_AS_DOUBLE(th.p);
      restore_first = true;
      return describe();
    }
    group = attr_i64(c, s_group, &ok);
    Ref sc(PyObject_GetAttr(c, s_scales)), pl(PyObject_GetAttr(c, s_plan));
    const Tensor* tc = sc.p ? plain(sc.p) : nullptr;
    if (!ok || !tc || !pl.p || !get_plan(pl.p, H, stored.device(), &p)) { PyErr_Clear(); return false; }
    scales = *tc;
    return describe();
  }
};
PyObject* wrap_or_none(const Tensor& t) {
  if (t.defined()) return THPVariable_Wrap(t);
  Py_RETURN_NONE;
}
PyObject* Saved::wrap(PyObject* plan) const {
  if (restore_first) {                                                 // (stored, row_ptr, cols, vals, threshold, scale, L, R, bits, M, H, S)
    Ref args(Py_BuildValue("NNNNdNNNLLLL", wrap_or_none(stored), wrap_or_none(row_ptr), wrap_or_none(cols), wrap_or_none(vals), threshold,
                           wrap_or_none(scale), wrap_or_none(L), wrap_or_none(R), (long long)bits, (long long)M, (long long)H, (long long)S));
    return args.p ? PyObject_CallObject(t_threshold, args.p) : nullptr;
  }
  Ref made(nullptr);
  if (!plan) {                                                         // (H, k, idx, plan, scale_rule)
    Ref args(Py_BuildValue("LLNNs", (long long)p.H, (long long)p.k, wrap_or_none(p.idx), wrap_or_none(p.plan),
                           p.rule == HYC_SCALE_ABSMAX ? "absmax" : "range"));
    if (!args.p || !(plan = made.p = PyObject_CallObject(t_plan, args.p))) return nullptr;
  }
  Ref a(THPVariable_Wrap(stored)), b(THPVariable_Wrap(vals)), c(THPVariable_Wrap(scales)), w(PyLong_FromLongLong(bits)), g(PyLong_FromLongLong(group)),
      m(PyLong_FromLongLong(M)), h(PyLong_FromLongLong(H));
  if (!a.p || !b.p || !c.p || !w.p || !g.p || !m.p || !h.p) return nullptr;
  PyObject* args[8] = {a.p, b.p, c.p, plan, w.p, g.p, m.p, h.p};      // (stored, vals, scales, plan, bits, group, M, H)
  return PyObject_Vectorcall(t_compressed, args, 8, nullptr);
}
// one of the channel scheme about to be written
struct Out : Saved {
  PyObject* plan;
  bool init(PyObject* plan_, PyObject* bits_, PyObject* group_, int64_t M_, int64_t H_, c10::Device device) {
    plan = plan_; M = M_; H = H_;
    if (!PyLong_CheckExact(bits_) || !PyLong_CheckExact(group_)) return false;
    bits = PyLong_AsLongLong(bits_);
    group = PyLong_AsLongLong(group_);
    if (hyc_check_shape(H, (int32_t)bits, (int32_t)group, HYC_MODE_CHANNEL) != 0 || !get_plan(plan, H, device, &p)) return false;
    p.describe(bits, group, &d);
    return true;
  }
  void alloc() {
    const auto opt = at::TensorOptions().device(p.plan.device());
    stored = at::empty({M, H * bits / 8}, opt.dtype(bits == 8 ? at::kChar : at::kByte));
    vals = at::empty({M, p.k}, opt.dtype(BF16));
    scales = at::empty({M, H / group}, opt.dtype(BF16));
  }
  PyObject* wrap() const { return Saved::wrap(plan); }
};

PyObject* none() { Py_RETURN_NONE; }
PyObject* tuple2(PyObject* a, PyObject* b) {
  if (!a || !b) { Py_XDECREF(a); Py_XDECREF(b); return nullptr; }
  PyObject* t = PyTuple_New(2);
  PyTuple_SET_ITEM(t, 0, a);
  PyTuple_SET_ITEM(t, 1, b);
  return t;
}
// the entry points' way out: a failed call goes through the interpreted form once more, which raises its error
#define OR_NONE(call_) do { if ((call_) != 0) return none(); } while (0)
#define ARGS(n_) do { if (nargs != (n_)) { PyErr_Format(PyExc_TypeError, "%s takes %d arguments", __func__, (n_)); return nullptr; } } while (0)

// ---- compress / decompress -----------------------------------------------------------------------------------
PyObject* compress_rows(const Tensor& x, PyObject* plan, PyObject* bits, PyObject* group) {    // nullptr without an error: not the plain case
  int64_t M, H, pitch;
  if (x.scalar_type() != BF16 || !spaced_rows(x, &M, &H, &pitch)) return nullptr;
  Out o;
  if (!o.init(plan, bits, group, M, H, x.device())) return nullptr;
  if (unlocked([&] {
        o.alloc();
        return hyc_compress_rows(x.data_ptr(), pitch, M, H, &o.d, o.stored.data_ptr(), o.vals.data_ptr(), o.scales.data_ptr(), nullptr, stream());
      }) != 0)
    return nullptr;
  return o.wrap();
}
PyObject* none_if_plain(PyObject* r) { return r || PyErr_Occurred() ? r : none(); }

// compress(x [M, H], plan, bits, group) -> ChannelCompressed
PyObject* compress(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ARGS(4);
  const Tensor* x = bf16(a[0]);
  return x && x->dim() == 2 ? none_if_plain(compress_rows(*x, a[1], a[2], a[3])) : none();
  END_HANDLE_TH_ERRORS
}
bool restore(PyObject* c, Tensor* x) {
  In in;
  return in.init(c) && unlocked([&] { return in.restore(x); });
}
// decompress(c) -> bf16 [M, H]; c of either scheme
PyObject* decompress(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ARGS(1);
  Tensor x;
  return restore(a[0], &x) ? THPVariable_Wrap(x) : none();
  END_HANDLE_TH_ERRORS
}

// ---- norms -----------------------------------------------------------------------------------------------------
bool weight_dtype(const Tensor& w, int64_t H, int* dtype) {
  if (!w.is_contiguous() || w.numel() != H) return false;
  if (w.scalar_type() == at::kFloat) *dtype = HYC_DTYPE_F32;
  else if (w.scalar_type() == BF16) *dtype = HYC_DTYPE_BF16;
  else return false;
  return true;
}
bool norm_weight(PyObject* o, int64_t H, const Tensor** w, int* dtype) {
  *w = plain(o);
  return *w && weight_dtype(**w, H, dtype);
}
struct NormOut {
  const Tensor *x, *w, *bias = nullptr;
  Out o;
  Tensor y, rstd, mean;
  // (x [..., H], w, bias or None, layer_norm, eps, plan, bits, group); false: not the plain case, or an error that is set
  bool init(PyObject* const* a) {
    int64_t M, H;
    x = bf16(a[0]);
    if (!x || !rows_of(*x, &M, &H) || !norm_weight(a[1], H, &w, &dtype)) return false;
    if (a[2] != Py_None) {
      bias = plain(a[2]);
      if (!bias || !bias->is_contiguous() || bias->numel() != H || bias->scalar_type() != w->scalar_type()) return false;
    }
    ln = a[3] == Py_True;
    eps = PyFloat_AsDouble(a[4]);
    return !PyErr_Occurred() && o.init(a[5], a[6], a[7], M, H, x->device());
  }
  int launch() {
    o.alloc();
    y = at::empty(x->sizes(), x->options());
    rstd = empty_like_on(*x, {o.M}, at::kFloat);
    if (!ln)
      return hyc_rmsnorm_fwd_compress(x->data_ptr(), w->data_ptr(), dtype, (float)eps, o.M, o.H, &o.d, y.data_ptr(), (float*)rstd.data_ptr(),
                                      o.stored.data_ptr(), o.vals.data_ptr(), o.scales.data_ptr(), nullptr, stream());
    mean = empty_like_on(*x, {o.M}, at::kFloat);
    return hyc_layernorm_fwd_compress(x->data_ptr(), w->data_ptr(), bias ? bias->data_ptr() : nullptr, dtype, (float)eps, o.M, o.H, &o.d, y.data_ptr(),
                                      (float*)mean.data_ptr(), (float*)rstd.data_ptr(), o.stored.data_ptr(), o.vals.data_ptr(), o.scales.data_ptr(),
                                      nullptr, stream());
  }
  int dtype;
  bool ln;
  double eps;
};
// norm_fwd(x [..., H], w, bias or None, layer_norm, eps, plan, bits, group) -> (y like x, mean or None, rstd, ChannelCompressed)
PyObject* norm_fwd(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ARGS(8);
  NormOut n;
  if (!n.init(a)) return none_if_plain(nullptr);
  OR_NONE(unlocked([&] { return n.launch(); }));
  PyObject* c = n.o.wrap();
  if (!c) return nullptr;
  PyObject* t = PyTuple_New(4);
  PyTuple_SET_ITEM(t, 0, THPVariable_Wrap(n.y));
  PyTuple_SET_ITEM(t, 1, wrap_or_none(n.mean));
  PyTuple_SET_ITEM(t, 2, THPVariable_Wrap(n.rstd));
  PyTuple_SET_ITEM(t, 3, c);
  return t;
  END_HANDLE_TH_ERRORS
}
// the statistics of M rows
bool row_stats(const Tensor& t, int64_t M) { return t.scalar_type() == at::kFloat && t.is_contiguous() && t.numel() == M; }
int norm_backward(const Tensor& dy, Saved& in, const Tensor& w, int dtype, const Tensor& mean, const Tensor& rstd, bool quirk, Tensor* dx, Tensor* dw) {
  const int64_t M = in.M, H = in.H;
  if (!in.ready()) return -1;
  const int64_t P = hyc_rmsnorm_bwd_partials(M, H);
  const Tensor partials = empty_like_on(dy, {P > 1 ? P : 1, H}, at::kFloat);
  *dx = at::empty(dy.sizes(), dy.options());
  *dw = empty_like_on(dy, {H}, w.scalar_type());
  if (mean.defined())
    return hyc_layernorm_bwd(dy.data_ptr(), in.codes(), in.values(), in.group_scales(), w.data_ptr(), dtype, (const float*)mean.data_ptr(),
                             (const float*)rstd.data_ptr(), M, H, &in.d, dx->data_ptr(), (float*)partials.data_ptr(), dw->data_ptr(), stream());
  return hyc_rmsnorm_bwd(dy.data_ptr(), in.codes(), in.values(), in.group_scales(), w.data_ptr(), dtype, (const float*)rstd.data_ptr(), M, H, &in.d,
                         quirk, dx->data_ptr(), (float*)partials.data_ptr(), dw->data_ptr(), stream());
}
// norm_bwd(dy [..., H], c, w, mean or None, rstd, quirk) -> (dx like dy, dw in w's dtype)
PyObject* norm_bwd(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ARGS(6);
  const Tensor *dy = bf16(a[0]), *w, *mean = nullptr, *rstd = plain(a[4]);
  int64_t M, H;
  int dtype;
  In in;
  if (!dy || !rows_of(*dy, &M, &H) || !norm_weight(a[2], H, &w, &dtype) || !in.init(a[1]) || in.M != M || in.H != H) return none();
  if (!rstd || !row_stats(*rstd, M)) return none();
  if (a[3] != Py_None) {
    mean = plain(a[3]);
    if (!mean || !row_stats(*mean, M)) return none();
  }
  const bool quirk = a[5] == Py_True;
  Tensor dx, dw;
  OR_NONE(unlocked([&] { return norm_backward(*dy, in, *w, dtype, mean ? *mean : Tensor(), *rstd, quirk, &dx, &dw); }));
  return tuple2(THPVariable_Wrap(dx), THPVariable_Wrap(dw));
  END_HANDLE_TH_ERRORS
}
int bias_backward(const Tensor& dy, int64_t M, int64_t H, bool f32, Tensor* db) {
  const int64_t P = hyc_bias_grad_partials(M, H);
  const Tensor partials = empty_like_on(dy, {P > 1 ? P : 1, H}, at::kFloat);
  *db = empty_like_on(dy, {H}, f32 ? at::kFloat : BF16);
  return hyc_bias_grad(dy.data_ptr(), M, H, (float*)partials.data_ptr(), db->data_ptr(), f32 ? HYC_DTYPE_F32 : HYC_DTYPE_BF16, stream());
}
// bias_grad(dy [..., H], fp32) -> db [H]
PyObject* bias_grad(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ARGS(2);
  const Tensor* dy = bf16(a[0]);
  int64_t M, H;
  if (!dy || !rows_of(*dy, &M, &H)) return none();
  const bool f32 = a[1] == Py_True;
  Tensor db;
  OR_NONE(unlocked([&] { return bias_backward(*dy, M, H, f32, &db); }));
  return THPVariable_Wrap(db);
  END_HANDLE_TH_ERRORS
}

// ---- the threshold scheme and kept probabilities: side data sized ahead of time ------------------------------------------
struct Csr {
  Tensor row_ptr, cols, vals, total;
  // room for `cap` entries
  void alloc(const Tensor& counts, int64_t rows, int64_t cap) {
    row_ptr = empty_like_on(counts, {rows + 1}, at::kInt);
    total = empty_like_on(counts, {}, at::kLong);
    cols = empty_like_on(counts, {cap}, at::kInt);
    vals = empty_like_on(counts, {cap}, BF16);
  }
  int64_t* all() const { return (int64_t*)total.data_ptr(); }
  // and offsets of the counts, cut off at that
  bool offsets(const Tensor& counts, int64_t rows, int64_t cap) {
    alloc(counts, rows, cap);
    return hyc_csr_offsets((const int32_t*)counts.data_ptr(), rows, cap, rp(), all(), stream()) == 0;
  }
  int32_t* rp() const { return (int32_t*)row_ptr.data_ptr(); }
  int32_t* co() const { return (int32_t*)cols.data_ptr(); }
};
PyObject* wrap_all(std::initializer_list<Tensor> ts) {
  PyObject* t = PyTuple_New((Py_ssize_t)ts.size());
  Py_ssize_t i = 0;
  for (const Tensor& x : ts) PyTuple_SET_ITEM(t, i++, x.defined() ? THPVariable_Wrap(x) : none());
  return t;
}
// threshold_fwd(x [..., H], norm, w or None, bias or None, eps, S, threshold, scale, bits, L or None, R or None, cap, slab entries per row)
//   -> (y like x or None, mean or None, rstd or None, stored, row_ptr, cols, vals, total); norm: 0 compress only, 1 rms, 2 layer
PyObject* threshold_fwd(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ARGS(13);
  const Tensor *x = bf16(a[0]), *w = nullptr, *bias = nullptr;
  const long norm = PyLong_AsLong(a[1]);
  const double eps = PyFloat_AsDouble(a[4]), thr = PyFloat_AsDouble(a[6]);
  const int64_t S = PyLong_AsLongLong(a[5]), bits = PyLong_AsLongLong(a[8]), cap = PyLong_AsLongLong(a[11]),
                slab_cap = PyLong_AsLongLong(a[12]);
  if (PyErr_Occurred()) return nullptr;
  int64_t M, H;
  int dtype = 0;
  Threshold t;
  if (!x || !rows_of(*x, &M, &H) || M == 0 || cap <= 0 || hyc_check_shape(H, (int32_t)bits, 0, HYC_MODE_THRESHOLD) != 0 ||
      !t.init(thr, a[7], bits, S, H, a[9], a[10]) || (norm && !norm_weight(a[2], H, &w, &dtype)))
    return none();
  if (norm == 2 && a[3] != Py_None) {
    bias = plain(a[3]);
    if (!bias || !bias->is_contiguous() || bias->numel() != H || bias->scalar_type() != w->scalar_type()) return none();
  }
  Tensor y, mean, rstd, stored;
  Csr csr;
  OR_NONE(unlocked([&]() -> int {
    stored = empty_like_on(*x, {M, H * bits / 8}, bits == 8 ? at::kChar : at::kByte);
    const Tensor counts = empty_like_on(*x, {M}, at::kInt);
    if (norm) {
      y = at::empty(x->sizes(), x->options());
      rstd = empty_like_on(*x, {M}, at::kFloat);
    }
    if (norm == 2) mean = empty_like_on(*x, {M}, at::kFloat);
    int32_t* n = (int32_t*)counts.data_ptr();
    const void* b = bias ? bias->data_ptr() : nullptr;
    Tensor slab;
    int rc = HYC_ENOTSUP;
    if (slab_cap > 0) {
      slab = empty_like_on(*x, {M, slab_cap}, at::kInt);
      rc = hyc_threshold_fwd((int32_t)norm, x->data_ptr(), norm ? w->data_ptr() : nullptr, b, dtype, (float)eps, M, H, &t.d, norm ? y.data_ptr() : nullptr,
                             norm == 2 ? (float*)mean.data_ptr() : nullptr, norm ? (float*)rstd.data_ptr() : nullptr, stored.data_ptr(), n,
                             (uint32_t*)slab.data_ptr(), slab_cap, stream());
    }
    const bool general = rc == HYC_ENOTSUP;
    if (general && norm == 2)
      rc = hyc_layernorm_fwd_compress(x->data_ptr(), w->data_ptr(), b, dtype, (float)eps, M, H, &t.d, y.data_ptr(), (float*)mean.data_ptr(),
                                      (float*)rstd.data_ptr(), stored.data_ptr(), nullptr, nullptr, n, stream());
    else if (general && norm)
      rc = hyc_rmsnorm_fwd_compress(x->data_ptr(), w->data_ptr(), dtype, (float)eps, M, H, &t.d, y.data_ptr(), (float*)rstd.data_ptr(), stored.data_ptr(),
                                    nullptr, nullptr, n, stream());
    else if (general)
      rc = hyc_compress(x->data_ptr(), M, H, &t.d, stored.data_ptr(), nullptr, nullptr, n, stream());
    if (rc != 0) return -1;
    if (general) {
      if (!csr.offsets(counts, M, cap)) return -1;
      return hyc_ref_outlier_fill(x->data_ptr(), M, H, &t.d, csr.rp(), csr.co(), csr.vals.data_ptr(), stream());
    }
    csr.alloc(counts, M, cap);
    return hyc_ref_outlier_csr_slab(x->data_ptr(), M, H, &t.d, n, (const uint32_t*)slab.data_ptr(), slab_cap, cap, csr.rp(), csr.all(), csr.co(),
                                    csr.vals.data_ptr(), stream());
  }));
  return wrap_all({y, mean, rstd, stored, csr.row_ptr, csr.cols, csr.vals, csr.total});
  END_HANDLE_TH_ERRORS
}
// softmax_fwd(x [..., N], threshold, slab entries per row, cap) -> (y, row_ptr, cols, vals, total)
PyObject* softmax_fwd(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ARGS(4);
  const Tensor* x = bf16(a[0]);
  const double thr = PyFloat_AsDouble(a[1]);
  const int64_t slab_cap = PyLong_AsLongLong(a[2]), cap = PyLong_AsLongLong(a[3]);
  if (PyErr_Occurred()) return nullptr;
  int64_t M, N;
  if (!x || !rows_of(*x, &M, &N) || M == 0 || slab_cap <= 0 || cap <= 0) return none();
  Tensor y;
  Csr csr;
  OR_NONE(unlocked([&]() -> int {
    y = at::empty(x->sizes(), x->options());
    const Tensor counts = empty_like_on(*x, {M}, at::kInt), slab = empty_like_on(*x, {M, slab_cap}, at::kInt);
    int32_t* n = (int32_t*)counts.data_ptr();
    uint32_t* sl = (uint32_t*)slab.data_ptr();
    const int rc = hyc_softmax_fwd_slab(x->data_ptr(), M, N, 0, (float)thr, y.data_ptr(), n, sl, slab_cap, stream());
    if (rc != 0) return -1;
    csr.alloc(counts, M, cap);
    return hyc_softmax_csr_slab(y.data_ptr(), M, N, (float)thr, n, sl, slab_cap, cap, csr.rp(), csr.all(), csr.co(), csr.vals.data_ptr(), stream());
  }));
  return wrap_all({y, csr.row_ptr, csr.cols, csr.vals, csr.total});
  END_HANDLE_TH_ERRORS
}
struct Sparse {                                                        // kernels.SparseRows about to be read
  Tensor row_ptr, cols, vals;
  bool init(PyObject* o) {
    if ((PyObject*)Py_TYPE(o) != t_sparse) return false;
    Ref r(PyObject_GetAttr(o, s_row_ptr)), c(PyObject_GetAttr(o, s_cols)), v(PyObject_GetAttr(o, s_vals));
    const Tensor *tr = attr_vec(r, at::kInt), *tc = attr_vec(c, at::kInt), *tv = attr_vec(v, BF16);
    if (!tr || !tc || !tv || tc->numel() == 0 || tc->numel() != tv->numel()) return false;
    row_ptr = *tr; cols = *tc; vals = *tv;
    return true;
  }
  int64_t rows() const { return row_ptr.numel() - 1; }
};
// softmax_bwd(g [..., N], kept) -> dx like g; the kept entries' row length is the caller's to check
PyObject* softmax_bwd(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ARGS(2);
  const Tensor* g = bf16(a[0]);
  int64_t M, N;
  Sparse sp;
  if (!g || !rows_of(*g, &M, &N) || M == 0 || !sp.init(a[1]) || sp.rows() != M) return none();
  Tensor dx;
  OR_NONE(unlocked([&] {
    dx = at::empty(g->sizes(), g->options());
    return hyc_softmax_bwd(g->data_ptr(), M, N, (const int32_t*)sp.row_ptr.data_ptr(), (const int32_t*)sp.cols.data_ptr(), sp.vals.data_ptr(),
                           dx.data_ptr(), stream());
  }));
  return THPVariable_Wrap(dx);
  END_HANDLE_TH_ERRORS
}

// ---- weight gradient, linear layer -------------------------------------------------------------------------------
// dW [N, H] = dy^T x_hat from rows of dy `pitch` apart; staged: through a restored x_hat
bool weight_grad(const void* dy, int64_t pitch, int64_t M, int64_t N, const Tensor& like, Saved& in, bool f32, bool staged, Tensor* out) {
  if (!(staged ? in.make_dense() : in.ready())) return false;
  *out = empty_like_on(like, {N, in.H}, f32 ? at::kFloat : BF16);
  const int64_t bytes = hyc_gradw_workspace_bytes(M, N, in.H);
  Tensor ws;
  if (bytes) ws = empty_like_on(like, {bytes / 4}, at::kFloat);
  return hyc_gradw_gemm(dy, M > 1 ? pitch : N, in.codes(), in.values(), in.group_scales(), M, N, in.H, &in.d, 1.f, 0.f, out->data_ptr(),
                        f32 ? HYC_DTYPE_F32 : HYC_DTYPE_BF16, bytes ? ws.data_ptr() : nullptr, stream()) == 0;
}
// gradw(dy [M, N], c, fp32, staged) -> dW [N, H]
PyObject* gradw(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ARGS(4);
  const Tensor* dy = bf16(a[0]);
  int64_t M, N, pitch;
  Tensor out;
  In in;
  const bool f32 = a[2] == Py_True, staged = a[3] == Py_True;
  if (!dy || dy->dim() != 2 || !spaced_rows(*dy, &M, &N, &pitch) || !in.init(a[1]) || in.M != M ||
      !unlocked([&] { return weight_grad(dy->data_ptr(), pitch, M, N, *dy, in, f32, staged, &out); }))
    return none();
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}
// sizes of x with another last one
std::vector<int64_t> with_last(const Tensor& x, int64_t n) {
  std::vector<int64_t> s = x.sizes().vec();
  s.back() = n;
  return s;
}
// a weight and rows that the kernels for few output features read as they lie, and a result in bf16
bool thin(const Tensor& rows, const Tensor& w, int64_t M, bool input_grad) {
  return hyc_thin_covers(M, w.size(1), w.size(0), input_grad) && aligned16(rows.data_ptr()) && aligned16(w.data_ptr()) && w.is_contiguous() &&
         rows.device() == w.device() && rows.device().index() == c10::hip::current_device() &&
         (!at::autocast::is_autocast_enabled(at::kCUDA) || at::autocast::get_autocast_dtype(at::kCUDA) == BF16);
}
// y = x w^T, into rows of its own shape (`view`: the library's result seen as that, or an alias of it that no view is tracked for)
int linear_forward(const Tensor& x, const Tensor& w, int64_t M, int64_t K, bool view, Tensor* y) {
  const auto sizes = with_last(x, w.size(0));
  if (!thin(x, w, M, false)) {
    *y = at::mm(x.view({M, K}), w.t());
    *y = view ? y->view(sizes) : at::_unsafe_view(*y, sizes);
    return 0;
  }
  *y = at::empty(sizes, x.options());
  const void* factor = w.data_ptr();
  return hyc_lora_down(x.data_ptr(), K, M, K, &factor, 1, (int32_t)w.size(0), y->data_ptr(), stream());
}
bool linear_operands(const Tensor* x, const Tensor* w, int64_t* M, int64_t* K) {
  return x && w && x->dim() >= 2 && w->dim() == 2 && x->numel() && rows_of(*x, M, K) && w->size(1) == *K;
}
// linear_fwd(x [..., K], w [N, K], plan or None, bits, group) -> (x w^T, ChannelCompressed or None)
PyObject* linear_fwd(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ARGS(5);
  const Tensor *x = bf16(a[0]), *w = bf16(a[1]);
  int64_t M, K;
  if (!linear_operands(x, w, &M, &K)) return none();
  PyObject* c = Py_None;
  if (a[2] == Py_None) Py_INCREF(c);
  else if (!(c = compress_rows(*x, a[2], a[3], a[4]))) return none_if_plain(nullptr);
  Ref hold(c);
  Tensor y;
  OR_NONE(unlocked([&] { return linear_forward(*x, *w, M, K, true, &y); }));
  Py_INCREF(c);
  return tuple2(THPVariable_Wrap(y), c);
  END_HANDLE_TH_ERRORS
}
int linear_backward(const Tensor& g, const Tensor& w, int64_t M, int64_t N, Saved* in, bool need_x, bool staged, Tensor* dx, Tensor* dw) {
  if (in && !weight_grad(g.data_ptr(), N, M, N, g, *in, false, staged, dw)) return -1;
  if (need_x && thin(g, w, M, true)) {
    *dx = at::empty(with_last(g, w.size(1)), g.options());
    return hyc_thin_dx(g.data_ptr(), N, M, w.data_ptr(), (int32_t)N, w.size(1), dx->data_ptr(), stream());
  }
  if (need_x) *dx = at::mm(g.view({M, N}), w).view(with_last(g, w.size(1)));
  return 0;
}
// linear_bwd(g [..., N], w [N, K], c or None, need_x, staged) -> (g w or None, dW bf16 or None)
PyObject* linear_bwd(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ARGS(5);
  const Tensor *g = bf16(a[0]), *w = bf16(a[1]);
  int64_t M, N;
  if (!g || !w || g->dim() < 2 || w->dim() != 2 || g->numel() == 0 || !rows_of(*g, &M, &N) || w->size(0) != N || c10::GradMode::is_enabled())
    return none();
  Tensor dw, dx;
  In in;
  const bool need_w = a[2] != Py_None, need_x = a[3] == Py_True, staged = a[4] == Py_True;
  if (need_w && (!in.init(a[2]) || in.M != M)) return none();
  OR_NONE(unlocked([&] { return linear_backward(*g, *w, M, N, need_w ? &in : nullptr, need_x, staged, &dx, &dw); }));
  return tuple2(wrap_or_none(dx), wrap_or_none(dw));
  END_HANDLE_TH_ERRORS
}

// ---- activations ---------------------------------------------------------------------------------------------------
struct ActOut {
  const Tensor* x;
  Out o;
  Tensor y;
  int32_t code;
  bool init(PyObject* const* a) {                                      // (code, x [..., H], plan, bits, group)
    int64_t M, H;
    x = bf16(a[1]);
    if (!x || !rows_of(*x, &M, &H) || !o.init(a[2], a[3], a[4], M, H, x->device())) return false;
    code = (int32_t)PyLong_AsLong(a[0]);
    return !PyErr_Occurred();
  }
  int launch() {
    o.alloc();
    y = at::empty(x->sizes(), x->options());
    return hyc_act_fwd_compress(code, x->data_ptr(), o.H, o.M, o.H, &o.d, y.data_ptr(), o.stored.data_ptr(), o.vals.data_ptr(), o.scales.data_ptr(),
                                stream());
  }
};
// act_fwd(code, x [..., H], plan, bits, group) -> (y like x, ChannelCompressed)
PyObject* act_fwd(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ARGS(5);
  ActOut f;
  if (!f.init(a)) return none_if_plain(nullptr);
  OR_NONE(unlocked([&] { return f.launch(); }));
  return tuple2(THPVariable_Wrap(f.y), f.o.wrap());
  END_HANDLE_TH_ERRORS
}
int act_backward(int32_t code, const Tensor& g, Saved& in, Tensor* dx) {
  if (!in.ready()) return -1;
  *dx = at::empty(g.sizes(), g.options());
  return hyc_act_bwd(code, g.data_ptr(), in.codes(), in.values(), in.group_scales(), in.M, in.H, &in.d, dx->data_ptr(), stream());
}
// act_bwd(code, g [..., H], c) -> dx like g
PyObject* act_bwd(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ARGS(3);
  const Tensor* g = bf16(a[1]);
  int64_t M, H;
  In in;
  if (!g || !rows_of(*g, &M, &H) || !in.init(a[2]) || in.M != M || in.H != H) return none();
  const int32_t code = (int32_t)PyLong_AsLong(a[0]);
  Tensor dx;
  OR_NONE(unlocked([&] { return act_backward(code, *g, in, &dx); }));
  return THPVariable_Wrap(dx);
  END_HANDLE_TH_ERRORS
}
struct GatedOut {
  const Tensor *gate, *up;
  Out o[3];
  Tensor h;
  int32_t code;
  int64_t pg, pu;
  bool init(PyObject* const* a) {                                      // (code, gate [..., H], up, plan_act, plan_up, plan_gate, bits, group)
    int64_t M, H, M2, H2;
    gate = bf16(a[1]);
    up = bf16(a[2]);
    if (!gate || !up || gate->sizes() != up->sizes() || !spaced_rows(*gate, &M, &H, &pg) || !spaced_rows(*up, &M2, &H2, &pu)) return false;
    for (int i = 0; i < 3; ++i)
      if (!o[i].init(a[3 + i], a[6], a[7], M, H, gate->device())) return false;
    code = (int32_t)PyLong_AsLong(a[0]);
    return !PyErr_Occurred();
  }
  int launch() {
    for (Out& out : o) out.alloc();
    h = at::empty(gate->sizes(), gate->options());
    return hyc_gated_act_fwd(code, gate->data_ptr(), pg, up->data_ptr(), pu, o[0].M, o[0].H, &o[0].d, &o[1].d, &o[2].d, h.data_ptr(),
                             o[0].stored.data_ptr(), o[0].vals.data_ptr(), o[0].scales.data_ptr(), o[1].stored.data_ptr(), o[1].vals.data_ptr(),
                             o[1].scales.data_ptr(), o[2].stored.data_ptr(), o[2].vals.data_ptr(), o[2].scales.data_ptr(), stream());
  }
};
// gated_fwd(code, gate [..., H], up, plan_act, plan_up, plan_gate, bits, group) -> (h [..., H], (c_act, c_up, c_gate))
PyObject* gated_fwd(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ARGS(8);
  GatedOut f;
  if (!f.init(a)) return none_if_plain(nullptr);
  OR_NONE(unlocked([&] { return f.launch(); }));
  PyObject* cs = PyTuple_New(3);
  for (int i = 0; i < 3; ++i) {
    PyObject* c = f.o[i].wrap();
    if (!c) { Py_DECREF(cs); return nullptr; }
    PyTuple_SET_ITEM(cs, i, c);
  }
  return tuple2(THPVariable_Wrap(f.h), cs);
  END_HANDLE_TH_ERRORS
}
// `n` matrices of [lead..., H] side by side in one [M, n H + room], or on their own (room < 0)
void side_by_side(const Tensor& like, int64_t n, int64_t M, int64_t H, int64_t room, Tensor* both, std::vector<Tensor>* parts, int64_t* pitch) {
  if (room < 0) {
    for (int64_t i = 0; i < n; ++i) parts->push_back(at::empty(with_last(like, H), like.options()));
    *pitch = H;
    return;
  }
  *pitch = n * H + room;
  *both = empty_like_on(like, {M, *pitch}, BF16);
  const auto lead = like.sizes().slice(0, like.dim() - 1);
  for (int64_t i = 0; i < n; ++i) parts->push_back(both->narrow(1, i * H, H).unflatten(0, lead));
}
PyObject* wrap_parts(const std::vector<Tensor>& parts, const Tensor& both) {
  PyObject* t = PyTuple_New((Py_ssize_t)parts.size() + 1);
  for (size_t i = 0; i < parts.size(); ++i) PyTuple_SET_ITEM(t, (Py_ssize_t)i, THPVariable_Wrap(parts[i]));
  PyTuple_SET_ITEM(t, (Py_ssize_t)parts.size(), both.defined() ? THPVariable_Wrap(both) : none());
  return t;
}
int64_t room_of(PyObject* o) { return o == Py_None ? -1 : PyLong_AsLongLong(o); }
template <class S>
int gated_backward(int32_t code, const Tensor& g, const S* in, int64_t room, Tensor* both, std::vector<Tensor>* d) {
  int64_t pitch;
  side_by_side(g, 2, in[0].M, in[0].H, room, both, d, &pitch);
  return hyc_gated_act_bwd_rows(code, g.data_ptr(), in[0].codes(), in[0].values(), in[0].group_scales(), &in[0].d, in[1].codes(), in[1].values(),
                                in[1].group_scales(), &in[1].d, in[2].codes(), in[2].values(), in[2].group_scales(), &in[2].d, in[0].M, in[0].H,
                                (*d)[0].data_ptr(), pitch, (*d)[1].data_ptr(), pitch, stream());
}
// gated_bwd(code, g [..., H], c_act, c_up, c_gate, room or None) -> (d_gate, d_up, their common matrix or None)
PyObject* gated_bwd(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ARGS(6);
  const Tensor* g = bf16(a[1]);
  int64_t M, H;
  In in[3];
  if (!g || g->dim() < 2 || !rows_of(*g, &M, &H)) return none();
  for (int i = 0; i < 3; ++i)
    if (!in[i].init(a[2 + i]) || in[i].M != M || in[i].H != H || in[i].restore_first) return none();
  const int32_t code = (int32_t)PyLong_AsLong(a[0]);
  const int64_t room = room_of(a[5]);
  Tensor both;
  std::vector<Tensor> d;
  OR_NONE(unlocked([&] { return gated_backward(code, *g, in, room, &both, &d); }));
  return wrap_parts(d, both);
  END_HANDLE_TH_ERRORS
}

// ---- LoRA groups -------------------------------------------------------------------------------------------------------
struct Factors {                                                       // a group's A (or B): bf16 [rows_i, cols_i], as the kernels read them
  int n = 0;
  const void* p[4];
  std::vector<const Tensor*> t;
  bool init(PyObject* seq, const Tensor& like) {
    if (!PyTuple_CheckExact(seq) || PyTuple_GET_SIZE(seq) < 1 || PyTuple_GET_SIZE(seq) > 4) return false;
    n = (int)PyTuple_GET_SIZE(seq);
    for (int i = 0; i < n; ++i) {
      const Tensor* f = bf16(PyTuple_GET_ITEM(seq, i));
      if (!f || f->dim() != 2 || !f->is_contiguous() || !aligned16(f->data_ptr()) || f->device() != like.device()) return false;
      p[i] = f->data_ptr();
      t.push_back(f);
    }
    return true;
  }
  bool shaped(int i, int64_t rows, int64_t cols) const { return t[i]->size(0) == rows && t[i]->size(1) == cols; }
};
bool widths(PyObject* seq, int n, int64_t* outs, int64_t* total) {
  if (!PyTuple_CheckExact(seq) || PyTuple_GET_SIZE(seq) != n) return false;
  *total = 0;
  for (int i = 0; i < n; ++i) {
    outs[i] = PyLong_AsLongLong(PyTuple_GET_ITEM(seq, i));
    if (outs[i] <= 0 || outs[i] % 8) return false;
    *total += outs[i];
  }
  return true;
}
bool base_weight(PyObject* packed, PyObject* absmax, const Tensor& like, int64_t n, const Tensor** p, const Tensor** m) {
  *p = plain(packed);
  *m = plain(absmax);
  return *p && *m && (*p)->scalar_type() == at::kByte && (*m)->scalar_type() == at::kFloat && (*p)->is_contiguous() && (*m)->is_contiguous() &&
         (*p)->numel() * 2 == n && (*m)->numel() * 64 == n && (*p)->device() == like.device() && (*m)->device() == like.device();
}
// out [M, N] = a b^T in one product, or in two at column `cut`
void product(const Tensor& out, const Tensor& a, const Tensor& b, int64_t cut) {
  const int64_t N = out.size(1), lo[2] = {0, cut}, hi[2] = {cut ? cut : N, N};
  for (int i = 0; i < (cut ? 2 : 1); ++i) {
    Tensor part = out.narrow(1, lo[i], hi[i] - lo[i]);
    at::mm_out(part, a, b.narrow(0, lo[i], hi[i] - lo[i]).t());
  }
}
// decoder_layer._parts of an [M, N] result: ranges of columns and rows
struct Part { int64_t c0, c1, r0, r1; };
bool parts_of(PyObject* seq, int64_t M, int64_t N, std::vector<Part>* out) {
  if (!PyTuple_CheckExact(seq)) return false;
  int64_t covered = 0;
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(seq); ++i) {
    PyObject* t = PyTuple_GET_ITEM(seq, i);
    if (!PyTuple_CheckExact(t) || PyTuple_GET_SIZE(t) != 4) return false;
    int64_t v[4];
    for (int j = 0; j < 4; ++j) v[j] = PyLong_AsLongLong(PyTuple_GET_ITEM(t, j));
    if (PyErr_Occurred()) { PyErr_Clear(); return false; }
    const Part p{v[0], v[1], v[2], v[3]};
    if (p.c0 < 0 || p.c0 >= p.c1 || p.c1 > N || p.r0 < 0 || p.r0 >= p.r1 || p.r1 > M) return false;
    covered += (p.c1 - p.c0) * (p.r1 - p.r0);
    out->push_back(p);
  }
  return covered == M * N;
}
// out += a b^T, part by part
void accumulate(const Tensor& out, const Tensor& a, const Tensor& b, const std::vector<Part>& parts) {
  for (const Part& p : parts)
    out.narrow(0, p.r0, p.r1 - p.r0).narrow(1, p.c0, p.c1 - p.c0).addmm_(a.narrow(0, p.r0, p.r1 - p.r0), b.narrow(0, p.c0, p.c1 - p.c0).t());
}
// lora_forward(x [..., K], (A_i), (B_i), scale, (out_i), packed, absmax, parts, plan or None, bits, group)
//   -> ((y_i [..., out_i]), h [M, n r], ChannelCompressed of x or None); the kernels' ranks and sizes are the caller's to check
PyObject* lora_forward(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ARGS(11);
  const Tensor *x = bf16(a[0]), *packed, *absmax;
  int64_t M, K, outs[4], total;
  Factors A, B;
  std::vector<Part> parts;
  if (!x || x->dim() < 2 || x->numel() == 0 || !rows_of(*x, &M, &K) || !aligned16(x->data_ptr()) || !A.init(a[1], *x) || !B.init(a[2], *x) || A.n != B.n ||
      !widths(a[4], A.n, outs, &total) || !base_weight(a[5], a[6], *x, total * K, &packed, &absmax) || !parts_of(a[7], M, total, &parts) ||
      c10::GradMode::is_enabled())
    return none();
  const int64_t r = A.t[0]->size(0);
  for (int i = 0; i < A.n; ++i)
    if (!A.shaped(i, r, K) || !B.shaped(i, outs[i], r)) return none();
  const double scale = PyFloat_AsDouble(a[3]);
  if (PyErr_Occurred()) return nullptr;
  Out o;
  const bool keep = a[8] != Py_None;
  if (keep && !o.init(a[8], a[9], a[10], M, K, x->device())) return none();
  bool few = hyc_few_rows_covers(M, K, total, 0);                      // kernels.few_rows_base
  for (int i = 0; i < A.n; ++i) few = few && outs[i] % 16 == 0;
  few = few && aligned16(packed->data_ptr()) && aligned16(absmax->data_ptr());
  Tensor x2, h, y;
  OR_NONE(unlocked([&] {
    x2 = x->view({M, K});
    h = empty_like_on(*x, {M, A.n * r}, BF16);
    y = empty_like_on(*x, {M, total}, BF16);
    int rc = hyc_lora_down(x->data_ptr(), K, M, K, A.p, A.n, (int32_t)r, h.data_ptr(), stream());
    if (!rc && few)
      rc = hyc_few_rows_nf4(x->data_ptr(), K, M, K, packed->data_ptr(), (const float*)absmax->data_ptr(), h.data_ptr(), B.p, outs, B.n, (int32_t)r,
                            (float)scale, y.data_ptr(), stream());
    else if (!rc)
      rc = hyc_lora_up(h.data_ptr(), M, B.p, outs, B.n, (int32_t)r, (float)scale, y.data_ptr(), stream());
    if (!rc && !few) {                                                 // (the weight's room is free again for the codes)
      const Tensor w = empty_like_on(*x, {total, K}, BF16);
      rc = hyc_nf4_dequantize(packed->data_ptr(), (const float*)absmax->data_ptr(), total * K, w.data_ptr(), stream());
      if (!rc) accumulate(y, x2, w, parts);
    }
    if (rc || !keep) return rc;
    o.alloc();
    return hyc_compress_rows(x->data_ptr(), K, M, K, &o.d, o.stored.data_ptr(), o.vals.data_ptr(), o.scales.data_ptr(), nullptr, stream());
  }));
  PyObject* c = keep ? o.wrap() : none();
  if (!c) return nullptr;
  const auto lead = x->sizes().slice(0, x->dim() - 1);
  PyObject* ys = PyTuple_New(A.n);
  int64_t col = 0;
  for (int i = 0; i < A.n; ++i) {
    PyTuple_SET_ITEM(ys, i, THPVariable_Wrap(y.narrow(1, col, outs[i]).unflatten(0, lead)));
    col += outs[i];
  }
  PyObject* t = PyTuple_New(3);
  PyTuple_SET_ITEM(t, 0, ys);
  PyTuple_SET_ITEM(t, 1, THPVariable_Wrap(h));
  PyTuple_SET_ITEM(t, 2, c);
  return t;
  END_HANDLE_TH_ERRORS
}
// lora_backward((g_i [..., out_i]), (A_i), (B_i), h, scale, (out_i), room, rows or None, packed, absmax, c, cut)
//   -> (dx [..., K], dA_0, ..., dB_0, ...); rows: the [M, total + room] matrix whose first columns the g_i are
PyObject* lora_backward(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ARGS(12);
  const Tensor *h = bf16(a[3]), *packed, *absmax;
  Factors A, B;
  int64_t outs[4], total, M = -1, pitches[4];
  if (!h || !h->is_contiguous() || h->dim() != 2 || !A.init(a[1], *h) || !B.init(a[2], *h) || A.n != B.n || !widths(a[5], A.n, outs, &total) ||
      !PyTuple_CheckExact(a[0]) || PyTuple_GET_SIZE(a[0]) != A.n || c10::GradMode::is_enabled())
    return none();
  const int n = A.n;
  const int64_t r = A.t[0]->size(0), K = A.t[0]->size(1), room = PyLong_AsLongLong(a[6]), cut = PyLong_AsLongLong(a[11]);
  const double scale = PyFloat_AsDouble(a[4]);
  if (PyErr_Occurred()) return nullptr;
  const void* dy[4];
  const Tensor* g0 = nullptr;
  for (int i = 0; i < n; ++i) {
    const Tensor* g = bf16(PyTuple_GET_ITEM(a[0], i));
    int64_t m, w;
    if (!g || g->device() != h->device() || !kernel_rows(*g, &m, &w, &pitches[i]) || w != outs[i] || (M >= 0 && m != M) || !A.shaped(i, r, K) ||
        !B.shaped(i, outs[i], r))
      return none();
    M = m;
    dy[i] = g->data_ptr();
    if (!i) g0 = g;
    const int64_t range = (M < 32768 ? M : 32768) + 63;                // kernels._lora_range_fits
    if (range / 64 * 64 * pitches[i] >= ((int64_t)1 << 30)) return none();
  }
  if (h->size(0) != M || h->size(1) != n * r || room < n * r || !base_weight(a[8], a[9], *h, total * K, &packed, &absmax)) return none();
  Tensor ext;
  const bool copy = a[7] == Py_None;
  if (!copy) {
    const Tensor* e = bf16(a[7]);
    if (!e || !e->is_contiguous() || e->dim() != 2 || e->size(0) != M || e->size(1) != total + room || e->device() != h->device()) return none();
    ext = *e;
  }
  In in;
  if (!in.init(a[10]) || in.M != M || in.H != K || in.restore_first) return none();
  std::vector<Tensor> dA, dB;
  Tensor dx;
  OR_NONE(unlocked([&] {
    if (copy) ext = empty_like_on(*h, {M, total + room}, BF16);
    const Tensor dh = empty_like_on(*h, {M, n * r}, BF16);
    void* pB[4];
    for (int i = 0; i < n; ++i) {
      dB.push_back(at::empty(B.t[i]->sizes(), B.t[i]->options()));
      pB[i] = dB[i].data_ptr();
    }
    int rc;
    {                                                                  // (the workspace's room is free again for the weight)
      const Tensor ws = empty_like_on(*h, {hyc_lora_up_bwd_workspace_bytes(M, outs, n, (int32_t)r) / 4}, at::kFloat);
      rc = hyc_lora_up_bwd(dy, pitches, M, outs, B.p, h->data_ptr(), n, (int32_t)r, (float)scale, dh.data_ptr(), ext.data_ptr(), total + room, room,
                           copy ? 1 : 0, pB, ws.data_ptr(), stream());
    }
    if (rc) return rc;
    // the dh of a group go through the weight gradient side by side, in as few calls as leave its sums in one order
    const int64_t per_call = hyc_gradw_rows_per_call(M, n * r, r, K, &in.d);
    for (int64_t c0 = 0; c0 < n * r; c0 += per_call) {
      const int64_t cols = c0 + per_call <= n * r ? per_call : n * r - c0;
      Tensor block;
      if (!weight_grad((const char*)dh.data_ptr() + 2 * c0, n * r, M, cols, dh, in, false, false, &block)) return -1;
      for (int64_t j = 0; j < cols; j += r) dA.push_back(block.narrow(0, j, r));
    }
    const Tensor wt = empty_like_on(*h, {K, total + room}, BF16);
    dx = empty_like_on(*h, {M, K}, BF16);
    rc = hyc_lora_weight_t(packed->data_ptr(), (const float*)absmax->data_ptr(), K, A.p, outs, n, (int32_t)r, room, wt.data_ptr(), stream());
    if (!rc && hyc_few_rows_covers(M, total + room, K, 1))
      rc = hyc_few_rows(ext.data_ptr(), total + room, M, total + room, wt.data_ptr(), K, dx.data_ptr(), stream());
    else if (!rc)
      product(dx, ext, wt, cut);
    return rc;
  }));
  PyObject* t = PyTuple_New(1 + 2 * n);
  PyTuple_SET_ITEM(t, 0, THPVariable_Wrap(dx.view(with_last(*g0, K))));
  for (int i = 0; i < n; ++i) {
    PyTuple_SET_ITEM(t, 1 + i, THPVariable_Wrap(dA[i]));
    PyTuple_SET_ITEM(t, 1 + n + i, THPVariable_Wrap(dB[i]));
  }
  return t;
  END_HANDLE_TH_ERRORS
}

// ---- attention -----------------------------------------------------------------------------------------------------------
struct Tokens {                                                        // bf16 [B, S, H], contiguous channels, evenly spaced tokens
  const Tensor* t;
  int64_t B, S, H, pitch;
  bool init(PyObject* o) {
    t = bf16(o);
    if (!t || t->dim() != 3 || t->numel() == 0 || t->stride(2) != 1) return false;
    B = t->size(0); S = t->size(1); H = t->size(2);
    pitch = S > 1 ? t->stride(1) : (B > 1 ? t->stride(0) : H);
    return B == 1 || t->stride(0) == S * pitch;
  }
  bool same(const Tokens& o) const { return B == o.B && S == o.S && H == o.H; }
};
bool tables(PyObject* cosv, PyObject* sinv, int64_t n, const Tensor** c, const Tensor** s) {
  *c = bf16(cosv);
  *s = bf16(sinv);
  return *c && *s && (*c)->is_contiguous() && (*s)->is_contiguous() && (*c)->numel() == n && (*s)->numel() == n;
}
// rope_attn_fwd(q, k, v, heads, cos, sin, scale, round_scores, plans of q, k, v (and out) or None, bits, group)
//   -> (q rows, k rows, out, lse, their ChannelCompressed or None): q and k rotated, attention on them, and with plans the codes
PyObject* rope_attn_fwd(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ARGS(11);
  Tokens t[3], &q = t[0], &v = t[2];
  const Tensor *cosv, *sinv;
  const int64_t heads = PyLong_AsLongLong(a[3]);
  const double scale = PyFloat_AsDouble(a[6]);
  if (PyErr_Occurred()) return nullptr;
  for (int i = 0; i < 3; ++i)
    if (!t[i].init(a[i]) || !q.same(t[i])) return none();
  if (heads <= 0 || q.H % heads || !tables(a[4], a[5], q.S * (q.H / heads), &cosv, &sinv)) return none();
  const int64_t hd = q.H / heads, M = q.B * q.S;
  const bool round_scores = a[7] == Py_True;
  Out o[4];
  const int sites = a[8] != Py_None && PyTuple_CheckExact(a[8]) ? (int)PyTuple_GET_SIZE(a[8]) : 0;
  if (a[8] != Py_None && sites != 3 && sites != 4) return none();
  for (int i = 0; i < sites; ++i)
    if (!o[i].init(PyTuple_GET_ITEM(a[8], i), a[9], a[10], M, q.H, q.t->device())) return none();
  Tensor rows[2], out, lse;
  OR_NONE(unlocked([&] {
    const auto opt = q.t->options();
    for (Tensor& r : rows) r = at::empty({q.B, q.S, q.H}, opt);
    const void* x[3] = {q.t->data_ptr(), t[1].t->data_ptr(), v.t->data_ptr()};
    const int64_t ldx[3] = {q.pitch, t[1].pitch, v.pitch};
    int rc = HYC_ENOTSUP;
    if (sites) {
      void *rp[3] = {rows[0].data_ptr(), rows[1].data_ptr(), nullptr}, *st[3], *va[3], *sc[3];
      hyc_desc d[3];
      for (int i = 0; i < 3; ++i) {
        o[i].alloc();
        st[i] = o[i].stored.data_ptr(); va[i] = o[i].vals.data_ptr(); sc[i] = o[i].scales.data_ptr(); d[i] = o[i].d;
      }
      rc = hyc_attn_sites_fwd(x, ldx, cosv->data_ptr(), sinv->data_ptr(), q.B, q.S, heads, hd, d, rp, st, va, sc, stream());
    }
    const bool one_by_one = rc == HYC_ENOTSUP;
    auto compress_site = [&](int i, const void* xi, int64_t ld) {
      return hyc_compress_rows(xi, ld, M, q.H, &o[i].d, o[i].stored.data_ptr(), o[i].vals.data_ptr(), o[i].scales.data_ptr(), nullptr, stream());
    };
    if (one_by_one) {
      rc = 0;
      for (int i = 0; i < 2 && !rc; ++i)
        rc = hyc_rope_to_heads(x[i], ldx[i], cosv->data_ptr(), sinv->data_ptr(), q.B, q.S, heads, hd, nullptr, rows[i].data_ptr(), stream());
      for (int i = 0; i < 3 && sites && !rc; ++i) rc = i < 2 ? compress_site(i, rows[i].data_ptr(), q.H) : compress_site(i, x[2], ldx[2]);
    }
    if (rc) return rc;
    out = at::empty({q.B, q.S, q.H}, opt);
    lse = empty_like_on(*q.t, {q.B, heads, q.S}, at::kFloat);
    rc = (round_scores ? hyc_attn_kept_fwd : hyc_attn_fwd)(rows[0].data_ptr(), q.H, rows[1].data_ptr(), q.H, v.t->data_ptr(), v.pitch, q.B, q.S, heads, hd,
                                                           (float)scale, out.data_ptr(), q.H, (float*)lse.data_ptr(), stream());
    if (rc || sites < 4) return rc;
    o[3].alloc();
    return compress_site(3, out.data_ptr(), q.H);
  }));
  PyObject* saved = sites ? PyTuple_New(sites) : none();
  for (int i = 0; i < sites; ++i) {
    PyObject* c = o[i].wrap();
    if (!c) { Py_DECREF(saved); return nullptr; }
    PyTuple_SET_ITEM(saved, i, c);
  }
  PyObject* r = PyTuple_New(5);
  PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(rows[0]));
  PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(rows[1]));
  PyTuple_SET_ITEM(r, 2, THPVariable_Wrap(out));
  PyTuple_SET_ITEM(r, 3, THPVariable_Wrap(lse));
  PyTuple_SET_ITEM(r, 4, saved);
  return r;
  END_HANDLE_TH_ERRORS
}
// q, k and v (and the row terms of the backward from the output's codes, with n = 4) out of their codes, in one launch where
// hyc_attn_sites_bwd covers them: HYC_ENOTSUP where not, before anything is launched
int restore_sites(In* in, int n, const Tokens& g, int64_t heads, const Tensor* lse, double scale, Tensor* x, Tensor* ws) {
  for (int i = 0; i < n; ++i)
    if (in[i].restore_first) return HYC_ENOTSUP;
  const void *st[4], *va[4], *sc[4];
  void* to[4] = {};
  hyc_desc d[4];
  for (int i = 0; i < n; ++i) {
    st[i] = in[i].codes(); va[i] = in[i].values(); sc[i] = in[i].group_scales(); d[i] = in[i].d;
    if (i >= 3) continue;
    x[i] = empty_like_on(in[i].stored, {in[i].M, in[i].H}, BF16);
    to[i] = x[i].data_ptr();
  }
  if (n == 4) *ws = empty_like_on(*g.t, {2 * g.B * heads * g.S}, at::kFloat);
  return hyc_attn_sites_bwd(st, va, sc, d, n, g.B, g.S, heads, g.H / heads, to, n == 4 ? g.t->data_ptr() : nullptr, g.H,
                            n == 4 ? (const float*)lse->data_ptr() : nullptr, (float)scale, n == 4 ? (float*)ws->data_ptr() : nullptr, stream());
}
// attn_bwd(g [B, S, H], [c_q, c_k, c_v, c_out], lse, heads, cos, sin, scale, room or None) -> (dq, dk, dv, their common matrix or None).
// The list is the call's to empty: once the four are restored their codes go, and the gradients take that room.
PyObject* attn_bwd(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ARGS(8);
  Tokens g;
  const Tensor *cosv, *sinv, *lse = plain(a[2]);
  const int64_t heads = PyLong_AsLongLong(a[3]);
  const double scale = PyFloat_AsDouble(a[6]);
  if (PyErr_Occurred()) return nullptr;
  if (!g.init(a[0]) || !g.t->is_contiguous() || !aligned16(g.t->data_ptr()) || heads <= 0 || g.H % heads ||
      !tables(a[4], a[5], g.S * (g.H / heads), &cosv, &sinv) || !aligned16(cosv->data_ptr()) || !aligned16(sinv->data_ptr()) || !lse ||
      lse->scalar_type() != at::kFloat || !lse->is_contiguous() || lse->numel() != g.B * heads * g.S || !PyList_CheckExact(a[1]) ||
      PyList_GET_SIZE(a[1]) != 4)
    return none();
  const int64_t room = room_of(a[7]);
  Tensor x[4], ws;
  bool terms = false;                                                  // the output went into the row terms, not into x[3]
  {
    In in[4];
    for (int i = 0; i < 4; ++i)
      if (!in[i].init(PyList_GET_ITEM(a[1], i)) || in[i].M != g.B * g.S || in[i].H != g.H) return none();
    if (!unlocked([&] {
          const int rc = restore_sites(in, 4, g, heads, lse, scale, x, &ws);
          terms = rc == 0;
          if (rc != HYC_ENOTSUP) return terms;
          for (int i = 0; i < 4; ++i)
            if (!in[i].restore(&x[i])) return false;
          return true;
        }))
      return none();
  }
  if (PyList_SetSlice(a[1], 0, 4, nullptr) != 0) return nullptr;
  Tensor both;
  std::vector<Tensor> d;
  const int rc = unlocked([&] {
    int64_t pitch;
    if (!terms) ws = empty_like_on(*g.t, {2 * g.B * heads * g.S}, at::kFloat);
    side_by_side(*g.t, 3, g.B * g.S, g.H, room, &both, &d, &pitch);
    if (terms)
      return hyc_attn_bwd_terms(g.t->data_ptr(), g.H, x[0].data_ptr(), g.H, x[1].data_ptr(), g.H, x[2].data_ptr(), g.H, cosv->data_ptr(),
                                sinv->data_ptr(), g.B, g.S, heads, g.H / heads, (float)scale, d[0].data_ptr(), pitch, d[1].data_ptr(), pitch,
                                d[2].data_ptr(), pitch, (float*)ws.data_ptr(), stream());
    return hyc_attn_bwd(g.t->data_ptr(), g.H, x[0].data_ptr(), g.H, x[1].data_ptr(), g.H, x[2].data_ptr(), g.H, x[3].data_ptr(), g.H,
                        (const float*)lse->data_ptr(), cosv->data_ptr(), sinv->data_ptr(), g.B, g.S, heads, g.H / heads, (float)scale, d[0].data_ptr(),
                        pitch, d[1].data_ptr(), pitch, d[2].data_ptr(), pitch, (float*)ws.data_ptr(), stream());
  });
  if (rc != 0) { PyErr_SetString(PyExc_RuntimeError, hyc_last_error()); return nullptr; }    // (no interpreted form to go on with)
  return wrap_parts(d, both);
  END_HANDLE_TH_ERRORS
}

// attn_kept(q rows [B, S, H], k rows, lse, heads, scale, threshold, slab entries per row, cap, first, matrices)
//   -> (row_ptr, cols, vals, total) of kernels.attn_kept
PyObject* attn_kept(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ARGS(10);
  Tokens q, k;
  const Tensor* lse = plain(a[2]);
  const int64_t heads = PyLong_AsLongLong(a[3]), slab_cap = PyLong_AsLongLong(a[6]), cap = PyLong_AsLongLong(a[7]), first = PyLong_AsLongLong(a[8]),
                matrices = PyLong_AsLongLong(a[9]);
  const double scale = PyFloat_AsDouble(a[4]), thr = PyFloat_AsDouble(a[5]);
  if (PyErr_Occurred()) return nullptr;
  if (!q.init(a[0]) || !k.init(a[1]) || !q.same(k) || heads <= 0 || q.H % heads || !lse || lse->scalar_type() != at::kFloat || !lse->is_contiguous() ||
      lse->numel() != q.B * heads * q.S || cap <= 0 || slab_cap <= 0 || matrices <= 0)
    return none();
  const int64_t rows = matrices * q.S, hd = q.H / heads;
  Csr csr;
  OR_NONE(unlocked([&]() -> int {
    const Tensor counts = empty_like_on(*q.t, {rows}, at::kInt), slab = empty_like_on(*q.t, {rows, slab_cap}, at::kInt);
    int32_t* n = (int32_t*)counts.data_ptr();
    uint32_t* sl = (uint32_t*)slab.data_ptr();
    const float* ls = (const float*)lse->data_ptr();
    const int rc = hyc_attn_kept(q.t->data_ptr(), q.pitch, k.t->data_ptr(), k.pitch, ls, q.B, q.S, heads, hd, (float)scale, (float)thr, first, matrices, n,
                                 sl, slab_cap, stream());
    if (rc != 0 || !csr.offsets(counts, rows, cap)) return -1;
    return hyc_attn_kept_fill(q.t->data_ptr(), q.pitch, k.t->data_ptr(), k.pitch, ls, q.B, q.S, heads, hd, (float)scale, (float)thr, first, matrices, n,
                              sl, slab_cap, csr.rp(), csr.co(), csr.vals.data_ptr(), stream());
  }));
  return wrap_all({csr.row_ptr, csr.cols, csr.vals, csr.total});
  END_HANDLE_TH_ERRORS
}
// attn_kept_bwd(g [B, S, H], c_q, c_k, c_v, [kept], heads, cos, sin, scale, room or None) -> (dq, dk, dv, their common matrix or None)
PyObject* attn_kept_bwd(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ARGS(10);
  Tokens g;
  const Tensor *cosv, *sinv;
  const int64_t heads = PyLong_AsLongLong(a[5]);
  const double scale = PyFloat_AsDouble(a[8]);
  if (PyErr_Occurred()) return nullptr;
  if (!g.init(a[0]) || !g.t->is_contiguous() || heads <= 0 || g.H % heads || !tables(a[6], a[7], g.S * (g.H / heads), &cosv, &sinv) || !PyList_CheckExact(a[4]))
    return none();
  std::vector<Sparse> kept((size_t)PyList_GET_SIZE(a[4]));
  int64_t rows = 0;
  for (size_t i = 0; i < kept.size(); ++i) {
    if (!kept[i].init(PyList_GET_ITEM(a[4], (Py_ssize_t)i)) || kept[i].rows() % g.S) return none();
    rows += kept[i].rows();
  }
  if (rows != g.B * heads * g.S) return none();
  In in[3];
  for (int i = 0; i < 3; ++i)
    if (!in[i].init(a[1 + i]) || in[i].M != g.B * g.S || in[i].H != g.H) return none();
  const int64_t room = room_of(a[9]);
  Tensor both;
  std::vector<Tensor> d;
  OR_NONE(unlocked([&] {
    Tensor x[3];
    int rc = restore_sites(in, 3, g, heads, nullptr, 0.0, x, nullptr);
    if (rc == HYC_ENOTSUP) {
      rc = 0;
      for (int i = 0; i < 3; ++i)
        if (!in[i].restore(&x[i])) rc = -1;
    }
    if (rc) return rc;
    int64_t pitch, first = 0;
    side_by_side(*g.t, 3, g.B * g.S, g.H, room, &both, &d, &pitch);
    for (const Sparse& sp : kept) {
      const int64_t matrices = sp.rows() / g.S;
      const Tensor records = empty_like_on(*g.t, {sp.cols.numel(), 2}, at::kInt);
      rc = hyc_attn_kept_bwd(g.t->data_ptr(), g.H, x[0].data_ptr(), g.H, x[1].data_ptr(), g.H, x[2].data_ptr(), g.H,
                             (const int32_t*)sp.row_ptr.data_ptr(), (const int32_t*)sp.cols.data_ptr(), sp.vals.data_ptr(), cosv->data_ptr(),
                             sinv->data_ptr(), g.B, g.S, heads, g.H / heads, (float)scale, first, matrices, d[0].data_ptr(), pitch,
                             d[1].data_ptr(), pitch, d[2].data_ptr(), pitch, records.data_ptr(), stream());
      if (rc) return rc;
      first += matrices;
    }
    return 0;
  }));
  return wrap_parts(d, both);
  END_HANDLE_TH_ERRORS
}

// ---- an operator's backward, recorded natively ---------------------------------------------------------------------------
// A short pass is bound by what torch.autograd.Function does around the calls above: the context and its attributes, argument tuples, the
// interpreter's lock in the engine's thread.  The *_node functions run the forward and record one node of this kind instead (us a pass: rms norm of 45 x
// 4096 82 -> 64, layer norm 31 x 117 x 1024 103 -> 81, LoRA-A 4096 x 4096 91 -> 69, the reference's rms norm 133 -> 104).  Like the
// contexts it replaces it keeps its tensors as they are (no saved-tensor hooks, nothing let go after a pass).  It holds no object of the
// interpreter, so that the engine's thread can run it and let go of it without the lock.  What the calls above do not cover, in a pass over it too
// (create_graph, gradients in a batch, of another type or layout), goes through `interpreted`, the Function's own backward as a function of
// (context, gradient), with a context made for it.  Whoever looks at what it keeps (grad_fn.saved and the like) or writes to it has it as a
// Function's context from then on: the same objects each time, and passes that go by them.
struct Lock {                                                          // the interpreter's lock
  PyGILState_STATE state = PyGILState_Ensure();
  ~Lock() { PyGILState_Release(state); }
};
struct Recorded : public torch::autograd::Node {
  enum Kind { NORM, LINEAR, ACT, GATED } kind;
  std::vector<Saved> saved;                                            // one activation; of the gated product act(gate), up and gate
  Tensor w, bias, mean, rstd;
  bool quirk = false, staged = false;
  bool needs[3] = {false, false, false};
  int32_t code = 0;
  std::string act, label;
  PyObject* interpreted = nullptr;                                     // lives as long as the process
  std::atomic<PyObject*> seen{nullptr};                                // a dict, once somebody has looked
  explicit Recorded(Kind k) : kind(k) {}
  ~Recorded() override {
    if (!seen.load() || !Py_IsInitialized()) return;
    Lock lock;
    Py_DECREF(seen.load());
  }
  std::string name() const override { return label; }

  bool native(const Tensor& g, torch::autograd::variable_list& out) const {
    int64_t M, H;
    int dtype;
    if (!dense_gpu(g) || g.scalar_type() != BF16 || g.unsafeGetTensorImpl()->is_python_dispatch() || !rows_of(g, &M, &H)) return false;
    std::vector<Saved> in = saved;                                     // (what is read as a restored matrix becomes one)
    for (Saved& c : in)
      if (M != c.M || (kind != LINEAR && H != c.H) || !c.describe()) return false;
    if (kind == GATED) {
      Tensor both;
      std::vector<Tensor> d;
      if (g.dim() < 2 || gated_backward(code, g, in.data(), -1, &both, &d) != 0) return false;
      out[0] = d[0];
      out[1] = d[1];
      return true;
    }
    if (kind == NORM) {
      if (!dense_gpu(w) || !weight_dtype(w, H, &dtype) || !dense_gpu(rstd) || !row_stats(rstd, M) ||
          (mean.defined() && (!dense_gpu(mean) || !row_stats(mean, M))) || norm_backward(g, in[0], w, dtype, mean, rstd, quirk, &out[0], &out[1])) return false;
      return !bias.defined() || bias_backward(g, M, H, bias.scalar_type() != BF16, &out[2]) == 0;
    }
    if (kind == ACT) return act_backward(code, g, in[0], &out[0]) == 0;
    return g.dim() >= 2 && g.numel() && dense_gpu(w) && w.scalar_type() == BF16 && w.dim() == 2 && w.size(0) == H &&
           linear_backward(g, w, M, H, in.empty() ? nullptr : &in[0], needs[0], staged, &out[0], &out[1]) == 0;
  }
  torch::autograd::variable_list apply(torch::autograd::variable_list&& grads) override {
    torch::autograd::variable_list out(num_outputs());
    if (!c10::GradMode::is_enabled() && !c10::impl::TorchDispatchModeTLS::any_modes_set() && !seen.load() && native(grads[0], out)) return out;
    const Tensor g = grads[0].defined() ? grads[0] : input_metadata(0).zeros_like();
    Lock lock;
    Ref names(seen.load() ? (Py_INCREF(seen.load()), seen.load()) : attributes()), none_(PyTuple_New(0)), ctx(names.p && none_.p ? PyObject_Call(t_namespace, none_.p, names.p) : nullptr),
        dy(ctx.p ? THPVariable_Wrap(g) : nullptr), r(dy.p ? PyObject_CallFunctionObjArgs(interpreted, ctx.p, dy.p, nullptr) : nullptr);
    if (!r.p || !PyTuple_Check(r.p) || PyTuple_GET_SIZE(r.p) < (Py_ssize_t)out.size()) {
      if (r.p) PyErr_SetString(PyExc_RuntimeError, "a backward returned something else than its gradients");
      python_error e;
      e.persist();
      throw e;
    }
    for (size_t i = 0; i < out.size(); ++i) {
      PyObject* d = PyTuple_GET_ITEM(r.p, (Py_ssize_t)i);
      out[i] = d == Py_None ? Tensor() : THPVariable_Unpack(d);
    }
    return out;
  }
  // what the Functions' contexts hold under these names
  PyObject* attributes() const {
    PyObject* c = kind == GATED ? Py_BuildValue("NNN", saved[0].wrap(nullptr), saved[1].wrap(nullptr), saved[2].wrap(nullptr))
                  : saved.empty() ? none() : saved[0].wrap(nullptr);
    if (!c) return nullptr;
    return Py_BuildValue("{s:N,s:N,s:N,s:N,s:N,s:N,s:N,s:d,s:N,s:N,s:O,s:s}", "saved", c, "weight", wrap_or_none(w), "w", wrap_or_none(w), "bias",
                         wrap_or_none(bias), "mean", wrap_or_none(mean), "rstd", wrap_or_none(rstd), "c2_quirk", PyBool_FromLong(quirk), "weight_offset",
                         0.0, "use_bias", PyBool_FromLong(0), "needs_input_grad",
                         Py_BuildValue("NNN", PyBool_FromLong(needs[0]), PyBool_FromLong(needs[1]), PyBool_FromLong(needs[2])), "grad_room", Py_None, "act",
                         act.c_str());
  }
  // them as somebody sees them, for `name` or, to write to, whatever it is; null without an error: there is none of the name
  PyObject* look(PyObject* name, bool write) {
    if (PyObject* d = seen.load()) return d;
    Ref all(attributes());
    if (!all.p) return nullptr;
    if (!write) {
      const int has = PyDict_Contains(all.p, name);
      if (has <= 0) return nullptr;
    }
    Py_INCREF(all.p);
    seen.store(all.p);
    return all.p;
  }
};
Recorded* node_of(PyObject* self) { return dynamic_cast<Recorded*>(reinterpret_cast<torch::autograd::THPCppFunction*>(self)->cdata.get()); }
// grad_fn.saved and the like
PyObject* node_attribute(PyObject* self, PyObject* name) {
  PyObject* v = PyObject_GenericGetAttr(self, name);
  if (v || !PyErr_ExceptionMatches(PyExc_AttributeError)) return v;
  Recorded* node = node_of(self);
  if (!node) return nullptr;
  PyObject *type, *value, *trace;
  PyErr_Fetch(&type, &value, &trace);
  PyObject* all = node->look(name, false);
  if (all && (v = PyDict_GetItemWithError(all, name))) Py_INCREF(v);
  if (!v && !PyErr_Occurred()) {
    PyErr_Restore(type, value, trace);
    return nullptr;
  }
  Py_XDECREF(type); Py_XDECREF(value); Py_XDECREF(trace);
  return v;
}
int set_node_attribute(PyObject* self, PyObject* name, PyObject* value) {
  Recorded* node = node_of(self);
  if (!node || PyObject_HasAttr((PyObject*)Py_TYPE(self), name)) return PyObject_GenericSetAttr(self, name, value);
  PyObject* all = node->look(name, true);
  if (!all) return -1;
  if (value) return PyDict_SetItem(all, name, value);
  if (PyDict_DelItem(all, name) == 0) return 0;
  if (PyErr_ExceptionMatches(PyExc_KeyError)) PyErr_SetObject(PyExc_AttributeError, name);
  return -1;
}
PyTypeObject node_type;

// whether a call on these may skip torch.autograd.Function: nothing watches it (a functorch transform, a trace, a dispatch mode) and no
// input carries a tangent
bool unwatched(std::initializer_list<const Tensor*> inputs) {
  if (c10::impl::TorchDispatchModeTLS::any_modes_set() || c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) ||
      c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Tracer))
    return false;
  for (const Tensor* t : inputs)
    if (t && (t->unsafeGetTensorImpl()->is_python_dispatch() || t->_fw_grad(0).defined())) return false;
  return true;
}
bool recording(std::initializer_list<const Tensor*> inputs) {
  if (!c10::GradMode::is_enabled()) return false;
  for (const Tensor* t : inputs)
    if (t && t->requires_grad()) return true;
  return false;
}
// functions of a module: there are a handful, and a node's reference must not need the interpreter's lock
PyObject* for_ever(PyObject* f) {
  static std::vector<PyObject*> known;
  for (PyObject* k : known)
    if (k == f) return f;
  Py_INCREF(f);
  known.push_back(f);
  return f;
}
std::shared_ptr<Recorded> new_node(Recorded::Kind kind, std::initializer_list<const Tensor*> inputs, PyObject* interpreted, PyObject* label) {
  std::shared_ptr<Recorded> node(new Recorded(kind), torch::autograd::deleteNode);
  torch::autograd::variable_list in;
  for (const Tensor* t : inputs) {
    if (!t) continue;
    node->needs[in.size()] = t->requires_grad();
    in.push_back(*t);
  }
  node->set_next_edges(torch::autograd::collect_next_edges(in));
  node->interpreted = for_ever(interpreted);
  const char* s = PyUnicode_AsUTF8(label);
  if (!s) throw python_error();
  node->label = s;
  return node;
}
// recordable(x, w, bias or None) -> True where norm_record can follow
PyObject* recordable(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ARGS(3);
  const Tensor *x = plain(a[0]), *w = plain(a[1]), *b = a[2] == Py_None ? nullptr : plain(a[2]);
  if (!x || !w || (a[2] != Py_None && !b) || !unwatched({x, w, b})) return none();
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}
// norm_record(y, x, w, bias or None, c, mean or None, rstd, quirk, interpreted, label) -> y, with its backward where one is recorded
PyObject* norm_record(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ARGS(10);
  const Tensor *y = bf16(a[0]), *x = bf16(a[1]), *w, *bias = a[3] == Py_None ? nullptr : plain(a[3]), *mean = a[5] == Py_None ? nullptr : plain(a[5]),
               *rstd = plain(a[6]);
  In in;
  int dtype;
  if (!y || !x || y->sizes() != x->sizes() || !in.init(a[4]) || !norm_weight(a[2], in.H, &w, &dtype) || !rstd || !row_stats(*rstd, in.M) ||
      (a[5] != Py_None && (!mean || !row_stats(*mean, in.M))) ||
      (a[3] != Py_None && (!bias || bias->scalar_type() != w->scalar_type())) || !unwatched({x, w, bias}))
    return none();
  if (recording({x, w, bias})) {
    auto node = new_node(Recorded::NORM, {x, w, bias}, a[8], a[9]);
    node->saved.push_back(in);
    node->w = *w;
    if (bias) node->bias = *bias;
    if (mean) node->mean = *mean;
    node->rstd = *rstd;
    node->quirk = a[7] == Py_True;
    torch::autograd::set_history(*y, node);
  }
  Py_INCREF(a[0]);
  return a[0];
  END_HANDLE_TH_ERRORS
}
// norm_node(norm_fwd's arguments, quirk, interpreted, label) -> y
PyObject* norm_node(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ARGS(11);
  NormOut n;
  if (!n.init(a)) return none_if_plain(nullptr);
  if (!unwatched({n.x, n.w, n.bias})) return none();
  OR_NONE(unlocked([&] { return n.launch(); }));
  if (recording({n.x, n.w, n.bias})) {
    auto node = new_node(Recorded::NORM, {n.x, n.w, n.bias}, a[9], a[10]);
    node->saved.push_back(n.o);
    node->w = *n.w;
    if (n.bias) node->bias = *n.bias;
    node->mean = n.mean;
    node->rstd = n.rstd;
    node->quirk = a[8] == Py_True;
    torch::autograd::set_history(n.y, node);
  }
  return THPVariable_Wrap(n.y);
  END_HANDLE_TH_ERRORS
}
// linear_node(x [..., K], w [N, K], plan, bits, group, staged, interpreted, label) -> x w^T; x is kept where w has a gradient
PyObject* linear_node(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ARGS(8);
  const Tensor *x = bf16(a[0]), *w = bf16(a[1]);
  int64_t M, K;
  if (!linear_operands(x, w, &M, &K) || !unwatched({x, w})) return none();
  const bool keep = w->requires_grad();
  Out o;
  if (keep && !o.init(a[2], a[3], a[4], M, K, x->device())) return none_if_plain(nullptr);
  Tensor y;
  OR_NONE(unlocked([&] {
    c10::AutoGradMode off(false);
    if (keep) {
      o.alloc();
      const int rc = hyc_compress_rows(x->data_ptr(), K, M, K, &o.d, o.stored.data_ptr(), o.vals.data_ptr(), o.scales.data_ptr(), nullptr, stream());
      if (rc) return rc;
    }
    return linear_forward(*x, *w, M, K, false, &y);
  }));
  if (recording({x, w})) {
    auto node = new_node(Recorded::LINEAR, {x, w}, a[6], a[7]);
    if (keep) node->saved.push_back(o);
    node->w = *w;
    node->staged = a[5] == Py_True;
    torch::autograd::set_history(y, node);
  }
  return THPVariable_Wrap(y);
  END_HANDLE_TH_ERRORS
}
// act_node(act_fwd's arguments, act, interpreted, label) -> act(x)
PyObject* act_node(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ARGS(8);
  ActOut f;
  if (!f.init(a)) return none_if_plain(nullptr);
  if (!unwatched({f.x})) return none();
  OR_NONE(unlocked([&] { return f.launch(); }));
  if (recording({f.x})) {
    auto node = new_node(Recorded::ACT, {f.x}, a[6], a[7]);
    node->saved.push_back(f.o);
    node->code = f.code;
    const char* s = PyUnicode_AsUTF8(a[5]);
    if (!s) return nullptr;
    node->act = s;
    torch::autograd::set_history(f.y, node);
  }
  return THPVariable_Wrap(f.y);
  END_HANDLE_TH_ERRORS
}

// gated_node(gated_fwd's arguments, act, interpreted, label) -> act(gate) up
PyObject* gated_node(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ARGS(11);
  GatedOut f;
  if (!f.init(a)) return none_if_plain(nullptr);
  if (!unwatched({f.gate, f.up})) return none();
  OR_NONE(unlocked([&] { return f.launch(); }));
  if (recording({f.gate, f.up})) {
    auto node = new_node(Recorded::GATED, {f.gate, f.up}, a[9], a[10]);
    node->saved.assign(f.o, f.o + 3);
    node->code = f.code;
    const char* s = PyUnicode_AsUTF8(a[8]);
    if (!s) return nullptr;
    node->act = s;
    torch::autograd::set_history(f.h, node);
  }
  return THPVariable_Wrap(f.h);
  END_HANDLE_TH_ERRORS
}

// rows(t [..., H]) -> (M, H, pitch) as spaced_rows has them, of a tensor on any device
PyObject* rows(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ARGS(1);
  int64_t M, H, pitch;
  if (!THPVariable_Check(a[0]) || !spaced_rows(THPVariable_Unpack(a[0]), &M, &H, &pitch)) return none();
  return Py_BuildValue("LLL", (long long)M, (long long)H, (long long)pitch);
  END_HANDLE_TH_ERRORS
}

// bind(Parameter, ChannelCompressed, ChannelPlan, ThresholdCompressed, SparseRows): the classes the functions above recognise
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  ARGS(5);
  PyObject** to[5] = {&t_parameter, &t_compressed, &t_plan, &t_threshold, &t_sparse};
  for (int i = 0; i < 5; ++i) {
    Py_INCREF(a[i]);
    Py_XDECREF(*to[i]);
    *to[i] = a[i];
  }
  return none();
}

#define ENTRY(f_) {#f_, (PyCFunction)(void (*)(void))f_, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {ENTRY(bind), ENTRY(rows), ENTRY(compress), ENTRY(decompress), ENTRY(norm_fwd), ENTRY(norm_bwd), ENTRY(bias_grad), ENTRY(gradw),
                         ENTRY(linear_fwd), ENTRY(linear_bwd), ENTRY(act_fwd), ENTRY(act_bwd), ENTRY(gated_fwd), ENTRY(gated_bwd), ENTRY(lora_forward),
                         ENTRY(lora_backward), ENTRY(rope_attn_fwd), ENTRY(attn_bwd), ENTRY(attn_kept), ENTRY(attn_kept_bwd),
                         ENTRY(threshold_fwd), ENTRY(softmax_fwd), ENTRY(softmax_bwd), ENTRY(norm_node), ENTRY(norm_record), ENTRY(recordable), ENTRY(linear_node),
                         ENTRY(act_node), ENTRY(gated_node), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_hyc_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__hyc_host() {
  struct { PyObject** to; const char* s; } names[] = {{&s_H, "H"}, {&s_M, "M"}, {&s_k, "k"}, {&s_idx, "idx"}, {&s_plan, "plan"},
                                                      {&s_scale_rule, "scale_rule"}, {&s_stored, "stored"}, {&s_vals, "vals"},
                                                      {&s_scales, "scales"}, {&s_bits, "bits"}, {&s_group, "group"},
                                                      {&s_S, "S"}, {&s_row_ptr, "row_ptr"}, {&s_cols, "cols"}, {&s_threshold, "threshold"},
                                                      {&s_scale, "scale"}, {&s_L, "L"}, {&s_R, "R"}};
  for (auto& n : names) *n.to = PyUnicode_InternFromString(n.s);
  HANDLE_TH_ERRORS
  Ref types(PyImport_ImportModule("types"));
  if (!types.p || !(t_namespace = PyObject_GetAttrString(types.p, "SimpleNamespace"))) return nullptr;
  node_type.tp_getattro = node_attribute;
  node_type.tp_setattro = set_node_attribute;
  torch::autograd::_initFunctionPyTypeObject(node_type, "CalibratedBackward", nullptr, nullptr);
  torch::autograd::registerCppFunction(typeid(Recorded), &node_type);
  END_HANDLE_TH_ERRORS
  return PyModule_Create(&module);
}

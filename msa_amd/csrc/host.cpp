// The host's side of the calls a prompt makes most: operands checked, results allocated and the kernel launched without Python in
// between.  A prompt of few tokens waits for the host, not for the kernels (122 tokens of four layers of 1024: 350 us of kernels, 610 to 650
// us in all through the interpreter, 385 to 430 so), and a call through the interpreter costs 9 to 14 us, of which the launch is 3 (us a
// call, in Python and here: a product 9.7 and 5.4, 0.2 of it for what is asked of its operands besides, a residual step with norm and shift
// 14.3 and 6.4, an RMS residual 8.9 and 4.4, a convolution 8.7 and 4.4, an opened sequence 23 and 6; eight of them together 7, and 26 with
// a view of every state's every row).
//
// Every function takes the operands as they come and answers None for whatever it does not take, without having launched anything: the
// caller's own path in Python then decides, with the checks and errors it has.  A code other than MSA_OK of the library is handed back.
#include <Python.h>

#include <algorithm>

#include <ATen/ATen.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>

#include "../../include/msa_amd.h"
#include "../../include/msa_seq.h"

namespace {

decltype(&msa_block_linear) block_linear;
decltype(&msa_block_linear_us) block_linear_us;
decltype(&msa_flow_linear) flow_linear;
decltype(&msa_flow_linear_us) flow_linear_us;
decltype(&msa_flow_workspace_bytes) flow_bytes;
decltype(&msa_seq_clear) clear_;
decltype(&msa_seq_ssd_chunked_norm) ssd_normed;
decltype(&msa_seq_ssd_norm_folds) ssd_folds;
decltype(&msa_seq_residual_norm) residual_norm_;
decltype(&msa_seq_rms_residual) rms_residual_;
decltype(&msa_seq_conv_silu) conv_silu_;
decltype(&msa_seq_group_rmsnorm) group_rmsnorm_;
decltype(&msa_seq_ssd_scan) ssd_scan;
decltype(&msa_seq_ssd_chunked) ssd_chunked;
decltype(&msa_seq_ssd_chunked_workspace_bytes) ssd_bytes;
decltype(&msa_seq_delta_scan) delta_scan;
decltype(&msa_seq_delta_chunked) delta_chunked;
decltype(&msa_seq_delta_chunked_workspace_bytes) delta_bytes;

// Lines of the products' dispatch, as the caller has them.
struct Lines {
  long long block_rows, block_depth, captured_rows, captured_depth;
  double block_us, captured_us;
} lines;

bool is_none(PyObject* o) { return o == nullptr || o == Py_None; }
const at::Tensor* tensor(PyObject* o) { return !is_none(o) && THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr; }
void* at_(const at::Tensor* t) { return t ? t->data_ptr() : nullptr; }
void* stream() { return c10::hip::getCurrentHIPStream().stream(); }
// The device that `stream` is of, or -1 without one.
int device() {
  int d = -1;
  if (hipGetDevice(&d) == hipSuccess) return d;
  (void)hipGetLastError();
  return -1;
}
int dtype_of(const at::Tensor& t) { return t.scalar_type() == at::kBFloat16 ? MSA_BF16 : t.scalar_type() == at::kFloat ? MSA_F32 : -1; }
bool dense(const at::Tensor* t) { return t && t->is_cuda() && t->is_contiguous(); }
// Whether nothing but the values is asked of a tensor: no gradient in either direction, no batch of vmap, no trace, no dispatch of a class
// or a mode of its own.  A launch would pass all of these by, without a word: what is not plain goes to torch's own call.
bool plain(PyObject* o, const at::Tensor* t) {
  using K = c10::DispatchKey;
  static const c10::DispatchKeySet of_tensor({K::Python, K::Functionalize, K::FuncTorchBatched, K::FuncTorchGradWrapper});
  static const c10::DispatchKeySet of_thread({K::Python, K::PythonDispatcher, K::Functionalize, K::Tracer, K::FuncTorchDynamicLayerFrontMode});
  return THPVariable_CheckExact(o) && !(t->requires_grad() && at::GradMode::is_enabled()) && !t->key_set().has_any(of_tensor) &&
         !c10::impl::tls_local_dispatch_key_set().included_.has_any(of_thread) && !t->_fw_grad(0).defined();
}
bool floats(const at::Tensor* t, int64_t n) { return dense(t) && t->scalar_type() == at::kFloat && t->numel() == n; }
// rows with unit column stride, and the stride between them
bool rows(const at::Tensor* t) { return t && t->is_cuda() && t->dim() == 2 && (t->size(1) <= 1 || t->stride(1) == 1); }
int64_t row_stride(const at::Tensor& t) { return t.size(0) > 1 ? t.stride(0) : std::max(t.stride(0), t.size(1)); }
bool aligned(const at::Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0; }

// The launch with the interpreter's lock given back, which is taken again however it ends.  It gets addresses, not tensors: data_ptr() of a
// tensor without storage (fake ones, wrappers of vmap) throws, and that has to be while the lock is held.
struct Unlocked {
  PyThreadState* state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
};
template <class Launch>
int run(Launch launch) {
  const Unlocked unlocked;
  return launch();
}
float* f32(const at::Tensor* t) { return static_cast<float*>(at_(t)); }
PyObject* none() { Py_RETURN_NONE; }
PyObject* wrap(const at::Tensor& t) { return THPVariable_Wrap(t); }

// ordinary(operands ...): whether all tensors among them are plain
PyObject* ordinary(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  for (Py_ssize_t i = 0; i < n; ++i) {
    const at::Tensor* t = tensor(args[i]);
    if (t && !plain(args[i], t)) Py_RETURN_FALSE;
  }
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// block_ok(x, w, end): the caller's rule (block_linear_ok has it, with its reasons).
PyObject* block_ok(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 3) return PyErr_Format(PyExc_TypeError, "block_ok takes 3 arguments");
  const at::Tensor *x = tensor(args[0]), *w = tensor(args[1]);
  if (!x || !w || !block_linear_us) return none();
  const bool end = PyObject_IsTrue(args[2]);
  if (x->dim() != 2 || w->dim() != 2 || !plain(args[0], x) || !plain(args[1], w)) Py_RETURN_FALSE;
  const int64_t T = x->size(0), K = x->size(1), N = w->size(0);
  if (!(T > 0 && x->is_cuda() && x->scalar_type() == at::kBFloat16 && w->scalar_type() == at::kBFloat16 && w->is_contiguous() && w->size(1) == K &&
        K % 64 == 0 && K >= 64 && K <= 32768 && N % 16 == 0 && N > 0 && N < 1 << 20 && T < 1 << 22 && (T <= lines.block_rows || K <= lines.block_depth)))
    Py_RETURN_FALSE;
  const double us = block_linear_us(T, (int32_t)K, (int32_t)N);
  if (us > lines.block_us) Py_RETURN_FALSE;
  if (!end && (us > lines.captured_us || T > lines.captured_rows || K > lines.captured_depth)) {
    hipStreamCaptureStatus status;
    if (hipStreamIsCapturing(c10::hip::getCurrentHIPStream().stream(), &status) != hipSuccess) return none();
    if (status != hipStreamCaptureStatusNone) Py_RETURN_FALSE;
  }
  return PyBool_FromLong((x->is_contiguous() || (x->stride(1) == 1 && x->stride(0) % 8 == 0 && K <= x->stride(0) && x->stride(0) < 1 << 21)) && aligned(*x) &&
                         aligned(*w) && w->device() == x->device());
  END_HANDLE_TH_ERRORS
}

// linear(x, w, mode, gelu_n, limit, alpha, shift): msa_block_linear of operands that block_ok took
PyObject* linear(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 7) return PyErr_Format(PyExc_TypeError, "linear takes 7 arguments");
  const at::Tensor *x = tensor(args[0]), *w = tensor(args[1]);
  const long mode = PyLong_AsLong(args[2]), gelu_n = PyLong_AsLong(args[3]);
  const msa_tile_end end{(int32_t)mode, (int32_t)gelu_n, (float)PyFloat_AsDouble(args[4]), (float)PyFloat_AsDouble(args[5]), (float)PyFloat_AsDouble(args[6])};
  if (PyErr_Occurred()) return nullptr;
  if (!x || !w || !block_linear || !x->is_cuda() || x->dim() != 2 || w->dim() != 2) return none();
  const int64_t T = x->size(0), K = x->size(1), N = w->size(0), ldx = T > 1 ? x->stride(0) : K;
  void *xp = at_(x), *wp = at_(w);
  at::Tensor out = at::empty({T, mode == MSA_TILE_GLU ? N / 2 : N}, x->options().requires_grad(false));
  void *to = out.data_ptr(), *st = stream();
  const int64_t ldo = out.size(1);
  const int rc = run([&] { return block_linear(xp, ldx, T, (int32_t)K, wp, (int32_t)N, &end, to, ldo, st); });
  return rc == MSA_OK ? wrap(out) : PyLong_FromLong(rc);
  END_HANDLE_TH_ERRORS
}

// flow(x, w, mode, gelu_n, limit, alpha, shift): msa_flow_linear where msa_flow_linear_us takes it, of plain operands
PyObject* flow(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 7) return PyErr_Format(PyExc_TypeError, "flow takes 7 arguments");
  const at::Tensor *x = tensor(args[0]), *w = tensor(args[1]);
  const long mode = PyLong_AsLong(args[2]), gelu_n = PyLong_AsLong(args[3]);
  const msa_tile_end end{(int32_t)mode, (int32_t)gelu_n, (float)PyFloat_AsDouble(args[4]), (float)PyFloat_AsDouble(args[5]), (float)PyFloat_AsDouble(args[6])};
  if (PyErr_Occurred()) return nullptr;
  if (!x || !w || !flow_linear || !x->is_cuda() || x->dim() != 2 || w->dim() != 2) return none();
  const int64_t T = x->size(0), K = x->size(1), N = w->size(0);
  if (!(plain(args[0], x) && plain(args[1], w) &&
        x->scalar_type() == at::kBFloat16 && w->scalar_type() == at::kBFloat16 && w->is_contiguous() && w->size(1) == K && K <= 32768 && N % 16 == 0 &&
        N < 1 << 20 && (x->is_contiguous() || (x->stride(1) == 1 && x->stride(0) % 8 == 0 && K <= x->stride(0) && x->stride(0) < 1 << 21)) && aligned(*x) &&
        aligned(*w) && w->device() == x->device() && gelu_n % 8 == 0 && gelu_n <= N &&
        flow_linear_us(T, (int32_t)K, (int32_t)N, (int32_t)mode) > 0.f))
    return none();
  at::Tensor out = at::empty({T, mode == MSA_TILE_GLU ? N / 2 : N}, x->options().requires_grad(false)), ws;
  const size_t need = flow_bytes(T, (int32_t)K, (int32_t)N, (int32_t)mode);
  if (need) ws = at::empty({(int64_t)need}, x->options().requires_grad(false).dtype(at::kByte));
  void *xp = at_(x), *wp = at_(w), *to = out.data_ptr(), *scratch = need ? ws.data_ptr() : nullptr, *st = stream();
  const int64_t ldx = x->stride(0), ldo = out.size(1);
  const int rc = run([&] { return flow_linear(xp, ldx, T, (int32_t)K, wp, (int32_t)N, &end, to, ldo, scratch, need, st); });
  return rc == MSA_OK ? wrap(out) : PyLong_FromLong(rc);
  END_HANDLE_TH_ERRORS
}

struct Batch {
  const msa_seq_batch* c;
  int64_t top;                 // its largest slot
  bool get(PyObject* address, PyObject* slot) {
    c = static_cast<const msa_seq_batch*>(PyLong_AsVoidPtr(address));
    top = PyLong_AsLongLong(slot);
    return c && !PyErr_Occurred();
  }
};

// residual_norm(batch address, its largest slot, x, y, gate, gate_bias, norm_w, norm_b, alpha, shift, prev, want_h, dtype): (x', h, h_shift)
PyObject* residual_norm(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 13) return PyErr_Format(PyExc_TypeError, "residual_norm takes 13 arguments");
  Batch b;
  if (!b.get(args[0], args[1])) return PyErr_Occurred() ? nullptr : none();
  const at::Tensor *x = tensor(args[2]), *y = tensor(args[3]), *gate = tensor(args[4]), *gate_bias = tensor(args[5]), *nw = tensor(args[6]),
                   *nb = tensor(args[7]), *shift = tensor(args[9]), *prev = tensor(args[10]);
  const msa_dyn_tanh norm{nw ? static_cast<const float*>(nw->data_ptr()) : nullptr, nb ? static_cast<const float*>(nb->data_ptr()) : nullptr,
                          (float)PyFloat_AsDouble(args[8]), 0};
  const long want_h = PyLong_AsLong(args[11]), dtype = PyLong_AsLong(args[12]);
  if (PyErr_Occurred()) return nullptr;
  if (!dense(x) || x->dim() != 2 || x->scalar_type() != at::kFloat || x->size(0) != b.c->rows || (!is_none(args[10]) && !dense(prev))) return none();
  const int64_t T = x->size(0), W = x->size(1);
  if ((!is_none(args[6]) || !is_none(args[7])) && !(floats(nw, W) && floats(nb, W))) return none();
  if (!is_none(args[3])) {
    if (!rows(y) || !rows(gate) || !floats(gate_bias, W) || y->sizes() != x->sizes() || gate->sizes() != x->sizes() || dtype_of(*y) != dtype || dtype_of(*gate) != dtype)
      return none();
  }
  if (!is_none(args[9]) && !(floats(shift, W) && prev && prev->scalar_type() == at::kFloat && prev->dim() == 2 && prev->size(1) == W && prev->size(0) > b.top)) return none();
  const auto wide = x->options().requires_grad(false), act = wide.dtype(dtype == MSA_BF16 ? at::kBFloat16 : at::kFloat);
  const float *xp = f32(x), *bias = f32(gate_bias), *shifts = f32(shift);
  float* before = f32(prev);
  void *yp = at_(y), *gp = at_(gate);
  const int64_t ldy = y ? row_stride(*y) : 0, ldg = gate ? row_stride(*gate) : 0;
  at::Tensor out, h, hs;
  if (y) out = at::empty({T, W}, wide);
  if (nw && want_h) h = at::empty({T, W}, act);
  if (shift) hs = at::empty({T, W}, act);
  float* sum = y ? f32(&out) : nullptr;
  void *hp = h.defined() ? h.data_ptr() : nullptr, *hsp = hs.defined() ? hs.data_ptr() : nullptr, *st = stream();
  const int rc = run([&] { return residual_norm_(xp, yp, ldy, gp, ldg, bias, sum, (int32_t)dtype, (int32_t)W, &norm, hp, shifts, before, hsp, b.c, st); });
  if (rc != MSA_OK) return PyLong_FromLong(rc);
  PyObject* first = y ? wrap(out) : (Py_INCREF(args[2]), args[2]);
  return Py_BuildValue("(NNN)", first, h.defined() ? wrap(h) : none(), hs.defined() ? wrap(hs) : none());
  END_HANDLE_TH_ERRORS
}

// rms_residual(x, y, w, eps, next_w, out, want_h, dtype): (x', h)
PyObject* rms_residual(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 8) return PyErr_Format(PyExc_TypeError, "rms_residual takes 8 arguments");
  const at::Tensor *x = tensor(args[0]), *y = tensor(args[1]), *w = tensor(args[2]), *next_w = tensor(args[4]), *out = tensor(args[5]);
  const double eps = PyFloat_AsDouble(args[3]);
  const long want_h = PyLong_AsLong(args[6]), dtype = PyLong_AsLong(args[7]);
  if (PyErr_Occurred()) return nullptr;
  if (!dense(x) || x->dim() != 2 || x->scalar_type() != at::kFloat || !y || !rows(y) || !floats(w, x->size(1)) || y->sizes() != x->sizes() || dtype_of(*y) != dtype ||
      !out || !dense(out) || out->sizes() != x->sizes() || out->scalar_type() != at::kFloat || (!is_none(args[4]) && !floats(next_w, x->size(1))))
    return none();
  const int64_t T = x->size(0), W = x->size(1);
  const float *xp = f32(x), *wp = f32(w), *next = f32(next_w);
  float* to = f32(out);
  void* yp = at_(y);
  const int64_t ldy = row_stride(*y);
  at::Tensor h;
  if (want_h || next_w) h = at::empty({T, W}, x->options().requires_grad(false).dtype(dtype == MSA_BF16 ? at::kBFloat16 : at::kFloat));
  void *hp = h.defined() ? h.data_ptr() : nullptr, *st = stream();
  const int rc = run([&] { return rms_residual_(xp, yp, ldy, wp, (float)eps, to, next, hp, (int32_t)dtype, (int32_t)T, (int32_t)W, st); });
  if (rc != MSA_OK) return PyLong_FromLong(rc);
  Py_INCREF(args[5]);
  return Py_BuildValue("(NN)", args[5], h.defined() ? wrap(h) : none());
  END_HANDLE_TH_ERRORS
}

// conv_silu(batch address, its largest slot, x, taps, bias, state): the convolved rows
PyObject* conv_silu(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 6) return PyErr_Format(PyExc_TypeError, "conv_silu takes 6 arguments");
  Batch b;
  if (!b.get(args[0], args[1])) return PyErr_Occurred() ? nullptr : none();
  const at::Tensor *x = tensor(args[2]), *taps = tensor(args[3]), *bias = tensor(args[4]), *state = tensor(args[5]);
  if (!rows(x) || dtype_of(*x) < 0 || !taps || taps->dim() != 2) return none();
  const int64_t T = x->size(0), Cn = x->size(1), K = taps->size(1);
  if (!floats(taps, Cn * K) || (!is_none(args[4]) && !floats(bias, Cn)) || !dense(state) || state->scalar_type() != at::kFloat || state->dim() != 3 ||
      state->size(1) != K - 1 || state->size(2) != Cn || state->size(0) <= b.top || T != b.c->rows)
    return none();
  const void* xp = at_(x);
  const float *tp = f32(taps), *bp = f32(bias);
  float* sp = f32(state);
  const int64_t ldx = row_stride(*x);
  const int dtype = dtype_of(*x);
  at::Tensor out = at::empty({T, Cn}, x->options().requires_grad(false));
  void *to = out.data_ptr(), *st = stream();
  const int rc = run([&] { return conv_silu_(xp, ldx, tp, bp, dtype, (int32_t)Cn, (int32_t)K, sp, to, Cn, b.c, st); });
  return rc == MSA_OK ? wrap(out) : PyLong_FromLong(rc);
  END_HANDLE_TH_ERRORS
}

// group_rmsnorm(v, w, parts, eps)
PyObject* group_rmsnorm(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 4) return PyErr_Format(PyExc_TypeError, "group_rmsnorm takes 4 arguments");
  const at::Tensor *v = tensor(args[0]), *w = tensor(args[1]);
  const long parts = PyLong_AsLong(args[2]);
  const double eps = PyFloat_AsDouble(args[3]);
  if (PyErr_Occurred()) return nullptr;
  if (!dense(v) || v->dim() != 2 || dtype_of(*v) < 0 || !floats(w, v->size(1))) return none();
  const int64_t T = v->size(0), W = v->size(1);
  const void* vp = at_(v);
  const float* wp = f32(w);
  const int dtype = dtype_of(*v);
  at::Tensor out = at::empty({T, W}, v->options().requires_grad(false));
  void *to = out.data_ptr(), *st = stream();
  const int rc = run([&] { return group_rmsnorm_(vp, dtype, (int32_t)T, (int32_t)W, (int32_t)parts, wp, (float)eps, to, st); });
  return rc == MSA_OK ? wrap(out) : PyLong_FromLong(rc);
  END_HANDLE_TH_ERRORS
}

// [slots, a, b, c] fp32 states that reach the step's slots
bool states(const at::Tensor* t, int64_t a, int64_t b, int64_t c, int64_t top) {
  return dense(t) && t->scalar_type() == at::kFloat && t->dim() == 4 && t->size(1) == a && t->size(2) == b && t->size(3) == c && t->size(0) > top;
}
bool block(const at::Tensor* t, int64_t r, int64_t c, at::ScalarType type) { return rows(t) && t->size(0) == r && t->size(1) == c && t->scalar_type() == type; }

// ssd(batch address, its largest slot, xbc, z, dt_raw, dt_bias, A_log, D, H, P, N, G, state, chunked[, w, parts, eps]): the gated output, or its norm
// where that is folded
PyObject* ssd(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 14 && n != 17) return PyErr_Format(PyExc_TypeError, "ssd takes 14 or 17 arguments");
  Batch b;
  if (!b.get(args[0], args[1])) return PyErr_Occurred() ? nullptr : none();
  const at::Tensor *xbc = tensor(args[2]), *z = tensor(args[3]), *dt = tensor(args[4]), *bias = tensor(args[5]), *a_log = tensor(args[6]), *d = tensor(args[7]),
                   *state = tensor(args[12]);
  const long H = PyLong_AsLong(args[8]), P = PyLong_AsLong(args[9]), N = PyLong_AsLong(args[10]), G = PyLong_AsLong(args[11]);
  const bool chunked = PyObject_IsTrue(args[13]);
  const at::Tensor* norm = n == 17 ? tensor(args[14]) : nullptr;
  const long parts = n == 17 ? PyLong_AsLong(args[15]) : 0;
  const double eps = n == 17 ? PyFloat_AsDouble(args[16]) : 0.0;
  if (PyErr_Occurred()) return nullptr;
  const int64_t T = b.c->rows;
  if (n == 17 && (!chunked || !floats(norm, H * P) || !aligned(*norm) ||
                  !ssd_folds(b.c->max_rows, b.c->n_seq, (int32_t)H, (int32_t)P, (int32_t)N, (int32_t)G, (int32_t)parts)))
    return none();
  if (!xbc || dtype_of(*xbc) < 0 || !floats(bias, H) || !floats(a_log, H) || !floats(d, H) || !states(state, H, N, P, b.top) ||
      !block(xbc, T, H * P + 2 * G * N, xbc->scalar_type()) || !block(z, T, H * P, xbc->scalar_type()) || !block(dt, T, H, xbc->scalar_type()))
    return none();
  const void *xp = at_(xbc), *zp = at_(z), *dp = at_(dt);
  const float *bp = f32(bias), *ap = f32(a_log), *skip = f32(d), *wp = f32(norm);
  float* sp = f32(state);
  const int64_t ldx = row_stride(*xbc), ldz = row_stride(*z), ldd = row_stride(*dt);
  const int dtype = dtype_of(*xbc);
  at::Tensor v = at::empty({T, H * P}, xbc->options().requires_grad(false)), ws;
  const size_t need = chunked ? ssd_bytes(b.c->max_rows, b.c->n_seq, (int32_t)H, (int32_t)P, (int32_t)N) : 0;
  if (need) ws = at::empty({(int64_t)need}, v.options().dtype(at::kByte));
  void *to = v.data_ptr(), *scratch = need ? ws.data_ptr() : nullptr, *st = stream();
  const int rc = run([&] {
    auto call = [&](auto fn, auto... more) {
      return fn(xp, ldx, zp, ldz, dp, ldd, bp, ap, skip, dtype, (int32_t)H, (int32_t)P, (int32_t)N, (int32_t)G, sp, to, b.c, more...);
    };
    if (norm) return call(ssd_normed, scratch, need, wp, (int32_t)parts, (float)eps, st);
    return chunked ? call(ssd_chunked, scratch, need, st) : call(ssd_scan, st);
  });
  return rc == MSA_OK ? wrap(v) : PyLong_FromLong(rc);
  END_HANDLE_TH_ERRORS
}

// delta(batch address, its largest slot, qkv, a, b, gate, A_log, dt_bias, norm, eps, H, G, D, E, state, chunked): normed and gated read-outs
PyObject* delta(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 16) return PyErr_Format(PyExc_TypeError, "delta takes 16 arguments");
  Batch b;
  if (!b.get(args[0], args[1])) return PyErr_Occurred() ? nullptr : none();
  const at::Tensor *qkv = tensor(args[2]), *a = tensor(args[3]), *beta = tensor(args[4]), *gate = tensor(args[5]), *a_log = tensor(args[6]), *bias = tensor(args[7]),
                   *norm = tensor(args[8]), *state = tensor(args[14]);
  const double eps = PyFloat_AsDouble(args[9]);
  const long H = PyLong_AsLong(args[10]), G = PyLong_AsLong(args[11]), D = PyLong_AsLong(args[12]), E = PyLong_AsLong(args[13]);
  const bool chunked = PyObject_IsTrue(args[15]);
  if (PyErr_Occurred()) return nullptr;
  const int64_t T = b.c->rows;
  if (!qkv || dtype_of(*qkv) < 0 || !floats(a_log, H) || !floats(bias, H * D) || !floats(norm, E) || !states(state, H, D, E, b.top)) return none();
  const auto type = qkv->scalar_type();
  if (!block(qkv, T, 2 * G * D + H * E, type) || !block(a, T, H * D, type) || !block(beta, T, H, type) || !block(gate, T, H * E, type)) return none();
  at::Tensor out = at::empty({T, H * E}, qkv->options().requires_grad(false)), ws;
  msa_delta_args c{};
  c.qkv = qkv->data_ptr(), c.a = a->data_ptr(), c.b = beta->data_ptr(), c.gate = gate->data_ptr();
  c.qkv_stride = row_stride(*qkv), c.a_stride = row_stride(*a), c.b_stride = row_stride(*beta), c.gate_stride = row_stride(*gate);
  c.A_log = f32(a_log), c.dt_bias = f32(bias), c.norm = f32(norm), c.state = f32(state), c.out = out.data_ptr();
  c.H = (int32_t)H, c.G = (int32_t)G, c.D = (int32_t)D, c.E = (int32_t)E, c.eps = (float)eps;
  const size_t need = chunked ? delta_bytes(&c, b.c->max_rows, b.c->n_seq) : 0;
  if (need) ws = at::empty({(int64_t)need}, out.options().dtype(at::kByte));
  void *scratch = need ? ws.data_ptr() : nullptr, *st = stream();
  const int dtype = dtype_of(*qkv);
  const int rc = run([&] { return chunked ? delta_chunked(&c, b.c, scratch, need, st) : delta_scan(&c, dtype, b.c, st); });
  return rc == MSA_OK ? wrap(out) : PyLong_FromLong(rc);
  END_HANDLE_TH_ERRORS
}

// pieces(words, places): the parts of an int64 vector, (first word, elements, whether of 32 bits) each
PyObject* pieces(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 2 || !PyList_Check(args[1])) return PyErr_Format(PyExc_TypeError, "pieces takes a tensor and a list");
  const at::Tensor* words = tensor(args[0]);
  if (!words || words->dim() != 1 || words->scalar_type() != at::kLong) return PyErr_Format(PyExc_TypeError, "pieces of an int64 vector");
  const Py_ssize_t count = PyList_GET_SIZE(args[1]);
  THPObjectPtr out(PyList_New(count));
  if (!out) return nullptr;
  const at::Tensor halves = words->view(at::kInt);
  for (Py_ssize_t i = 0; i < count; ++i) {
    long long at, len;
    int small;
    if (!PyArg_ParseTuple(PyList_GET_ITEM(args[1], i), "LLp", &at, &len, &small)) return nullptr;
    PyObject* part = wrap(small ? halves.narrow(0, 2 * at, len) : words->narrow(0, at, len));
    if (!part) return nullptr;
    PyList_SET_ITEM(out.get(), i, part);
  }
  return out.release();
  END_HANDLE_TH_ERRORS
}

// clear(tensors, slot): zeroes the tensors' rows of that slot, or of a list of slots, in one launch or a few.  Tensors of another device than
// the current one go to the library's call, which switches to theirs: a launch from here would be of the current device and its stream.
PyObject* clear(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 2 || !PyList_Check(args[0])) return PyErr_Format(PyExc_TypeError, "clear takes a list and a slot");
  std::vector<int64_t> slots;
  const bool several = PyList_Check(args[1]);
  for (Py_ssize_t i = 0; i < (several ? PyList_GET_SIZE(args[1]) : 1); ++i) slots.push_back(PyLong_AsLongLong(several ? PyList_GET_ITEM(args[1], i) : args[1]));
  if (PyErr_Occurred()) return nullptr;
  std::vector<const at::Tensor*> tensors;
  std::vector<void*> base;
  std::vector<int64_t> bytes;
  const int here = device();
  const auto [least, most] = std::minmax_element(slots.begin(), slots.end());
  bool dense = clear_ != nullptr;
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(args[0]); ++i) {
    PyObject* o = PyList_GET_ITEM(args[0], i);
    const at::Tensor* t = tensor(o);
    if (!t) return PyErr_Format(PyExc_TypeError, "clear: not a tensor");
    tensors.push_back(t);
    dense = dense && t->is_cuda() && t->device().index() == here && t->is_contiguous() && plain(o, t) && t->dim() > 0 &&
            (slots.empty() || (*least >= 0 && *most < t->size(0)));
    if (!dense || t->numel() == 0) continue;
    base.push_back(t->data_ptr());
    bytes.push_back((int64_t)t->nbytes() / t->size(0));
  }
  if (dense && !base.empty()) {
    void* st = stream();
    const int rc = run([&] { return clear_(base.data(), bytes.data(), (int32_t)base.size(), slots.data(), (int32_t)slots.size(), st); });
    if (rc == MSA_OK) Py_RETURN_NONE;
  }
  // (a view a tensor and slot costs as much as a launch where there are some of both: only here)
  std::vector<at::Tensor> rows;
  for (const at::Tensor* t : tensors)
    for (const int64_t slot : slots) rows.push_back(t->select(0, slot));
  if (!rows.empty()) at::_foreach_zero_(rows);
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

template <class F>
bool resolve(void* lib, const char* name, F& f) {
  f = reinterpret_cast<F>(dlsym(lib, name));
  if (!f) PyErr_Format(PyExc_ImportError, "%s is not in the library", name);
  return f != nullptr;
}
// bind(libmsa_amd.so or None, libmsa_seq.so, (lines ...)): once, in front of everything else.  The libraries stay apart: both have some
// names.  Without the first, which a checkout that only runs the decoders of mixed layers has not built, products are declined.
PyObject* bind(PyObject*, PyObject* args) {
  const char *amd, *seq;
  Lines l;
  if (!PyArg_ParseTuple(args, "zs(LLLLdd)", &amd, &seq, &l.block_rows, &l.block_depth, &l.captured_rows, &l.captured_depth, &l.block_us,
                        &l.captured_us))
    return nullptr;
  void *a = amd ? dlopen(amd, RTLD_NOW | RTLD_LOCAL) : nullptr, *s = dlopen(seq, RTLD_NOW | RTLD_LOCAL);
  if ((amd && !a) || !s) return PyErr_Format(PyExc_ImportError, "%s", dlerror());
  if (a && (!resolve(a, "msa_block_linear", block_linear) || !resolve(a, "msa_block_linear_us", block_linear_us) || !resolve(a, "msa_flow_linear", flow_linear) ||
            !resolve(a, "msa_flow_linear_us", flow_linear_us) || !resolve(a, "msa_flow_workspace_bytes", flow_bytes))) return nullptr;
  if (!resolve(s, "msa_seq_clear", clear_) || !resolve(s, "msa_seq_residual_norm", residual_norm_) || !resolve(s, "msa_seq_rms_residual", rms_residual_) ||
      !resolve(s, "msa_seq_conv_silu", conv_silu_) || !resolve(s, "msa_seq_group_rmsnorm", group_rmsnorm_) ||
      !resolve(s, "msa_seq_ssd_scan", ssd_scan) || !resolve(s, "msa_seq_ssd_chunked", ssd_chunked) || !resolve(s, "msa_seq_ssd_chunked_norm", ssd_normed) ||
      !resolve(s, "msa_seq_ssd_norm_folds", ssd_folds) ||
      !resolve(s, "msa_seq_ssd_chunked_workspace_bytes", ssd_bytes) || !resolve(s, "msa_seq_delta_scan", delta_scan) ||
      !resolve(s, "msa_seq_delta_chunked", delta_chunked) || !resolve(s, "msa_seq_delta_chunked_workspace_bytes", delta_bytes))
    return nullptr;
  lines = l;
  Py_RETURN_NONE;
}

#define MSA_FAST(f) {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {{"bind", bind, METH_VARARGS, nullptr}, MSA_FAST(ordinary), MSA_FAST(block_ok), MSA_FAST(linear), MSA_FAST(flow), MSA_FAST(residual_norm), MSA_FAST(rms_residual), MSA_FAST(conv_silu),
                         MSA_FAST(group_rmsnorm), MSA_FAST(ssd), MSA_FAST(delta), MSA_FAST(pieces), MSA_FAST(clear), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() { return PyModule_Create(&module); }

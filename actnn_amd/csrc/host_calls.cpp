// The host side of the calls a training step makes most often: allocation of the results, the generator's
// (seed, offset), the current stream and the call into the kernels' C library, in one native function each
// instead of a dozen calls out of Python.  A module of its own beside the C library (which knows no tensors): what it
// allocates, draws and launches is what the Python functions of cpp_extension document, and those still check the
// arguments that users hand in.
//
// What it is for: calls of a few microseconds, where Python was slower than the GPU.  compress + restore of bf16
// [32, 64, 56, 56] took 47.7 us, of them 26 us of kernels and the rest host time behind them (eight torch.empty, two calls of 11
// and 22 converted arguments, checks); 34.8 now, QDropout's two passes over bf16 [128, 4096] 86.6 and 62.9.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/Context.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/actnn_hip.h"

namespace {

using at::Tensor;

// ---------------------------------------------------------------------------- arguments
struct Args {
  PyObject* const* at;
  Py_ssize_t n, i = 0;
  Args(PyObject* const* a, Py_ssize_t count, Py_ssize_t want) : at(a), n(count) {
    TORCH_CHECK(count == want, "expected ", want, " arguments, got ", count);
  }
  PyObject* tensor_object() {
    PyObject* o = at[i++];
    TORCH_CHECK_TYPE(THPVariable_Check(o), "argument ", i, " must be a tensor");
    return o;
  }
  const Tensor& tensor() { return THPVariable_Unpack(tensor_object()); }
  // whether the next `count` arguments are tensors
  bool tensors(int count) const {
    for (int k = 0; k < count; ++k)
      if (!THPVariable_Check(at[i + k])) return false;
    return true;
  }
  // (an undefined tensor for None)
  Tensor optional() { return at[i] == Py_None ? (++i, Tensor()) : tensor(); }
  int64_t integer() {
    const int64_t v = PyLong_AsLongLong(at[i++]);
    if (v == -1 && PyErr_Occurred()) throw python_error();
    return v;
  }
  double number() {
    const double v = PyFloat_AsDouble(at[i++]);
    if (v == -1.0 && PyErr_Occurred()) throw python_error();
    return v;
  }
  bool flag() {
    const int v = PyObject_IsTrue(at[i++]);
    if (v < 0) throw python_error();
    return v != 0;
  }
};

PyObject* wrap(const Tensor& t) {
  if (!t.defined()) Py_RETURN_NONE;
  return THPVariable_Wrap(t);
}
template <typename... Ts> PyObject* tuple_of(const Ts&... ts) {
  PyObject* out = PyTuple_New(sizeof...(ts));
  if (!out) throw python_error();
  Py_ssize_t i = 0;
  auto put = [&](const Tensor& t) {
    PyObject* o = wrap(t);
    if (!o) {
      Py_DECREF(out);
      throw python_error();
    }
    PyTuple_SET_ITEM(out, i++, o);
  };
  (put(ts), ...);
  return out;
}

// ---------------------------------------------------------------------------- plumbing
int code_of(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return ACTNN_F32;
    case at::kHalf: return ACTNN_F16;
    case at::kBFloat16: return ACTNN_BF16;
    default: TORCH_CHECK(false, "unsupported dtype ", t);
  }
}
at::ScalarType type_of(int64_t code) {
  TORCH_CHECK(code >= ACTNN_F32 && code <= ACTNN_BF16, "unknown dtype code ", code);
  return code == ACTNN_F32 ? at::kFloat : code == ACTNN_F16 ? at::kHalf : at::kBFloat16;
}
void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
float* f32(const Tensor& t) { return static_cast<float*>(ptr(t)); }
int32_t* i32(const Tensor& t) { return static_cast<int32_t*>(ptr(t)); }
void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
// Runs a call into the C library without the interpreter's lock (a launch may wait for room in its queue).
template <typename F> void launch(const char* what, F f) {
  int rc;
  {
    struct Unlocked {
      PyThreadState* state = PyEval_SaveThread();
      ~Unlocked() { PyEval_RestoreThread(state); }
    } unlocked;
    rc = f();
  }
  TORCH_CHECK(rc == ACTNN_OK, what, " failed: ", actnn_strerror(rc), " (code ", rc, ")");
}
Tensor empty(at::IntArrayRef size, const Tensor& like, at::ScalarType dtype) {
  return at::empty(size, at::TensorOptions().dtype(dtype).device(like.device()));
}

// A tensor argument with the Python object it came as.  What makes a new tensor of it goes through Python where its class may
// have a say, and the object goes along with the tensor: the next step works on the same one the kernel reads or writes.
class Given {
 public:
  explicit Given(PyObject* o) : object_(o), tensor_(THPVariable_Unpack(o)) { Py_INCREF(object_); }
  Given(const Given&) = delete;
  Given& operator=(const Given&) = delete;
  ~Given() { Py_DECREF(object_); }
  const Tensor& tensor() const { return tensor_; }
  void make_contiguous() {
    if (plain()) tensor_ = tensor_.contiguous();
    else replace(PyObject_CallMethod(object_, "contiguous", nullptr));
  }
  // (the kernels use 16-byte accesses; only views with a storage offset are not aligned)
  void make_aligned() {
    if (reinterpret_cast<uintptr_t>(tensor_.data_ptr()) % 16 == 0) return;
    if (plain()) tensor_ = tensor_.clone();
    else replace(PyObject_CallMethod(object_, "clone", nullptr));
  }
  Tensor empty_like() const {
    if (plain()) return at::empty_like(tensor_);
    PyObject* torch = PyImport_ImportModule("torch");
    if (!torch) throw python_error();
    PyObject* made = PyObject_CallMethod(torch, "empty_like", "O", object_);
    Py_DECREF(torch);
    const Tensor out = unpacked(made);
    Py_DECREF(made);
    return out;
  }

 private:
  // (a plain object_ stays when its tensor is replaced: only its class counts)
  bool plain() const { return THPVariable_CheckExact(object_); }
  static Tensor unpacked(PyObject* made) {
    if (!made) throw python_error();
    if (!THPVariable_Check(made)) {
      Py_DECREF(made);
      TORCH_CHECK_TYPE(false, "a tensor's class made something that is no tensor");
    }
    return THPVariable_Unpack(made);
  }
  void replace(PyObject* made) {
    tensor_ = unpacked(made);
    Py_DECREF(object_);
    object_ = made;
  }
  PyObject* object_;
  Tensor tensor_;
};

// (seed, offset) of the device's default generator, advancing the offset by 4 under its lock
struct Draw {
  uint64_t seed, offset;
  explicit Draw(const Tensor& t) {
    at::Generator gen = at::globalContext().defaultGenerator(t.device());
    std::lock_guard<std::mutex> lock(gen.mutex());
    seed = gen.current_seed();
    offset = gen.get_offset();
    gen.set_offset(offset + 4);
  }
};

// the sensitivity's multiplier: nothing, one device scalar or one fp32 value per sample on the same device
struct Mult {
  Tensor held;
  int per_sample = 0;
  Mult(Tensor mult, int64_t N, const Tensor& like) {
    if (!mult.defined()) return;
    TORCH_CHECK(mult.scalar_type() == at::kFloat && mult.device() == like.device() && (mult.numel() == 1 || mult.numel() == N),
                "the sensitivity's multiplier must be fp32 on the same device with 1 or N values");
    held = mult.contiguous();
    per_sample = mult.numel() == N && N != 1;
  }
};

constexpr int64_t kMaskBlock = 512;
int64_t mask_words(int64_t n) { return (n + kMaskBlock - 1) / kMaskBlock * 16; }
int64_t single_packed_bytes(int64_t N, int64_t G, int64_t bits) {
  const int64_t per = 8 / bits, rounded = (N + per - 1) / per * per;
  return (bits * rounded * G * 256 + 8) / 8;
}

// ---------------------------------------------------------------------------- compress / restore
// rows, N, mn | None, mx | None, factor, mult | None, initial, target, total, sens | None, stored dtype
//   -> packed, bits, scale, stored minimum, prefix
PyObject* quantize_rows(PyObject* const* a, Py_ssize_t n) {
  Args args(a, n, 11);
  const Tensor rows = args.tensor();
  const int64_t N = args.integer();
  Tensor mn = args.optional(), mx = args.optional();
  const double factor = args.number();
  const Mult mult(args.optional(), N, rows);
  const int64_t initial = args.integer(), target = args.integer(), total = args.integer();
  Tensor sens = args.optional();
  const auto dtype = rows.scalar_type();
  const auto store = type_of(args.integer());
  TORCH_CHECK(N > 0 && total >= 0, "quantize_rows: no samples");
  const int64_t F = rows.numel() / N, G = (F + 255) / 256;
  const bool known = mn.defined();
  const c10::DeviceGuard guard(rows.device());
  if (!known) {
    mn = empty({N * G}, rows, dtype);
    mx = empty({N * G}, rows, dtype);
  }
  const Tensor stored = store == dtype ? mn : empty({N * G}, rows, store);
  if (!sens.defined()) sens = empty({N}, rows, at::kFloat);
  const Tensor bits = empty({N}, rows, at::kInt), prefix = empty({N + 1}, rows, at::kInt);
  const Tensor packed = empty({total * G * 8}, rows, at::kInt), scale = empty({N, G, 1}, rows, store);
  const Draw draw(rows);
  launch("quantize_activation", [&] {
      return actnn_quantize_rows(ptr(rows), ptr(mn), ptr(mx), known, (float)factor, f32(mult.held), mult.per_sample, f32(sens),
                           i32(bits), i32(prefix), (int)initial, target, ptr(scale), ptr(stored), i32(packed), draw.seed,
                           draw.offset, N, F, code_of(dtype), code_of(store), stream_of(rows));
  });
  return tuple_of(packed, bits, scale, stored, prefix);
}

// rows [N, F], width, mn | None, mx | None (of whole groups), stored dtype -> packed, scale, minimum
PyObject* quantize_rows_fixed(PyObject* const* a, Py_ssize_t n) {
  Args args(a, n, 5);
  const Tensor rows = args.tensor();
  const int64_t bits = args.integer();
  const Tensor known_mn = args.optional(), known_mx = args.optional();
  const auto dtype = rows.scalar_type();
  const auto store = type_of(args.integer());
  TORCH_CHECK(rows.dim() == 2, "quantize_rows_fixed: rows must have two dimensions, got ", rows.dim());
  TORCH_CHECK(bits >= 1 && bits <= 8 && 8 % bits == 0, "quantize_rows_fixed: 8 % bits must be 0, got ", bits);
  const int64_t N = rows.size(0), F = rows.size(1), G = (F + 255) / 256;
  const c10::DeviceGuard guard(rows.device());
  const Tensor packed = empty({single_packed_bytes(N, G, bits)}, rows, at::kChar), scale = empty({N, G, 1}, rows, store);
  const bool keeps = known_mn.defined() && store == known_mn.scalar_type();       // the given minimum is what is stored
  const Tensor mn = keeps ? known_mn.view({N, G, 1}) : empty({N, G, 1}, rows, store);
  const Draw draw(rows);
  launch("quantize_fixed", [&] {
      return actnn_quantize_fixed(ptr(rows), ptr(known_mn), ptr(known_mx), (int)bits, ptr(scale), keeps ? nullptr : ptr(mn),
                            static_cast<int8_t*>(ptr(packed)), draw.seed, draw.offset, N, F, code_of(dtype), code_of(store),
                            stream_of(rows));
  });
  return tuple_of(packed, scale, mn);
}

bool holds(const Tensor& t, at::ScalarType dtype, int64_t dim) {
  return t.is_cuda() && t.is_contiguous() && t.dim() == dim && t.scalar_type() == dtype;
}
bool holds_float(const Tensor& t, int64_t dim) {
  return t.is_cuda() && t.is_contiguous() && t.dim() == dim &&
         (t.scalar_type() == at::kFloat || t.scalar_type() == at::kHalf || t.scalar_type() == at::kBFloat16);
}

// packed, bits, prefix, sum of the widths, scale, mn, N, F, dtype -> [N, F], or None for arguments that do not fit
// together (the caller's own checks then say which)
PyObject* unpack_rows_mixed(PyObject* const* a, Py_ssize_t n) {
  Args args(a, n, 9);
  if (!args.tensors(3) || !THPVariable_Check(a[4]) || !THPVariable_Check(a[5])) Py_RETURN_NONE;
  const Tensor packed = args.tensor(), bits = args.tensor(), prefix = args.tensor();
  const int64_t total = args.integer();
  const Tensor scale = args.tensor(), mn = args.tensor();
  const int64_t N = args.integer(), F = args.integer(), G = (F + 255) / 256;
  const auto dtype = type_of(args.integer());
  if (!(holds(packed, at::kInt, 1) && holds(bits, at::kInt, 1) && holds_float(scale, 3) && holds_float(mn, 3) &&
        mn.scalar_type() == scale.scalar_type() && scale.numel() == N * G && mn.numel() == N * G && bits.numel() == N &&
        packed.numel() >= total * G * 8))
    Py_RETURN_NONE;
  const c10::DeviceGuard guard(packed.device());
  const Tensor out = empty({N, F}, packed, dtype);
  launch("unpack_mixed_precision", [&] {
      return actnn_unpack_mixed_rows(i32(packed), i32(bits), i32(prefix), ptr(scale), ptr(mn), ptr(out), N, F, code_of(dtype),
                               code_of(scale.scalar_type()), stream_of(packed));
  });
  return wrap(out);
}

// packed, width, scale, mn, N, F, dtype -> [N, F], or None as above
PyObject* unpack_rows_fixed(PyObject* const* a, Py_ssize_t n) {
  Args args(a, n, 7);
  if (!args.tensors(1) || !THPVariable_Check(a[2]) || !THPVariable_Check(a[3])) Py_RETURN_NONE;
  const Tensor packed = args.tensor();
  const int64_t bits = args.integer();
  const Tensor scale = args.tensor(), mn = args.tensor();
  const int64_t N = args.integer(), F = args.integer(), G = (F + 255) / 256;
  const auto dtype = type_of(args.integer());
  if (!(bits >= 1 && bits <= 8 && 8 % bits == 0 && holds(packed, at::kChar, 1) && holds_float(scale, 3) && holds_float(mn, 3) &&
        mn.scalar_type() == scale.scalar_type() && scale.numel() == N * G && mn.numel() == N * G &&
        packed.numel() >= single_packed_bytes(N, G, bits) - 1))
    Py_RETURN_NONE;
  const c10::DeviceGuard guard(packed.device());
  const Tensor out = empty({N, F}, packed, dtype);
  launch("unpack_single_precision", [&] {
      return actnn_unpack_single_rows(static_cast<int8_t*>(ptr(packed)), (int)bits, ptr(scale), ptr(mn), ptr(out), N, F, code_of(dtype),
                                code_of(scale.scalar_type()), stream_of(packed));
  });
  return wrap(out);
}

// ---------------------------------------------------------------------------- masks
// x -> relu(x), mask;  x, p -> dropout(x), mask
PyObject* mask_forward(Args& args, bool dropout) {
  Given given(args.tensor_object());
  given.make_aligned();
  const Tensor& x = given.tensor();
  TORCH_CHECK(x.is_cuda(), "input must be a CUDA tensor!");
  const double p = dropout ? args.number() : 0.0;
  const int64_t count = x.numel();
  const c10::DeviceGuard guard(x.device());
  const Tensor y = given.empty_like(), mask = empty({mask_words(count)}, x, at::kInt);
  const int code = code_of(x.scalar_type());
  if (dropout) {
    const Draw draw(x);
    launch("dropout_forward", [&] {
      return actnn_dropout_forward(ptr(x), ptr(y), i32(mask), count, (float)p, draw.seed, draw.offset, code, stream_of(x));
  });
  } else {
    launch("relu_forward", [&] {
      return actnn_relu_forward(ptr(x), ptr(y), i32(mask), count, code, stream_of(x));
  });
  }
  return tuple_of(y, mask);
}
PyObject* relu_forward(PyObject* const* a, Py_ssize_t n) {
  Args args(a, n, 1);
  return mask_forward(args, false);
}
PyObject* dropout_forward(PyObject* const* a, Py_ssize_t n) {
  Args args(a, n, 2);
  return mask_forward(args, true);
}

// grad, mask[, p] -> gradient of the input
PyObject* mask_backward(Args& args, bool dropout) {
  Given given(args.tensor_object());
  given.make_contiguous();                             // (the order the kernel reads and writes in: before the result is made)
  given.make_aligned();
  const Tensor& grad = given.tensor();
  const Tensor mask = args.tensor();
  TORCH_CHECK(grad.is_cuda() && mask.is_cuda(), "grad_output must be a CUDA tensor!");
  const double p = dropout ? args.number() : 0.0;
  const c10::DeviceGuard guard(grad.device());
  const Tensor out = given.empty_like();
  const int code = code_of(grad.scalar_type());
  if (dropout)
    launch("dropout_backward", [&] {
      return actnn_dropout_backward(ptr(grad), i32(mask), ptr(out), out.numel(), (float)p, code, stream_of(grad));
  });
  else
    launch("relu_backward", [&] {
      return actnn_relu_backward(ptr(grad), i32(mask), ptr(out), out.numel(), code, stream_of(grad));
  });
  return wrap(out);
}
PyObject* relu_backward(PyObject* const* a, Py_ssize_t n) {
  Args args(a, n, 2);
  return mask_backward(args, false);
}
PyObject* dropout_backward(PyObject* const* a, Py_ssize_t n) {
  Args args(a, n, 3);
  return mask_backward(args, true);
}

// ---------------------------------------------------------------------------- batch norm
// x[, parameters] -> (N, C, HW, channels last) of a dense tensor the batch-norm kernels take, or None.  With parameters (None
// or tensors): None as well unless x is 16-byte aligned and each of them dense fp32 on a GPU.
PyObject* batch_norm_geometry(PyObject* const* a, Py_ssize_t n) {
  TORCH_CHECK(n >= 1, "expected a tensor");
  if (!THPVariable_Check(a[0])) Py_RETURN_NONE;
  const Tensor& x = THPVariable_Unpack(a[0]);
  const auto dtype = x.scalar_type();
  if (!x.is_cuda() || x.dim() < 2 || (dtype != at::kFloat && dtype != at::kHalf && dtype != at::kBFloat16)) Py_RETURN_NONE;
  const bool dense = x.is_contiguous();
  const bool cl = !dense && ((x.dim() == 4 && x.is_contiguous(at::MemoryFormat::ChannelsLast)) ||
                             (x.dim() == 5 && x.is_contiguous(at::MemoryFormat::ChannelsLast3d)));
  if (!dense && !cl) Py_RETURN_NONE;
  const int64_t N = x.size(0), C = x.size(1);
  int64_t HW = 1;
  for (int64_t d = 2; d < x.dim(); ++d) HW *= x.size(d);
  if (N * C * HW == 0 || actnn_batch_norm_workspace_bytes(N, C, HW, code_of(dtype), cl) < 0) Py_RETURN_NONE;
  if (n > 1 && reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 != 0) Py_RETURN_NONE;
  for (Py_ssize_t i = 1; i < n; ++i) {
    if (a[i] == Py_None) continue;
    if (!THPVariable_Check(a[i])) Py_RETURN_NONE;
    const Tensor& t = THPVariable_Unpack(a[i]);
    if (t.scalar_type() != at::kFloat || !t.is_cuda() || !t.is_contiguous()) Py_RETURN_NONE;
  }
  return Py_BuildValue("(LLLO)", (long long)N, (long long)C, (long long)HW, cl ? Py_True : Py_False);
}

struct BnGeometry {
  int64_t N, C, HW;
  int code, channels_last;
  BnGeometry(Args& args, const Tensor& x) {
    N = args.integer();
    C = args.integer();
    HW = args.integer();
    channels_last = args.flag();
    code = code_of(x.scalar_type());
  }
  int64_t workspace() const { return actnn_batch_norm_workspace_bytes(N, C, HW, code, channels_last); }
  int64_t sumsq_entries() const { return actnn_batch_norm_backward_sumsq_entries(N, C, HW, code, channels_last); }
};

// x, N, C, HW, channels last, weight, bias, running mean, running variance (None or fp32), momentum, eps, factor,
// mult | None, initial, target, total, sens | None, relu, residual | None
//   -> y, mean, invstd, mn, mx, bits, packed, scale, prefix, mask, mn of y, mx of y (the last three None without relu)
PyObject* batch_norm_forward_quantize(PyObject* const* a, Py_ssize_t n) {
  Args args(a, n, 19);
  const Tensor x = args.tensor();
  const BnGeometry g(args, x);
  const Tensor weight = args.optional(), bias = args.optional(), running_mean = args.optional(), running_var = args.optional();
  const double momentum = args.number(), eps = args.number(), factor = args.number();
  const Mult mult(args.optional(), g.N, x);
  const int64_t initial = args.integer(), target = args.integer(), total = args.integer();
  Tensor sens = args.optional();
  const bool relu = args.flag();
  const Tensor residual = args.optional();
  const auto dtype = x.scalar_type();
  const int64_t G = g.C * g.HW / 256, ws_bytes = g.workspace();
  const c10::DeviceGuard guard(x.device());
  const Tensor ws = empty({ws_bytes / 4}, x, at::kFloat), mean = empty({g.C}, x, at::kFloat), invstd = empty({g.C}, x, at::kFloat);
  const Tensor mn = empty({g.N * G}, x, dtype), mx = empty({g.N * G}, x, dtype), y = Given(a[0]).empty_like();
  if (!sens.defined()) sens = empty({g.N}, x, at::kFloat);
  const Tensor bits = empty({g.N}, x, at::kInt), prefix = empty({g.N + 1}, x, at::kInt);
  const Tensor packed = empty({total * G * 8}, x, at::kInt), scale = empty({g.N, G, 1}, x, dtype);
  Tensor mask, ymn, ymx;
  if (relu) {
    mask = empty({mask_words(g.N * g.C * g.HW)}, x, at::kInt);
    ymn = empty({g.N * G}, x, dtype);
    ymx = empty({g.N * G}, x, dtype);
  }
  const Draw draw(x);
  launch("batch_norm_forward_quantize", [&] {
      return actnn_batch_norm_forward_quantize(
           ptr(x), f32(weight), f32(bias), f32(running_mean), f32(running_var), ptr(y), f32(mean), f32(invstd), ptr(mn), ptr(mx),
           ptr(ws), ws_bytes, (float)factor, f32(mult.held), mult.per_sample, f32(sens), i32(bits), i32(prefix), (int)initial,
           target, ptr(scale), i32(packed), draw.seed, draw.offset, i32(mask), ptr(ymn), ptr(ymx), ptr(residual), g.N, g.C, g.HW,
           momentum, eps, g.code, g.channels_last, stream_of(x));
  });
  return tuple_of(y, mean, invstd, mn, mx, bits, packed, scale, prefix, mask, ymn, ymx);
}

// x, N, C, HW, channels last, weight, bias, running mean, running variance, momentum, eps, group ranges too
//   -> y, mean, invstd, mn, mx (None without)
PyObject* batch_norm_forward(PyObject* const* a, Py_ssize_t n) {
  Args args(a, n, 12);
  const Tensor x = args.tensor();
  const BnGeometry g(args, x);
  const Tensor weight = args.optional(), bias = args.optional(), running_mean = args.optional(), running_var = args.optional();
  const double momentum = args.number(), eps = args.number();
  const bool ranges = args.flag();
  const int64_t ws_bytes = g.workspace();
  const c10::DeviceGuard guard(x.device());
  const Tensor ws = empty({ws_bytes / 4}, x, at::kFloat), y = Given(a[0]).empty_like();
  const Tensor mean = empty({g.C}, x, at::kFloat), invstd = empty({g.C}, x, at::kFloat);
  Tensor mn, mx;
  if (ranges) {
    const int64_t groups = g.N * (g.C * g.HW / 256);
    mn = empty({groups}, x, x.scalar_type());
    mx = empty({groups}, x, x.scalar_type());
  }
  launch("batch_norm_forward", [&] {
      return actnn_batch_norm_forward(ptr(x), f32(weight), f32(bias), f32(running_mean), f32(running_var), ptr(y), f32(mean), f32(invstd),
                                ptr(mn), ptr(mx), ptr(ws), ws_bytes, g.N, g.C, g.HW, momentum, eps, g.code, g.channels_last,
                                stream_of(x));
  });
  return tuple_of(y, mean, invstd, mn, mx);
}

// x, dy, N, C, HW, channels last, weight | None, mean, invstd, sumsq -> dx, dweight, dbias, squares of dx (None without)
PyObject* batch_norm_backward(PyObject* const* a, Py_ssize_t n) {
  Args args(a, n, 10);
  const Tensor x = args.tensor(), dy = args.tensor();
  const BnGeometry g(args, x);
  const Tensor weight = args.optional(), mean = args.tensor(), invstd = args.tensor();
  const int64_t entries = args.flag() ? g.sumsq_entries() : 0, ws_bytes = g.workspace();
  const c10::DeviceGuard guard(x.device());
  const Tensor ws = empty({ws_bytes / 4 + entries}, x, at::kFloat), dx = Given(a[0]).empty_like();
  const Tensor dweight = empty({g.C}, x, at::kFloat), dbias = empty({g.C}, x, at::kFloat);
  launch("batch_norm_backward", [&] {
      return actnn_batch_norm_backward(ptr(x), ptr(dy), f32(weight), f32(mean), f32(invstd), ptr(dx), f32(dweight), f32(dbias), ptr(ws),
                                 ws_bytes, entries ? f32(ws) + ws_bytes / 4 : nullptr, entries, g.N, g.C, g.HW, g.code,
                                 g.channels_last, stream_of(x));
  });
  return tuple_of(dx, dweight, dbias, entries ? ws.narrow(0, ws_bytes / 4, entries) : Tensor());
}

// packed, bits, prefix, scale, mn, dy, N, C, HW, channels last, weight | None, mean, invstd, sumsq, mask | None,
// masked | None -> dx, dweight, dbias, squares of dx (None without)
PyObject* batch_norm_backward_packed(PyObject* const* a, Py_ssize_t n) {
  Args args(a, n, 16);
  const Tensor packed = args.tensor(), bits = args.tensor(), prefix = args.tensor(), scale = args.tensor(), mn = args.tensor();
  const Tensor dy = args.tensor();
  const BnGeometry g(args, dy);
  const Tensor weight = args.optional(), mean = args.tensor(), invstd = args.tensor();
  const int64_t entries = args.flag() ? g.sumsq_entries() : 0, ws_bytes = g.workspace();
  const Tensor mask = args.optional(), masked = args.optional();
  const c10::DeviceGuard guard(dy.device());
  const Tensor ws = empty({ws_bytes / 4 + entries}, dy, at::kFloat), dx = Given(a[5]).empty_like();
  const Tensor dweight = empty({g.C}, dy, at::kFloat), dbias = empty({g.C}, dy, at::kFloat);
  float* squares = entries ? f32(ws) + ws_bytes / 4 : nullptr;
  if (mask.defined())
    launch("batch_norm_backward_packed_relu", [&] {
      return actnn_batch_norm_backward_packed_add_relu(
             i32(packed), i32(bits), i32(prefix), ptr(scale), ptr(mn), ptr(dy), i32(mask), ptr(masked), f32(weight), f32(mean),
             f32(invstd), ptr(dx), f32(dweight), f32(dbias), ptr(ws), ws_bytes, squares, entries, g.N, g.C, g.HW, g.code,
             g.channels_last, stream_of(dy));
  });
  else
    launch("batch_norm_backward_packed", [&] {
      return actnn_batch_norm_backward_packed(
             i32(packed), i32(bits), i32(prefix), ptr(scale), ptr(mn), ptr(dy), f32(weight), f32(mean), f32(invstd), ptr(dx),
             f32(dweight), f32(dbias), ptr(ws), ws_bytes, squares, entries, g.N, g.C, g.HW, g.code, g.channels_last,
             stream_of(dy));
  });
  return tuple_of(dx, dweight, dbias, entries ? ws.narrow(0, ws_bytes / 4, entries) : Tensor());
}

// ---------------------------------------------------------------------------- max-pool
// x (dense in its format), channels last, window, stride, padding, dilation (two each), two indices a byte -> y, indices
PyObject* max_pool2d_forward(PyObject* const* a, Py_ssize_t n) {
  Args args(a, n, 11);
  const Tensor x = args.tensor();
  const bool cl = args.flag();
  int64_t v[8];
  for (int64_t& q : v) q = args.integer();
  const bool nibble = args.flag();
  TORCH_CHECK(x.is_cuda() && x.dim() == 4, "The dimension of input is not correct!");
  const int64_t N = x.size(0), C = x.size(1), H = x.size(2), W = x.size(3);
  // (rounded down, as Python's division does, also for windows larger than the padded image)
  auto out = [](int64_t size, int64_t k, int64_t s, int64_t p, int64_t d) {
    const int64_t room = size + 2 * p - d * (k - 1) - 1;
    TORCH_CHECK(s != 0, "stride must not be zero");
    return room / s - (room % s != 0 && (room < 0) != (s < 0)) + 1;
  };
  const int64_t Ho = out(H, v[0], v[2], v[4], v[6]), Wo = out(W, v[1], v[3], v[5], v[7]);
  const auto format = cl ? at::MemoryFormat::ChannelsLast : at::MemoryFormat::Contiguous;
  const c10::DeviceGuard guard(x.device());
  const auto options = at::TensorOptions().device(x.device()).memory_format(format);
  const Tensor y = at::empty({N, C, Ho, Wo}, options.dtype(x.scalar_type()));
  const Tensor idx = nibble ? empty({(N * C * Ho * Wo + 1) / 2}, x, at::kByte) : at::empty({N, C, Ho, Wo}, options.dtype(at::kChar));
  const int code = code_of(x.scalar_type());
  launch("max_pool2d_forward", [&] {
    auto to = [&](auto f, auto* index) {
      return f(ptr(x), ptr(y), index, N, C, H, W, Ho, Wo, (int)v[0], (int)v[1], (int)v[2], (int)v[3], (int)v[4], (int)v[5], code,
               stream_of(x));
    };
    if (nibble)
      return to(cl ? actnn_max_pool2d_forward_cl_nibble : actnn_max_pool2d_forward_nibble, static_cast<uint8_t*>(ptr(idx)));
    return to(cl ? actnn_max_pool2d_forward_cl : actnn_max_pool2d_forward, static_cast<int8_t*>(ptr(idx)));
  });
  return tuple_of(y, idx);
}

// grad (dense in its format), indices, channels last, two indices a byte, N, C, H, W, window, stride, padding -> gradient
PyObject* max_pool2d_backward(PyObject* const* a, Py_ssize_t n) {
  Args args(a, n, 14);
  const Tensor grad = args.tensor(), idx = args.tensor();
  const bool cl = args.flag(), nibble = args.flag();
  int64_t size[4], v[6];
  for (int64_t& q : size) q = args.integer();
  for (int64_t& q : v) q = args.integer();
  TORCH_CHECK(grad.is_cuda() && grad.dim() == 4, "The dimension of grad_output is not correct!");
  const c10::DeviceGuard guard(grad.device());
  const Tensor out = at::empty({size[0], size[1], size[2], size[3]},
                               at::TensorOptions().device(grad.device()).dtype(grad.scalar_type()).memory_format(
                                   cl ? at::MemoryFormat::ChannelsLast : at::MemoryFormat::Contiguous));
  const int code = code_of(grad.scalar_type());
  launch("max_pool2d_backward", [&] {
    auto to = [&](auto f, auto* index) {
      return f(ptr(grad), index, ptr(out), size[0], size[1], size[2], size[3], grad.size(2), grad.size(3), (int)v[0], (int)v[1],
               (int)v[2], (int)v[3], (int)v[4], (int)v[5], code, stream_of(grad));
    };
    if (nibble)
      return to(cl ? actnn_max_pool2d_backward_cl_nibble : actnn_max_pool2d_backward_nibble, static_cast<uint8_t*>(ptr(idx)));
    return to(cl ? actnn_max_pool2d_backward_cl : actnn_max_pool2d_backward, static_cast<int8_t*>(ptr(idx)));
  });
  return wrap(out);
}

template <PyObject* (*F)(PyObject* const*, Py_ssize_t)>
PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  return F(args, n);
  END_HANDLE_TH_ERRORS
}
#define ACTNN_CALL(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&call<name>)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    ACTNN_CALL(quantize_rows), ACTNN_CALL(quantize_rows_fixed), ACTNN_CALL(unpack_rows_mixed), ACTNN_CALL(unpack_rows_fixed),
    ACTNN_CALL(relu_forward), ACTNN_CALL(relu_backward), ACTNN_CALL(dropout_forward), ACTNN_CALL(dropout_backward),
    ACTNN_CALL(batch_norm_geometry), ACTNN_CALL(batch_norm_forward_quantize), ACTNN_CALL(batch_norm_forward), ACTNN_CALL(batch_norm_backward),
    ACTNN_CALL(batch_norm_backward_packed), ACTNN_CALL(max_pool2d_forward), ACTNN_CALL(max_pool2d_backward), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) { return PyModule_Create(&module); }

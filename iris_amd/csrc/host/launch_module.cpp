// The Python launchers' way to the C-ABI (include/iris_amd.h): a CPython module that checks the operands, fills the
// argument struct and launches on torch's current stream without going through Python for any of it.
//
// A launch of a few rows is 7 us of GPU work.  Checked and filled in Python (nine tensors, some sixty attribute
// reads, a ctypes struct, a device context) it cost 15 us of host time a launch, and a stream of such launches ran at the
// host's pace; here it costs what the runtime's launch call does.
//
// Every function takes the ordinary, well-formed call and nothing else.  Anything it is not sure of (a tensor of
// another type, a subclass, a wrong extent, another current device) it declines before anything is launched, and
// the Python code behind it runs the full checks, which raise what they always did.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/core/grad_mode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include "../../../include/iris_amd.h"

namespace {

constexpr int DECLINED = -1;

// Read off the file by iris_amd/build.py and iris_amd/_native.py before it is loaded.
__attribute__((used)) const char built_for[] = "iris_amd._launch built for " IRIS_BUILT_FOR;

// A plain strided tensor of the device, or (for None) nothing.  False: not for this module.
struct Operand {
  const at::Tensor* t = nullptr;
  explicit operator bool() const { return t != nullptr; }
  void* ptr() const { return t ? t->data_ptr() : nullptr; }
};

bool plain(const at::Tensor& t) {
  using c10::DispatchKey;
  static const c10::DispatchKeySet wrapped({DispatchKey::Python, DispatchKey::Functionalize, DispatchKey::Conjugate,
                                            DispatchKey::Negative, DispatchKey::ZeroTensor, DispatchKey::FuncTorchBatched,
                                            DispatchKey::FuncTorchGradWrapper});
  return t.defined() && t.layout() == c10::kStrided && t.has_storage() && !t.key_set().has_any(wrapped);
}

// Whether this thread is being traced, or inside a transform or a dispatch mode (torch.func, functionalization,
// make_fx, ...): autograd's apply records a function there, or refuses it, and a launch of our own would pass it by.
bool watched() {
  using c10::DispatchKey;
  static const c10::DispatchKeySet modes({DispatchKey::FuncTorchDynamicLayerFrontMode, DispatchKey::FuncTorchDynamicLayerBackMode,
                                          DispatchKey::FuncTorchVmapMode, DispatchKey::FuncTorchBatched,
                                          DispatchKey::FuncTorchGradWrapper, DispatchKey::Functionalize, DispatchKey::Python,
                                          DispatchKey::PythonTLSSnapshot, DispatchKey::PythonDispatcher, DispatchKey::PreDispatch,
                                          DispatchKey::Tracer});
  return torch::jit::tracer::isTracing() || c10::impl::tls_local_dispatch_key_set().included_.has_any(modes);
}

// Whether autograd has business with a tensor among the arguments: a gradient, or a tangent (forward mode).
bool differentiated(PyObject* const* x, Py_ssize_t n) {
  for (Py_ssize_t i = 0; i < n; ++i) {
    // (what most arguments are: the check for a tensor asks its metaclass about each of these)
    if (x[i] == Py_None || PyLong_Check(x[i]) || PyUnicode_Check(x[i]) || !THPVariable_Check(x[i])) continue;
    const at::Tensor& t = THPVariable_Unpack(x[i]);
    if (!plain(t) || (at::GradMode::is_enabled() && t.requires_grad()) || t._fw_grad(/*level=*/0).defined()) return true;
  }
  return false;
}

bool operand(PyObject* o, int device, Operand* out) {
  if (o == Py_None) return true;
  if (!THPVariable_CheckExact(o)) return false;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!plain(t) || !t.is_cuda() || t.get_device() != device) return false;
  out->t = &t;
  return true;
}

// Python ints (bools too) only: anything else is left to the Python code's conversions.
bool integer(PyObject* o, int64_t lo, int64_t hi, int64_t* out) {
  if (!PyLong_Check(o)) return false;
  int overflow = 0;
  const long long v = PyLong_AsLongLongAndOverflow(o, &overflow);
  if (overflow || v < lo || v > hi) return false;
  *out = v;
  return true;
}
bool int32(PyObject* o, int32_t* out) {
  int64_t v;
  if (!integer(o, INT32_MIN, INT32_MAX, &v)) return false;
  *out = (int32_t)v;
  return true;
}
bool ticks(PyObject* o, uint64_t* out) {
  int64_t v;
  if (!integer(o, 0, INT64_MAX, &v)) return false;
  *out = (uint64_t)v;
  return true;
}

int dtype_code(const at::Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return IRIS_DTYPE_F32;
    case at::kHalf: return IRIS_DTYPE_F16;
    case at::kBFloat16: return IRIS_DTYPE_BF16;
    default: return -1;
  }
}

bool matrix_of(const Operand& t, int64_t rows, int64_t cols) {
  return t && t.t->dim() == 2 && t.t->size(0) >= rows && t.t->size(1) >= cols;
}

bool contiguous(const Operand& t, at::ScalarType type, int64_t numel) {
  return t.t->scalar_type() == type && t.t->numel() >= numel && t.t->is_contiguous();
}

int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

bool flags_ok(const Operand& flags, int64_t tiles) { return !flags || contiguous(flags, at::kInt, tiles); }

bool bases_ok(const Operand& bases, int64_t ranks) {
  if (!bases) return ranks <= 1;
  const auto type = bases.t->scalar_type();
  return (type == at::kUInt64 || type == at::kLong) && bases.t->numel() >= ranks;
}

// The device a launch's tensors must share: the first one's, which must be the current one too.
int launch_device(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return -1;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!plain(t) || !t.is_cuda()) return -1;
  int current = -1;
  if (hipGetDevice(&current) != hipSuccess || current != t.get_device()) return -1;
  return current;
}

void* current_stream(int device) { return c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream(); }

template <class Launch>
int unlocked(Launch launch) {
  int err;
  Py_BEGIN_ALLOW_THREADS;
  err = launch();
  Py_END_ALLOW_THREADS;
  return err;
}

struct GemmOperands {
  Operand a, b, c, c_global, flags, bases, ts_begin, ts_end, status, partials, locks;
};

// The tensors' share of iris_gemm_args, checked as ops.gemm_launch documents it; `g` holds the numbers already.
bool fill_gemm(const GemmOperands& t, iris_gemm_args* g) {
  if (!t.a || !t.b || t.a.t->dim() != 2 || t.b.t->dim() != 2) return false;
  const int64_t M = t.a.t->size(0), K = t.a.t->size(1), N = t.b.t->size(1);
  if (t.b.t->size(0) != K || M > INT32_MAX || N > INT32_MAX || K > INT32_MAX) return false;
  const int dt = dtype_code(*t.a.t);
  if (dt < 0 || t.b.t->scalar_type() != t.a.t->scalar_type()) return false;
  if (g->block_m <= 0 || g->block_n <= 0 || g->group_size_m <= 0 || g->num_sms <= 0 || g->world_size <= 0) return false;
  const int64_t tiles = cdiv(M, g->block_m) * cdiv(N, g->block_n);
  switch (g->epilogue) {
    case IRIS_EPI_ALL_SCATTER:
      if (!matrix_of(t.c_global, M, N * g->world_size)) return false;
      break;
    case IRIS_EPI_ATOMIC_ADD:
      if (!matrix_of(t.c_global, M, N)) return false;
      break;
    case IRIS_EPI_ONE_SHOT:
      if (!matrix_of(t.c, M, N) || !matrix_of(t.c_global, M, N)) return false;
      break;
    default: return false;
  }
  if (!flags_ok(t.flags, tiles) || !bases_ok(t.bases, g->world_size)) return false;
  if (t.ts_begin && !contiguous(t.ts_begin, at::kLong, tiles)) return false;
  if (t.ts_end && !contiguous(t.ts_end, at::kLong, tiles)) return false;
  if (t.status && !((t.status.t->scalar_type() == at::kInt || t.status.t->scalar_type() == at::kUInt32) && t.status.t->numel() >= 1))
    return false;
  g->a = t.a.ptr();
  g->b = t.b.ptr();
  g->c = t.c.ptr();
  g->c_global = t.c_global.ptr();
  g->tile_completed = static_cast<int32_t*>(t.flags.ptr());
  g->heap_bases = static_cast<const uint64_t*>(t.bases.ptr());
  g->mm_begin_timestamp = static_cast<int64_t*>(t.ts_begin.ptr());
  g->mm_end_timestamp = static_cast<int64_t*>(t.ts_end.ptr());
  g->status = static_cast<uint32_t*>(t.status.ptr());
  g->M = (int32_t)M;
  g->N = (int32_t)N;
  g->K = (int32_t)K;
  g->stride_am = t.a.t->stride(0);
  g->stride_ak = t.a.t->stride(1);
  g->stride_bk = t.b.t->stride(0);
  g->stride_bn = t.b.t->stride(1);
  g->ab_dtype = dt;
  if (t.c) {
    if (t.c.t->dim() != 2 || (g->c_dtype = dtype_code(*t.c.t)) < 0) return false;
    g->stride_cm = t.c.t->stride(0);
    g->stride_cn = t.c.t->stride(1);
  }
  if (t.c_global) {
    if ((g->c_global_dtype = dtype_code(*t.c_global.t)) < 0) return false;
    g->stride_cm_global = t.c_global.t->stride(0);
    g->stride_cn_global = t.c_global.t->stride(1);
  }
  if (t.locks) {
    if (!contiguous(t.locks, at::kInt, g->num_sms)) return false;
    g->locks = static_cast<int32_t*>(t.locks.ptr());
  }
  if (t.partials) {
    if (!t.locks || t.partials.t->scalar_type() != at::kFloat || t.partials.t->dim() != 2 || !t.partials.t->is_contiguous() ||
        t.partials.t->size(0) < g->num_sms)
      return false;
    g->partials = static_cast<float*>(t.partials.ptr());
    g->partials_slot_elems = t.partials.t->size(1);
  } else if (g->split_k > 1 || g->split_k == IRIS_GEMM_SPLIT_STREAM_K) {
    return false;
  }
  return true;
}

// gemm(a, b, c, c_global, tile_completed, heap_bases, mm_begin_timestamp, mm_end_timestamp, status, partials, locks,
//      rank, world_size, num_sms, BLK_M, BLK_N, BLK_K, gsize_m, epilogue, phase, notify, num_xcds, scope, variant,
//      spin_timeout_ticks, split_k, split_handover, flag_sem, touch_ahead)
// -> hipError_t of the launch, or -1: declined, nothing launched.
PyObject* gemm(PyObject*, PyObject* const* v, Py_ssize_t n) {
  if (n != 29) {
    PyErr_SetString(PyExc_TypeError, "gemm takes 29 arguments");
    return nullptr;
  }
  const int device = launch_device(v[0]);
  GemmOperands t;
  iris_gemm_args g{};
  int32_t notify = PyObject_IsTrue(v[20]);
  const bool ok =
      device >= 0 && operand(v[0], device, &t.a) && operand(v[1], device, &t.b) && operand(v[2], device, &t.c) &&
      operand(v[3], device, &t.c_global) && operand(v[4], device, &t.flags) && operand(v[5], device, &t.bases) &&
      operand(v[6], device, &t.ts_begin) && operand(v[7], device, &t.ts_end) && operand(v[8], device, &t.status) &&
      operand(v[9], device, &t.partials) && operand(v[10], device, &t.locks) && int32(v[11], &g.cur_rank) &&
      int32(v[12], &g.world_size) && int32(v[13], &g.num_sms) && int32(v[14], &g.block_m) && int32(v[15], &g.block_n) &&
      int32(v[16], &g.block_k) && int32(v[17], &g.group_size_m) && int32(v[18], &g.epilogue) && int32(v[19], &g.phase) &&
      notify >= 0 && int32(v[21], &g.num_xcds) && int32(v[22], &g.scope) && int32(v[23], &g.variant) &&
      ticks(v[24], &g.spin_timeout_ticks) && int32(v[25], &g.split_k) && int32(v[26], &g.split_handover) &&
      int32(v[27], &g.flag_sem) && int32(v[28], &g.touch_ahead);
  g.notify = notify;
  PyErr_Clear();
  if (!ok || !fill_gemm(t, &g)) return PyLong_FromLong(DECLINED);
  void* stream = current_stream(device);
  return PyLong_FromLong(unlocked([&] { return iris_gemm_launch(&g, stream); }));
}

// The wrappers' P / locks buffers (benchmark.py:136-142) where they have the reference's shapes, else neither.
void workspace(PyObject* P, PyObject* locks, int device, iris_gemm_args* g, GemmOperands* t) {
  Operand p, l;
  if (!operand(P, device, &p) || !operand(locks, device, &l) || !p || !l) return;
  if (p.t->scalar_type() != at::kFloat || p.t->dim() != 2 || !p.t->is_contiguous() || p.t->size(0) < g->num_sms ||
      p.t->size(1) < (int64_t)g->block_m * g->block_n || !contiguous(l, at::kInt, g->num_sms))
    return;
  t->partials = p;
  t->locks = l;
}

// Class attributes of a `matmul` class that steer its launch.
PyObject *s_debug, *s_notify, *s_phase, *s_scope, *s_variant, *s_status, *s_ticks, *s_split_k;

struct Attr {
  PyObject* o;
  Attr(PyObject* cls, PyObject* name) : o(PyObject_GetAttr(cls, name)) {}
  ~Attr() { Py_XDECREF(o); }
  Attr(const Attr&) = delete;
  bool truth(int32_t* out) const { return o && (*out = PyObject_IsTrue(o)) >= 0; }
};

// matmul_apply(cls, epilogue, args): the positional `matmul.apply(*args)` of a wrapper class, when it is not in debug
// mode, no operand wants a gradient or carries a tangent, and nothing traces or transforms the call.  -> what autograd's
// apply returns (a view of `c`, or None); NotImplemented: declined, nothing launched, the caller takes the long way; or the
// hipError_t of a launch that failed (its first kernel may have run, so it is not tried again).
PyObject* matmul_apply(PyObject*, PyObject* const* v, Py_ssize_t n) {
  if (n != 3 || !PyTuple_Check(v[2])) {
    PyErr_SetString(PyExc_TypeError, "matmul_apply(cls, epilogue, args)");
    return nullptr;
  }
  PyObject* const cls = v[0];
  PyObject* const* x = &PyTuple_GET_ITEM(v[2], 0);
  const Py_ssize_t nx = PyTuple_GET_SIZE(v[2]);
  auto decline = [] {
    PyErr_Clear();
    Py_RETURN_NOTIMPLEMENTED;
  };
  // a, b, c, c_global, bias, P, locks, tile_completed, rank, world_size, grid, BLK_M, BLK_N, BLK_K, gsize_m, two_tiles,
  // num_stages, num_warps, waves_per_eu, mfmaInstrSize, kpack, heap_bases_ptr, cu_count, COLLECT_TIMESTAMPS, begin, end
  if (nx < 22 || nx > 26) return decline();
  const int device = launch_device(x[0]);
  if (device < 0) return decline();
  const Attr debug(cls, s_debug), notify(cls, s_notify), phase(cls, s_phase), scope(cls, s_scope), variant(cls, s_variant),
      status(cls, s_status), spin(cls, s_ticks), split_k(cls, s_split_k);
  GemmOperands t;
  iris_gemm_args g{};
  int32_t debug_on, cu_count = 304, collect = 0;
  if (!debug.truth(&debug_on) || debug_on || !notify.truth(&g.notify) || !phase.o || !int32(phase.o, &g.phase) || !scope.o ||
      !int32(scope.o, &g.scope) || !variant.o || !int32(variant.o, &g.variant) || !status.o ||
      !operand(status.o, device, &t.status) || !spin.o || !ticks(spin.o, &g.spin_timeout_ticks) || !split_k.o ||
      !int32(split_k.o, &g.split_k))
    return decline();
  if (!operand(x[0], device, &t.a) || !operand(x[1], device, &t.b) || !operand(x[2], device, &t.c) ||
      !operand(x[3], device, &t.c_global) || !operand(x[7], device, &t.flags) || !int32(x[8], &g.cur_rank) ||
      !int32(x[9], &g.world_size) || !int32(x[10], &g.num_sms) || !int32(x[11], &g.block_m) || !int32(x[12], &g.block_n) ||
      !int32(x[13], &g.block_k) || !int32(x[14], &g.group_size_m) || !operand(x[21], device, &t.bases) || !int32(v[1], &g.epilogue))
    return decline();
  if (nx > 22 && !int32(x[22], &cu_count)) return decline();
  if (nx > 23 && (collect = PyObject_IsTrue(x[23])) < 0) return decline();
  if (collect && ((nx > 24 && !operand(x[24], device, &t.ts_begin)) || (nx > 25 && !operand(x[25], device, &t.ts_end))))
    return decline();
  if (watched() || differentiated(x, nx)) return decline();
  // (ops.default_num_xcds)
  g.num_xcds = (cu_count == 304 || cu_count == 256) && g.num_sms % 8 == 0 ? 8 : 1;
  if (g.num_sms > 0 && g.block_m > 0 && g.block_n > 0) workspace(x[5], x[6], device, &g, &t);
  if (!fill_gemm(t, &g)) return decline();
  void* stream = current_stream(device);
  const int err = unlocked([&] { return iris_gemm_launch(&g, stream); });
  if (err != hipSuccess) return PyLong_FromLong(err);
  if (!t.c) Py_RETURN_NONE;
  try {
    at::NoGradGuard guard;
    return THPVariable_Wrap(t.c.t->view_as(*t.c.t));
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

// one_shot_reduce(c, c_global, tile_completed, heap_bases, status, rank, world_size, BLK_M, BLK_N, gsize_m, num_sms,
//                 num_xcds, scope, wait_flags, variant, spin_timeout_ticks, flag_sem)
PyObject* one_shot_reduce(PyObject*, PyObject* const* v, Py_ssize_t n) {
  if (n != 17) {
    PyErr_SetString(PyExc_TypeError, "one_shot_reduce takes 17 arguments");
    return nullptr;
  }
  const int device = launch_device(v[0]);
  Operand c, c_global, flags, bases, status;
  iris_reduce_args r{};
  r.wait_flags = PyObject_IsTrue(v[13]);
  const bool ok = device >= 0 && operand(v[0], device, &c) && operand(v[1], device, &c_global) && operand(v[2], device, &flags) &&
                  operand(v[3], device, &bases) && operand(v[4], device, &status) && int32(v[5], &r.cur_rank) &&
                  int32(v[6], &r.world_size) && int32(v[7], &r.block_m) && int32(v[8], &r.block_n) &&
                  int32(v[9], &r.group_size_m) && int32(v[10], &r.num_sms) && int32(v[11], &r.num_xcds) &&
                  int32(v[12], &r.scope) && r.wait_flags >= 0 && int32(v[14], &r.variant) &&
                  ticks(v[15], &r.spin_timeout_ticks) && int32(v[16], &r.flag_sem);
  PyErr_Clear();
  if (!ok || c.t->dim() != 2 || !matrix_of(c_global, c.t->size(0), c.t->size(1)) || c.t->size(0) > INT32_MAX ||
      c.t->size(1) > INT32_MAX || r.block_m <= 0 || r.block_n <= 0 || r.group_size_m <= 0 || r.num_sms < 0)
    return PyLong_FromLong(DECLINED);
  const int64_t tiles = cdiv(c.t->size(0), r.block_m) * cdiv(c.t->size(1), r.block_n);
  r.c_dtype = dtype_code(*c.t);
  r.c_global_dtype = dtype_code(*c_global.t);
  if (r.c_dtype < 0 || r.c_global_dtype < 0 || (r.wait_flags && r.world_size > 1 && !flags) || !flags_ok(flags, tiles) ||
      !bases_ok(bases, r.world_size))
    return PyLong_FromLong(DECLINED);
  r.c = c.ptr();
  r.c_global = c_global.ptr();
  r.tile_completed = static_cast<int32_t*>(flags.ptr());
  r.heap_bases = static_cast<const uint64_t*>(bases.ptr());
  r.status = static_cast<uint32_t*>(status.ptr());
  r.M = (int32_t)c.t->size(0);
  r.N = (int32_t)c.t->size(1);
  r.stride_cm = c.t->stride(0);
  r.stride_cn = c.t->stride(1);
  r.stride_cm_global = c_global.t->stride(0);
  r.stride_cn_global = c_global.t->stride(1);
  void* stream = current_stream(device);
  return PyLong_FromLong(unlocked([&] { return iris_one_shot_reduce_launch(&r, stream); }));
}

// memset_i32(tensor, value)
PyObject* memset_i32(PyObject*, PyObject* const* v, Py_ssize_t n) {
  if (n != 2) {
    PyErr_SetString(PyExc_TypeError, "memset_i32(tensor, value)");
    return nullptr;
  }
  const int device = launch_device(v[0]);
  Operand t;
  int32_t value;
  if (device < 0 || !operand(v[0], device, &t) || t.t->scalar_type() != at::kInt || !t.t->is_contiguous() || !int32(v[1], &value))
    return PyLong_FromLong(DECLINED);
  int32_t* p = static_cast<int32_t*>(t.ptr());
  const int64_t count = t.t->numel();
  void* stream = current_stream(device);
  return PyLong_FromLong(unlocked([&] { return iris_memset_i32_launch(p, value, count, stream); }));
}

PyMethodDef methods[] = {
    {"gemm", (PyCFunction)(void (*)(void))gemm, METH_FASTCALL, "launch a shard GEMM; -1: declined"},
    {"matmul_apply", (PyCFunction)(void (*)(void))matmul_apply, METH_FASTCALL, "matmul.apply; NotImplemented: declined, int: failed"},
    {"one_shot_reduce", (PyCFunction)(void (*)(void))one_shot_reduce, METH_FASTCALL, "launch the reduce; -1: declined"},
    {"memset_i32", (PyCFunction)(void (*)(void))memset_i32, METH_FASTCALL, "int32 fill; -1: declined"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_launch", "launches through the C-ABI on torch's current stream", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__launch(void) {
  s_debug = PyUnicode_InternFromString("_debug");
  s_notify = PyUnicode_InternFromString("notify");
  s_phase = PyUnicode_InternFromString("phase");
  s_scope = PyUnicode_InternFromString("scope");
  s_variant = PyUnicode_InternFromString("variant");
  s_status = PyUnicode_InternFromString("status");
  s_ticks = PyUnicode_InternFromString("spin_timeout_ticks");
  s_split_k = PyUnicode_InternFromString("split_k");
  return PyModule_Create(&module);
}

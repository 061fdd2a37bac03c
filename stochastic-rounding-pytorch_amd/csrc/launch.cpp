// Native entries of the launches: the standalone cast, the functional AdamW
// and momentum-SGD updates, and the optimizers' multi-tensor launches.
//
// A launch over up to a few million elements is bound by the host: the HIP
// launch itself costs about 2.2 us, and reaching it through a Python wrapper
// and ctypes added about 4 us to a cast (tensor checks, argument conversion,
// the foreign call) and more to an update.  This CPython extension takes the
// tensors directly, makes the tensor checks the Python wrappers made, with
// their messages, and calls the C ABI's entry points through the addresses
// the Python side binds once.
//
// bind(cast, adamw_step, sgdm_step[, adamw_multi, sgdm_multi])
//   Keep the addresses of sr_cast, sr_adamw_step, sr_sgdm_step,
//   sr_adamw_multi and sr_sgdm_multi, taken from the loaded library.
//
// cast_new(x, dtype_code, rule, seed, offset, threads, stream) -> tensor, int or None
//   cast() into a new contiguous tensor of x's shape and device, allocated
//   here by the call that torch.empty_like makes: about 1.5 us less per call than
//   allocating in Python.  Returns the tensor, or the entry's status where
//   that is not 0.  None, with nothing allocated, for an x that is not
//   exactly a torch.Tensor or Parameter, or under a __torch_function__ mode:
//   there the allocation belongs to the subclass or the mode.
//
// adamw_multi(rows, tile_rows, row_scalars, nrows, total_tiles, p, g, m,
//             m_rule, v, v_rule, hparams, seed, rng_step, block_size, device,
//             stream) -> int
// sgdm_multi(rows, tile_rows, nrows, total_tiles, p, g, u, u_rule, hparams,
//            seed, rng_step, block_size, device, stream) -> int
//   sr_adamw_multi and sr_sgdm_multi with GPU number `device` current; tables
//   and hparams are addresses (row_scalars 0 for none), borrowed for the call.
//   Through ctypes the same call costs 3 us more.
//
// cast(x, out, dtype_code, rule, seed, offset, threads, stream) -> int
//   x: contiguous FP32 tensor; out: contiguous tensor of x's shape and
//   device with the dtype of `dtype_code` (sr_dtype), sharing no byte with
//   x.  Raises ValueError when out breaks that, or when x is not a
//   contiguous FP32 GPU tensor, before anything is launched.
//
// adamw_step(p, g, m, v, m_code, m_rule, v_code, v_rule, scalars, key,
//            offset, block_size, stream) -> int
// sgdm_step(p, g, u, u_code, u_rule, scalars, key, offset, block_size,
//           stream) -> int
//   The tensor checks of the fused single-tensor updates
//   (sr_states/triton/_optimizer.py:24-60): GPU tensors on one device, of
//   one shape, contiguous; FP32 or BF16 parameter and gradient; no byte of
//   the parameter or a state shared with another operand (the gradient is
//   only read).  `scalars` is the tuple of the launch's FP32 scalars as the
//   host computed them (sr_adamw_hparams' eight fields in order, or
//   sr_sgdm_hparams' two), each rounded to FP32 here as ctypes rounds a
//   Python float.  Raises TypeError or ValueError before anything is
//   launched; nothing is launched for empty tensors.
//
// Each tensor entry calls the C ABI with the first tensor's device current (set and
// restored only when it is not) and the GIL released, and returns its
// status.  Non-empty tensors without device memory (wrapper subclasses) are
// refused with ValueError.  seed, key and offset are taken modulo 2^32;
// `stream` is the raw handle of a stream on that device.

#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/ops/empty_like.h>
#include <c10/core/DeviceGuard.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <exception>
#include <initializer_list>
#include <string>

#include "../../include/sr_states_hip.h"

namespace {

using CastFn = int (*)(const void*, void*, int64_t, int, int, uint32_t, uint32_t, int, void*);
using AdamWFn = int (*)(void*, const void*, void*, void*, int64_t, int, int, int, int, int, int,
                        const sr_adamw_hparams*, uint32_t, uint32_t, int, void*);
using SgdmFn = int (*)(void*, const void*, void*, int64_t, int, int, int, int, const sr_sgdm_hparams*, uint32_t,
                       uint32_t, int, void*);
using AdamWMultiFn = int (*)(const sr_row*, const uint32_t*, const float*, int, uint32_t, int, int, int, int, int, int,
                             const sr_adamw_hparams*, uint64_t, uint64_t, int, void*);
using SgdmMultiFn = int (*)(const sr_row*, const uint32_t*, int, uint32_t, int, int, int, int, const sr_sgdm_hparams*,
                            uint64_t, uint64_t, int, void*);
CastFn g_cast = nullptr;
AdamWFn g_adamw = nullptr;
SgdmFn g_sgdm = nullptr;
AdamWMultiFn g_adamw_multi = nullptr;
SgdmMultiFn g_sgdm_multi = nullptr;

// sr_dtype codes of include/sr_states_hip.h.
bool dtype_matches(int code, c10::ScalarType type) {
  switch (code) {
    case SR_F32: return type == c10::ScalarType::Float;
    case SR_BF16: return type == c10::ScalarType::BFloat16;
    case SR_F16: return type == c10::ScalarType::Half;
    case SR_E4M3: return type == c10::ScalarType::Float8_e4m3fn;
    case SR_E5M2: return type == c10::ScalarType::Float8_e5m2;
    default: return false;
  }
}

PyObject* fail(PyObject* type, const char* message) {
  PyErr_SetString(type, message);
  return nullptr;
}

void* address(unsigned long long value) { return reinterpret_cast<void*>(static_cast<uintptr_t>(value)); }

PyObject* bind(PyObject*, PyObject* args) {
  unsigned long long cast = 0, adamw = 0, sgdm = 0, adamw_multi = 0, sgdm_multi = 0;
  if (!PyArg_ParseTuple(args, "KKK|KK", &cast, &adamw, &sgdm, &adamw_multi, &sgdm_multi)) return nullptr;
  if (!cast || !adamw || !sgdm) return fail(PyExc_ValueError, "null entry point address");
  g_cast = reinterpret_cast<CastFn>(address(cast));
  g_adamw = reinterpret_cast<AdamWFn>(address(adamw));
  g_sgdm = reinterpret_cast<SgdmFn>(address(sgdm));
  g_adamw_multi = reinterpret_cast<AdamWMultiFn>(address(adamw_multi));
  g_sgdm_multi = reinterpret_cast<SgdmMultiFn>(address(sgdm_multi));
  Py_RETURN_NONE;
}

bool tensors(std::initializer_list<PyObject*> objects) {
  for (PyObject* object : objects) {
    if (!THPVariable_Check(object)) return false;
  }
  return true;
}

// Calls `launch` with `device` current and the GIL released, as torch's
// own operators and a ctypes call do (a launch can wait for room in the
// device queue).  False, with a RuntimeError set, for a C++ exception, such
// as a device that the guard cannot select.  The tensors stay alive through
// the caller's argument tuple.
template <class Launch>
bool run_on_device(const c10::Device& device, Launch launch) {
  bool failed = false;
  std::string message;
  Py_BEGIN_ALLOW_THREADS
  try {
    const c10::DeviceGuard guard(device);
    launch();
  } catch (const std::exception& error) {
    failed = true;
    message = error.what();
  } catch (...) {
    failed = true;
    message = "unknown C++ exception in a native launch";
  }
  Py_END_ALLOW_THREADS
  if (failed) fail(PyExc_RuntimeError, message.c_str());
  return !failed;
}

// The same for a launch that returns its status.
template <class Launch>
PyObject* on_device(const c10::Device& device, Launch launch) {
  int status = 0;
  if (!run_on_device(device, [&] { status = launch(); })) return nullptr;
  return PyLong_FromLong(status);
}

PyObject* cast(PyObject*, PyObject* args) {
  PyObject *x_obj, *out_obj;
  int code, rule, threads;
  unsigned long long seed, offset, stream;
  if (!PyArg_ParseTuple(args, "OOiiKKiK", &x_obj, &out_obj, &code, &rule, &seed, &offset, &threads, &stream)) {
    return nullptr;
  }
  if (!tensors({x_obj, out_obj})) return fail(PyExc_TypeError, "x and out must be tensors");
  const at::Tensor& x = THPVariable_Unpack(x_obj);
  const at::Tensor& out = THPVariable_Unpack(out_obj);
  // The output first: workgroups read x and write out concurrently, so any
  // shared byte would make the result depend on their timing.
  if (!dtype_matches(code, out.scalar_type()) || out.sizes() != x.sizes() || out.device() != x.device() ||
      !out.is_contiguous()) {
    return fail(PyExc_ValueError, "out must be a contiguous tensor of the requested dtype, shape and device");
  }
  const int64_t n = x.numel();
  if (n) {
    const auto x_start = reinterpret_cast<uintptr_t>(x.const_data_ptr());
    const auto out_start = reinterpret_cast<uintptr_t>(out.const_data_ptr());
    if (!x_start || !out_start) return fail(PyExc_ValueError, "tensors without device memory cannot be cast");
    if (x_start < out_start + out.nbytes() && out_start < x_start + x.nbytes()) {
      return fail(PyExc_ValueError, "out must not overlap the input");
    }
  }
  if (!x.is_cuda() || x.scalar_type() != c10::ScalarType::Float || !x.is_contiguous()) {
    return fail(PyExc_ValueError, "the cast input must be a contiguous FP32 tensor on the GPU");
  }
  if (n == 0) return PyLong_FromLong(0);
  if (g_cast == nullptr) return fail(PyExc_RuntimeError, "the native entries are not bound to the library");
  return on_device(x.device(), [&] {
    return g_cast(x.const_data_ptr(), out.data_ptr(), n, code, rule, static_cast<uint32_t>(seed),
                  static_cast<uint32_t>(offset), threads, address(stream));
  });
}

c10::ScalarType scalar_type(int code) {
  switch (code) {
    case SR_BF16: return c10::ScalarType::BFloat16;
    case SR_F16: return c10::ScalarType::Half;
    case SR_E4M3: return c10::ScalarType::Float8_e4m3fn;
    case SR_E5M2: return c10::ScalarType::Float8_e5m2;
    default: return c10::ScalarType::Float;
  }
}

// Torch's own translation of its exceptions around the allocation: an
// allocator that is out of memory raises torch.OutOfMemoryError.
PyObject* cast_new(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  PyObject* x_obj;
  int code, rule, threads;
  unsigned long long seed, offset, stream;
  if (!PyArg_ParseTuple(args, "OiiKKiK", &x_obj, &code, &rule, &seed, &offset, &threads, &stream)) return nullptr;
  if (!THPVariable_CheckExact(x_obj) || at::impl::torch_function_mode_enabled()) Py_RETURN_NONE;
  const at::Tensor& x = THPVariable_Unpack(x_obj);
  if (code < SR_F32 || code > SR_E5M2) return fail(PyExc_ValueError, "unknown cast dtype");
  if (!x.is_cuda() || x.scalar_type() != c10::ScalarType::Float || !x.is_contiguous()) {
    return fail(PyExc_ValueError, "the cast input must be a contiguous FP32 tensor on the GPU");
  }
  if (g_cast == nullptr) return fail(PyExc_RuntimeError, "the native entries are not bound to the library");
  at::Tensor out;
  {
    const pybind11::gil_scoped_release no_gil;
    // The options torch.empty_like(x, dtype=, memory_format=) passes on.
    out = at::empty_like(x, at::TensorOptions().dtype(scalar_type(code)).pinned_memory(false),
                         at::MemoryFormat::Contiguous);
  }
  const int64_t n = x.numel();
  if (n == 0) return THPVariable_Wrap(std::move(out));
  const void* source = x.const_data_ptr();
  void* target = out.data_ptr();
  if (!source || !target) return fail(PyExc_ValueError, "tensors without device memory cannot be cast");
  int status = 0;
  if (!run_on_device(x.device(), [&] {
        status = g_cast(source, target, n, code, rule, static_cast<uint32_t>(seed), static_cast<uint32_t>(offset),
                        threads, address(stream));
      })) {
    return nullptr;
  }
  return status ? PyLong_FromLong(status) : THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// The tensor checks of the fused updates, in the validating order of
// sr_states/triton/_optimizer.py:24-60; ts[0] is the parameter, ts[1] the
// gradient (only read).  Returns false with the Python error set.
bool check_update_tensors(std::initializer_list<const at::Tensor*> ts) {
  const at::Tensor& p = **ts.begin();
  const at::Tensor& g = **(ts.begin() + 1);
  if (!p.is_cuda()) {
    fail(PyExc_ValueError, "fused state updates require GPU tensors");
    return false;
  }
  for (const at::Tensor* t : ts) {
    if (t->device() != p.device()) {
      fail(PyExc_ValueError, "all tensors must be on the same GPU device");
      return false;
    }
    if (t->sizes() != p.sizes()) {
      fail(PyExc_ValueError, "all tensors must have identical shapes");
      return false;
    }
    if (!t->is_contiguous()) {
      fail(PyExc_ValueError, "fused state updates require contiguous tensors");
      return false;
    }
  }
  const auto float_or_bf16 = [](const at::Tensor& t) {
    return t.scalar_type() == c10::ScalarType::Float || t.scalar_type() == c10::ScalarType::BFloat16;
  };
  if (!float_or_bf16(p) || !float_or_bf16(g)) {
    fail(PyExc_TypeError, "parameter and gradient must be FP32 or BF16");
    return false;
  }
  if (p.numel() == 0) return true;
  for (const at::Tensor* t : ts) {
    if (t->const_data_ptr() == nullptr) {
      fail(PyExc_ValueError, "fused state updates require tensors that hold device memory");
      return false;
    }
  }
  // Every written span (all but the gradient) disjoint from every other
  // span: with one read-only tensor, every pair holds a written one.
  int i = 0;
  for (const at::Tensor* a : ts) {
    int j = 0;
    for (const at::Tensor* b : ts) {
      if (j > i) {
        const auto a0 = reinterpret_cast<uintptr_t>(a->const_data_ptr());
        const auto b0 = reinterpret_cast<uintptr_t>(b->const_data_ptr());
        if (a0 < b0 + b->nbytes() && b0 < a0 + a->nbytes()) {
          fail(PyExc_ValueError, "parameter, gradient, and state must not overlap optimizer writes");
          return false;
        }
      }
      ++j;
    }
    ++i;
  }
  return true;
}

int pg_code(const at::Tensor& t) { return t.scalar_type() == c10::ScalarType::Float ? SR_F32 : SR_BF16; }

bool state_matches(int code, const at::Tensor& t) {
  if (dtype_matches(code, t.scalar_type())) return true;
  fail(PyExc_ValueError, "state dtype does not match its state format");
  return false;
}

PyObject* adamw_step(PyObject*, PyObject* args) {
  PyObject *p_obj, *g_obj, *m_obj, *v_obj;
  int m_code, m_rule, v_code, v_rule, block;
  double s[8];
  unsigned long long key, offset, stream;
  if (!PyArg_ParseTuple(args, "OOOOiiii(dddddddd)KKiK", &p_obj, &g_obj, &m_obj, &v_obj, &m_code, &m_rule, &v_code,
                        &v_rule, &s[0], &s[1], &s[2], &s[3], &s[4], &s[5], &s[6], &s[7], &key, &offset, &block,
                        &stream)) {
    return nullptr;
  }
  if (!tensors({p_obj, g_obj, m_obj, v_obj})) return fail(PyExc_TypeError, "parameter, gradient and states must be tensors");
  const at::Tensor& p = THPVariable_Unpack(p_obj);
  const at::Tensor& g = THPVariable_Unpack(g_obj);
  const at::Tensor& m = THPVariable_Unpack(m_obj);
  const at::Tensor& v = THPVariable_Unpack(v_obj);
  if (!state_matches(m_code, m) || !state_matches(v_code, v) || !check_update_tensors({&p, &g, &m, &v})) {
    return nullptr;
  }
  if (p.numel() == 0) return PyLong_FromLong(0);
  if (g_adamw == nullptr) return fail(PyExc_RuntimeError, "the native entries are not bound to the library");
  const sr_adamw_hparams hp = {static_cast<float>(s[0]), static_cast<float>(s[1]), static_cast<float>(s[2]),
                               static_cast<float>(s[3]), static_cast<float>(s[4]), static_cast<float>(s[5]),
                               static_cast<float>(s[6]), static_cast<float>(s[7])};
  return on_device(p.device(), [&] {
    return g_adamw(p.data_ptr(), g.const_data_ptr(), m.data_ptr(), v.data_ptr(), p.numel(), pg_code(p), pg_code(g),
                   m_code, m_rule, v_code, v_rule, &hp, static_cast<uint32_t>(key), static_cast<uint32_t>(offset),
                   block, address(stream));
  });
}

PyObject* sgdm_step(PyObject*, PyObject* args) {
  PyObject *p_obj, *g_obj, *u_obj;
  int u_code, u_rule, block;
  double s[2];
  unsigned long long key, offset, stream;
  if (!PyArg_ParseTuple(args, "OOOii(dd)KKiK", &p_obj, &g_obj, &u_obj, &u_code, &u_rule, &s[0], &s[1], &key, &offset,
                        &block, &stream)) {
    return nullptr;
  }
  if (!tensors({p_obj, g_obj, u_obj})) return fail(PyExc_TypeError, "parameter, gradient and states must be tensors");
  const at::Tensor& p = THPVariable_Unpack(p_obj);
  const at::Tensor& g = THPVariable_Unpack(g_obj);
  const at::Tensor& u = THPVariable_Unpack(u_obj);
  if (!state_matches(u_code, u) || !check_update_tensors({&p, &g, &u})) return nullptr;
  if (p.numel() == 0) return PyLong_FromLong(0);
  if (g_sgdm == nullptr) return fail(PyExc_RuntimeError, "the native entries are not bound to the library");
  const sr_sgdm_hparams hp = {static_cast<float>(s[0]), static_cast<float>(s[1])};
  return on_device(p.device(), [&] {
    return g_sgdm(p.data_ptr(), g.const_data_ptr(), u.data_ptr(), p.numel(), pg_code(p), pg_code(g), u_code, u_rule,
                  &hp, static_cast<uint32_t>(key), static_cast<uint32_t>(offset), block, address(stream));
  });
}

PyObject* adamw_multi(PyObject*, PyObject* args) {
  unsigned long long rows, tile_rows, row_scalars, hparams, seed, rng_step, stream;
  unsigned int total_tiles;
  int nrows, p, g, m, m_rule, v, v_rule, block, device;
  if (!PyArg_ParseTuple(args, "KKKiIiiiiiiKKKiiK", &rows, &tile_rows, &row_scalars, &nrows, &total_tiles, &p, &g, &m,
                        &m_rule, &v, &v_rule, &hparams, &seed, &rng_step, &block, &device, &stream)) {
    return nullptr;
  }
  if (g_adamw_multi == nullptr) return fail(PyExc_RuntimeError, "the native entries are not bound to the library");
  return on_device(c10::Device(c10::DeviceType::CUDA, static_cast<c10::DeviceIndex>(device)), [&] {
    return g_adamw_multi(static_cast<const sr_row*>(address(rows)), static_cast<const uint32_t*>(address(tile_rows)),
                         static_cast<const float*>(address(row_scalars)), nrows, total_tiles, p, g, m, m_rule, v,
                         v_rule, static_cast<const sr_adamw_hparams*>(address(hparams)), seed, rng_step, block,
                         address(stream));
  });
}

PyObject* sgdm_multi(PyObject*, PyObject* args) {
  unsigned long long rows, tile_rows, hparams, seed, rng_step, stream;
  unsigned int total_tiles;
  int nrows, p, g, u, u_rule, block, device;
  if (!PyArg_ParseTuple(args, "KKiIiiiiKKKiiK", &rows, &tile_rows, &nrows, &total_tiles, &p, &g, &u, &u_rule,
                        &hparams, &seed, &rng_step, &block, &device, &stream)) {
    return nullptr;
  }
  if (g_sgdm_multi == nullptr) return fail(PyExc_RuntimeError, "the native entries are not bound to the library");
  return on_device(c10::Device(c10::DeviceType::CUDA, static_cast<c10::DeviceIndex>(device)), [&] {
    return g_sgdm_multi(static_cast<const sr_row*>(address(rows)), static_cast<const uint32_t*>(address(tile_rows)),
                        nrows, total_tiles, p, g, u, u_rule, static_cast<const sr_sgdm_hparams*>(address(hparams)),
                        seed, rng_step, block, address(stream));
  });
}

// Every entry behind one guard: a C++ exception from torch (a tensor
// without storage refuses its data pointer) becomes a RuntimeError instead
// of escaping into the interpreter.
template <PyObject* (*Entry)(PyObject*, PyObject*)>
PyObject* guarded(PyObject* self, PyObject* args) {
  try {
    return Entry(self, args);
  } catch (const std::exception& error) {
    return fail(PyExc_RuntimeError, error.what());
  } catch (...) {
    return fail(PyExc_RuntimeError, "unknown C++ exception in a native entry");
  }
}

PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, "Keep the addresses of the C ABI's entry points."},
    {"cast_new", cast_new, METH_VARARGS, "Cast into a new tensor; returns it, a nonzero status, or None."},
    {"adamw_multi", guarded<adamw_multi>, METH_VARARGS, "Call sr_adamw_multi on a device; returns its status."},
    {"sgdm_multi", guarded<sgdm_multi>, METH_VARARGS, "Call sr_sgdm_multi on a device; returns its status."},
    {"cast", guarded<cast>, METH_VARARGS, "Check the tensors and call sr_cast; returns its status."},
    {"adamw_step", guarded<adamw_step>, METH_VARARGS,
     "Check the tensors and call sr_adamw_step; returns its status."},
    {"sgdm_step", guarded<sgdm_step>, METH_VARARGS, "Check the tensors and call sr_sgdm_step; returns its status."},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_launch", "Native entries of the launches.", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__launch(void) { return PyModule_Create(&module); }

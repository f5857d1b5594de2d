// gdnr_host.cpp -- the CPython extension module _gdnr_host: the host path of
// one entry-point call (tensors -> gdnr_tensor descriptors, device and stream,
// the C call) and the slot cache's step metadata, without interpreter work per
// tensor. An eager fused step of one sequence (16 tensors) took 41 us a call
// with ctypes descriptors, ten times its kernel; 19 with this module. A step
// of the slot cache (40 entries) 75 us, now 31, its metadata packed here into
// one pinned buffer and one copy.
//
// The entry points themselves stay those of libgdnreplay.so (include/gdnr.h),
// reached through the addresses gdnr_lib.py binds. Checks and their errors
// are the Python layer's: every tensor on one GPU, rank and dtype accepted; a
// nonzero status raises the bound error class with the library's message.
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <Python.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <array>
#include <string>
#include <utility>
#include <vector>

#include "gdnr.h"

namespace {

constexpr int kMaxTensors = 17, kMaxInts = 3, kMaxFloats = 1;

using Invoke = int (*)(void*, const gdnr_tensor* const*, const int32_t*, const float*, void*);

template <size_t>
using TensorArg = const gdnr_tensor*;
template <size_t>
using IntArg = int32_t;
template <size_t>
using FloatArg = float;

template <size_t... T, size_t... I, size_t... F>
int invoke_as(void* fn, const gdnr_tensor* const* t, const int32_t* i, const float* f, void* stream,
              std::index_sequence<T...>, std::index_sequence<I...>, std::index_sequence<F...>) {
  (void)i, (void)f;
  return reinterpret_cast<int (*)(TensorArg<T>..., IntArg<I>..., FloatArg<F>..., void*)>(fn)(t[T]..., i[I]..., f[F]...,
                                                                                            stream);
}
template <int NT, int NI, int NF>
int invoke(void* fn, const gdnr_tensor* const* t, const int32_t* i, const float* f, void* stream) {
  return invoke_as(fn, t, i, f, stream, std::make_index_sequence<NT>{}, std::make_index_sequence<NI>{},
                   std::make_index_sequence<NF>{});
}

struct Signature {
  int nt, ni, nf;
  Invoke invoke;
};
template <int NT, int NI, int NF = 0>
constexpr Signature signature() {
  return {NT, NI, NF, &invoke<NT, NI, NF>};
}
// the argument counts of the entry points (include/gdnr.h)
constexpr Signature kSignatures[] = {
    signature<1, 1>(),  signature<3, 0>(),  signature<3, 2>(),  signature<4, 0>(),     signature<4, 2>(),
    signature<7, 0>(),  signature<9, 3>(),  signature<10, 1>(), signature<11, 1>(),    signature<11, 3>(),
    signature<16, 1>(), signature<17, 1>(), signature<8, 0, 1>(),
};

struct Entry {
  const Signature* sig;
  void* fn;
};
std::vector<Entry> g_entries;
const char* (*g_last_error)() = nullptr;
PyObject* g_error_class = nullptr;

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kBFloat16: return GDNR_DTYPE_BF16;
    case at::kHalf: return GDNR_DTYPE_F16;
    case at::kFloat: return GDNR_DTYPE_F32;
    case at::kFloat8_e4m3fn: return GDNR_DTYPE_FP8E4M3FN;
    case at::kByte: return GDNR_DTYPE_U8;
    case at::kInt: return GDNR_DTYPE_I32;
    case at::kLong: return GDNR_DTYPE_I64;
    case at::kBool: return GDNR_DTYPE_BOOL;
    case at::kChar: return GDNR_DTYPE_I8;
    default: return -1;
  }
}

// the interpreter lock released for a scope (exceptions leave it held again)
struct Unlocked {
  PyThreadState* state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
};

// C++ exceptions (torch's) become Python ones at every function's edge
template <class Fn>
PyObject* guarded(Fn&& fn) {
  try {
    return fn();
  } catch (const c10::Error& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what_without_backtrace());
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
  }
  return nullptr;
}

// bind(error_class, last_error_address, [(address, tensors, ints, floats), ...])
PyObject* host_bind(PyObject*, PyObject* args) {
  PyObject *error_class, *list;
  unsigned long long last_error;
  if (!PyArg_ParseTuple(args, "OKO!", &error_class, &last_error, &PyList_Type, &list)) return nullptr;
  std::vector<Entry> entries;
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(list); ++i) {
    unsigned long long address;
    int nt, ni, nf;
    if (!PyArg_ParseTuple(PyList_GET_ITEM(list, i), "Kiii", &address, &nt, &ni, &nf)) return nullptr;
    const Signature* found = nullptr;
    for (const Signature& s : kSignatures)
      if (s.nt == nt && s.ni == ni && s.nf == nf) found = &s;
    if (!found) {
      PyErr_Format(PyExc_RuntimeError, "entry point %zd: no call of %d tensors, %d ints and %d floats", i, nt, ni, nf);
      return nullptr;
    }
    entries.push_back({found, reinterpret_cast<void*>(address)});
  }
  Py_INCREF(error_class);
  Py_XSETREF(g_error_class, error_class);
  g_last_error = reinterpret_cast<const char* (*)()>(last_error);
  g_entries = std::move(entries);
  Py_RETURN_NONE;
}

// require(names, tensors): every tensor (None skipped) is on one GPU
PyObject* host_require(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 2 || !PyTuple_Check(args[0]) || !PyTuple_Check(args[1]) ||
      PyTuple_GET_SIZE(args[0]) != PyTuple_GET_SIZE(args[1])) {
    PyErr_SetString(PyExc_TypeError, "require(names, tensors): two tuples of one length");
    return nullptr;
  }
  return guarded([&]() -> PyObject* {
    c10::optional<at::Device> device;
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(args[1]); ++i) {
      PyObject* o = PyTuple_GET_ITEM(args[1], i);
      if (o == Py_None) continue;
      if (!THPVariable_Check(o) || !THPVariable_Unpack(o).is_cuda()) {
        PyErr_Format(PyExc_ValueError, "%U must be a tensor on the GPU", PyTuple_GET_ITEM(args[0], i));
        return nullptr;
      }
      const at::Device d = THPVariable_Unpack(o).device();
      if (!device) {
        device = d;
      } else if (d != *device) {
        PyErr_Format(PyExc_ValueError, "%U is on %s, expected %s", PyTuple_GET_ITEM(args[0], i), d.str().c_str(),
                     device->str().c_str());
        return nullptr;
      }
    }
    Py_RETURN_NONE;
  });
}

// empty(like, shape): a new contiguous tensor of like's dtype and device
PyObject* host_empty(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 2 || !THPVariable_Check(args[0]) || !PyTuple_Check(args[1])) {
    PyErr_SetString(PyExc_TypeError, "empty(like, shape)");
    return nullptr;
  }
  return guarded([&]() -> PyObject* {
    const at::Tensor& like = THPVariable_Unpack(args[0]);
    c10::SmallVector<int64_t, GDNR_MAX_DIMS> shape;
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(args[1]); ++i) {
      shape.push_back(PyLong_AsLongLong(PyTuple_GET_ITEM(args[1], i)));
      if (PyErr_Occurred()) return nullptr;
    }
    const auto options = at::TensorOptions().dtype(like.dtype()).device(like.device());
    // (an allocation may wait for the device, and that for another thread)
    return THPVariable_Wrap([&] {
      Unlocked unlocked;
      return at::empty(shape, options);
    }());
  });
}

// call(entry, tensors, ints, floats, stream): the entry point with the tensors'
// descriptors on the first tensor's device, on `stream` (None: torch's current
// stream there)
PyObject* host_call(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 5 || !PyTuple_Check(args[1]) || !PyTuple_Check(args[2]) || !PyTuple_Check(args[3])) {
    PyErr_SetString(PyExc_TypeError, "call(entry, tensors, ints, floats, stream)");
    return nullptr;
  }
  const long id = PyLong_AsLong(args[0]);
  if (id == -1 && PyErr_Occurred()) return nullptr;
  if (id < 0 || (size_t)id >= g_entries.size()) {
    PyErr_Format(PyExc_RuntimeError, "entry point %ld is not bound", id);
    return nullptr;
  }
  const Entry e = g_entries[id];
  if (PyTuple_GET_SIZE(args[1]) != e.sig->nt || PyTuple_GET_SIZE(args[2]) != e.sig->ni ||
      PyTuple_GET_SIZE(args[3]) != e.sig->nf) {
    PyErr_Format(PyExc_TypeError, "entry point %ld takes %d tensors, %d ints and %d floats", id, e.sig->nt, e.sig->ni,
                 e.sig->nf);
    return nullptr;
  }
  return guarded([&]() -> PyObject* {
    std::array<gdnr_tensor, kMaxTensors> desc;
    std::array<const gdnr_tensor*, kMaxTensors> ptr;
    std::array<int32_t, kMaxInts> ints{};
    std::array<float, kMaxFloats> floats{};
    c10::optional<at::Device> device;
    for (int i = 0; i < e.sig->nt; ++i) {
      PyObject* o = PyTuple_GET_ITEM(args[1], i);
      ptr[i] = nullptr;
      if (o == Py_None) continue;
      if (!THPVariable_Check(o)) {
        PyErr_SetString(PyExc_TypeError, "expected a tensor");
        return nullptr;
      }
      const at::Tensor& t = THPVariable_Unpack(o);
      if (t.dim() > GDNR_MAX_DIMS) {
        PyErr_Format(PyExc_ValueError, "tensors of rank %d are not accepted", (int)t.dim());
        return nullptr;
      }
      gdnr_tensor& d = desc[i];
      d = {};
      d.dtype = dtype_code(t.scalar_type());
      if (d.dtype < 0) {
        PyObject* dtype = PyObject_GetAttrString(o, "dtype");
        if (!dtype) return nullptr;
        PyErr_Format(PyExc_TypeError, "dtype %S is not accepted by libgdnreplay", dtype);
        Py_DECREF(dtype);
        return nullptr;
      }
      d.ndim = (int32_t)t.dim();
      const auto sizes = t.sizes(), strides = t.strides();
      for (int k = 0; k < d.ndim; ++k) {
        d.shape[k] = sizes[k];
        d.strides[k] = strides[k];
      }
      d.data = t.numel() ? t.data_ptr() : nullptr;
      ptr[i] = &d;
      if (!device) device = t.device();
    }
    for (int i = 0; i < e.sig->ni; ++i) {
      PyObject* number = PyNumber_Long(PyTuple_GET_ITEM(args[2], i));
      if (!number) return nullptr;
      const long long v = PyLong_AsLongLong(number);
      Py_DECREF(number);
      if (v == -1 && PyErr_Occurred()) return nullptr;
      ints[i] = (int32_t)v;
    }
    for (int i = 0; i < e.sig->nf; ++i) {
      floats[i] = (float)PyFloat_AsDouble(PyTuple_GET_ITEM(args[3], i));
      if (PyErr_Occurred()) return nullptr;
    }
    c10::OptionalDeviceGuard guard;
    if (device && device->is_cuda()) guard.reset_device(*device);
    void* stream = nullptr;
    if (args[4] != Py_None) {
      stream = reinterpret_cast<void*>(PyLong_AsUnsignedLongLong(args[4]));
      if (PyErr_Occurred()) return nullptr;
    } else if (device && device->is_cuda()) {
      stream = c10::hip::getCurrentHIPStream(device->index()).stream();
    }
    int status;
    std::string message;
    {
      Unlocked unlocked;
      status = e.sig->invoke(e.fn, ptr.data(), ints.data(), floats.data(), stream);
      if (status) message = g_last_error();  // (thread-local in the library)
    }
    if (status == 0) Py_RETURN_NONE;
    PyObject* error = PyObject_CallFunction(g_error_class, "is", status, message.c_str());
    if (error) {
      PyErr_SetObject(g_error_class, error);
      Py_DECREF(error);
    }
    return nullptr;
  });
}

// A buffer of contiguous items behind a Python object: int64 (T = int64_t) or
// bytes (T = uint8_t). The format is checked and not only its size: a float64
// or uint64 array has 8-byte items too.
template <class T>
struct Buffer {
  Py_buffer view{};
  bool ok;
  Buffer(PyObject* o, bool writable) {
    ok = PyObject_GetBuffer(o, &view, PyBUF_ND | PyBUF_FORMAT | (writable ? PyBUF_WRITABLE : 0)) == 0;
    if (!ok) return;
    const char* f = view.format ? view.format : "B";
    if (*f == '@' || *f == '=') ++f;
    const bool fits = sizeof(T) == 8 ? (*f == 'l' || *f == 'q') && !f[1] : (*f == 'B' || *f == '?') && !f[1];
    if (fits && view.itemsize == (Py_ssize_t)sizeof(T)) return;
    PyErr_Format(PyExc_TypeError, "expected a buffer of %s, got %zd-byte items of format '%s'",
                 sizeof(T) == 8 ? "8-byte signed integers" : "bytes", view.itemsize, view.format ? view.format : "B");
    ok = false;
  }
  ~Buffer() {
    if (view.obj) PyBuffer_Release(&view);
  }
  T* data() const { return (T*)view.buf; }
  Py_ssize_t count() const { return view.len / view.itemsize; }
};

// slot_metadata(fill, slots, window, out): checks a batch's slots (int64, 0 =
// padding) against the ring fills (int64, one a slot) and writes the step's
// metadata into out (bytes): int32 slot, pos and valid_len of each entry, then
// one flush byte each
PyObject* host_slot_metadata(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 4) {
    PyErr_SetString(PyExc_TypeError, "slot_metadata(fill, slots, window, out)");
    return nullptr;
  }
  const long long window = PyLong_AsLongLong(args[2]);
  if (window == -1 && PyErr_Occurred()) return nullptr;
  const Buffer<int64_t> fill(args[0], false);
  if (!fill.ok) return nullptr;
  const Buffer<int64_t> slots(args[1], false);
  if (!slots.ok) return nullptr;
  const Buffer<uint8_t> out(args[3], true);
  if (!out.ok) return nullptr;
  return guarded([&]() -> PyObject* {
    const Py_ssize_t n = slots.count(), total = fill.count();
    const int64_t *f = fill.data(), *s = slots.data();
    if (out.count() < 13 * n) {
      PyErr_SetString(PyExc_ValueError, "out is too small");
      return nullptr;
    }
    int32_t* o = (int32_t*)out.data();
    uint8_t* flush = (uint8_t*)(o + 3 * n);
    std::vector<bool> seen(total);
    for (Py_ssize_t i = 0; i < n; ++i)
      if (s[i] < 0 || s[i] >= total) {
        PyErr_Format(PyExc_ValueError, "slots outside 0..%zd", total - 1);
        return nullptr;
      }
    for (Py_ssize_t i = 0; i < n; ++i) {
      const int64_t k = s[i];
      if (k != 0 && seen[k]) {
        PyErr_SetString(PyExc_ValueError, "a non-null slot appears twice in the batch");
        return nullptr;
      }
      seen[k] = true;
      o[i] = (int32_t)k;
      o[n + i] = k ? (int32_t)f[k] : -1;
      o[2 * n + i] = k ? (int32_t)f[k] + 1 : 0;
      flush[i] = k && f[k] + 1 == window;
    }
    Py_RETURN_NONE;
  });
}

// advance(fill, slots, window): the fills after a step (a flushed ring restarts)
PyObject* host_advance(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 3) {
    PyErr_SetString(PyExc_TypeError, "advance(fill, slots, window)");
    return nullptr;
  }
  const long long window = PyLong_AsLongLong(args[2]);
  if (window == -1 && PyErr_Occurred()) return nullptr;
  const Buffer<int64_t> fill(args[0], true);
  if (!fill.ok) return nullptr;
  const Buffer<int64_t> slots(args[1], false);
  if (!slots.ok) return nullptr;
  int64_t* f = fill.data();
  const int64_t* s = slots.data();
  const Py_ssize_t total = fill.count();
  for (Py_ssize_t i = 0; i < slots.count(); ++i)
    if (s[i] > 0 && s[i] < total) f[s[i]] = f[s[i]] + 1 == window ? 0 : f[s[i]] + 1;
  Py_RETURN_NONE;
}

PyMethodDef kMethods[] = {
    {"bind", host_bind, METH_VARARGS, nullptr},
    {"require", (PyCFunction)(void (*)())host_require, METH_FASTCALL, nullptr},
    {"empty", (PyCFunction)(void (*)())host_empty, METH_FASTCALL, nullptr},
    {"call", (PyCFunction)(void (*)())host_call, METH_FASTCALL, nullptr},
    {"slot_metadata", (PyCFunction)(void (*)())host_slot_metadata, METH_FASTCALL, nullptr},
    {"advance", (PyCFunction)(void (*)())host_advance, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_gdnr_host", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__gdnr_host(void) { return PyModule_Create(&kModule); }

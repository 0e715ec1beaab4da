// CPython binding of the entry points that launch work: torch tensors in, tri_* call, status out.
//
// What it replaces and why: filling the tri_tensor structs from Python through ctypes took 0.7 us per tensor and 8 to
// 25 us per call, more than most kernels of a decode step run (RMSNorm of 16 rows: 10.2 us a call of which the GPU
// worked 3.0).  Reading sizes and strides from the tensor object takes some 20 ns.
//
// Every function takes the tensors (or descriptors of them) in the order of the C entry point (None where it allows
// NULL), then its scalars, then the stream as an integer, and returns the status; trinity_amd/ext.py turns a status into
// an exception.
#include <torch/csrc/autograd/python_variable.h>

#include <cstring>

#include "../../include/trinity_amd.h"

namespace {

constexpr int kMaxTensors = 12;

struct Tensors {
  tri_tensor v[kMaxTensors];
  tri_tensor* p[kMaxTensors];
};

// a[i] = tensor, None, or a tensor's descriptor as ext.as_tri makes it
bool to_tri(PyObject* o, tri_tensor& v, tri_tensor*& p) {
  if (o == Py_None) {
    p = nullptr;
    return true;
  }
  if (!THPVariable_Check(o)) {
    Py_buffer b;
    if (strcmp(Py_TYPE(o)->tp_name, "TriTensor") != 0 || PyObject_GetBuffer(o, &b, PyBUF_SIMPLE) != 0) {
      PyErr_Format(PyExc_TypeError, "expected a tensor or None, got %.100s", Py_TYPE(o)->tp_name);
      return false;
    }
    const bool whole = b.len == (Py_ssize_t)sizeof v;
    if (whole) memcpy(&v, b.buf, sizeof v);
    else PyErr_SetString(PyExc_TypeError, "not the TriTensor of this library");
    PyBuffer_Release(&b);
    p = &v;
    return whole;
  }
  const at::Tensor& t = THPVariable_Unpack(o);
  switch (t.scalar_type()) {
    case at::kHalf: v.dtype = TRI_F16; break;
    case at::kBFloat16: v.dtype = TRI_BF16; break;
    case at::kFloat: v.dtype = TRI_F32; break;
    case at::kByte: v.dtype = TRI_U8; break;
    case at::kFloat8_e4m3fn: v.dtype = TRI_FP8_E4M3; break;
    default: PyErr_Format(PyExc_TypeError, "unsupported dtype %s", at::toString(t.scalar_type())); return false;
  }
  const int64_t nd = t.dim();
  if (nd > 4) {
    PyErr_SetString(PyExc_ValueError, "at most 4 dimensions");
    return false;
  }
  v.ptr = t.data_ptr();
  v.ndim = (int32_t)nd;
  for (int i = 0; i < 4; ++i) {
    v.shape[i] = i < nd ? t.size(i) : 0;
    v.stride[i] = i < nd ? t.stride(i) : 0;
  }
  p = &v;
  return true;
}

bool marshal(PyObject* const* args, Py_ssize_t nargs, int ntensors, int nscalars, Tensors& t) {
  if (nargs != ntensors + nscalars + 1) {
    PyErr_Format(PyExc_TypeError, "expected %d arguments, got %zd", ntensors + nscalars + 1, nargs);
    return false;
  }
  for (int i = 0; i < ntensors; ++i) {
    if (!to_tri(args[i], t.v[i], t.p[i])) return false;
  }
  return true;
}

// the bytes of a ctypes structure (tri_attn_params)
struct Params {
  Py_buffer buf{};
  const tri_attn_params* p = nullptr;
  explicit Params(PyObject* o) {
    if (PyObject_GetBuffer(o, &buf, PyBUF_SIMPLE) != 0) return;
    if (buf.len == (Py_ssize_t)sizeof(tri_attn_params)) p = static_cast<const tri_attn_params*>(buf.buf);
    else PyErr_SetString(PyExc_TypeError, "expected TriAttnParams");
  }
  ~Params() { if (buf.obj != nullptr) PyBuffer_Release(&buf); }
};

void* stream_of(PyObject* o) { return PyLong_AsVoidPtr(o); }

// Other Python threads run while the library works (a launch may wait for room in a stream's queue, and what that queue
// waits for may need the interpreter: a host callback in Python, a thread that feeds another stream).
struct NoGil {
  PyThreadState* state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};
template <class F>
int call(F f) {
  if (PyErr_Occurred() != nullptr) return 0;
  const NoGil nogil;
  return f();
}

template <class F>
PyObject* run(F f) {
  try {
    const int st = f();
    return PyErr_Occurred() != nullptr ? nullptr : PyLong_FromLong(st);
  } catch (const std::exception& e) {  // (a tensor without storage, for instance)
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

#define TRI_BIND(name) PyObject* name(PyObject*, PyObject* const* a, Py_ssize_t n)

TRI_BIND(rmsnorm) {
  return run([&] {
    Tensors t;
    if (!marshal(a, n, 3, 1, t)) return 0;
    const double eps = PyFloat_AsDouble(a[3]);
    void* s = stream_of(a[4]);
    return call([&] { return tri_rmsnorm(t.p[0], t.p[1], t.p[2], (float)eps, s); });
  });
}
TRI_BIND(ffn_swiglu) {
  return run([&] {
    Tensors t;
    if (!marshal(a, n, 7, 0, t)) return 0;
    void* s = stream_of(a[7]);
    return call([&] { return tri_ffn_swiglu(t.p[0], t.p[1], t.p[2], t.p[3], t.p[4], t.p[5], t.p[6], s); });
  });
}
TRI_BIND(gateup_swiglu) {
  return run([&] {
    Tensors t;
    if (!marshal(a, n, 6, 0, t)) return 0;
    void* s = stream_of(a[6]);
    return call([&] { return tri_gateup_swiglu(t.p[0], t.p[1], t.p[2], t.p[3], t.p[4], t.p[5], s); });
  });
}
TRI_BIND(matmul) {
  return run([&] {
    Tensors t;
    if (!marshal(a, n, 5, 0, t)) return 0;
    void* s = stream_of(a[5]);
    return call([&] { return tri_matmul(t.p[0], t.p[1], t.p[2], t.p[3], t.p[4], s); });
  });
}
TRI_BIND(ffn_gelu) {
  return run([&] {
    Tensors t;
    if (!marshal(a, n, 6, 0, t)) return 0;
    void* s = stream_of(a[6]);
    return call([&] { return tri_ffn_gelu(t.p[0], t.p[1], t.p[2], t.p[3], t.p[4], t.p[5], s); });
  });
}
TRI_BIND(ffn_block) {
  return run([&] {
    Tensors t;
    if (!marshal(a, n, 12, 0, t)) return 0;
    void* s = stream_of(a[12]);
    return call([&] {
      return tri_ffn_block(t.p[0], t.p[1], t.p[2], t.p[3], t.p[4], t.p[5], t.p[6], t.p[7], t.p[8], t.p[9], t.p[10], t.p[11], s);
    });
  });
}
TRI_BIND(qkv_attention) {
  return run([&] {
    Tensors t;
    if (!marshal(a, n, 10, 1, t)) return 0;
    const Params p(a[10]);
    void* s = stream_of(a[11]);
    return call([&] {
      return tri_qkv_attention(t.p[0], t.p[1], t.p[2], t.p[3], t.p[4], t.p[5], t.p[6], t.p[7], t.p[8], t.p[9], p.p, s);
    });
  });
}
TRI_BIND(qkv_attention_static) {
  return run([&] {
    Tensors t;
    if (!marshal(a, n, 9, 1, t)) return 0;
    const Params p(a[9]);
    void* s = stream_of(a[10]);
    return call([&] {
      return tri_qkv_attention_static(t.p[0], t.p[1], t.p[2], t.p[3], t.p[4], t.p[5], t.p[6], t.p[7], t.p[8], p.p, s);
    });
  });
}
TRI_BIND(keyformer) {
  return run([&] {
    Tensors t;
    if (!marshal(a, n, 11, 1, t)) return 0;
    const Params p(a[11]);
    void* s = stream_of(a[12]);
    return call([&] {
      return tri_keyformer(t.p[0], t.p[1], t.p[2], t.p[3], t.p[4], t.p[5], t.p[6], t.p[7], t.p[8], t.p[9], t.p[10], p.p, s);
    });
  });
}
TRI_BIND(roco) {  // (as_mean_var comes before the parameters, as in the C entry point)
  return run([&] {
    Tensors t;
    if (!marshal(a, n, 11, 2, t)) return 0;
    const long mean_var = PyLong_AsLong(a[11]);
    const Params p(a[12]);
    void* s = stream_of(a[13]);
    return call([&] {
      return tri_roco(t.p[0], t.p[1], t.p[2], t.p[3], t.p[4], t.p[5], t.p[6], t.p[7], t.p[8], t.p[9], t.p[10],
                      (int32_t)mean_var, p.p, s);
    });
  });
}
#undef TRI_BIND

PyObject* qkv_scratch_bytes(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 2) return PyErr_Format(PyExc_TypeError, "expected 2 arguments, got %zd", n);
  const Params p(a[0]);
  const long long n_model = PyLong_AsLongLong(a[1]);
  if (PyErr_Occurred() != nullptr) return nullptr;
  return PyLong_FromLongLong(tri_qkv_scratch_bytes(p.p, n_model));
}
template <int64_t (*F)(int64_t, int64_t, int64_t)>
PyObject* workspace_bytes(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 3) return PyErr_Format(PyExc_TypeError, "expected 3 arguments, got %zd", n);
  const long long x = PyLong_AsLongLong(a[0]), y = PyLong_AsLongLong(a[1]), z = PyLong_AsLongLong(a[2]);
  if (PyErr_Occurred() != nullptr) return nullptr;
  return PyLong_FromLongLong(F(x, y, z));
}

#define TRI_METHOD(name, fn) {name, (PyCFunction)(void (*)(void))(PyObject* (*)(PyObject*, PyObject* const*, Py_ssize_t))(fn), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    TRI_METHOD("rmsnorm", rmsnorm), TRI_METHOD("ffn_swiglu", ffn_swiglu), TRI_METHOD("gateup_swiglu", gateup_swiglu),
    TRI_METHOD("matmul", matmul), TRI_METHOD("ffn_gelu", ffn_gelu), TRI_METHOD("ffn_block", ffn_block),
    TRI_METHOD("qkv_attention", qkv_attention), TRI_METHOD("qkv_attention_static", qkv_attention_static),
    TRI_METHOD("keyformer", keyformer), TRI_METHOD("roco", roco), TRI_METHOD("qkv_scratch_bytes", qkv_scratch_bytes),
    TRI_METHOD("gemm_workspace_bytes", workspace_bytes<tri_gemm_workspace_bytes>),
    TRI_METHOD("ffn_workspace_bytes", workspace_bytes<tri_ffn_workspace_bytes>),
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&module); }

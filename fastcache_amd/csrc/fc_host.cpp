// Host path of the calls a model makes once per layer or once per step: a CPython module that takes torch tensors,
// fills the C ABI's descriptors and enqueues, without a Python statement per field.  Built as fastcache_amd/_host.so
// next to the kernel library it calls; there is no Python fallback for what it does.
//
// What it saves, measured on the host of an MI355X box: a view built field by field in Python costs 2.5 to 4 us, a
// ctypes call with its arguments 4 us, torch.cuda.current_stream() 8 us, so a decode layer (two views per plane, two
// calls) spent 40 us on the host for 16 us of kernels.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/InferenceMode.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <string>
#include <vector>

#include "../../include/fastcache_hip.h"

namespace {

PyObject* g_error = nullptr;      // FastcacheError

// Python exception already set, or to be set from a C++ one
struct PyFailed {};

[[noreturn]] void fail(const std::string& text) {
  PyErr_SetString(g_error ? g_error : PyExc_RuntimeError, text.c_str());
  throw PyFailed();
}

void check(int rc, const char* what) {
  if (rc != 0) fail(std::string(what) + " failed (code " + std::to_string(rc) + "): " + fc_last_error());
}

// A module function: `body` runs with C++ exceptions turned into Python ones.
template <typename F>
PyObject* guarded(F&& body) {
  try {
    return body();
  } catch (const PyFailed&) {
    return nullptr;
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

bool is_tensor(PyObject* o) { return THPVariable_Check(o); }

const at::Tensor& tensor(PyObject* o, const char* name) {
  if (!is_tensor(o)) fail(std::string(name) + " must be a tensor");
  return THPVariable_Unpack(o);
}

void require_gpu(const at::Tensor& t, const char* name) {
  if (!t.is_cuda())
    fail(std::string(name) + " must live on the GPU (got device " + t.device().str() + "); libfastcache_hip has no CPU path");
}

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return FC_F32;
    case at::kHalf: return FC_F16;
    case at::kBFloat16: return FC_BF16;
    default: fail(std::string("unsupported KV dtype ") + c10::toString(t) + "; expected float32, float16 or bfloat16");
  }
}

void* stream_of(const at::Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

long long as_int(PyObject* o) {
  const long long v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) throw PyFailed();
  return v;
}

PyObject* wrap(at::Tensor t) { return THPVariable_Wrap(std::move(t)); }

void need_args(Py_ssize_t got, Py_ssize_t want, const char* who) {
  if (got != want) fail(std::string(who) + ": " + std::to_string(got) + " arguments, expected " + std::to_string(want));
}

// dense [B, H, S, D] tensor (any strides with contiguous D); size-1 axes have arbitrary strides
fc_kv_view dense_view(const at::Tensor& t, int64_t layers, int64_t stride_layer) {
  fc_kv_view v{};
  v.base = t.data_ptr();
  v.stride_layer = layers > 1 ? stride_layer : 0;
  v.stride_batch = t.size(0) > 1 ? t.stride(0) : 0;
  v.stride_head = t.size(1) > 1 ? t.stride(1) : 0;
  v.stride_token = t.size(2) > 1 ? t.stride(2) : 0;
  v.block_size = 1;
  v.dtype = dtype_code(t.scalar_type());
  v.num_layers = (int32_t)layers;
  v.batch = (int32_t)t.size(0);
  v.num_kv_heads = (int32_t)t.size(1);
  v.head_dim = (int32_t)t.size(3);
  v.max_seq_len = (int32_t)t.size(2);
  return v;
}

// ---- parameters of a module: unchanged since they were packed? ------------------------------------------------------
// A watch holds (dict, key, object) of every step from a module list to its parameters, and of every parameter its
// version counter and address.  192 parameters walked in Python cost about 180 us, here about 4.
struct Watch {
  struct Entry {
    PyObject *dict, *key, *value;
    bool param;
    int64_t version;
    const void* ptr;
  };
  std::vector<Entry> entries;
  ~Watch() {
    for (Entry& e : entries) {
      Py_DECREF(e.dict);
      Py_DECREF(e.key);
      Py_DECREF(e.value);
    }
  }
};

const char* const kWatch = "fastcache_amd.Watch";

int64_t version_of(const at::Tensor& t) { return t.is_inference() ? 0 : (int64_t)t._version(); }

// watch([(dict, key), ...]) -> capsule, or None when a key is missing
PyObject* py_watch(PyObject*, PyObject* list) {
  return guarded([&]() -> PyObject* {
    if (!PyList_Check(list)) fail("watch: a list of (dict, key) pairs expected");
    auto w = std::make_unique<Watch>();
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(list); ++i) {
      PyObject* pair = PyList_GET_ITEM(list, i);
      if (!PyTuple_Check(pair) || PyTuple_GET_SIZE(pair) != 2 || !PyDict_Check(PyTuple_GET_ITEM(pair, 0)))
        fail("watch: a list of (dict, key) pairs expected");
      PyObject *d = PyTuple_GET_ITEM(pair, 0), *k = PyTuple_GET_ITEM(pair, 1);
      PyObject* v = PyDict_GetItemWithError(d, k);
      if (!v) {
        if (PyErr_Occurred()) throw PyFailed();
        Py_RETURN_NONE;
      }
      Py_INCREF(d);
      Py_INCREF(k);
      Py_INCREF(v);
      Watch::Entry e{d, k, v, is_tensor(v), 0, nullptr};
      if (e.param) {
        const at::Tensor& t = THPVariable_Unpack(v);
        e.version = version_of(t);
        e.ptr = t.const_data_ptr();
      }
      w->entries.push_back(e);
    }
    PyObject* cap = PyCapsule_New(w.get(), kWatch, [](PyObject* c) { delete (Watch*)PyCapsule_GetPointer(c, kWatch); });
    if (cap) w.release();
    return cap;
  });
}

PyObject* py_unchanged(PyObject*, PyObject* cap) {
  return guarded([&]() -> PyObject* {
    auto* w = (Watch*)PyCapsule_GetPointer(cap, kWatch);
    if (!w) throw PyFailed();
    for (const Watch::Entry& e : w->entries) {
      if (PyDict_GetItemWithError(e.dict, e.key) != e.value) {
        if (PyErr_Occurred()) throw PyFailed();
        Py_RETURN_FALSE;
      }
      if (e.param) {
        const at::Tensor& t = THPVariable_Unpack(e.value);
        if (version_of(t) != e.version || t.const_data_ptr() != e.ptr) Py_RETURN_FALSE;
      }
    }
    Py_RETURN_TRUE;
  });
}

// ---- MLP compressors over a list of per-layer tensors ------------------------------------------------------------------
bool same_geometry(const at::Tensor& a, const at::Tensor& b) {
  return a.sizes() == b.sizes() && a.strides() == b.strides() && a.scalar_type() == b.scalar_type() && a.device() == b.device();
}

// ccm_layers(pairs, weights, segments, out_len, factor, min_rows) -> [(k, v), ...] or None when the list does not share
// one geometry (its layers then go one by one).  weights: one tuple of six stacked tensors per (segment, plane);
// segments: (start, length, destination) each.
PyObject* py_ccm_layers(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  return guarded([&]() -> PyObject* {
    need_args(nargs, 6, "ccm_layers");
    if (!PyTuple_Check(args[1]) || !PyTuple_Check(args[2])) fail("ccm_layers: tuples of weights and segments expected");
    PyObject* fast = PySequence_Fast(args[0], "ccm_layers: a list of (key, value) pairs expected");
    if (!fast) throw PyFailed();
    struct Drop {
      PyObject* o;
      ~Drop() { Py_DECREF(o); }
    } drop{fast};
    const Py_ssize_t L = PySequence_Fast_GET_SIZE(fast);
    const int nseg = (int)PyTuple_GET_SIZE(args[2]);
    if (L < 1 || L > 64 || nseg < 1 || nseg > 2 || PyTuple_GET_SIZE(args[1]) != 2 * nseg) Py_RETURN_NONE;
    const void* ptr[2][64];
    const at::Tensor* first[2] = {nullptr, nullptr};
    for (Py_ssize_t l = 0; l < L; ++l) {
      PyObject* kv = PySequence_Fast_GET_ITEM(fast, l);
      if (!PyTuple_Check(kv) || PyTuple_GET_SIZE(kv) != 2) Py_RETURN_NONE;
      for (int p = 0; p < 2; ++p) {
        if (!is_tensor(PyTuple_GET_ITEM(kv, p))) Py_RETURN_NONE;
        const at::Tensor& t = THPVariable_Unpack(PyTuple_GET_ITEM(kv, p));
        if (!first[p]) first[p] = &t;
        if (!same_geometry(t, *first[p])) Py_RETURN_NONE;
        ptr[p][l] = t.const_data_ptr();
      }
    }
    const at::Tensor &k0 = *first[0], &v0 = *first[1];
    if (!k0.is_cuda() || k0.dim() != 4 || k0.sizes() != v0.sizes() || k0.scalar_type() != v0.scalar_type() ||
        k0.device() != v0.device() || k0.stride(3) != 1 || v0.stride(3) != 1)
      Py_RETURN_NONE;
    fc_mlp_weights w[4];
    for (int i = 0; i < 2 * nseg; ++i) {
      PyObject* six = PyTuple_GET_ITEM(args[1], i);
      if (!PyTuple_Check(six) || PyTuple_GET_SIZE(six) != 6) fail("ccm_layers: six tensors per weight group expected");
      const void* q[6];
      for (int j = 0; j < 6; ++j) {
        const at::Tensor& t = tensor(PyTuple_GET_ITEM(six, j), "weights");
        if (t.device() != k0.device() || t.scalar_type() != k0.scalar_type() || !t.is_contiguous() || t.size(0) < L)
          fail("ccm_layers: weights must be stacked, contiguous and in the KV dtype");
        q[j] = t.const_data_ptr();
      }
      w[i] = {q[0], q[1], q[2], q[3], q[4], q[5]};
    }
    int32_t start[2], len[2], dst[2];
    for (int s = 0; s < nseg; ++s) {
      PyObject* seg = PyTuple_GET_ITEM(args[2], s);
      if (!PyTuple_Check(seg) || PyTuple_GET_SIZE(seg) != 3) fail("ccm_layers: (start, length, destination) expected");
      start[s] = (int32_t)as_int(PyTuple_GET_ITEM(seg, 0));
      len[s] = (int32_t)as_int(PyTuple_GET_ITEM(seg, 1));
      dst[s] = (int32_t)as_int(PyTuple_GET_ITEM(seg, 2));
    }
    const int64_t C = as_int(args[3]), B = k0.size(0), H = k0.size(1), D = k0.size(3);
    // one allocation for all layers: what the caller gets are contiguous tensors inside it
    at::Tensor all = at::empty({2 * (int64_t)L, B, H, C, D}, k0.options());
    if (all.numel() > 0) {
      fc_kv_view ks = dense_view(k0, L, 0), vs = dense_view(v0, L, 0);
      fc_kv_view kd = dense_view(all.select(0, 0), L, B * H * C * D), vd = kd;
      vd.base = (char*)all.data_ptr() + (int64_t)L * B * H * C * D * all.element_size();
      check(fc_ccm_mlp_layers(ptr[0], ptr[1], &ks, &vs, &kd, &vd, w, nseg, start, len, dst, (int32_t)as_int(args[4]),
                              (int32_t)as_int(args[5]), stream_of(k0)),
            "fc_ccm_mlp_layers");
    }
    std::vector<at::Tensor> parts = all.unbind(0);
    PyObject* out = PyList_New(L);
    if (!out) throw PyFailed();
    for (Py_ssize_t l = 0; l < L; ++l) {
      PyObject* kv = PyTuple_New(2);
      PyTuple_SET_ITEM(kv, 0, wrap(std::move(parts[l])));
      PyTuple_SET_ITEM(kv, 1, wrap(std::move(parts[L + l])));
      PyList_SET_ITEM(out, l, kv);
    }
    return out;
  });
}

PyObject* py_init(PyObject*, PyObject* error) {
  Py_XDECREF(g_error);
  Py_INCREF(error);
  g_error = error;
  Py_RETURN_NONE;
}

PyMethodDef kMethods[] = {
    {"init", py_init, METH_O, "init(error class)"},
    {"watch", py_watch, METH_O, "watch([(dict, key), ...]) -> capsule or None"},
    {"unchanged", py_unchanged, METH_O, "unchanged(capsule) -> bool"},
    {"ccm_layers", (PyCFunction)(void (*)(void))py_ccm_layers, METH_FASTCALL,
     "ccm_layers(pairs, weights, segments, out_len, factor, min_rows) -> list of pairs, or None"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_host", "host path of fastcache_amd", -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) { return PyModule_Create(&kModule); }

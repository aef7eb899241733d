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
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <memory>
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

// inference tensors keep no version, so a write to one would not be seen: _version() raises for them
int64_t version_of(const at::Tensor& t) { return (int64_t)t._version(); }

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
    // a tensor per layer and plane, as the layers one by one would give: each can be saved, resized or dropped by itself
    std::vector<at::Tensor> parts(2 * L);
    void* to[2][64];
    for (int p = 0; p < 2; ++p)
      for (Py_ssize_t l = 0; l < L; ++l) {
        at::Tensor& t = parts[p * L + l];
        t = at::empty({B, H, C, D}, k0.options());
        to[p][l] = t.data_ptr();
      }
    if (parts[0].numel() > 0) {
      const fc_kv_view ks = dense_view(k0, L, 0), vs = dense_view(v0, L, 0), kd = dense_view(parts[0], L, 0);
      check(fc_ccm_mlp_layers_into(ptr[0], ptr[1], to[0], to[1], &ks, &vs, &kd, &kd, w, nseg, start, len, dst,
                                   (int32_t)as_int(args[4]), (int32_t)as_int(args[5]), stream_of(k0)),
            "fc_ccm_mlp_layers_into");
    }
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

// ---- presses on one layer's dense tensors -------------------------------------------------------------------------------------
// [B, H, S, D] K and V of one geometry on one GPU, and a kept count the out-of-place kernels take
bool press_takes(const at::Tensor& k, const at::Tensor& v, int64_t n) {
  return k.is_cuda() && v.device() == k.device() && k.dim() == 4 && k.sizes() == v.sizes() &&
         k.scalar_type() == v.scalar_type() && k.stride(3) == 1 && v.stride(3) == 1 && n > 0 && n <= k.size(2) &&
         k.numel() > 0 && k.size(2) <= FC_SELECT_MAX_KEYS;
}

PyObject* pair(at::Tensor a, at::Tensor b) {
  PyObject* out = PyTuple_New(2);
  if (!out) throw PyFailed();
  PyTuple_SET_ITEM(out, 0, wrap(std::move(a)));
  PyTuple_SET_ITEM(out, 1, wrap(std::move(b)));
  return out;
}

// Scratch for the kept positions when selection and gather are to be launches of their own, else undefined.
at::Tensor gather_apart(const at::Tensor& k, int64_t n) {
  if (!fc_press_gather_apart((int32_t)(k.size(0) * k.size(1)), (int32_t)k.size(2), (int32_t)n)) return at::Tensor();
  return at::empty({k.size(0), k.size(1), n}, k.options().dtype(at::kInt));
}

// knorm_into(keys, values, n) -> (k, v) [B, H, n, D], or None
PyObject* py_knorm_into(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  return guarded([&]() -> PyObject* {
    need_args(nargs, 3, "knorm_into");
    if (!is_tensor(args[0]) || !is_tensor(args[1])) Py_RETURN_NONE;
    const at::Tensor &k = THPVariable_Unpack(args[0]), &v = THPVariable_Unpack(args[1]);
    const int64_t n = as_int(args[2]);
    if (!press_takes(k, v, n)) Py_RETURN_NONE;
    const int64_t B = k.size(0), H = k.size(1), S = k.size(2), D = k.size(3);
    at::Tensor ok = at::empty({B, H, n, D}, k.options()), ov = at::empty({B, H, n, D}, k.options()), scores;
    const fc_kv_view kv = dense_view(k, 1, 0), vv = dense_view(v, 1, 0), dk = dense_view(ok, 1, 0), dv = dense_view(ov, 1, 0);
    // Short columns are scored by the workgroups that gather them, each for itself; longer ones by the whole chip first, in a
    // launch and a tensor more.  us per hook, half kept, one launch against norms first, bf16 columns of 333 / 500 / 600 /
    // 1000 keys: 8 columns 9.2 11.0, 10.4 11.1, 11.4 10.4, 14.4 11.0; 32 of one prompt 9.5 11.3, 10.8 10.9, 11.9 11.2, 17.7
    // 12.1; 32 of four 9.5 11.3, 10.8 11.3, 12.3 11.9, 17.8 12.6; 256 16.3 17.0, 21.9 21.5, 26.2 25.3, 40.6 37.9.
    float* sp = nullptr;
    if (S > 512) {
      scores = at::empty({B, H, S}, k.options().dtype(at::kFloat));
      sp = scores.data_ptr<float>();
    }
    const at::Tensor idx = gather_apart(k, n);
    check(fc_knorm_press_into(&kv, &vv, &dk, &dv, (int32_t)n, sp, (int32_t)S, idx.defined() ? idx.data_ptr<int32_t>() : nullptr,
                              stream_of(k)),
          "fc_knorm_press_into");
    return pair(std::move(ok), std::move(ov));
  });
}

// snapkv_into(keys, values, queries, lse or None, n, window, kernel_size, causal, scale, out_scale) -> (k, v), or None
PyObject* py_snapkv_into(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  return guarded([&]() -> PyObject* {
    need_args(nargs, 10, "snapkv_into");
    for (int i = 0; i < 3; ++i)
      if (!is_tensor(args[i])) Py_RETURN_NONE;
    const at::Tensor &k = THPVariable_Unpack(args[0]), &v = THPVariable_Unpack(args[1]), &q = THPVariable_Unpack(args[2]);
    const int64_t n = as_int(args[4]), W = as_int(args[5]), ksz = as_int(args[6]), causal = as_int(args[7]);
    const double scale = PyFloat_AsDouble(args[8]), out_scale = PyFloat_AsDouble(args[9]);
    if (PyErr_Occurred()) throw PyFailed();
    if (!press_takes(k, v, n) || q.dim() != 4 || q.device() != k.device() || q.scalar_type() != k.scalar_type() ||
        !q.is_contiguous() || (k.scalar_type() != at::kHalf && k.scalar_type() != at::kBFloat16))
      Py_RETURN_NONE;
    const int64_t B = k.size(0), H = k.size(1), S = k.size(2), D = k.size(3), hq = q.size(1);
    if (q.size(0) != B || q.size(2) != W || q.size(3) != D || hq % H || (hq / H) * ((W + 31) / 32) > 16 || n <= W ||
        S - W <= ksz || ksz < 1 || !(ksz & 1) || ksz > 63)
      Py_RETURN_NONE;
    const float* lse = nullptr;
    if (args[3] != Py_None) {
      const at::Tensor& t = tensor(args[3], "lse");
      if (t.device() != k.device() || t.scalar_type() != at::kFloat || !t.is_contiguous() || t.numel() != B * hq * W) Py_RETURN_NONE;
      lse = t.const_data_ptr<float>();
    }
    at::Tensor ok = at::empty({B, H, n, D}, k.options()), ov = at::empty({B, H, n, D}, k.options());
    const fc_kv_view kv = dense_view(k, 1, 0), vv = dense_view(v, 1, 0), dk = dense_view(ok, 1, 0), dv = dense_view(ov, 1, 0);
    const bool once = !lse && fc_snapkv_once_pays(&kv, (int32_t)hq, (int32_t)W, (int32_t)S);
    const int32_t nsplit = once ? 0 : fc_snapkv_select_splits(&kv, (int32_t)hq, (int32_t)W);
    const int64_t bytes = once ? fc_snapkv_once_workspace_bytes(&kv, (int32_t)hq, (int32_t)W)
                               : fc_snapkv_select_workspace_bytes(1, (int32_t)B, (int32_t)hq, (int32_t)H, (int32_t)W, (int32_t)S, nsplit);
    at::Tensor ws = at::empty({bytes}, k.options().dtype(at::kByte));
    const at::Tensor idx = gather_apart(k, n);
    int32_t* apart = idx.defined() ? idx.data_ptr<int32_t>() : nullptr;
    if (once)
      check(fc_snapkv_press_into_once(&kv, &vv, &dk, &dv, q.const_data_ptr(), (int32_t)hq, (int32_t)W, (int32_t)ksz, (int32_t)causal,
                                      (float)scale, (float)out_scale, (int32_t)n, apart, 0, ws.data_ptr(), bytes, stream_of(k)),
            "fc_snapkv_press_into_once");
    else
      check(fc_snapkv_press_into(&kv, &vv, &dk, &dv, q.const_data_ptr(), lse, (int32_t)hq, (int32_t)W, (int32_t)ksz,
                                 (int32_t)causal, (float)scale, (float)out_scale, (int32_t)n, apart, nsplit, ws.data_ptr(), bytes,
                                 stream_of(k)),
            "fc_snapkv_press_into");
    return pair(std::move(ok), std::move(ov));
  });
}

// ---- quantisers ----------------------------------------------------------------------------------------------------------
at::ScalarType fp8_type(int64_t kind) { return kind == FC_QUANT_E5M2 ? at::kFloat8_e5m2 : at::kFloat8_e4m3fn; }

// quantize_pair(kind, keys, values, group_size) -> ((codes, scale), (codes, scale)) with one launch for both tensors (two for
// float8), or None (the caller's general path then serves or refuses the arguments)
PyObject* py_quantize_pair(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  return guarded([&]() -> PyObject* {
    need_args(nargs, 4, "quantize_pair");
    if (!is_tensor(args[1]) || !is_tensor(args[2])) Py_RETURN_NONE;
    const int64_t kind = as_int(args[0]), group = as_int(args[3]);
    at::Tensor x[2] = {THPVariable_Unpack(args[1]), THPVariable_Unpack(args[2])};
    const at::ScalarType dt = x[0].scalar_type();
    if (!x[0].is_cuda() || x[1].device() != x[0].device() || x[1].scalar_type() != dt || x[0].sizes() != x[1].sizes() ||
        x[0].dim() < 1 || x[0].numel() == 0 || (dt != at::kFloat && dt != at::kHalf && dt != at::kBFloat16))
      Py_RETURN_NONE;
    const bool fp8 = kind == FC_QUANT_E4M3 || kind == FC_QUANT_E5M2, bits4 = kind == FC_QUANT_INT4 || kind == FC_QUANT_NF4;
    const int64_t last = x[0].size(-1), d = bits4 ? group : last, n = x[0].numel();
    if (bits4 && (group < 2 || group % 2 || last % group)) Py_RETURN_NONE;
    for (at::Tensor& t : x) t = t.contiguous();
    std::vector<int64_t> shape = x[0].sizes().vec(), lead = shape;
    if (bits4) shape.back() = last / 2;
    lead.back() = bits4 ? last / group : 1;
    at::Tensor codes[2], scale[2];
    for (int i = 0; i < 2; ++i) {
      codes[i] = at::empty(shape, x[0].options().dtype(kind == FC_QUANT_INT8 ? at::kChar : fp8 ? fp8_type(kind) : at::kByte));
      scale[i] = fp8 ? at::empty({}, x[0].options()) : at::empty(lead, x[0].options());
    }
    const int64_t bytes = fc_quantize_pair_workspace_bytes((int32_t)kind);
    at::Tensor ws;
    if (bytes) ws = at::empty({bytes}, x[0].options().dtype(at::kByte));
    check(fc_quantize_pair((int32_t)kind, x[0].const_data_ptr(), x[1].const_data_ptr(), n / d, (int32_t)d, dtype_code(dt),
                           codes[0].data_ptr(), codes[1].data_ptr(), scale[0].data_ptr(), scale[1].data_ptr(),
                           bytes ? ws.data_ptr() : nullptr, bytes, stream_of(x[0])),
          "fc_quantize_pair");
    PyObject* out[2];
    for (int i = 0; i < 2; ++i) out[i] = pair(std::move(codes[i]), fp8 ? scale[i].expand(lead) : std::move(scale[i]));
    return Py_BuildValue("(NN)", out[0], out[1]);
  });
}

// dequantize(kind, codes, scale, dtype, group_size) -> tensor, or None (likewise)
PyObject* py_dequantize(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  return guarded([&]() -> PyObject* {
    need_args(nargs, 5, "dequantize");
    if (!is_tensor(args[1]) || !is_tensor(args[2]) || !THPDtype_Check(args[3])) Py_RETURN_NONE;
    const int64_t kind = as_int(args[0]), group = as_int(args[4]);
    const at::Tensor &q = THPVariable_Unpack(args[1]), &s = THPVariable_Unpack(args[2]);
    const at::ScalarType dt = reinterpret_cast<THPDtype*>(args[3])->scalar_type;
    const bool fp8 = kind == FC_QUANT_E4M3 || kind == FC_QUANT_E5M2, bits4 = kind == FC_QUANT_INT4 || kind == FC_QUANT_NF4;
    if (!q.is_cuda() || s.device() != q.device() || s.scalar_type() != dt || !q.is_contiguous() || q.dim() < 1 || q.numel() == 0 ||
        s.numel() == 0 || (dt != at::kFloat && dt != at::kHalf && dt != at::kBFloat16))
      Py_RETURN_NONE;
    if (q.scalar_type() != (kind == FC_QUANT_INT8 ? at::kChar : bits4 ? at::kByte : fp8_type(kind))) Py_RETURN_NONE;
    const int64_t n = bits4 ? 2 * q.numel() : q.numel(), d = bits4 ? group : q.size(-1);
    if (!fp8 && (d < 1 || n % d || s.numel() != n / d || !s.is_contiguous())) Py_RETURN_NONE;
    std::vector<int64_t> shape = q.sizes().vec();
    if (bits4) shape.back() *= 2;
    at::Tensor out = at::empty(shape, q.options().dtype(dt));
    const int32_t code = dtype_code(dt);
    void* st = stream_of(q);
    if (fp8)
      check(fc_dequantize_fp8((const uint8_t*)q.const_data_ptr(), s.const_data_ptr(), n, kind == FC_QUANT_E5M2, code, code, out.data_ptr(), st),
            "fc_dequantize_fp8");
    else if (bits4)
      check(fc_dequantize_group4((const uint8_t*)q.const_data_ptr(), s.const_data_ptr(), n / d, (int32_t)d, code, code,
                                 kind == FC_QUANT_NF4, out.data_ptr(), st),
            "fc_dequantize_group4");
    else
      check(fc_dequantize_rows((const int8_t*)q.const_data_ptr(), s.const_data_ptr(), n / d, (int32_t)d, code, code, out.data_ptr(), st),
            "fc_dequantize_rows");
    return wrap(std::move(out));
  });
}

// The counters of a stream's decode launches: the index of the stream among those seen on its device, or -1 where a
// launch of its own must merge.  A graph under capture may be replayed on another stream; a stream that is not torch's
// own may be destroyed and its handle given to the next one while it still runs.
int decode_turn(const at::Tensor& t, const c10::hip::HIPStream& stream) {
  constexpr int kDevices = 64;
  static std::vector<c10::StreamId> seen[kDevices];     // under the interpreter's lock
  const int dev = t.get_device();
  const c10::StreamId id = stream.id();
  if (dev < 0 || dev >= kDevices || (id != 0 && !(id & 1))) return -1;
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream.stream(), &capture) != hipSuccess) {
    (void)hipGetLastError();
    return -1;
  }
  if (capture != hipStreamCaptureStatusNone) return -1;
  auto& ids = seen[dev];
  const auto at = std::find(ids.begin(), ids.end(), id);
  if (at != ids.end()) return (int)(at - ids.begin());
  if (ids.size() >= FC_DECODE_TURNS) return -1;
  ids.push_back(id);
  return (int)ids.size() - 1;
}

// ---- one attention layer of a decode step ---------------------------------------------------------------------------------
// decode_layer(q, k, v, k_cache, v_cache, slot_mapping, context_lens, block_tables, scale, q_heads, kv_heads, head_dim,
//              workspace or None, out or None, arrivals or None) -> out [n, q_heads * head_dim], or None when the arguments
// are not the plain decode step (the caller's general path then serves or refuses them).  arrivals: FC_DECODE_ARRIVALS zeros,
// counted on only beside the workspace they come with: a launch whose partial results lie elsewhere may run beside theirs.
PyObject* py_decode_layer(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  return guarded([&]() -> PyObject* {
    need_args(nargs, 15, "decode_layer");
    for (int i = 0; i < 8; ++i)
      if (!is_tensor(args[i])) Py_RETURN_NONE;
    const at::Tensor &q = THPVariable_Unpack(args[0]), &k = THPVariable_Unpack(args[1]), &v = THPVariable_Unpack(args[2]);
    const at::Tensor &kc = THPVariable_Unpack(args[3]), &vc = THPVariable_Unpack(args[4]);
    const at::Tensor &slots = THPVariable_Unpack(args[5]), &lens = THPVariable_Unpack(args[6]), &tables = THPVariable_Unpack(args[7]);
    const double scale = PyFloat_AsDouble(args[8]);
    if (scale == -1.0 && PyErr_Occurred()) throw PyFailed();
    const int64_t hq = as_int(args[9]), hkv = as_int(args[10]), d = as_int(args[11]);
    const at::ScalarType dt = kc.scalar_type();
    if (!q.is_cuda() || (dt != at::kHalf && dt != at::kBFloat16) || kc.dim() != 4 || tables.dim() != 2 || d <= 0) Py_RETURN_NONE;
    const auto dev = q.device();
    const int64_t n = tables.size(0), row = hkv * d;
    for (const at::Tensor* t : {&k, &v, &kc, &vc, &slots, &lens, &tables})
      if (t->device() != dev) Py_RETURN_NONE;
    for (const at::Tensor* t : {&q, &k, &v, &vc})
      if (t->scalar_type() != dt) Py_RETURN_NONE;
    for (const at::Tensor* t : {&slots, &lens, &tables})
      if (t->scalar_type() != at::kInt || !t->is_contiguous()) Py_RETURN_NONE;
    if (n == 0 || slots.numel() != n || lens.numel() != n || q.numel() != n * hq * d || !q.is_contiguous()) Py_RETURN_NONE;
    // new rows: [n, ...] with the row's elements adjacent
    int64_t stride[2];
    int i = 0;
    for (const at::Tensor* t : {&k, &v}) {
      if (t->numel() != n * row) Py_RETURN_NONE;
      if (t->is_contiguous()) stride[i] = row;
      else if (t->dim() == 2 && t->size(0) == n && t->stride(1) == 1) stride[i] = t->stride(0);
      else Py_RETURN_NONE;
      ++i;
    }
    if (kc.sizes() != vc.sizes() || kc.size(2) != hkv || kc.size(3) != d || !kc.is_contiguous() || !vc.is_contiguous())
      Py_RETURN_NONE;
    fc_kv_view kv{};
    kv.base = kc.data_ptr();
    kv.stride_token = row;
    kv.stride_head = hkv > 1 ? d : 0;
    kv.stride_block = kc.size(0) > 1 ? kc.size(1) * row : 0;
    kv.block_tables = (const int32_t*)tables.const_data_ptr();
    kv.table_stride = (int32_t)tables.size(1);
    kv.block_size = (int32_t)kc.size(1);
    kv.dtype = dtype_code(dt);
    kv.num_layers = 1;
    kv.batch = (int32_t)n;
    kv.num_kv_heads = (int32_t)hkv;
    kv.head_dim = (int32_t)d;
    kv.max_seq_len = (int32_t)(tables.size(1) * kc.size(1));
    fc_kv_view vv = kv;
    vv.base = vc.data_ptr();
    const int64_t need = fc_decode_layer_workspace_bytes(&kv, &vv, (int32_t)hq);
    if (need < 0) Py_RETURN_NONE;
    at::Tensor ws;
    void* wsp = nullptr;
    int64_t ws_bytes = 0;
    bool callers = false;        // the workspace is
    if (need > 0) {
      if (args[12] != Py_None) ws = tensor(args[12], "workspace");
      callers = ws.defined() && ws.device() == dev && ws.scalar_type() == at::kByte && ws.is_contiguous() && ws.numel() >= need;
      // the allocator hands blocks out per stream, so a workspace of this call is safe with any number of them
      if (!callers) ws = at::empty({need}, q.options().dtype(at::kByte));
      wsp = ws.data_ptr();
      ws_bytes = ws.numel();
    }
    at::Tensor out;
    if (args[13] != Py_None) {
      if (!is_tensor(args[13])) Py_RETURN_NONE;
      out = THPVariable_Unpack(args[13]);
      if (out.device() != dev || out.scalar_type() != dt || out.dim() != 2 || out.size(0) != n || out.size(1) != hq * d ||
          !out.is_contiguous() || ((uintptr_t)out.const_data_ptr() & 15) != 0)
        Py_RETURN_NONE;
    } else {
      out = at::empty({n, hq * d}, q.options());
    }
    const c10::hip::HIPStream stream = c10::hip::getCurrentHIPStream(q.get_device());
    const int32_t *sp = (const int32_t*)slots.const_data_ptr(), *lp = (const int32_t*)lens.const_data_ptr();
    if (callers && args[14] != Py_None) {
      const at::Tensor& arr = tensor(args[14], "arrivals");
      if (arr.device() != dev || arr.scalar_type() != at::kInt || !arr.is_contiguous() || arr.numel() < FC_DECODE_ARRIVALS)
        fail("decode_layer: arrivals must be contiguous int32 words on the device of q");
      check(fc_decode_layer_arrivals(&kv, &vv, q.const_data_ptr(), k.const_data_ptr(), stride[0], v.const_data_ptr(), stride[1], sp,
                                     out.data_ptr(), (int32_t)hq, lp, (float)scale, wsp, ws_bytes,
                                     (uint32_t*)arr.data_ptr(), (void*)stream.stream()),
            "fc_decode_layer");
    } else {
      check(fc_decode_layer_turn(&kv, &vv, q.const_data_ptr(), k.const_data_ptr(), stride[0], v.const_data_ptr(), stride[1], sp,
                                 out.data_ptr(), (int32_t)hq, lp, (float)scale, wsp, ws_bytes,
                                 ws_bytes ? decode_turn(q, stream) : -1, (void*)stream.stream()),
            "fc_decode_layer");
    }
    return wrap(std::move(out));
  });
}

// stage_decode(q, k, v, slots, lens, tables, q_static, k_static, v_static, slots_static, lens_static, tables_static) ->
// True, or False when a tensor is not of the plain form (the caller then copies piece by piece)
PyObject* py_stage_decode(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  return guarded([&]() -> PyObject* {
    need_args(nargs, 12, "stage_decode");
    const at::Tensor* t[12];
    for (int i = 0; i < 12; ++i) {
      if (!is_tensor(args[i])) Py_RETURN_FALSE;
      t[i] = &THPVariable_Unpack(args[i]);
      if (!t[i]->is_cuda() || t[i]->device() != t[0]->device()) Py_RETURN_FALSE;
    }
    const at::Tensor& gq = *t[6];
    const int64_t L = gq.size(0), bs = t[0]->dim() == 3 ? t[0]->size(1) : 0;
    for (int i = 0; i < 3; ++i) {
      const at::Tensor &x = *t[i], &g = *t[6 + i];
      if (x.dim() != 3 || g.dim() != 3 || x.scalar_type() != gq.scalar_type() || g.scalar_type() != gq.scalar_type() ||
          x.size(0) != L || g.size(0) != L || x.size(1) != bs || g.size(1) != gq.size(1) || x.size(2) != g.size(2) ||
          x.stride(2) != 1 || !g.is_contiguous())
        Py_RETURN_FALSE;
      const int64_t eb = x.element_size();
      if ((x.stride(0) * eb) % 16 || (x.stride(1) * eb) % 16 || (x.size(2) * eb) % 16 || ((uintptr_t)x.const_data_ptr() & 15))
        Py_RETURN_FALSE;
    }
    if (t[1]->size(2) != t[2]->size(2)) Py_RETURN_FALSE;
    for (int i = 3; i < 6; ++i)
      for (const at::Tensor* x : {t[i], t[6 + i]})
        if (x->scalar_type() != at::kInt || !x->is_contiguous()) Py_RETURN_FALSE;
    const at::Tensor &tab = *t[5], &gtab = *t[11];
    if (bs < 1 || bs > gq.size(1) || t[3]->numel() != bs || t[4]->numel() != bs || tab.dim() != 2 || tab.size(0) != bs ||
        gtab.dim() != 2 || gtab.size(0) != gq.size(1) || tab.size(1) < 1 || tab.size(1) > gtab.size(1) ||
        t[9]->numel() != gq.size(1) || t[10]->numel() != gq.size(1))
      Py_RETURN_FALSE;
    const auto ints = [](const at::Tensor& x) { return (int32_t*)x.data_ptr(); };
    check(fc_stage_decode(t[0]->const_data_ptr(), t[0]->stride(0), t[0]->stride(1), t[1]->const_data_ptr(), t[1]->stride(0),
                          t[1]->stride(1), t[2]->const_data_ptr(), t[2]->stride(0), t[2]->stride(1), (int32_t)L, (int32_t)bs,
                          (int32_t)t[0]->size(2), (int32_t)t[1]->size(2), dtype_code(gq.scalar_type()), ints(*t[3]),
                          ints(*t[4]), ints(tab), (int32_t)tab.size(1), t[6]->data_ptr(), t[7]->data_ptr(), t[8]->data_ptr(),
                          ints(*t[9]), ints(*t[10]), ints(gtab), (int32_t)gq.size(1), (int32_t)gtab.size(1), stream_of(gq)),
          "fc_stage_decode");
    Py_RETURN_TRUE;
  });
}

// ---- a step's numbers to the device -----------------------------------------------------------------------------------------
// Up to FC_UPLOAD_MAX bytes travel as a kernel's arguments, more (and what a stream under capture is given, which the
// callers refuse or torch does, and what is not for a GPU) as a copy from pinned memory.
struct Packed {
  at::Tensor host, dev;
  std::vector<char> small;
  int64_t at = 0;
  void* stream = nullptr;      // of `small`
  Packed(int64_t bytes, const c10::Device& device)
      : dev(at::empty({bytes}, at::TensorOptions().dtype(at::kByte).device(device))) {
    if (device.is_cuda() && bytes <= FC_UPLOAD_MAX && bytes % 4 == 0) {
      const hipStream_t st = c10::hip::getCurrentHIPStream(device.index()).stream();
      hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
      if (hipStreamIsCapturing(st, &capture) != hipSuccess) {
        (void)hipGetLastError();
      } else if (capture == hipStreamCaptureStatusNone) {
        small.resize(std::max<int64_t>(bytes, 1));
        stream = (void*)st;
      }
    }
    if (small.empty()) host = at::empty({bytes}, at::TensorOptions().dtype(at::kByte).pinned_memory(true));
  }
  template <typename T>
  T* take(int64_t n) {
    T* p = (T*)((small.empty() ? (char*)host.data_ptr() : small.data()) + at);
    at += n * (int64_t)sizeof(T);
    return p;
  }
  void send() {
    if (small.empty()) {
      dev.copy_(host, true);
    } else if (dev.numel() > 0) {
      const c10::DeviceGuard guard(dev.device());
      check(fc_upload(dev.data_ptr(), small.data(), (int32_t)dev.numel(), stream), "fc_upload");
    }
  }
  at::Tensor part(int64_t byte, int64_t n, at::ScalarType t) { return dev.narrow(0, byte, n * (int64_t)c10::elementSize(t)).view(t); }
};

c10::Device device_arg(PyObject* o) { return tensor(o, "device reference").device(); }

// rows of Python ints, right-padded with -1
int64_t table_width(PyObject* tables, Py_ssize_t n) {
  int64_t width = 0;
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* row = PyList_GET_ITEM(tables, i);
    if (!PyList_Check(row)) fail("a block table is a list of page numbers");
    width = std::max<int64_t>(width, PyList_GET_SIZE(row));
  }
  return width;
}

void fill_tables(PyObject* tables, Py_ssize_t n, int64_t width, int32_t* out) {
  for (Py_ssize_t i = 0; i < n; ++i, out += width) {
    PyObject* row = PyList_GET_ITEM(tables, i);
    const Py_ssize_t len = PyList_GET_SIZE(row);
    for (Py_ssize_t j = 0; j < len; ++j) out[j] = (int32_t)as_int(PyList_GET_ITEM(row, j));
    for (int64_t j = len; j < width; ++j) out[j] = -1;
  }
}

// decode_inputs(ids, lens, tables, block_size, ref) -> (input_ids, positions, slots, context_lens, block_tables) on the
// device of `ref`: one upload instead of five
PyObject* py_decode_inputs(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  return guarded([&]() -> PyObject* {
    need_args(nargs, 5, "decode_inputs");
    for (int i = 0; i < 3; ++i)
      if (!PyList_Check(args[i])) fail("decode_inputs: lists expected");
    const Py_ssize_t n = PyList_GET_SIZE(args[0]);
    if (n == 0 || PyList_GET_SIZE(args[1]) != n || PyList_GET_SIZE(args[2]) != n) fail("decode_inputs: lists of one length expected");
    const int64_t bs = as_int(args[3]), width = table_width(args[2], n);
    Packed pk(n * 16 + n * 8 + n * width * 4, device_arg(args[4]));
    int64_t *ids = pk.take<int64_t>(n), *pos = pk.take<int64_t>(n);
    int32_t *slots = pk.take<int32_t>(n), *lens = pk.take<int32_t>(n), *tab = pk.take<int32_t>(n * width);
    for (Py_ssize_t i = 0; i < n; ++i) {
      ids[i] = as_int(PyList_GET_ITEM(args[0], i));
      const int64_t len = as_int(PyList_GET_ITEM(args[1], i));
      pos[i] = len;
      lens[i] = (int32_t)len;
      PyObject* row = PyList_GET_ITEM(args[2], i);
      const Py_ssize_t pages = PyList_GET_SIZE(row);
      if (pages == 0) {
        PyErr_SetString(PyExc_IndexError, "sequence without pages");
        throw PyFailed();
      }
      const int64_t page = as_int(PyList_GET_ITEM(row, std::min<int64_t>(len / bs, pages - 1)));
      slots[i] = (int32_t)(page * bs + len % bs);
    }
    fill_tables(args[2], n, width, tab);
    pk.send();
    PyObject* out = PyTuple_New(5);
    PyTuple_SET_ITEM(out, 0, wrap(pk.part(0, n, at::kLong)));
    PyTuple_SET_ITEM(out, 1, wrap(pk.part(n * 8, n, at::kLong)));
    PyTuple_SET_ITEM(out, 2, wrap(pk.part(n * 16, n, at::kInt)));
    PyTuple_SET_ITEM(out, 3, wrap(pk.part(n * 20, n, at::kInt)));
    PyTuple_SET_ITEM(out, 4, wrap(pk.part(n * 24, n * width, at::kInt).view({n, width})));
    return out;
  });
}

// upload_tables(tables, rows, ref) -> (block_tables [n, width], then one int32 tensor per list of `rows`)
PyObject* py_upload_tables(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  return guarded([&]() -> PyObject* {
    need_args(nargs, 3, "upload_tables");
    if (!PyList_Check(args[0]) || !PyTuple_Check(args[1])) fail("upload_tables: a list of tables and a tuple of lists expected");
    const Py_ssize_t n = PyList_GET_SIZE(args[0]), extra = PyTuple_GET_SIZE(args[1]);
    const int64_t width = table_width(args[0], n);
    int64_t total = n * width;
    for (Py_ssize_t i = 0; i < extra; ++i) {
      if (!PyList_Check(PyTuple_GET_ITEM(args[1], i))) fail("upload_tables: lists of ints expected");
      total += PyList_GET_SIZE(PyTuple_GET_ITEM(args[1], i));
    }
    Packed pk(total * 4, device_arg(args[2]));
    fill_tables(args[0], n, width, pk.take<int32_t>(n * width));
    for (Py_ssize_t i = 0; i < extra; ++i) {
      PyObject* row = PyTuple_GET_ITEM(args[1], i);
      const Py_ssize_t len = PyList_GET_SIZE(row);
      int32_t* p = pk.take<int32_t>(len);
      for (Py_ssize_t j = 0; j < len; ++j) p[j] = (int32_t)as_int(PyList_GET_ITEM(row, j));
    }
    pk.send();
    PyObject* out = PyTuple_New(1 + extra);
    PyTuple_SET_ITEM(out, 0, wrap(pk.part(0, n * width, at::kInt).view({n, width})));
    int64_t byte = n * width * 4;
    for (Py_ssize_t i = 0; i < extra; ++i) {
      const int64_t len = PyList_GET_SIZE(PyTuple_GET_ITEM(args[1], i));
      PyTuple_SET_ITEM(out, 1 + i, wrap(pk.part(byte, len, at::kInt)));
      byte += len * 4;
    }
    return out;
  });
}

// ---- presses of a paged pool whose caller wants the moved rows alone ------------------------------------------------------------
// One plane of a pool [2, L, blocks, block_size, Hkv, D] as the views of _lib.paged_view
fc_kv_view paged_view(const at::Tensor& pool, int plane, const at::Tensor& tables, const at::Tensor& lens, int64_t max_len) {
  const auto stride = [&](int i) { return pool.size(i) > 1 ? pool.stride(i) : 0; };
  fc_kv_view v{};
  v.base = (char*)pool.data_ptr() + plane * pool.stride(0) * (int64_t)pool.element_size();
  v.stride_layer = stride(1);
  v.stride_block = stride(2);
  v.stride_token = stride(3);
  v.stride_head = stride(4);
  v.block_tables = tables.data_ptr<int32_t>();
  v.table_stride = (int32_t)tables.size(1);
  v.block_size = (int32_t)pool.size(3);
  v.dtype = dtype_code(pool.scalar_type());
  v.num_layers = (int32_t)pool.size(1);
  v.batch = (int32_t)tables.size(0);
  v.num_kv_heads = (int32_t)pool.size(4);
  v.head_dim = (int32_t)pool.size(5);
  v.max_seq_len = (int32_t)max_len;
  v.seq_lens = lens.data_ptr<int32_t>();
  return v;
}

// A device block cut into pieces that start on 256 bytes
struct Scratch {
  at::Tensor mem;
  int64_t at = 0;
  static int64_t room(int64_t bytes) { return (bytes + 255) / 256 * 256; }
  Scratch(int64_t bytes, const at::Tensor& ref) : mem(at::empty({bytes}, ref.options().dtype(at::kByte))) {}
  void* take(int64_t bytes) {
    void* p = (char*)mem.data_ptr() + at;
    at += room(bytes);
    return p;
  }
};

// press_rows(pool, tables, lens, max_len, width, counts or None, order or None, snapkv or None) -> True, or None (the
// caller's general path then serves or refuses the arguments).  The kept rows of every column move to the front of its pages;
// scores and indices are scratch.  counts: kept rows per sequence where they differ; order: the sequences, longest first.
// snapkv = (queries, window, kernel_size, causal, scale, out_scale, fits, mean length): one launch where the shape fits one and cutting
// the columns does not pay, else key ranges, selection and compaction; None: the Knorm press in one launch; False: its norms, selection and compaction.  Views, scratch and uploads in Python cost 25 to 45 us before the launch,
// with the GPU idle behind the last pass's synchronisation: 13 sequences of 200 to 2300 tokens (SnapKV, 28 layers) 500 -> 475 us.
PyObject* py_press_rows(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  return guarded([&]() -> PyObject* {
    need_args(nargs, 8, "press_rows");
    for (int i = 0; i < 3; ++i)
      if (!is_tensor(args[i])) Py_RETURN_NONE;
    const at::Tensor &pool = THPVariable_Unpack(args[0]), &tables = THPVariable_Unpack(args[1]), &lens = THPVariable_Unpack(args[2]);
    const int64_t S = as_int(args[3]), width = as_int(args[4]);
    if (!pool.is_cuda() || pool.dim() != 6 || pool.size(0) != 2 || pool.stride(5) != 1 || tables.device() != pool.device() ||
        lens.device() != pool.device() || tables.scalar_type() != at::kInt || lens.scalar_type() != at::kInt ||
        tables.dim() != 2 || !tables.is_contiguous() || !lens.is_contiguous() || lens.numel() != tables.size(0) ||
        tables.size(0) == 0 || width <= 0 || S <= 0)
      Py_RETURN_NONE;
    if (pool.numel() == 0) Py_RETURN_NONE;
    const int64_t L = pool.size(1), B = tables.size(0), H = pool.size(4), D = pool.size(5), cols = L * B * H;
    const fc_kv_view kv = paged_view(pool, 0, tables, lens, S), vv = paged_view(pool, 1, tables, lens, S);
    at::Tensor q;
    int64_t W = 0, ksz = 0, causal = 0, hq = 0;
    int32_t nsplit = 1;
    bool one = true, once = false;
    double scale = 0, out_scale = 0;
    const bool norms_apart = args[7] == Py_False;
    if (args[7] != Py_None && !norms_apart) {
      if (!PyTuple_Check(args[7]) || PyTuple_GET_SIZE(args[7]) != 8) fail("press_rows: the SnapKV arguments are a tuple of eight");
      const auto item = [&](int i) { return PyTuple_GET_ITEM(args[7], i); };
      q = tensor(item(0), "queries");
      W = as_int(item(1));
      ksz = as_int(item(2));
      causal = as_int(item(3));
      scale = PyFloat_AsDouble(item(4));
      out_scale = PyFloat_AsDouble(item(5));
      const bool fits = as_int(item(6)) != 0;
      if (PyErr_Occurred()) throw PyFailed();
      if (q.device() != pool.device() || q.scalar_type() != pool.scalar_type() || !q.is_contiguous() || q.dim() != 5 ||
          q.size(0) != L || q.size(1) != B || q.size(3) != W || q.size(4) != D || W <= 0 || q.size(2) % H)
        Py_RETURN_NONE;
      hq = q.size(2);
      nsplit = fc_snapkv_rows_route(&kv, (int32_t)hq, (int32_t)W, fits, (int32_t)as_int(item(7)));
      if (nsplit < 0) Py_RETURN_NONE;
      once = fc_snapkv_rows_once_pays(&kv, (int32_t)hq, (int32_t)W, (int32_t)as_int(item(7)), (int32_t)width, nsplit) != 0;
      one = nsplit == 0 && !once;
    }
    const int32_t *counts = nullptr, *order = nullptr;
    at::Tensor numbers;      // kept until the launches are enqueued
    if (args[5] != Py_None) {
      const bool ordered = args[6] != Py_None && one;      // (the one launch's columns start in that order)
      if (!PyList_Check(args[5]) || PyList_GET_SIZE(args[5]) != B || (ordered && (!PyList_Check(args[6]) || PyList_GET_SIZE(args[6]) != B)))
        fail("press_rows: one count per sequence expected");
      Packed pk((ordered ? 2 : 1) * B * 4, pool.device());
      int32_t* p = pk.take<int32_t>((ordered ? 2 : 1) * B);
      for (Py_ssize_t i = 0; i < B; ++i) {
        p[i] = (int32_t)as_int(PyList_GET_ITEM(args[5], i));
        if (ordered) p[B + i] = (int32_t)as_int(PyList_GET_ITEM(args[6], i));
      }
      pk.send();
      numbers = pk.dev;
      counts = (const int32_t*)numbers.data_ptr();
      if (ordered) order = counts + B;
    }
    void* stream = stream_of(pool);
    const int64_t idx_bytes = cols * width * 4;
    if (!one) {
      const int64_t ws = once ? fc_snapkv_once_workspace_bytes(&kv, (int32_t)hq, (int32_t)W)
                              : fc_snapkv_select_workspace_bytes((int32_t)L, (int32_t)B, (int32_t)hq, (int32_t)H, (int32_t)W, (int32_t)S, nsplit);
      Scratch mem(Scratch::room(idx_bytes) + ws, pool);
      int32_t* idx = (int32_t*)mem.take(idx_bytes);
      if (once)
        check(fc_snapkv_select_once(&kv, q.const_data_ptr(), (int32_t)hq, (int32_t)W, (int32_t)ksz, (int32_t)causal, (float)scale,
                                    (float)out_scale, (int32_t)width, counts, idx, (int32_t)width, 0, mem.take(ws), ws, stream),
              "fc_snapkv_select_once");
      else check(fc_snapkv_select(&kv, q.const_data_ptr(), nullptr, (int32_t)hq, (int32_t)W, (int32_t)ksz, (int32_t)causal,
                             (float)scale, (float)out_scale, (int32_t)width, counts, idx, (int32_t)width, nsplit,
                             mem.take(ws), ws, stream),
            "fc_snapkv_select");
      check(fc_compact(&kv, &vv, &kv, &vv, idx, (int32_t)width, (int32_t)H, (int32_t)width, counts, stream), "fc_compact");
      Py_RETURN_TRUE;
    }
    Scratch mem(Scratch::room(idx_bytes) + Scratch::room(cols * S * 4) + cols * 4, pool);
    int32_t* idx = (int32_t*)mem.take(idx_bytes);
    float* scores = (float*)mem.take(cols * S * 4);
    if (norms_apart) {
      check(fc_knorm_score(&kv, scores, (int32_t)S, stream), "fc_knorm_score");
      check(fc_topk_select(scores, (int32_t)S, (int32_t)cols, (int32_t)S, counts ? lens.data_ptr<int32_t>() : nullptr, (int32_t)H,
                           counts ? (int32_t)B : 1, (int32_t)width, counts, idx, (int32_t)width, stream),
            "fc_topk_select");
      check(fc_compact(&kv, &vv, &kv, &vv, idx, (int32_t)width, (int32_t)H, (int32_t)width, counts, stream), "fc_compact");
    } else if (!q.defined()) {
      check(fc_knorm_press(&kv, &vv, scores, (int32_t)S, (int32_t)width, counts, idx, (int32_t)width, stream), "fc_knorm_press");
    } else if (order) {
      check(fc_snapkv_press_ordered(&kv, &vv, q.const_data_ptr(), nullptr, (int32_t)hq, (int32_t)W, (int32_t)ksz, (int32_t)causal,
                                    (float)scale, (float)out_scale, scores, (int32_t)S, (float*)mem.take(cols * 4), (int32_t)width,
                                    counts, idx, (int32_t)width, order, stream),
            "fc_snapkv_press_ordered");
    } else {
      check(fc_snapkv_press(&kv, &vv, q.const_data_ptr(), nullptr, (int32_t)hq, (int32_t)W, (int32_t)ksz, (int32_t)causal,
                            (float)scale, (float)out_scale, scores, (int32_t)S, (float*)mem.take(cols * 4), (int32_t)width, counts,
                            idx, (int32_t)width, stream),
            "fc_snapkv_press");
    }
    Py_RETURN_TRUE;
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
    {"decode_layer", (PyCFunction)(void (*)(void))py_decode_layer, METH_FASTCALL,
     "decode_layer(q, k, v, k_cache, v_cache, slots, lens, tables, scale, q_heads, kv_heads, head_dim, workspace) -> out or None"},
    {"stage_decode", (PyCFunction)(void (*)(void))py_stage_decode, METH_FASTCALL,
     "stage_decode(q, k, v, slots, lens, tables, and the six static buffers) -> bool"},
    {"decode_inputs", (PyCFunction)(void (*)(void))py_decode_inputs, METH_FASTCALL,
     "decode_inputs(ids, lens, tables, block_size, ref) -> five device tensors"},
    {"upload_tables", (PyCFunction)(void (*)(void))py_upload_tables, METH_FASTCALL,
     "upload_tables(tables, (list, ...), ref) -> device tensors"},
    {"press_rows", (PyCFunction)(void (*)(void))py_press_rows, METH_FASTCALL,
     "press_rows(pool, tables, lens, max_len, width, counts, order, snapkv) -> True or None"},
    {"quantize_pair", (PyCFunction)(void (*)(void))py_quantize_pair, METH_FASTCALL,
     "quantize_pair(kind, keys, values, group_size) -> ((codes, scale), (codes, scale)) or None"},
    {"dequantize", (PyCFunction)(void (*)(void))py_dequantize, METH_FASTCALL,
     "dequantize(kind, codes, scale, dtype, group_size) -> tensor or None"},
    {"knorm_into", (PyCFunction)(void (*)(void))py_knorm_into, METH_FASTCALL, "knorm_into(keys, values, n) -> (k, v) or None"},
    {"snapkv_into", (PyCFunction)(void (*)(void))py_snapkv_into, METH_FASTCALL,
     "snapkv_into(keys, values, queries, lse, n, window, kernel_size, causal, scale, out_scale) -> (k, v) or None"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_host", "host path of fastcache_amd", -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) { return PyModule_Create(&kModule); }

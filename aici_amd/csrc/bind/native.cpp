// CPython binding of the hot entry points of libhipattn.so: aici_amd/_native.so.
//
// A generation step makes about ten calls per layer, and with few rows the device finishes a layer in some hundred
// microseconds, so what the host spends per call decides the time of a step.  Through ctypes a call with eight tensors cost
// 30 to 40 us (a Structure filled field by field from tensor methods, the current stream looked up in Python); here a
// tensor argument is one call of torch's DLPack exchange function -- the tensor's own size and stride arrays, no
// Python objects made -- and the stream comes from the same table.
//
// Every wrapper is generated from the C prototype in hipattn.h: the parameter types say how an argument is converted.
// The stream, always the last parameter, is not passed from Python: it is torch's current stream on the device of
// the call's first GPU tensor.  Errors are raised as aici_amd._lib.HipAttnError with the library's message.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/dlpack.h>

#include <cstring>
#include <string>
#include <tuple>
#include <utility>
#include <vector>

#include "../../../include/hipattn.h"

namespace {

PyObject *g_error = nullptr;                     // HipAttnError
PyTypeObject *g_tensor_type = nullptr;           // torch.Tensor
const DLPackExchangeAPI *g_exchange = nullptr;   // torch's table

struct Call {
  const char *fn;      // entry point, for messages
  const char *names;   // parameter names, comma separated
  int device_type = -1, device = 0;  // of the first GPU tensor
};

// The i-th of a comma-separated list (error path only).
std::string name_at(const char *names, int i) {
  const char *p = names;
  for (; i > 0 && *p; p++)
    if (*p == ',') i--;
  const char *e = strchr(p, ',');
  return e ? std::string(p, e) : std::string(p);
}

bool dtype_of(const DLDataType &t, int32_t *out) {
  if (t.lanes != 1) return false;
  switch (t.code) {
    case kDLFloat: if (t.bits == 32) *out = HIPATTN_F32; else if (t.bits == 16) *out = HIPATTN_F16; else return false; return true;
    case kDLBfloat: if (t.bits != 16) return false; *out = HIPATTN_BF16; return true;
    case kDLInt: if (t.bits == 32) *out = HIPATTN_I32; else if (t.bits == 64) *out = HIPATTN_I64; else return false; return true;
    case kDLUInt: if (t.bits != 8) return false; *out = HIPATTN_U8; return true;
    default: return false;
  }
}

bool describe(PyObject *o, int index, Call &c, hipattn_tensor *d) {
  if (Py_TYPE(o) != g_tensor_type && !PyObject_TypeCheck(o, g_tensor_type)) {
    PyErr_Format(PyExc_TypeError, "%s: expected a torch.Tensor or None, got %s", name_at(c.names, index).c_str(),
                 Py_TYPE(o)->tp_name);
    return false;
  }
  DLTensor t;
  if (g_exchange->dltensor_from_py_object_no_sync(o, &t) != 0) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, "the tensor cannot be described");
    return false;
  }
  if (!dtype_of(t.dtype, &d->dtype)) {
    PyObject *dt = PyObject_GetAttrString(o, "dtype");
    PyErr_Format(g_error, "%s: unsupported dtype %S", name_at(c.names, index).c_str(), dt ? dt : Py_None);
    Py_XDECREF(dt);
    return false;
  }
  if (t.device.device_type != kDLROCM && t.device.device_type != kDLCUDA) {
    PyObject *dev = PyObject_GetAttrString(o, "device");
    PyErr_Format(g_error, "%s: expected a GPU tensor, got one on %S", name_at(c.names, index).c_str(), dev ? dev : Py_None);
    Py_XDECREF(dev);
    return false;
  }
  if (t.ndim > HIPATTN_MAX_DIMS) {
    PyErr_Format(g_error, "%s: at most %d dims", name_at(c.names, index).c_str(), HIPATTN_MAX_DIMS);
    return false;
  }
  d->data = static_cast<char *>(t.data) + t.byte_offset;
  d->ndim = t.ndim;
  int64_t dense = 1;
  for (int i = t.ndim - 1; i >= 0; i--) {
    d->sizes[i] = t.shape[i];
    d->strides[i] = t.strides ? t.strides[i] : dense;
    dense *= t.shape[i];
  }
  if (c.device_type < 0) {
    c.device_type = t.device.device_type;
    c.device = t.device.device_id;
  }
  return true;
}

bool to_i64(PyObject *o, int64_t *v) {
  if (PyLong_CheckExact(o)) {
    *v = PyLong_AsLongLong(o);
  } else {  // whatever int() takes
    PyObject *n = PyNumber_Long(o);
    if (n == nullptr) return false;
    *v = PyLong_AsLongLong(n);
    Py_DECREF(n);
  }
  return !(*v == -1 && PyErr_Occurred());
}

// Arg<T>: one parameter.  `from` takes the Python argument it consumes; `value` is what the C call gets.
template <typename T>
struct Arg;

template <>
struct Arg<hipattn_tensor *> {
  static constexpr bool kFromPython = true;
  hipattn_tensor d;
  hipattn_tensor *p = nullptr;
  bool from(PyObject *o, int index, Call &c) {
    if (o == Py_None) return true;
    p = &d;
    return describe(o, index, c, &d);
  }
  bool finish(Call &) { return true; }
  hipattn_tensor *value() { return p; }
};
template <>
struct Arg<const hipattn_tensor *> : Arg<hipattn_tensor *> {};

template <>
struct Arg<int64_t> {
  static constexpr bool kFromPython = true;
  int64_t v = 0;
  bool from(PyObject *o, int, Call &) { return to_i64(o, &v); }
  bool finish(Call &) { return true; }
  int64_t value() { return v; }
};
template <>
struct Arg<int> {
  static constexpr bool kFromPython = true;
  int v = 0;
  bool from(PyObject *o, int index, Call &c) {
    int64_t w;
    if (!to_i64(o, &w)) return false;
    if (w < INT32_MIN || w > INT32_MAX) {
      PyErr_Format(PyExc_OverflowError, "%s does not fit 32 bits", name_at(c.names, index).c_str());
      return false;
    }
    v = (int)w;
    return true;
  }
  bool finish(Call &) { return true; }
  int value() { return v; }
};
template <>
struct Arg<float> {
  static constexpr bool kFromPython = true;
  float v = 0.f;
  bool from(PyObject *o, int, Call &) {
    const double d = PyFloat_AsDouble(o);
    v = (float)d;
    return !(d == -1.0 && PyErr_Occurred());
  }
  bool finish(Call &) { return true; }
  float value() { return v; }
};
template <>
struct Arg<bool> {
  static constexpr bool kFromPython = true;
  bool v = false;
  bool from(PyObject *o, int, Call &) {
    const int t = PyObject_IsTrue(o);
    v = t == 1;
    return t >= 0;
  }
  bool finish(Call &) { return true; }
  bool value() { return v; }
};
// The stream: torch's current one on the device of the first GPU tensor.
template <>
struct Arg<void *> {
  static constexpr bool kFromPython = false;
  void *s = nullptr;
  bool from(PyObject *, int, Call &) { return true; }
  bool finish(Call &c) {
    if (c.device_type < 0) return true;  // no tensor at all: the library says what is missing
    if (g_exchange->current_work_stream((DLDeviceType)c.device_type, c.device, &s) != 0) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, "no current stream");
      return false;
    }
    return true;
  }
  void *value() { return s; }
};

template <auto Fn>
struct Binding;

template <typename... A, char *(*Fn)(A...)>
struct Binding<Fn> {
  static const char *fn, *names;
  static constexpr int kArgs = ((Arg<A>::kFromPython ? 1 : 0) + ...);

  static PyObject *call(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != kArgs) {
      PyErr_Format(PyExc_TypeError, "%s takes %d arguments (%s), got %zd", fn, kArgs, names, n);
      return nullptr;
    }
    return go(args, std::index_sequence_for<A...>{});
  }
  template <size_t... I>
  static PyObject *go(PyObject *const *args, std::index_sequence<I...>) {
    std::tuple<Arg<A>...> a;
    Call c{fn, names};
    int at = 0;
    const bool ok = ([&] {
      auto &x = std::get<I>(a);
      if (!std::remove_reference_t<decltype(x)>::kFromPython) return true;
      const int i = at++;
      return x.from(args[i], i, c);
    }() && ...) && (std::get<I>(a).finish(c) && ...);
    if (!ok) return nullptr;
    char *err;
    Py_BEGIN_ALLOW_THREADS
    err = Fn(std::get<I>(a).value()...);
    Py_END_ALLOW_THREADS
    if (err != nullptr) {
      PyErr_Format(g_error, "hipattn_%s: %s", fn, err);
      hipattn_free_error(err);
      return nullptr;
    }
    Py_RETURN_NONE;
  }
};
template <typename... A, char *(*Fn)(A...)>
const char *Binding<Fn>::fn = "";
template <typename... A, char *(*Fn)(A...)>
const char *Binding<Fn>::names = "";

template <auto Fn>
PyMethodDef method(const char *fn, const char *names) {
  Binding<Fn>::fn = fn;
  Binding<Fn>::names = names;
  return {fn, (PyCFunction)(void (*)(void))Binding<Fn>::call, METH_FASTCALL, names};
}

// copy_blocks(key_caches, value_caches, pairs): lists of every layer's caches and of src, dst, src, dst, ...  True if done;
// False where the caches are not what hipattn_copy_blocks_host takes (the caller then has its own checks).
PyObject *copy_blocks(PyObject *, PyObject *const *args, Py_ssize_t n) {
  if (n != 3) {
    PyErr_Format(PyExc_TypeError, "copy_blocks takes 3 arguments (key_caches,value_caches,pairs), got %zd", n);
    return nullptr;
  }
  Call c{"copy_blocks", "key_caches,value_caches,pairs"};
  std::vector<void *> ptrs[2];
  hipattn_tensor first{};
  int64_t bytes = 1;
  PyObject *held[3] = {nullptr, nullptr, nullptr};
  struct Release {
    PyObject **held;
    ~Release() {
      for (int i = 0; i < 3; i++) Py_XDECREF(held[i]);
    }
  } release{held};
  for (int i = 0; i < 3; i++)
    if ((held[i] = PySequence_Fast(args[i], "copy_blocks: expected sequences")) == nullptr) return nullptr;
  for (int side = 0; side < 2; side++) {
    const Py_ssize_t layers = PySequence_Fast_GET_SIZE(held[side]);
    for (Py_ssize_t l = 0; l < layers; l++) {
      PyObject *o = PySequence_Fast_GET_ITEM(held[side], l);
      hipattn_tensor d{};
      DLTensor t;
      if (!PyObject_TypeCheck(o, g_tensor_type) || g_exchange->dltensor_from_py_object_no_sync(o, &t) != 0) {
        PyErr_Clear();
        Py_RETURN_FALSE;
      }
      if ((t.device.device_type != kDLROCM && t.device.device_type != kDLCUDA) || t.ndim < 1 || t.ndim > HIPATTN_MAX_DIMS ||
          !dtype_of(t.dtype, &d.dtype) || (d.dtype != HIPATTN_F16 && d.dtype != HIPATTN_BF16) || !describe(o, side, c, &d)) {
        PyErr_Clear();
        Py_RETURN_FALSE;
      }
      int64_t dense = 1, all = 1;
      bool contiguous = true;
      for (int i = d.ndim - 1; i >= 0; i--) {
        contiguous = contiguous && (d.sizes[i] == 1 || d.strides[i] == dense);
        dense *= d.sizes[i];
        if (i > 0) all *= d.sizes[i];
      }
      if (side == 0 && l == 0) {
        first = d;
        bytes = all * 2;
      }
      int64_t first_numel = 1;
      for (int i = 0; i < first.ndim; i++) first_numel *= first.sizes[i];
      if (!contiguous || dense != first_numel || t.device.device_id != c.device ||
          (reinterpret_cast<uintptr_t>(d.data) & 15) != 0) Py_RETURN_FALSE;
      ptrs[side].push_back(d.data);
    }
  }
  if (bytes <= 0 || bytes % 16 != 0 || bytes > (1 << 26) || ptrs[0].size() != ptrs[1].size() || ptrs[0].empty()) Py_RETURN_FALSE;
  const Py_ssize_t count = PySequence_Fast_GET_SIZE(held[2]);
  std::vector<int64_t> pairs((size_t)count);
  for (Py_ssize_t i = 0; i < count; i++)
    if (!to_i64(PySequence_Fast_GET_ITEM(held[2], i), &pairs[(size_t)i])) return nullptr;
  for (Py_ssize_t i = 0; i + 1 < count; i += 2) {
    const int64_t src = pairs[(size_t)i], dst = pairs[(size_t)i + 1], blocks = first.sizes[0];
    if (src < 0 || src >= blocks || dst < 0 || dst >= blocks) {
      PyErr_Format(g_error, "copy_blocks: pair %lld -> %lld out of range, the caches have %lld blocks", (long long)src, (long long)dst,
                   (long long)blocks);
      return nullptr;
    }
  }
  if (first.sizes[0] > INT32_MAX) Py_RETURN_FALSE;
  void *stream = nullptr;
  if (g_exchange->current_work_stream((DLDeviceType)c.device_type, c.device, &stream) != 0) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, "no current stream");
    return nullptr;
  }
  char *err;
  Py_BEGIN_ALLOW_THREADS
  err = hipattn_copy_blocks_host(ptrs[0].data(), ptrs[1].data(), (int64_t)ptrs[0].size(), pairs.data(), count / 2, bytes, stream);
  Py_END_ALLOW_THREADS
  if (err != nullptr) {
    PyErr_Format(g_error, "hipattn_copy_blocks_host: %s", err);
    hipattn_free_error(err);
    return nullptr;
  }
  Py_RETURN_TRUE;
}
#define BIND(name, names) method<hipattn_##name>(#name, names)

PyMethodDef g_methods[] = {
    BIND(mha_varlen_fwd, "q,k,v,seqlens_q,seqlens_k,seqused_k,max_seqlen_q,max_seqlen_k,p_dropout,softmax_scale,"
                         "zero_tensors,causal,window_left,window_right,out,lse"),
    BIND(mha_varlen_fwd_paged, "q,key_cache,value_cache,block_tables,cu_seqlens_q,context_lens,max_seqlen_q,max_seqlen_k,"
                               "softmax_scale,causal,out,lse"),
    BIND(paged_attention_v1, "out,query,key_cache,value_cache,num_kv_heads,scale,block_tables,context_lens,block_size,"
                             "max_context_len,alibi"),
    BIND(paged_attention_v1_static, "out,query,key_cache,value_cache,num_kv_heads,scale,block_tables,context_lens,"
                                    "block_size,max_context_len,alibi"),
    BIND(paged_attention_v2, "out,exp_sums,max_logits,tmp_out,query,key_cache,value_cache,num_kv_heads,scale,"
                             "block_tables,context_lens,block_size,max_context_len,alibi"),
    BIND(reshape_and_cache, "key,value,key_cache,value_cache,slot_mapping"),
    BIND(gather_cached_kv, "key,value,key_cache,value_cache,slot_mapping"),
    {"copy_blocks", (PyCFunction)(void (*)(void))copy_blocks, METH_FASTCALL, "key_caches,value_caches,pairs"},
    BIND(rotary_embedding, "positions,query,key,head_size,cos_sin_cache,is_neox"),
    BIND(rotary_embedding_and_cache, "positions,query,key,value,head_size,cos_sin_cache,is_neox,key_cache,value_cache,"
                                     "slot_mapping"),
    BIND(rms_norm, "out,input,weight,epsilon"),
    BIND(fused_add_rms_norm, "input,residual,weight,epsilon"),
    BIND(add_rms_norm, "out,input,residual,weight,epsilon"),
    BIND(linear, "out,x,weight,bias,residual,workspace"),
    BIND(linear_silu_and_mul, "out,x,weight,workspace"),
    BIND(linear_rms_norm, "out,norm_out,x,weight,bias,residual,norm_weight,epsilon,workspace"),
    BIND(rms_norm_linear, "out,x,norm_weight,epsilon,weight,silu_and_mul"),
    BIND(qkv_linear, "out,x,norm_weight,epsilon,weight,positions,cos_sin_cache,key_cache,value_cache,slot_mapping"),
    BIND(silu_and_mul, "out,input"),
    BIND(gelu_new, "out,input"),
    BIND(gelu_fast, "out,input"),
    BIND(bias_argmax, "logits,bias,mask,bias_rows,out_tokens,out_logits"),
    BIND(bias_sample, "logits,bias,mask,bias_rows,temperature,top_p,uniforms,out_tokens"),
    BIND(varlen_attn, "q,k,v,key_cache,value_cache,slot_mapping,gather_mapping,seqlens_q,seqlens_k,q_multi,max_seqlen_q,"
                      "max_seqlen_k,paged_block_tables,paged_context_lens,paged_block_size,paged_max_context_len,"
                      "softmax_scale,gather_k,gather_v,y"),
    BIND(varlen_attn_paged, "q,k,v,key_cache,value_cache,slot_mapping,multi_block_tables,seqlens_q,multi_context_lens,"
                            "q_multi,max_seqlen_q,max_seqlen_k,paged_block_tables,paged_context_lens,paged_block_size,"
                            "paged_max_context_len,softmax_scale,y"),
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_native", "Bindings of libhipattn.so's hot entry points.", -1, g_methods,
                        nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) {
  PyObject *lib = PyImport_ImportModule("aici_amd._lib");
  if (lib == nullptr) return nullptr;
  g_error = PyObject_GetAttrString(lib, "HipAttnError");
  Py_DECREF(lib);
  PyObject *torch = PyImport_ImportModule("torch");
  if (g_error == nullptr || torch == nullptr) return nullptr;
  PyObject *type = PyObject_GetAttrString(torch, "Tensor");
  Py_DECREF(torch);
  if (type == nullptr) return nullptr;
  g_tensor_type = reinterpret_cast<PyTypeObject *>(type);
  PyObject *capsule = PyObject_GetAttrString(type, "__dlpack_c_exchange_api__");
  if (capsule == nullptr) return nullptr;
  g_exchange = static_cast<const DLPackExchangeAPI *>(PyCapsule_GetPointer(capsule, "dlpack_exchange_api"));
  Py_DECREF(capsule);
  if (g_exchange == nullptr) return nullptr;
  if (g_exchange->header.version.major != DLPACK_MAJOR_VERSION || g_exchange->dltensor_from_py_object_no_sync == nullptr ||
      g_exchange->current_work_stream == nullptr) {
    PyErr_SetString(PyExc_ImportError, "this torch's DLPack exchange table is not the one the extension was built for");
    return nullptr;
  }
  return PyModule_Create(&g_module);
}

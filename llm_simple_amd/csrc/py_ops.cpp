// Python face of the operator entry points: the hip_*_layer functions of llm_simple_amd.ops.
//
// A decode step of a small model takes the GPU 4-7 us, and a ctypes call with its wrapper took 1.0-1.8 us of the
// host's 4-5 beside the launch; parsed here it takes 0.3-0.5 us, most of it the data_ptr() of each tensor.
// Arguments are positional or by name; a device buffer is None, an address or anything with data_ptr(); the stream is
// None, an address (0 by default) or what ctypes takes for a void pointer, as the c_void_p that llmhip_stream_create
// fills or a torch.cuda.Stream.  A status other than 0 raises LlmHipError(status, name).
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <string.h>

#include "../../include/llmhip.h"

namespace {

PyObject *g_error = nullptr;     // ops.LlmHipError
PyObject *g_data_ptr = nullptr;  // "data_ptr"
PyObject *g_cast = nullptr;      // ctypes.cast
PyObject *g_void_p = nullptr;    // ctypes.c_void_p

enum Kind : char { P = 'p', S = 's', I = 'i', L = 'l', B = 'b' };  // buffer, stream, int, 64-bit int, truth value

struct Arg {
  const char *name;
  Kind kind;
};
union Value {
  void *p;
  long long i;
};
constexpr int kMaxArgs = 16;

bool to_value(PyObject *o, Kind kind, Value *out) {
  if (kind == B) {
    const int t = PyObject_IsTrue(o);
    out->i = t;
    return t >= 0;
  }
  if (kind == P || kind == S) {
    out->p = nullptr;
    if (o == Py_None) return true;
    PyObject *a = o;
    if (PyLong_Check(o)) {
      Py_INCREF(a);
    } else if (kind == P) {
      a = PyObject_CallMethodNoArgs(o, g_data_ptr);
    } else {
      PyObject *handle = PyObject_CallFunctionObjArgs(g_cast, o, g_void_p, nullptr);
      a = handle ? PyObject_GetAttrString(handle, "value") : nullptr;  // None for a null pointer
      Py_XDECREF(handle);
    }
    if (a && a != Py_None) out->p = PyLong_AsVoidPtr(a);
    Py_XDECREF(a);
    return !PyErr_Occurred();
  }
  out->i = PyLong_AsLongLong(o);
  return out->i != -1 || !PyErr_Occurred();
}

// `optional`: how many of the last arguments may be left out (they are 0 then).
bool parse(const char *fn, const Arg *spec, int count, int optional, PyObject *const *args, Py_ssize_t nargs,
           PyObject *kwnames, Value *out) {
  if (nargs > count) {
    PyErr_Format(PyExc_TypeError, "%s() takes at most %d arguments (%zd given)", fn, count, nargs);
    return false;
  }
  for (Py_ssize_t i = 0; i < nargs; ++i)
    if (!to_value(args[i], spec[i].kind, out + i)) return false;
  unsigned have = (1u << nargs) - 1;
  const Py_ssize_t nkw = kwnames ? PyTuple_GET_SIZE(kwnames) : 0;
  for (Py_ssize_t j = 0; j < nkw; ++j) {
    PyObject *name = PyTuple_GET_ITEM(kwnames, j);
    int at = 0;
    while (at < count && PyUnicode_CompareWithASCIIString(name, spec[at].name) != 0) ++at;
    if (at == count || (have >> at & 1)) {
      PyErr_Format(PyExc_TypeError, "%s() got %s argument '%U'", fn, at == count ? "an unexpected" : "twice the", name);
      return false;
    }
    if (!to_value(args[nargs + j], spec[at].kind, out + at)) return false;
    have |= 1u << at;
  }
  for (int i = 0; i < count; ++i)
    if (!(have >> i & 1)) {
      if (i < count - optional) {
        PyErr_Format(PyExc_TypeError, "%s() missing argument '%s'", fn, spec[i].name);
        return false;
      }
      out[i].p = nullptr;
    }
  return true;
}

PyObject *result(int status, const char *fn) {
  if (status == 0) Py_RETURN_NONE;
  PyObject *e = g_error ? PyObject_CallFunction(g_error, "is", status, fn) : nullptr;
  if (e) {
    PyErr_SetObject(g_error, e);
    Py_DECREF(e);
  } else if (!PyErr_Occurred()) {
    PyErr_Format(PyExc_RuntimeError, "%s: status %d", fn, status);
  }
  return nullptr;
}

inline int as_int(const Value &v) { return (int)v.i; }

#define OPERATOR(FN, CALL, ...)                                                                              \
  PyObject *py_##FN(PyObject *, PyObject *const *args, Py_ssize_t nargs, PyObject *kwnames) {                \
    static const Arg spec[] = {__VA_ARGS__};                                                                 \
    constexpr int count = sizeof(spec) / sizeof(spec[0]);                                                    \
    static_assert(count <= kMaxArgs, "");                                                                    \
    Value v[kMaxArgs];                                                                                       \
    if (!parse(#FN, spec, count, 1, args, nargs, kwnames, v)) return nullptr;                                \
    int status;                                                                                              \
    Py_BEGIN_ALLOW_THREADS /* a full queue may block the launch */                                           \
    status = CALL;                                                                                           \
    Py_END_ALLOW_THREADS                                                                                     \
    return result(status, #FN);                                                                              \
  }

OPERATOR(hip_flash_attn_layer,
         llmhip_flash_attn(v[0].p, v[1].p, v[2].p, v[3].p, as_int(v[4]), as_int(v[5]), as_int(v[6]), as_int(v[7]),
                           as_int(v[8]), as_int(v[9]), v[10].p),
         {"output_dev", P}, {"q_dev", P}, {"k_dev", P}, {"v_dev", P}, {"m", I}, {"n", I}, {"offset", I},
         {"head_num", I}, {"head_dim", I}, {"dt", I}, {"stream", S})

OPERATOR(hip_flash_attn_gqa_layer,
         llmhip_flash_attn_gqa(v[0].p, v[1].p, v[2].p, v[3].p, as_int(v[4]), as_int(v[5]), as_int(v[6]), as_int(v[7]),
                               as_int(v[8]), as_int(v[9]), as_int(v[10]), v[11].p),
         {"output_dev", P}, {"q_dev", P}, {"k_dev", P}, {"v_dev", P}, {"m", I}, {"n", I}, {"offset", I},
         {"group_size", I}, {"kv_head_num", I}, {"head_dim", I}, {"dt", I}, {"stream", S})

OPERATOR(hip_flash_attn_opt_prefill_layer,
         llmhip_flash_attn_opt_prefill(v[0].p, v[1].p, v[2].p, v[3].p, as_int(v[4]), as_int(v[5]), as_int(v[6]),
                                       as_int(v[7]), as_int(v[8]), as_int(v[9]), v[10].p),
         {"output_dev", P}, {"q_dev", P}, {"k_dev", P}, {"v_dev", P}, {"m", I}, {"n", I}, {"offset", I},
         {"head_num", I}, {"head_dim", I}, {"dt", I}, {"stream", S})

OPERATOR(hip_flash_decode_gqa_layer,
         llmhip_flash_decode_gqa(v[0].p, v[1].p, v[2].p, v[3].p, v[4].p, (size_t)v[5].i, as_int(v[6]), as_int(v[7]),
                                 v[8].i, as_int(v[9]), as_int(v[10]), as_int(v[11]), as_int(v[12]), as_int(v[13]),
                                 v[14].p),
         {"output_dev", P}, {"q_dev", P}, {"k_cache_dev", P}, {"v_cache_dev", P}, {"workspace_dev", P},
         {"workspace_bytes", L}, {"batch", I}, {"n", I}, {"kv_seq_stride", L}, {"group_size", I}, {"kv_head_num", I},
         {"head_dim", I}, {"num_splits", I}, {"dt", I}, {"stream", S})

OPERATOR(hip_flash_decode_gqa_static_layer,
         llmhip_flash_decode_gqa_static(v[0].p, v[1].p, v[2].p, v[3].p, as_int(v[4]), as_int(v[5]), v[6].i,
                                        as_int(v[7]), as_int(v[8]), as_int(v[9]), as_int(v[10]), as_int(v[11]),
                                        v[12].p),
         {"output_dev", P}, {"q_dev", P}, {"k_cache_dev", P}, {"v_cache_dev", P}, {"batch", I}, {"n", I},
         {"kv_seq_stride", L}, {"group_size", I}, {"kv_head_num", I}, {"head_dim", I}, {"num_splits", I}, {"dt", I},
         {"stream", S})

OPERATOR(hip_decode_step_gqa_layer,
         llmhip_decode_step_gqa(v[0].p, v[1].p, v[2].p, v[3].p, v[4].p, v[5].p, v[6].p, as_int(v[7]), as_int(v[8]),
                                as_int(v[9]), as_int(v[10]), as_int(v[11]), as_int(v[12]), v[13].p),
         {"output_dev", P}, {"k_cache_dev", P}, {"v_cache_dev", P}, {"freqs_cis_dev", P}, {"input_q_dev", P},
         {"input_k_dev", P}, {"input_v_dev", P}, {"pos", I}, {"group_size", I}, {"kv_head_num", I}, {"head_dim", I},
         {"is_neox_style", B}, {"dt", I}, {"stream", S})

OPERATOR(hip_matmul_layer,
         llmhip_matmul(v[0].p, v[1].p, v[2].p, as_int(v[3]), as_int(v[4]), as_int(v[5]), as_int(v[6]), v[7].p),
         {"output_dev", P}, {"lhs_dev", P}, {"weight_dev", P}, {"m", I}, {"n", I}, {"k", I}, {"dt", I}, {"stream", S})

OPERATOR(hip_matmul_bias_layer,
         llmhip_matmul_bias(v[0].p, v[1].p, v[2].p, v[3].p, as_int(v[4]), as_int(v[5]), as_int(v[6]), as_int(v[7]),
                            v[8].p),
         {"output_dev", P}, {"lhs_dev", P}, {"weight_dev", P}, {"bias_dev", P}, {"m", I}, {"n", I}, {"k", I},
         {"dt", I}, {"stream", S})

OPERATOR(hip_add_layer, llmhip_add(v[0].p, v[1].p, v[2].p, v[3].i, as_int(v[4]), v[5].p),
         {"output_dev", P}, {"lhs_dev", P}, {"rhs_dev", P}, {"total_size", L}, {"dt", I}, {"stream", S})

OPERATOR(hip_rope_layer,
         llmhip_rope(v[0].p, v[1].p, v[2].p, v[3].p, v[4].p, as_int(v[5]), as_int(v[6]), as_int(v[7]), as_int(v[8]),
                     as_int(v[9]), as_int(v[10]), v[11].p),
         {"output_q_dev", P}, {"output_k_dev", P}, {"freqs_cis_dev", P}, {"input_q_dev", P}, {"input_k_dev", P},
         {"start_pos", I}, {"cur_size", I}, {"n_heads", I}, {"hidden_dim", I}, {"is_neox_style", B}, {"dt", I},
         {"stream", S})

OPERATOR(hip_rope_single_layer,
         llmhip_rope_single(v[0].p, v[1].p, v[2].p, as_int(v[3]), as_int(v[4]), as_int(v[5]), as_int(v[6]),
                            as_int(v[7]), as_int(v[8]), v[9].p),
         {"output_x_dev", P}, {"freqs_cis_dev", P}, {"input_x_dev", P}, {"start_pos", I}, {"cur_size", I},
         {"n_heads", I}, {"hidden_dim", I}, {"is_neox_style", B}, {"dt", I}, {"stream", S})

OPERATOR(hip_rope_kv_append_layer,
         llmhip_rope_kv_append(v[0].p, v[1].p, v[2].p, v[3].p, v[4].p, v[5].p, v[6].p, as_int(v[7]), as_int(v[8]),
                               as_int(v[9]), as_int(v[10]), as_int(v[11]), as_int(v[12]), as_int(v[13]), v[14].p),
         {"output_q_dev", P}, {"k_cache_dev", P}, {"v_cache_dev", P}, {"freqs_cis_dev", P}, {"input_q_dev", P},
         {"input_k_dev", P}, {"input_v_dev", P}, {"start_pos", I}, {"cur_size", I}, {"n_heads", I}, {"n_kv_heads", I},
         {"head_dim", I}, {"is_neox_style", B}, {"dt", I}, {"stream", S})

PyObject *set_error(PyObject *, PyObject *cls) {
  Py_INCREF(cls);
  Py_XDECREF(g_error);
  g_error = cls;
  Py_RETURN_NONE;
}

#define METHOD(FN, SIGNATURE, DOC)                                                                    \
  {#FN, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(py_##FN)), METH_FASTCALL | METH_KEYWORDS, \
   #FN SIGNATURE "\n--\n\n" DOC}

PyMethodDef methods[] = {
    METHOD(hip_flash_attn_layer,
           "(output_dev, q_dev, k_dev, v_dev, m, n, offset, head_num, head_dim, dt, stream=0)",
           "npu_flash_attn_layer (prebuild/npu_ops.h:6-8)."),
    METHOD(hip_flash_attn_gqa_layer,
           "(output_dev, q_dev, k_dev, v_dev, m, n, offset, group_size, kv_head_num, head_dim, dt, stream=0)",
           "npu_flash_attn_gqa_layer (prebuild/npu_ops.h:10-13)."),
    METHOD(hip_flash_attn_opt_prefill_layer,
           "(output_dev, q_dev, k_dev, v_dev, m, n, offset, head_num, head_dim, dt, stream=0)",
           "npu_flash_attn_opt_prefill_layer (prebuild/npu_ops.h:15-18)."),
    METHOD(hip_flash_decode_gqa_layer,
           "(output_dev, q_dev, k_cache_dev, v_cache_dev, workspace_dev, workspace_bytes, batch, n, kv_seq_stride, "
           "group_size, kv_head_num, head_dim, num_splits, dt, stream=0)",
           "Batched split-KV decode (no counterpart in the reference header: decode there\n"
           "is npu_flash_attn_gqa_layer with m = 1, src/llama2_layer_npu.cpp:866-869)."),
    METHOD(hip_flash_decode_gqa_static_layer,
           "(output_dev, q_dev, k_cache_dev, v_cache_dev, batch, n, kv_seq_stride, group_size, kv_head_num, head_dim, "
           "num_splits, dt, stream=0)",
           "hip_flash_decode_gqa_layer without a workspace: the partials live in a fixed 4 MiB array\n"
           "inside the library and the call allocates nothing."),
    METHOD(hip_decode_step_gqa_layer,
           "(output_dev, k_cache_dev, v_cache_dev, freqs_cis_dev, input_q_dev, input_k_dev, input_v_dev, pos, "
           "group_size, kv_head_num, head_dim, is_neox_style, dt, stream=0)",
           "One decode step in one pass over the cache: rope(q), rope(k) -> k_cache[pos], v -> v_cache[pos] and\n"
           "attention over rows [0, pos], fused into the decode kernel (src/llama2_layer_npu.cpp:790-869 does it\n"
           "with four calls)."),
    METHOD(hip_matmul_layer, "(output_dev, lhs_dev, weight_dev, m, n, k, dt, stream=0)",
           "npu_matmul_nz_layer (prebuild/npu_ops.h:87-88) with the weight as W[n][k] row-major."),
    METHOD(hip_matmul_bias_layer, "(output_dev, lhs_dev, weight_dev, bias_dev, m, n, k, dt, stream=0)",
           "npu_matmul_bias_nz_layer (prebuild/npu_ops.h:90-92): fp32 bias added before the rounding."),
    METHOD(hip_add_layer, "(output_dev, lhs_dev, rhs_dev, total_size, dt, stream=0)",
           "npu_add_layer (prebuild/npu_ops.h:81-82)."),
    METHOD(hip_rope_layer,
           "(output_q_dev, output_k_dev, freqs_cis_dev, input_q_dev, input_k_dev, start_pos, cur_size, n_heads, "
           "hidden_dim, is_neox_style, dt, stream=0)",
           "npu_rope_layer (prebuild/npu_ops.h:39-42)."),
    METHOD(hip_rope_single_layer,
           "(output_x_dev, freqs_cis_dev, input_x_dev, start_pos, cur_size, n_heads, hidden_dim, is_neox_style, dt, "
           "stream=0)",
           "npu_rope_single_layer (prebuild/npu_ops.h:44-47)."),
    METHOD(hip_rope_kv_append_layer,
           "(output_q_dev, k_cache_dev, v_cache_dev, freqs_cis_dev, input_q_dev, input_k_dev, input_v_dev, start_pos, "
           "cur_size, n_heads, n_kv_heads, head_dim, is_neox_style, dt, stream=0)",
           "rope(Q), rope(K) -> k_cache[start_pos:], V -> v_cache[start_pos:] in one launch\n"
           "(src/llama2_layer_npu.cpp:790-798 + :830-844)."),
    {"set_error", set_error, METH_O, "The exception class of a failed call."},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_operators", "Operator calls of libllmhip.so.", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__operators(void) {
  PyObject *ctypes = PyImport_ImportModule("ctypes");
  if (ctypes) {
    g_cast = PyObject_GetAttrString(ctypes, "cast");
    g_void_p = PyObject_GetAttrString(ctypes, "c_void_p");
    Py_DECREF(ctypes);
  }
  g_data_ptr = PyUnicode_InternFromString("data_ptr");
  if (!g_cast || !g_void_p || !g_data_ptr) return nullptr;
  return PyModule_Create(&module);
}

// The kernel library's entry points and the checks of their operands as Python functions, in native code: a step of few tokens
// puts a hundred kernels on the stream, and what the interpreter does for each was longer than most of them run. A call with twenty
// arguments takes 0.5 us here where ctypes takes 2; a check of a tensor 0.1 where the same lines of Python take 0.5.
//
// open(path) takes the entry points out of the library; call(name) gives an entry as a function. Its arguments are converted by the
// types of its declaration in pyre_api.h: pointers from None, an integer or a tensor on a GPU, numbers from numbers. A result that is not
// zero raises KernelError with the library's message. The interpreter's lock is free while an entry runs.
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <dlfcn.h>

#include <exception>
#include <string>
#include <type_traits>
#include <unordered_map>

#include "pyre_api.h"

namespace {

PyObject* kernel_error = nullptr;  // the exception class, handed over when the module is set up
const char* (*last_error)() = nullptr;

// Every entry point that work is put on the stream with.
#define PYRE_ENTRIES(X)                                                                                                          \
  X(read_probe) X(embed) X(add_rmsnorm) X(rope_kv_write) X(silu_mul) X(reduce_partials) X(fill_rows) X(gemm_generic)             \
  X(gemm_f32) X(attn_generic) X(attn_prefill_f32) X(attn_decode_work_bf16) X(attn_decode_work_rope_bf16) X(attn_prefill_bf16)    \
  X(attn_prefill_work_bf16) X(argmax) X(argmax_static) X(argmax_static_init) X(gemm_skinny_bf16) X(gemm_skinny_silu_bf16)        \
  X(gemm_mid_bf16) X(gemm_mid_silu_bf16) X(sample) X(feed_tokens) X(gemm_skinny_glu_bf16) X(gemm_f32_whole) X(gemm_tile_choice)  \
  X(gemm_tile_bf16) X(gemm_tile_glu_bf16) X(gemm_mid_glu_bf16) X(add_layernorm) X(clipped_glu) X(scale) X(stream_norm)           \
  X(poly_norm) X(unit_qkv_write) X(attn_biased_tile) X(attn_biased_single) X(gla_prepare) X(gla_scan) X(gla_chunks)              \
  X(gla_finish) X(add_tanhnorm) X(softcap) X(rope_tied_write) X(latent_rows) X(head_matmul) X(latent_attn_tile)                  \
  X(latent_attn_single) X(gemm_tile_paged_bf16) X(latent_heads) X(route_topk) X(expert_act) X(add_rms_terms) X(bigram_embed)     \
  X(conv_qkv_write) X(retention_prepare) X(gla_finish_wide) X(ssm_conv) X(ssm_low) X(ssm_scan) X(ssm_step) X(route_grouped)      \
  X(expert_glu_act) X(add_weighted_rows) X(wide_norm_qkv_write) X(gdr_prepare) X(gdr_scan) X(gdr_finish) X(token_side_gate)

bool raise(const std::string& what) {
  PyErr_SetString(kernel_error ? kernel_error : PyExc_RuntimeError, what.c_str());
  return false;
}

const at::Tensor* tensor(PyObject* o) {
  if (THPVariable_Check(o)) return &THPVariable_Unpack(o);
  PyErr_Format(PyExc_TypeError, "a tensor is expected, not %s", Py_TYPE(o)->tp_name);
  return nullptr;
}

bool on_gpu(const at::Tensor& t) { return t.is_cuda() || raise("kernel operand is not on a GPU (there is no CPU path)"); }

// ---- an argument as the entry's declaration has it

template <typename T>
bool convert(PyObject* o, T& out) {
  if constexpr (std::is_pointer_v<T>) {
    if (o == Py_None) {
      out = nullptr;
    } else if (THPVariable_Check(o)) {
      const at::Tensor& t = THPVariable_Unpack(o);
      if (!on_gpu(t)) return false;
      out = static_cast<T>(t.data_ptr());
    } else {
      out = static_cast<T>(PyLong_AsVoidPtr(o));
    }
  } else if constexpr (std::is_floating_point_v<T>) {
    out = static_cast<T>(PyFloat_AsDouble(o));
  } else if constexpr (std::is_unsigned_v<T>) {
    out = static_cast<T>(PyLong_AsUnsignedLongLongMask(o));
  } else {
    const long v = PyLong_AsLong(o);
    out = static_cast<T>(v);
    if (out != v && !PyErr_Occurred()) PyErr_Format(PyExc_OverflowError, "%ld does not fit the entry's argument", v);
  }
  return !PyErr_Occurred();
}

// The interpreter's lock, given up for the lifetime: an exception out of an entry takes it back too.
struct Unlocked {
  PyThreadState* const state = PyEval_SaveThread();
  Unlocked() = default;
  Unlocked(const Unlocked&) = delete;
  ~Unlocked() { PyEval_RestoreThread(state); }
};

template <typename F>
struct Entry;
template <typename... A>
struct Entry<int (*)(A...)> {
  template <size_t... I>
  static PyObject* run(int (*fn)(A...), PyObject* const* args, std::index_sequence<I...>) {
    std::tuple<A...> v;
    if (!(convert(args[I], std::get<I>(v)) && ...)) return nullptr;
    int rc;
    {
      Unlocked unlocked;
      rc = fn(std::get<I>(v)...);
    }
    if (rc == 0) Py_RETURN_NONE;
    raise(last_error());
    return nullptr;
  }
  static PyObject* call(int (*fn)(A...), const char* name, PyObject* const* args, Py_ssize_t n) {
    if (!fn) return raise(std::string(name) + ": the library is not open"), nullptr;
    if (n != static_cast<Py_ssize_t>(sizeof...(A)))
      return PyErr_Format(PyExc_TypeError, "%s takes %zu arguments, %zd given", name, sizeof...(A), n);
    try {
      return run(fn, args, std::index_sequence_for<A...>{});
    } catch (const std::exception& e) {  // of torch, about a tensor without memory, or of the entry
      return PyErr_SetString(PyExc_RuntimeError, e.what()), nullptr;
    }
  }
};

#define PYRE_DEFINE(name)                                                                    \
  decltype(&pyre_##name) fn_##name = nullptr;                                                \
  PyObject* call_##name(PyObject*, PyObject* const* args, Py_ssize_t n) {                    \
    return Entry<decltype(&pyre_##name)>::call(fn_##name, "pyre_" #name, args, n);           \
  }
PYRE_ENTRIES(PYRE_DEFINE)

// ---- checks

#define PYRE_GUARDED(...)                                   \
  try {                                                     \
    __VA_ARGS__                                             \
  } catch (const std::exception& e) {                       \
    return PyErr_SetString(PyExc_RuntimeError, e.what()), nullptr; \
  }

bool takes(const char* name, Py_ssize_t n, Py_ssize_t least, Py_ssize_t most) {
  if (n >= least && n <= most) return true;
  PyErr_Format(PyExc_TypeError, "%s takes %zd to %zd arguments, %zd given", name, least, most, n);
  return false;
}

std::string text(PyObject* o) {
  const char* s = PyUnicode_Check(o) ? PyUnicode_AsUTF8(o) : nullptr;
  PyErr_Clear();
  return s ? s : "operand";
}

// dev(*tensors): every one that is not None lies on a GPU.
PyObject* dev(PyObject*, PyObject* const* args, Py_ssize_t n) {
  for (Py_ssize_t i = 0; i < n; ++i) {
    if (args[i] == Py_None) continue;
    const at::Tensor* t = tensor(args[i]);
    if (!t || !on_gpu(*t)) return nullptr;
  }
  Py_RETURN_NONE;
}

// contig(name, tensor)
PyObject* contig(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (!takes("contig", n, 2, 2)) return nullptr;
  const at::Tensor* t = tensor(args[1]);
  if (!t) return nullptr;
  PYRE_GUARDED(if (!t->is_contiguous()) return raise(text(args[0]) + " must be contiguous"), nullptr;)
  Py_RETURN_NONE;
}

const char* type_name(at::ScalarType s) { return c10::toString(s); }

// i32(name, tensor[, entries]): int32, contiguous, of that many entries at least
PyObject* i32(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (!takes("i32", n, 2, 3)) return nullptr;
  const at::Tensor* t = tensor(args[1]);
  if (!t) return nullptr;
  if (t->scalar_type() != at::kInt) return raise(text(args[0]) + " must be int32, got " + type_name(t->scalar_type())), nullptr;
  PYRE_GUARDED(if (!t->is_contiguous()) return raise(text(args[0]) + " must be contiguous"), nullptr;)
  if (n == 3 && args[2] != Py_None) {
    const long want = PyLong_AsLong(args[2]);
    if (PyErr_Occurred()) return nullptr;
    if (t->numel() < want)
      return raise(text(args[0]) + " holds " + std::to_string(t->numel()) + " entries, " + std::to_string(want) + " needed"), nullptr;
  }
  Py_RETURN_NONE;
}

long code_of(at::ScalarType s) { return s == at::kFloat ? 0 : s == at::kBFloat16 ? 1 : -1; }

bool code(PyObject* o, long& out) {
  at::ScalarType s;
  if (THPDtype_Check(o)) {
    s = reinterpret_cast<THPDtype*>(o)->scalar_type;
  } else {
    const at::Tensor* t = tensor(o);
    if (!t) return false;
    s = t->scalar_type();
  }
  out = code_of(s);
  return out >= 0 || raise(std::string("unsupported element type ") + type_name(s) + "; kernels take float32 and bfloat16");
}

// dtype_code(tensor or dtype)
PyObject* dtype_code(PyObject*, PyObject* o) {
  long c;
  return code(o, c) ? PyLong_FromLong(c) : nullptr;
}

// ptr(tensor or None)
PyObject* ptr(PyObject*, PyObject* o) {
  if (o == Py_None) Py_RETURN_NONE;
  const at::Tensor* t = tensor(o);
  if (!t) return nullptr;
  PYRE_GUARDED(return PyLong_FromVoidPtr(t->data_ptr());)
}

// product(x, w, m): the operands of a 16-bit product of x's first m rows, as the entries take them, and its columns and k:
// (x, ldx, w, ldw), (N, K).
PyObject* product(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (!takes("product", n, 3, 3)) return nullptr;
  const at::Tensor *x = tensor(args[0]), *w = x ? tensor(args[1]) : nullptr;
  const long m = w ? PyLong_AsLong(args[2]) : 0;
  if (!w || PyErr_Occurred() || !on_gpu(*x) || !on_gpu(*w)) return nullptr;
  PYRE_GUARDED(
    if (x->scalar_type() != at::kBFloat16 || w->scalar_type() != at::kBFloat16) return raise("gemm_skinny: bfloat16 operands expected"), nullptr;
    if (x->dim() != 2 || w->dim() != 2 || x->size(1) != w->size(1) || x->size(0) < m)
      return raise("gemm_skinny: x " + c10::str(x->sizes()) + " and w " + c10::str(w->sizes()) + " do not fit " + std::to_string(m) + " rows"), nullptr;
    if (x->stride(1) != 1 || w->stride(1) != 1) return raise("gemm_skinny: rows must be contiguous"), nullptr;
    return Py_BuildValue("(NlNl)(ll)", PyLong_FromVoidPtr(x->data_ptr()), static_cast<long>(x->stride(0)), PyLong_FromVoidPtr(w->data_ptr()),
                         static_cast<long>(w->stride(0)), static_cast<long>(w->size(0)), static_cast<long>(w->size(1)));)
}

// sums(out, elements): whether out is contiguous float32 on a GPU of that many elements at least
PyObject* sums(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (!takes("sums", n, 2, 2)) return nullptr;
  const at::Tensor* t = tensor(args[0]);
  const long want = t ? PyLong_AsLong(args[1]) : 0;
  if (!t || PyErr_Occurred()) return nullptr;
  PYRE_GUARDED(return PyBool_FromLong(t->scalar_type() == at::kFloat && t->is_cuda() && t->is_contiguous() && t->numel() >= want);)
}

// partials(data, bias or None, width): (data, its type, parts, elements of a part, bias, its type)
PyObject* partials(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (!takes("partials", n, 3, 3)) return nullptr;
  const at::Tensor* d = tensor(args[0]);
  const at::Tensor* b = d && args[1] != Py_None ? tensor(args[1]) : nullptr;
  const long width = d ? PyLong_AsLong(args[2]) : 0;
  long dt, bt = 0;
  if (!d || (args[1] != Py_None && !b) || PyErr_Occurred() || !code(args[0], dt)) return nullptr;
  PYRE_GUARDED(
    if (d->size(2) != width) return raise("partials are " + std::to_string(d->size(2)) + " wide, " + std::to_string(width) + " expected"), nullptr;
    if (b && b->numel() != width) return raise("bias has " + std::to_string(b->numel()) + " entries, " + std::to_string(width) + " expected"), nullptr;
    if (b && !code(args[1], bt)) return nullptr;
    PyObject* bias = Py_None;
    if (b) bias = PyLong_FromVoidPtr(b->data_ptr());
    else Py_INCREF(bias);
    return Py_BuildValue("NlllNl", PyLong_FromVoidPtr(d->data_ptr()), dt, static_cast<long>(d->size(0)), static_cast<long>(d->stride(0)), bias, bt);)
}

// ---- the module

PyObject* setup(PyObject*, PyObject* error) {
  Py_INCREF(error);
  kernel_error = error;
  Py_RETURN_NONE;
}

PyObject* open_library(PyObject*, PyObject* path) {
  const char* p = PyUnicode_AsUTF8(path);
  if (!p) return nullptr;
  void* const h = dlopen(p, RTLD_NOW | RTLD_LOCAL);
  if (!h) return raise(std::string("cannot open the kernel library: ") + dlerror()), nullptr;
  last_error = reinterpret_cast<decltype(last_error)>(dlsym(h, "pyre_last_error"));
  bool whole = last_error != nullptr;
#define PYRE_FIND(name) whole &= (fn_##name = reinterpret_cast<decltype(fn_##name)>(dlsym(h, "pyre_" #name))) != nullptr;
  PYRE_ENTRIES(PYRE_FIND)
  if (!whole) return raise("the kernel library lacks an entry point: it was built from other sources"), nullptr;
  Py_RETURN_NONE;
}

#define PYRE_METHOD(name) {"pyre_" #name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(call_##name)), METH_FASTCALL, nullptr},
#define PYRE_FAST(name, fn) {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(fn)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {PYRE_ENTRIES(PYRE_METHOD){"setup", setup, METH_O, nullptr},
                         {"open", open_library, METH_O, nullptr},
                         {"dtype_code", dtype_code, METH_O, nullptr},
                         {"ptr", ptr, METH_O, nullptr},
                         PYRE_FAST("dev", dev),
                         PYRE_FAST("contig", contig),
                         PYRE_FAST("i32", i32),
                         PYRE_FAST("product", product),
                         PYRE_FAST("sums", sums),
                         PYRE_FAST("partials", partials),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "pyre_binding", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_pyre_binding() { return PyModule_Create(&module); }

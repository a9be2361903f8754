// Host side of the one-launch operators, in C++ over the entry points of include/lego_hip.h.
//
// A transpose, softmax, stencil or product over a small matrix takes the GPU 2 to 5 us, and its launch the host some 3; the checks,
// the allocation of the result and the call in Python took another 3 to 6.  These take the same checks, ask for the same tensors and
// call the same entry points on the current stream.  us a call, in Python / here, where the GPU takes less: softmax 5.9 / 3.7, transpose
// 6.5 / 3.8, stencil 6.4 / 3.9, a product 7.4 / 3.9, against a .T view 9.3 / 4.6, eight grouped ones 25.7 / 9.5.
// They take what needs nothing else: plain GPU tensors in the layouts that the kernels take, with no dispatch or function mode,
// tracer or transform in between.  Everything else, errors included, returns None, and the caller goes on in Python.
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>
#include <torch/extension.h>

#include <vector>

#include "lego_hip.h"

namespace {

void* current_stream() { return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream(); }

// what of a key set is beyond another one (a difference keeps backend bits, which say nothing by themselves)
bool beyond(c10::DispatchKeySet keys, c10::DispatchKeySet known) { return (keys - known).highestFunctionalityKey() != c10::DispatchKey::Undefined; }

bool nothing_in_between()
{
  return !beyond(c10::impl::tls_local_dispatch_key_set().included_, c10::default_included_set) && at::impl::PythonTorchFunctionTLS::stack_len() == 0;
}

// A plain GPU tensor of `dims` dimensions that has elements, or null.
const at::Tensor* plain(PyObject* object, int64_t dims)
{
  if (!THPVariable_CheckExact(object)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(object);
  constexpr c10::DispatchKeySet known({c10::DispatchKey::CUDA, c10::DispatchKey::AutogradCUDA, c10::DispatchKey::ADInplaceOrView, c10::DispatchKey::AutocastCUDA});
  if (!t.defined() || !t.is_cuda() || beyond(t.key_set(), known) || t.dim() != dims || t.numel() == 0 || t._fw_grad(0).defined()) return nullptr;
  for (const int64_t size : t.sizes())
    if (size > INT_MAX) return nullptr;
  return &t;
}

PyObject* nothing() { Py_RETURN_NONE; }

// `run`, without the interpreter's lock, gives the result, or an undefined tensor: nothing was enqueued, and the call is Python's.
template <class Run>
PyObject* result(const Run& run)
{
  HANDLE_TH_ERRORS
  at::Tensor out;
  {
    pybind11::gil_scoped_release nothing_here_needs_it;
    out = run();
  }
  return out.defined() ? THPVariable_Wrap(std::move(out)) : nothing();
  END_HANDLE_TH_ERRORS
}

at::TensorOptions options_of(const at::Tensor& t) { return at::TensorOptions(t.device()).dtype(t.scalar_type()); }

// transpose(x)
PyObject* transpose(PyObject*, PyObject* const* args, Py_ssize_t count)
{
  const at::Tensor* const x = count == 1 && nothing_in_between() ? plain(args[0], 2) : nullptr;
  if (!x || !x->is_contiguous() || (x->element_size() != 2 && x->element_size() != 4)) return nothing();
  return result([&] {
    const int64_t rows = x->size(0), cols = x->size(1);
    at::Tensor out = at::empty({cols, rows}, options_of(*x));
    const auto entry = x->element_size() == 4 ? lego_hip_transpose_f32 : lego_hip_transpose_f16;
    return entry(x->const_data_ptr(), out.mutable_data_ptr(), (int)rows, (int)cols, current_stream()) == 0 ? out : at::Tensor();
  });
}

// softmax(x)
PyObject* softmax(PyObject*, PyObject* const* args, Py_ssize_t count)
{
  const at::Tensor* const x = count == 1 && nothing_in_between() ? plain(args[0], 2) : nullptr;
  if (!x || !x->is_contiguous()) return nothing();
  const at::ScalarType type = x->scalar_type();
  const auto entry = type == at::kHalf ? lego_hip_softmax_f16 : type == at::kBFloat16 ? lego_hip_softmax_bf16 : type == at::kFloat ? lego_hip_softmax_f32 : nullptr;
  if (!entry) return nothing();
  return result([&] {
    at::Tensor out = at::empty(x->sizes(), options_of(*x));
    return entry(x->const_data_ptr(), out.mutable_data_ptr(), (int)x->size(0), (int)x->size(1), current_stream()) == 0 ? out : at::Tensor();
  });
}

// stencil(x, c, radius, bricks, dense), with a result of its own; the caller has looked at c's shape
PyObject* stencil(PyObject*, PyObject* const* args, Py_ssize_t count)
{
  if (count != 5 || !nothing_in_between() || !PyLong_CheckExact(args[2]) || !PyBool_Check(args[3])) return nothing();
  const bool dense = args[4] == Py_True;
  const at::Tensor *const x = plain(args[0], 3), *const c = plain(args[1], dense ? 3 : 1);
  int overflow = 0;
  const long radius = PyLong_AsLongAndOverflow(args[2], &overflow);
  if (!x || !c || overflow || radius < 0 || radius > INT_MAX || !x->is_contiguous() || !c->is_contiguous() || x->scalar_type() != at::kFloat || c->scalar_type() != at::kFloat ||
      x->size(0) != x->size(1) || x->size(0) != x->size(2))
    return nothing();
  return result([&] {
    at::Tensor out = at::empty(x->sizes(), options_of(*x));
    const auto entry = dense ? lego_hip_stencil_f3d_f32_zeros : lego_hip_stencil_laplacian_f32_zeros;
    return entry(x->const_data_ptr<float>(), out.mutable_data_ptr<float>(), c->const_data_ptr<float>(), (int)x->size(0), (int)radius, args[3] == Py_True, current_stream()) == 0
               ? out : at::Tensor();
  });
}

// A row-major or column-major matrix, as `ops._operand` tells them apart.
bool stored(const at::Tensor& t, int& transposed)
{
  transposed = 0;
  if (t.is_contiguous()) return true;
  transposed = 1;
  return (t.stride(0) == 1 || t.size(0) == 1) && (t.stride(1) == t.size(0) || t.size(1) == 1);
}

// matmul(a, b, activation, out_dtype)
PyObject* matmul(PyObject*, PyObject* const* args, Py_ssize_t count)
{
  if (count != 4 || !nothing_in_between() || !PyUnicode_CheckExact(args[2]) || !THPDtype_Check(args[3])) return nothing();
  const at::Tensor *const a = plain(args[0], 2), *const b = plain(args[1], 2);
  int ta, tb;
  if (!a || !b || a->scalar_type() != b->scalar_type() || a->size(1) != b->size(0) || !stored(*a, ta) || !stored(*b, tb)) return nothing();
  const int activation = PyUnicode_GET_LENGTH(args[2]) == 0 ? 0 : PyUnicode_CompareWithASCIIString(args[2], "leaky_relu") == 0 ? 1 : -1;
  const at::ScalarType type = a->scalar_type(), out_type = reinterpret_cast<THPDtype*>(args[3])->scalar_type;
  const bool eight = type == at::kFloat8_e4m3fn || type == at::kFloat8_e5m2, half = type == at::kHalf, brain = type == at::kBFloat16;
  if (activation < 0 || !(eight || half || brain) || (!eight && out_type != at::kHalf && out_type != type)) return nothing();
  const int M = (int)a->size(0), N = (int)b->size(1), K = (int)a->size(1);
  unsigned long long need = 0;
  const bool ragged = eight && (N % 16 || (ta ? M : K) % 16 || (tb && K % 16));      // copies, where they gain
  if (eight) {
    if (lego_hip_gemm_layout_workspace_bytes(M, N, K, ta, tb, 1, &need) != 0) return nothing();
  } else if ((ta && M % 8) || lego_hip_gemm_layout_workspace_bytes(M, N, K, ta, tb, 2, &need) != 0) {
    return nothing();       // a column-major A of such columns may be stored row-major first
  }
  return result([&] {
    at::Tensor out = at::empty({M, N}, options_of(*a).dtype(eight ? at::kHalf : out_type)), workspace;
    if (need) workspace = at::empty({(int64_t)((need + 3) / 4)}, options_of(*a).dtype(at::kFloat));
    const void *const pa = a->const_data_ptr(), *const pb = b->const_data_ptr();
    void *const pc = out.mutable_data_ptr(), *const stream = current_stream();
    const bool mixed = brain && out_type == at::kHalf;
    const int code = eight && need ? (ragged ? lego_hip_gemm_fp8_padded : lego_hip_gemm_fp8_ex_ws)(pa, pb, pc, M, N, K, ta, tb, activation, type == at::kFloat8_e5m2,
                                                                                                   workspace.mutable_data_ptr(), need, stream)
                     : eight ? lego_hip_gemm_fp8_ex(pa, pb, pc, M, N, K, ta, tb, activation, type == at::kFloat8_e5m2, stream)
                     : need ? lego_hip_gemm_ex_ws(half ? 0 : mixed ? 4 : 1, pa, pb, pc, M, N, K, ta, tb, activation, workspace.mutable_data_ptr(), need, stream)
                            : (half ? lego_hip_gemm_f16_ex : mixed ? lego_hip_gemm_bf16_f16_ex : lego_hip_gemm_bf16_ex)(pa, pb, pc, M, N, K, ta, tb, activation, stream);
    return code == 0 ? out : at::Tensor();
  });
}

// group(as, bs): the grouped launch of two lists of row-major fp16 matrices
PyObject* group(PyObject*, PyObject* const* args, Py_ssize_t count)
{
  HANDLE_TH_ERRORS
  constexpr int kMost = 64;       // pointers kept on the stack; longer lists are Python's
  if (count != 2 || !nothing_in_between() || !PyList_CheckExact(args[0]) || !PyList_CheckExact(args[1])) return nothing();
  const Py_ssize_t groups = PyList_GET_SIZE(args[0]);
  if (groups == 0 || groups > kMost || PyList_GET_SIZE(args[1]) != groups) return nothing();
  std::vector<at::Tensor> as, bs, cs;       // held while the interpreter's lock is not
  std::vector<int> sizes;
  bool ragged = false, deep = false;
  for (Py_ssize_t g = 0; g < groups; ++g) {
    const at::Tensor *const a = plain(PyList_GET_ITEM(args[0], g), 2), *const b = plain(PyList_GET_ITEM(args[1], g), 2);
    if (!a || !b || a->scalar_type() != at::kHalf || b->scalar_type() != at::kHalf || !a->is_contiguous() || !b->is_contiguous() || a->size(1) != b->size(0))
      return nothing();
    const int N = (int)b->size(1), K = (int)a->size(1);
    ragged = ragged || N % 8 || K % 8;
    if (ragged && groups == 1) return nothing();       // a product of its own
    deep = deep || ((N % 8 || K % 8) && K > 1984);      // 31 k-tiles: lego_hip_grouped_gemm_f16_apart looks at none of fewer
    as.push_back(*a);
    bs.push_back(*b);
    sizes.insert(sizes.end(), {(int)a->size(0), N, K});
  }
  unsigned long long need = 0;
  int limit = 0;
  if (lego_hip_grouped_gemm_f16_room(sizes.data(), (int)groups, &need, &limit) != 0 || (deep && limit == 0)) return nothing();      // some may be products of their own
  {
    pybind11::gil_scoped_release nothing_here_needs_it;
    const void *pa[kMost], *pb[kMost];
    void* pc[kMost];
    for (Py_ssize_t g = 0; g < groups; ++g) {
      cs.push_back(at::empty({sizes[3 * g], sizes[3 * g + 1]}, options_of(as[g])));
      pa[g] = as[g].const_data_ptr();
      pb[g] = bs[g].const_data_ptr();
      pc[g] = cs[g].mutable_data_ptr();
    }
    at::Tensor workspace;
    if (need) workspace = at::empty({(int64_t)((need + 3) / 4)}, options_of(cs.back()).dtype(at::kFloat));
    const int code = need ? lego_hip_grouped_gemm_f16_ws(pa, pb, pc, sizes.data(), (int)groups, workspace.mutable_data_ptr(), need, current_stream())
                          : lego_hip_grouped_gemm_f16(pa, pb, pc, sizes.data(), (int)groups, current_stream());
    if (code != 0) cs.clear();
  }
  if (cs.empty()) return nothing();
  THPObjectPtr list(PyList_New(groups));
  if (!list) return nullptr;
  for (Py_ssize_t g = 0; g < groups; ++g) {
    PyObject* const c = THPVariable_Wrap(std::move(cs[g]));
    if (!c) return nullptr;
    PyList_SET_ITEM(list.get(), g, c);
  }
  return list.release();
  END_HANDLE_TH_ERRORS
}

template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyMethodDef method(const char* name) { return {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(F)), METH_FASTCALL, nullptr}; }

PyMethodDef methods[] = {method<transpose>("transpose"), method<softmax>("softmax"), method<stencil>("stencil"), method<matmul>("matmul"), method<group>("group"), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "host_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_host_calls() { return PyModule_Create(&module); }

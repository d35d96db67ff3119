// _fast: the fused entry points for callers that hold torch tensors, as a CPython module.
//
// A short call is bound by its host side: the b2b product [8192, 64] x [64, 256] x [256, 64] takes 4 us on the device and
// took 11 us through ctypes, of which the launch is 2 (argument objects, the stream looked up through torch.cuda, a
// dozen attribute look-ups per tensor).  Here a call is checked, its output allocated and its kernel launched in one
// native function.
//
// The functions take what is certainly right and return None for everything else, without having done anything: the
// caller (_core.py) then goes through its own checks, which name what is wrong.
#include <ATen/core/Tensor.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <climits>
#include <cmath>
#include <vector>

#include "../../include/ftk.h"

namespace {

PyObject* g_counts = nullptr;   // dict: calls by name
PyObject* g_raise = nullptr;    // callable: raises for a return code of the library

bool is_tensor(PyObject* o) { return THPVariable_Check(o); }
const at::Tensor& tensor_of(PyObject* o) { return THPVariable_Unpack(o); }

// a dense tensor on the GPU of one type
bool plain(PyObject* o, at::ScalarType type) {
  if (!is_tensor(o)) return false;
  const at::Tensor& t = tensor_of(o);
  return t.is_cuda() && t.scalar_type() == type && t.is_contiguous();
}

bool count(const char* name) {
  PyObject* key = PyUnicode_InternFromString(name);
  if (!key) return false;
  PyObject* old = PyDict_GetItem(g_counts, key);
  PyObject* now = PyLong_FromLong((old ? PyLong_AsLong(old) : 0) + 1);
  const bool ok = now && PyDict_SetItem(g_counts, key, now) == 0;
  Py_XDECREF(now);
  Py_DECREF(key);
  return ok;
}

PyObject* raise(int rc) {
  PyObject* r = PyObject_CallFunction(g_raise, "i", rc);
  Py_XDECREF(r);
  if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, "libftkernels: an error code that raised nothing");
  return nullptr;
}

at::Tensor empty(at::IntArrayRef shape, at::ScalarType type, const at::Tensor& like) {
  return at::detail::empty_cuda(shape, type, like.device(), std::nullopt);
}

void* stream() { return c10::hip::getCurrentHIPStream().stream(); }

int dim(const at::Tensor& t, int i) { return (int)t.size(i); }

template <typename F>
PyObject* guarded(F&& f) {
  try {
    return f();
  } catch (const std::exception& e) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

// Other Python threads run while one is in the library: a launch may wait for the lock that orders launches of several streams,
// or for the device.
struct WithoutGil {
  PyThreadState* state = PyEval_SaveThread();
  ~WithoutGil() { PyEval_RestoreThread(state); }
};
template <typename F>
int in_library(F&& f) {
  WithoutGil released;
  return f();
}

PyObject* init(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 2 || !PyDict_Check(args[0]) || !PyCallable_Check(args[1])) {
    PyErr_SetString(PyExc_TypeError, "init(counts, raise)");
    return nullptr;
  }
  Py_INCREF(args[0]);
  Py_INCREF(args[1]);
  Py_XDECREF(g_counts);
  Py_XDECREF(g_raise);
  g_counts = args[0];
  g_raise = args[1];
  Py_RETURN_NONE;
}

// b2b_gemm(A [G,M,K], B_nk [G,N,K], C_pn [G,P,N], out or None)
PyObject* b2b_gemm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    constexpr auto f16 = at::kHalf;
    if (n != 4 || !plain(a[0], f16) || !plain(a[1], f16) || !plain(a[2], f16)) Py_RETURN_NONE;
    const at::Tensor &A = tensor_of(a[0]), &B = tensor_of(a[1]), &C = tensor_of(a[2]);
    if (A.dim() != 3 || B.dim() != 3 || C.dim() != 3) Py_RETURN_NONE;
    const int G = dim(A, 0), M = dim(A, 1), K = dim(A, 2), N = dim(B, 1), P = dim(C, 1);
    if (dim(B, 0) != G || dim(B, 2) != K || dim(C, 0) != G || dim(C, 2) != N) Py_RETURN_NONE;
    at::Tensor D;
    if (a[3] == Py_None) {
      D = empty({G, M, P}, f16, A);
    } else {
      if (!plain(a[3], f16)) Py_RETURN_NONE;
      D = tensor_of(a[3]);
      if (D.dim() != 3 || dim(D, 0) != G || dim(D, 1) != M || dim(D, 2) != P) Py_RETURN_NONE;
    }
    if (!count("b2b_gemm")) return nullptr;
    void *const ap = A.data_ptr(), *const bp = B.data_ptr(), *const cp = C.data_ptr(), *const dp = D.data_ptr(), *const s = stream();
    const int rc = in_library([&] { return ftk_b2b_gemm_f16(ap, bp, cp, dp, G, M, N, K, P, s); });
    return rc ? raise(rc) : THPVariable_Wrap(std::move(D));
  });
}

// flash_attention(half, Q [B,Hd,Sq,D], K, V [B,Hd,Skv,D], scale or None, out or None, workspace or None, split_keys)
PyObject* flash_attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 8) Py_RETURN_NONE;
    const bool half = a[0] == Py_True;
    const auto type = half ? at::kHalf : at::kFloat;
    if (!plain(a[1], type) || !plain(a[2], type) || !plain(a[3], type)) Py_RETURN_NONE;
    const at::Tensor &Q = tensor_of(a[1]), &K = tensor_of(a[2]), &V = tensor_of(a[3]);
    if (Q.dim() != 4 || K.dim() != 4 || V.dim() != 4 || K.sizes() != V.sizes()) Py_RETURN_NONE;
    const int B = dim(Q, 0), Hd = dim(Q, 1), Sq = dim(Q, 2), D = dim(Q, 3), Skv = dim(K, 2);
    if (dim(K, 0) != B || dim(K, 1) != Hd || dim(K, 3) != D) Py_RETURN_NONE;
    double scale = 1.0 / std::sqrt((double)D);
    if (a[4] != Py_None) {
      if (!PyFloat_Check(a[4]) && !PyLong_Check(a[4])) Py_RETURN_NONE;
      scale = PyFloat_AsDouble(a[4]);
    }
    at::Tensor O, ws;
    if (a[5] == Py_None) {
      O = empty(Q.sizes(), type, Q);
    } else {
      if (!plain(a[5], type)) Py_RETURN_NONE;
      O = tensor_of(a[5]);
      if (O.sizes() != Q.sizes()) Py_RETURN_NONE;
    }
    if (a[7] != Py_True && a[7] != Py_False) Py_RETURN_NONE;
    const size_t need = !half              ? ftk_flash_attn_f32_workspace_bytes(B, Hd, Sq, Skv, D)
                        : a[7] == Py_True ? ftk_flash_attn_f16_workspace_bytes(B, Hd, Sq, Skv, D)
                                          : 0;
    if (a[6] != Py_None) {
      if (!is_tensor(a[6]) || !tensor_of(a[6]).is_cuda() || !tensor_of(a[6]).is_contiguous()) Py_RETURN_NONE;
      ws = tensor_of(a[6]);
    } else if (need) {
      ws = empty({(int64_t)need}, at::kByte, Q);
    }
    const size_t bytes = ws.defined() ? ws.nbytes() : 0;
    if (!count(half ? "flash_attention" : "flash_attention_f32")) return nullptr;
    if (half && need && !count("flash_attention_split_keys")) return nullptr;
    void *const qp = Q.data_ptr(), *const kp = K.data_ptr(), *const vp = V.data_ptr(), *const op = O.data_ptr();
    void *const wp = ws.defined() ? ws.data_ptr() : nullptr, *const s = stream();
    const int rc = in_library([&] {
      if (!half) return ftk_flash_attn_f32((const float*)qp, (const float*)kp, (const float*)vp, (float*)op, B, Hd, Sq, Skv, D, (float)scale, wp, bytes, s);
      if (need) return ftk_flash_attn_ws_f16(qp, kp, vp, op, B, Hd, Sq, Skv, D, (float)scale, wp, bytes, s);
      return ftk_flash_attn_f16(qp, kp, vp, op, B, Hd, Sq, Skv, D, (float)scale, s);
    });
    return rc ? raise(rc) : THPVariable_Wrap(std::move(O));
  });
}

// flash_attention_f32_flat(q, k, v, B, Hd, Sq, Skv, D, scale) -> o: fp32 attention on the one-dimensional buffers of [B,Hd,Sq,D] and
// [B,Hd,Skv,D].  (Three views of the operands and one of the result are 3 of the 17 us of host time of a short attention program.)
PyObject* flash_attention_f32_flat(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 9 || !plain(a[0], at::kFloat) || !plain(a[1], at::kFloat) || !plain(a[2], at::kFloat) || !PyFloat_Check(a[8])) Py_RETURN_NONE;
    int64_t size[5];
    for (int i = 0; i < 5; ++i) {
      if (!PyLong_Check(a[3 + i])) Py_RETURN_NONE;
      size[i] = PyLong_AsLongLong(a[3 + i]);
      if (size[i] <= 0 || size[i] > INT_MAX) {
        PyErr_Clear();
        Py_RETURN_NONE;
      }
    }
    const int B = (int)size[0], Hd = (int)size[1], Sq = (int)size[2], Skv = (int)size[3], D = (int)size[4];
    const at::Tensor &Q = tensor_of(a[0]), &K = tensor_of(a[1]), &V = tensor_of(a[2]);
    __int128 of_q = (__int128)B * Hd * Sq * D, of_k = (__int128)B * Hd * Skv * D;
    if (Q.dim() != 1 || K.dim() != 1 || V.dim() != 1 || Q.numel() != of_q || K.numel() != of_k || V.numel() != of_k) Py_RETURN_NONE;
    at::Tensor O = empty(Q.sizes(), at::kFloat, Q), ws;
    const size_t bytes = ftk_flash_attn_f32_workspace_bytes(B, Hd, Sq, Skv, D);
    if (bytes) ws = empty({(int64_t)bytes}, at::kByte, Q);
    if (!count("flash_attention_f32")) return nullptr;
    void *const qp = Q.data_ptr(), *const kp = K.data_ptr(), *const vp = V.data_ptr(), *const op = O.data_ptr();
    void *const wp = ws.defined() ? ws.data_ptr() : nullptr, *const s = stream();
    const float scale = (float)PyFloat_AsDouble(a[8]);
    const int rc = in_library([&] {
      return ftk_flash_attn_f32((const float*)qp, (const float*)kp, (const float*)vp, (float*)op, B, Hd, Sq, Skv, D, scale, wp, bytes, s);
    });
    return rc ? raise(rc) : THPVariable_Wrap(std::move(O));
  });
}

// stacked_lstm(half, xs [T,B,H], WU [L,2H,4H], bias [L,4H] or None, dilations or None, (h, c) or None, workspace or None,
//              products, check or None, small) -> (h, c, small states met)
// products: a code of ftk_lstm_options (-1: the process-wide mode).  check: wait for the stream and raise if the launch gave
// up a wait (None: if the workspace is allocated here).  small: wait and say whether small states were met.
PyObject* stacked_lstm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 10) Py_RETURN_NONE;
    const bool half = a[0] == Py_True;
    const auto type = half ? at::kHalf : at::kFloat;
    if (!plain(a[1], type) || !plain(a[2], type) || !(a[3] == Py_None || plain(a[3], at::kFloat))) Py_RETURN_NONE;
    const at::Tensor &xs = tensor_of(a[1]), &WU = tensor_of(a[2]);
    if (xs.dim() != 3 || WU.dim() != 3) Py_RETURN_NONE;
    const int T = dim(xs, 0), B = dim(xs, 1), H = dim(xs, 2), L = dim(WU, 0);
    if (dim(WU, 1) != 2 * H || dim(WU, 2) != 4 * H) Py_RETURN_NONE;
    const float* bias = nullptr;
    if (a[3] != Py_None) {
      const at::Tensor& b = tensor_of(a[3]);
      if (b.dim() != 2 || dim(b, 0) != L || dim(b, 1) != 4 * H) Py_RETURN_NONE;
      bias = b.data_ptr<float>();
    }
    std::vector<int> dil;
    if (a[4] != Py_None) {
      if (!PyList_Check(a[4]) && !PyTuple_Check(a[4])) Py_RETURN_NONE;
      if (PySequence_Fast_GET_SIZE(a[4]) != L) Py_RETURN_NONE;
      for (int l = 0; l < L; ++l) {
        PyObject* v = PySequence_Fast_GET_ITEM(a[4], l);
        if (!PyLong_Check(v)) Py_RETURN_NONE;
        const long d = PyLong_AsLong(v);
        if (d < 1 || d > (1 << 30)) Py_RETURN_NONE;
        dil.push_back((int)d);
      }
    }
    at::Tensor h, c, ws;
    if (a[5] == Py_None) {
      h = empty({L, T, B, H}, type, xs);
      c = empty({L, T, B, H}, type, xs);
    } else {
      if (!PyTuple_Check(a[5]) || PyTuple_GET_SIZE(a[5]) != 2) Py_RETURN_NONE;
      for (int i = 0; i < 2; ++i) {
        PyObject* o = PyTuple_GET_ITEM(a[5], i);
        if (!plain(o, type)) Py_RETURN_NONE;
        const at::Tensor& t = tensor_of(o);
        if (t.dim() != 4 || dim(t, 0) != L || dim(t, 1) != T || dim(t, 2) != B || dim(t, 3) != H) Py_RETURN_NONE;
        (i ? c : h) = t;
      }
    }
    if (!PyLong_Check(a[7]) || (a[8] != Py_None && a[8] != Py_True && a[8] != Py_False) || (a[9] != Py_True && a[9] != Py_False))
      Py_RETURN_NONE;
    bool check = a[8] == Py_True;
    if (a[6] == Py_None) {
      const size_t need = half ? ftk_stacked_lstm_f16_workspace_bytes(L, T, B, H) : ftk_stacked_lstm_workspace_bytes(L, T, B, H);
      ws = empty({(int64_t)need}, at::kByte, xs);
      if (a[8] == Py_None) check = true;
    } else {
      if (!is_tensor(a[6]) || !tensor_of(a[6]).is_cuda() || !tensor_of(a[6]).is_contiguous()) Py_RETURN_NONE;
      ws = tensor_of(a[6]);
    }
    if (!count(half ? "stacked_lstm_f16" : "stacked_lstm")) return nullptr;
    const int* dp = dil.empty() ? nullptr : dil.data();
    const ftk_lstm_options options = {(int)PyLong_AsLong(a[7]), 0};
    void *const xp = xs.data_ptr(), *const up = WU.data_ptr(), *const hp = h.data_ptr(), *const cp = c.data_ptr(), *const wp = ws.data_ptr();
    void* const s = stream();
    const size_t bytes = ws.nbytes();
    const bool small_asked = a[9] == Py_True;
    int small = 0;
    const int rc = in_library([&] {
      const int rc = half ? ftk_stacked_lstm_f16(xp, up, bias, dp, nullptr, hp, cp, L, T, B, H, wp, bytes, s)
                          : ftk_stacked_lstm_opts_f32((const float*)xp, (const float*)up, bias, dp, nullptr, (float*)hp, (float*)cp, L, T, B, H,
                                                      &options, wp, bytes, s);
      if (rc || !(check || small_asked)) return rc;
      const int waited = ftk_stacked_lstm_result(wp, &small, s);
      return waited == FTK_ERR_TIMEOUT && !check ? FTK_OK : waited;
    });
    if (rc) return raise(rc);
    PyObject* out = PyTuple_New(3);
    if (!out) return nullptr;
    PyTuple_SET_ITEM(out, 0, THPVariable_Wrap(std::move(h)));
    PyTuple_SET_ITEM(out, 1, THPVariable_Wrap(std::move(c)));
    PyTuple_SET_ITEM(out, 2, PyBool_FromLong(small));
    return out;
  });
}

// stacked_lstm_result(workspace): waits for the current stream, raises if the last stack on this workspace gave up a wait, and
// says whether it met small states.
PyObject* stacked_lstm_result(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 1 || !is_tensor(a[0]) || !tensor_of(a[0]).is_cuda()) {
      PyErr_SetString(PyExc_TypeError, "stacked_lstm_result(workspace on the GPU)");
      return nullptr;
    }
    const at::Tensor& ws = tensor_of(a[0]);
    void *const wp = ws.data_ptr(), *const s = stream();
    int small = 0;
    const int rc = in_library([&] { return ftk_stacked_lstm_result(wp, &small, s); });
    return rc ? raise(rc) : PyBool_FromLong(small);
  });
}

// stacked_lstm_workspace(half, xs [T,B,H], WU [L,2H,4H]): the workspace of their stack.
PyObject* stacked_lstm_workspace(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 3 || !is_tensor(a[1]) || !is_tensor(a[2]) || tensor_of(a[1]).dim() != 3 || tensor_of(a[2]).dim() != 3) {
      PyErr_SetString(PyExc_TypeError, "stacked_lstm_workspace(half, xs [T,B,H], WU [L,2H,4H])");
      return nullptr;
    }
    const at::Tensor& xs = tensor_of(a[1]);
    const int L = dim(tensor_of(a[2]), 0), T = dim(xs, 0), B = dim(xs, 1), H = dim(xs, 2);
    const size_t need = a[0] == Py_True ? ftk_stacked_lstm_f16_workspace_bytes(L, T, B, H) : ftk_stacked_lstm_workspace_bytes(L, T, B, H);
    return THPVariable_Wrap(empty({(int64_t)need}, at::kByte, xs));
  });
}

PyMethodDef methods[] = {
    {"init", (PyCFunction)(void*)init, METH_FASTCALL, "init(counts, raise)"},
    {"b2b_gemm", (PyCFunction)(void*)b2b_gemm, METH_FASTCALL, "b2b_gemm(A, B_nk, C_pn, out)"},
    {"flash_attention", (PyCFunction)(void*)flash_attention, METH_FASTCALL,
     "flash_attention(half, Q, K, V, scale, out, workspace, split_keys)"},
    {"flash_attention_f32_flat", (PyCFunction)(void*)flash_attention_f32_flat, METH_FASTCALL,
     "flash_attention_f32_flat(q, k, v, B, Hd, Sq, Skv, D, scale)"},
    {"stacked_lstm", (PyCFunction)(void*)stacked_lstm, METH_FASTCALL,
     "stacked_lstm(half, xs, WU, bias, dilations, out, workspace, products, check, small)"},
    {"stacked_lstm_result", (PyCFunction)(void*)stacked_lstm_result, METH_FASTCALL, "stacked_lstm_result(workspace)"},
    {"stacked_lstm_workspace", (PyCFunction)(void*)stacked_lstm_workspace, METH_FASTCALL, "stacked_lstm_workspace(half, xs, WU)"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fast", "the fused entry points on torch tensors", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fast(void) { return PyModule_Create(&module); }

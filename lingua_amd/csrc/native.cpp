// The linear's host path for an interpreter that calls it per layer: checks, allocations and library calls of one forward or
// backward pass in one function.  Bound by the host: from Python a forward + backward of a small linear was some thirty
// crossings of the language boundary and eleven allocations at 1.5 to 2 us each around thirteen kernels that take 90 us.
// us per pass, [1021,2048].[2048,2048] with a bias, forward + backward 271 / 148; one token through a kept [2048,2048]
// weight 14.9 / 8.6.
//
// Every function returns None where its operands are not the plain ones (other types, devices, strides that need a copy,
// empty problems, a dispatch mode): the Python form in lingua_amd/float8.py then runs, with its error messages.  The memos
// and the weight cache stay there too; nothing is kept here between calls.
#include <ATen/ATen.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>

#include "../../include/lingua_fp8.h"

namespace {

using at::Tensor;

// The library's entries, taken from the handle that lingua_amd._lib loaded (bind): one copy of the library per process.
struct Library {
#define L8_ENTRY(name) decltype(&::name) name = nullptr;
#define L8_ENTRIES(X)                                                                                                        \
  X(l8_last_error) X(l8_linear_fwd_rows) X(l8_linear_fwd_rows_workspace) X(l8_cast_rowwise) X(l8_cast_rowwise_workspace)               \
  X(l8_cast_tensorwise) X(l8_cast_tensorwise_t_rows) X(l8_amax_reduce) X(l8_cast_colwise_transposed_pad) X(l8_cast_transposed_many) X(l8_col_amax) X(l8_col_sum) X(l8_col_sum_workspace) X(l8_gemm_nt) X(l8_linear_bwd_casts) X(l8_linear_bwd_casts_pays)
  L8_ENTRIES(L8_ENTRY)
#undef L8_ENTRY
} lib;

void check(int code, const char *what) {
  if (code != L8_OK) throw std::runtime_error(std::string(what) + " failed (" + std::to_string(code) + "): " + lib.l8_last_error());
}

// A bf16 matrix as the kernels take it: `rows` rows of `cols` elements, `ld` apart.
struct Rows {
  const void *p = nullptr;
  int64_t rows = 0, cols = 0, ld = 0;
};

bool plain_type(PyObject *o) {
  return THPVariable_CheckExact(o) || Py_TYPE(o) == reinterpret_cast<PyTypeObject *>(ParameterClass);
}

// Leading dimensions of a contiguous tensor count as one; a view that would need a copy is not taken.
bool as_rows(const Tensor &t, int device, Rows &m) {
  if (t.scalar_type() != at::kBFloat16 || t.layout() != at::kStrided || !t.is_cuda() || t.get_device() != device || t.dim() < 2) return false;
  m.cols = t.size(-1);
  if (t.dim() == 2) {
    m.rows = t.size(0);
    if (m.rows < 1 || m.cols < 1 || t.stride(1) != 1 || t.stride(0) < m.cols) return false;
    m.ld = m.rows > 1 ? t.stride(0) : m.cols;
  } else {
    if (t.numel() < 1 || !t.is_contiguous()) return false;
    m.rows = t.numel() / m.cols;
    m.ld = m.cols;
  }
  m.p = t.const_data_ptr();
  return true;
}

// A dense tensor of `n` elements of one type (quantised copies, scales, amaxes, bias).
bool dense(const Tensor &t, at::ScalarType type, int64_t n, int device) {
  return t.defined() && t.scalar_type() == type && t.layout() == at::kStrided && t.is_cuda() && t.get_device() == device && t.numel() == n && t.is_contiguous();
}

// A quantised operand handed in: rows x cols bytes, rows any stride apart (0: not one).
int64_t fp8_rows(const Tensor &t, int64_t rows, int64_t cols, int device) {
  if (!t.defined() || t.scalar_type() != at::kFloat8_e4m3fn || t.layout() != at::kStrided || !t.is_cuda() || t.get_device() != device ||
      t.dim() != 2 || t.size(0) != rows || t.size(1) != cols || t.stride(1) != 1 || (rows > 1 && t.stride(0) < cols))
    return 0;
  return rows > 1 ? t.stride(0) : cols;
}
// A new one, its rows on 128-byte lines (figures in linear.cpp) or dense.
Tensor empty_fp8(int64_t rows, int64_t cols, const at::TensorOptions &o, bool on_lines = true) {
  return at::empty_strided({rows, cols}, {on_lines ? (cols + 127) / 128 * 128 : cols, 1}, o.dtype(at::kFloat8_e4m3fn));
}

Tensor arg(PyObject *o) { return o == Py_None ? Tensor() : THPVariable_Unpack(o); }
PyObject *wrap(const Tensor &t) {
  if (!t.defined()) Py_RETURN_NONE;
  return THPVariable_Wrap(t);
}
bool truth(PyObject *o) {  // as `if` takes it: a switch of the configuration may hold any number
  const int t = PyObject_IsTrue(o);
  if (t < 0) throw python_error();
  return t != 0;
}
bool tensors(PyObject *const *args, int n) {  // Tensor or Parameter with memory of its own (not a batch under vmap) or None, and no mode that wants to see what is done to them
  for (int i = 0; i < n; ++i)
    if (args[i] != Py_None && !(plain_type(args[i]) && THPVariable_Unpack(args[i]).has_storage())) return false;
  return !c10::impl::dispatch_mode_enabled();
}
PyObject *tuple_of(std::initializer_list<Tensor> ts) {
  PyObject *out = PyTuple_New((Py_ssize_t)ts.size());
  if (!out) throw python_error();
  Py_ssize_t i = 0;
  for (const Tensor &t : ts) PyTuple_SET_ITEM(out, i++, wrap(t));
  return out;
}

// Work space of one call: freed into the caching allocator on return, as a Python temporary's would be.
struct Space {
  Tensor t;
  Space(const Tensor &like, int64_t bytes) {
    if (bytes > 0) t = at::empty({bytes}, like.options().dtype(at::kByte));
  }
  void *p() const { return t.defined() ? t.mutable_data_ptr() : nullptr; }
};

// linear_fwd(x, w, bias, qx, sx, x_ready, want_qx, want_col, qw, sw, want_amax, algo) -> (y, qx, sx, col amax, w's row amax) or None.
// The casts and the product of l8_linear_fwd_rows.  qx / sx: x already quantised (x_ready); want_qx: hand the quantised x out.
PyObject *linear_fwd(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 12) throw std::runtime_error("linear_fwd: 12 arguments");
  if (!tensors(args, 5) || !tensors(args + 8, 2) || args[0] == Py_None || args[1] == Py_None) Py_RETURN_NONE;
  const Tensor &x = THPVariable_Unpack(args[0]), &w = THPVariable_Unpack(args[1]);
  const Tensor bias = arg(args[2]), qx_in = arg(args[3]), sx_in = arg(args[4]), qw = arg(args[8]), sw = arg(args[9]);
  const bool x_ready = truth(args[5]), want_qx = truth(args[6]), want_col = truth(args[7]), want_amax = truth(args[10]);
  const int64_t algo = PyLong_AsLongLong(args[11]);
  if (!x.is_cuda()) Py_RETURN_NONE;
  const int device = x.get_device();
  Rows rx, rw;
  if (!as_rows(x, device, rx) || !as_rows(w, device, rw) || w.dim() != 2 || rx.cols != rw.cols || rx.cols % 16 || rw.rows % 16 ||
      c10::hip::current_device() != device)
    Py_RETURN_NONE;
  const int64_t M = rx.rows, N = rw.rows, K = rx.cols;
  int64_t ldqx = x_ready ? fp8_rows(qx_in, M, K, device) : K, ldqw = qw.defined() ? fp8_rows(qw, N, K, device) : K;
  if ((bias.defined() && !dense(bias, at::kBFloat16, N, device)) || !ldqx || !ldqw || (x_ready && !dense(sx_in, at::kFloat, M, device)) ||
      (qw.defined() && !dense(sw, at::kFloat, N, device)))
    Py_RETURN_NONE;
  Tensor y, qx, sx, col, amax;
  {
    pybind11::gil_scoped_release no_gil;
    const auto o = x.options();
    if (x.dim() == 2) {
      y = at::empty({M, N}, o);
    } else {
      at::DimVector shape(x.sizes().begin(), x.sizes().end());
      shape.back() = N;
      y = at::empty(shape, o);
    }
    qx = qx_in;
    sx = sx_in;
    if (!x_ready && want_qx) {
      qx = empty_fp8(M, K, o);
      ldqx = qx.stride(0);
      sx = at::empty({M, 1}, o.dtype(at::kFloat));
    }
    if (want_col) col = at::empty({K}, o.dtype(at::kFloat));
    if (want_amax) amax = at::empty({N, 1}, o);
    l8_linear_fwd_args a{};
    a.x = rx.p, a.M = M, a.K = K, a.ldx = rx.ld;
    a.w = rw.p, a.N = N, a.ldw = rw.ld;
    a.bias = bias.defined() ? bias.const_data_ptr() : nullptr;
    a.y = y.mutable_data_ptr(), a.ldy = N;
    if (qx.defined()) a.qx = qx.mutable_data_ptr(), a.sx = sx.mutable_data_ptr<float>(), a.x_ready = x_ready;
    if (col.defined()) a.col_amax_x = col.mutable_data_ptr<float>();
    if (qw.defined()) a.qw = qw.mutable_data_ptr(), a.sw = sw.mutable_data_ptr<float>(), a.w_ready = 1;
    if (amax.defined()) a.amax_w = amax.mutable_data_ptr();
    a.algo = algo;
    a.stream = c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream();
    const int64_t need = lib.l8_linear_fwd_rows_workspace(&a, ldqx, ldqw);
    const Space ws(x, need);  // a negative size is an error that the call below reports
    a.workspace = ws.p(), a.workspace_bytes = need > 0 ? need : 0;
    check(lib.l8_linear_fwd_rows(&a, ldqx, ldqw), "l8_linear_fwd");
  }
  return tuple_of({y, qx, sx, col, amax});
  END_HANDLE_TH_ERRORS
}

// A matrix quantised along its rows' direction, padded to 16 of them, in the layout that the weight gradient multiplies with.
void cast_colwise_t(const Tensor &like, const Rows &m, const Tensor &col, bool on_lines, Tensor &q, Tensor &s, void *stream) {
  const auto o = like.options();
  const int64_t padded = (m.rows + 15) / 16 * 16;
  q = empty_fp8(m.cols, padded, o, on_lines);
  s = at::empty({m.cols, 1}, o.dtype(at::kFloat));
  check(lib.l8_cast_colwise_transposed_pad(m.p, m.rows, m.cols, m.ld, col.const_data_ptr<float>(), q.mutable_data_ptr(), q.stride(0), padded,
                                           s.mutable_data_ptr<float>(), stream), "l8_cast_colwise_transposed_pad");
}

// linear_bwd(g, a, w, w's row amax, a's col amax, qat, sat, qwt, swt, need_a, need_b, need_bias, algo)
//   -> (grad a, grad w, grad bias, qat, sat) or None.  fp8 weight gradient.  qat / sat: a already quantised along the tokens
// (then a may be None); qwt / swt: w already quantised tensor-wise and transposed.
PyObject *linear_bwd(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 13) throw std::runtime_error("linear_bwd: 13 arguments");
  if (!tensors(args, 9) || args[0] == Py_None || args[2] == Py_None || args[3] == Py_None) Py_RETURN_NONE;
  const Tensor &g = THPVariable_Unpack(args[0]), &w = THPVariable_Unpack(args[2]), &amax = THPVariable_Unpack(args[3]);
  const Tensor a = arg(args[1]), a_col_in = arg(args[4]), qat_in = arg(args[5]), sat_in = arg(args[6]), qwt_in = arg(args[7]), swt_in = arg(args[8]);
  const bool need_a = truth(args[9]), need_b = truth(args[10]), need_bias = truth(args[11]);
  const int algo = (int)PyLong_AsLongLong(args[12]);
  if (!g.is_cuda()) Py_RETURN_NONE;
  const int device = g.get_device();
  Rows rg, rw, ra;
  if (g.dim() != 2 || w.dim() != 2 || !as_rows(g, device, rg) || !as_rows(w, device, rw) || c10::hip::current_device() != device) Py_RETURN_NONE;
  const int64_t M = rg.rows, N = rg.cols, K = rw.cols, padded = (M + 15) / 16 * 16;
  if (rw.rows != N || N % 16 || K % 16 || !dense(amax, at::kBFloat16, N, device) ||
      (need_bias && (rg.ld % 8 || reinterpret_cast<uintptr_t>(rg.p) % 16)))
    Py_RETURN_NONE;
  if (need_b && !qat_in.defined() && !(a.defined() && a.dim() == 2 && as_rows(a, device, ra) && ra.rows == M && ra.cols == K)) Py_RETURN_NONE;
  if ((qat_in.defined() && !(fp8_rows(qat_in, K, padded, device) && dense(sat_in, at::kFloat, K, device))) ||
      (qwt_in.defined() && !(fp8_rows(qwt_in, K, N, device) && dense(swt_in, at::kFloat, 1, device))) ||
      (a_col_in.defined() && !dense(a_col_in, at::kFloat, K, device)))
    Py_RETURN_NONE;
  Tensor ga, gb, gbias, qat = qat_in, sat = sat_in, qwt = qwt_in, swt = swt_in;
  {
    pybind11::gil_scoped_release no_gil;
    const auto o = g.options();
    void *stream = c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream();
    Tensor g_col, qg, sg, qgt, sgt;
    // the casts of a small pass in two launches
    const bool together = need_a && need_b && !(need_b && !qat.defined() && !a_col_in.defined()) &&
                          (reinterpret_cast<uintptr_t>(amax.const_data_ptr()) % 16) == 0 && lib.l8_linear_bwd_casts_pays(M, N, K);
    if (together) {
      l8_linear_bwd_casts_args c{};
      qg = empty_fp8(M, N, o), sg = at::empty({M, 1}, o.dtype(at::kFloat));
      qgt = empty_fp8(N, padded, o), sgt = at::empty({N, 1}, o.dtype(at::kFloat));
      c.g = rg.p, c.M = M, c.N = N, c.ldg = rg.ld, c.K = K, c.Mp = padded, c.stream = stream;
      c.qg = qg.mutable_data_ptr(), c.ldqg = qg.stride(0), c.sg = sg.mutable_data_ptr<float>();
      c.qgt = qgt.mutable_data_ptr(), c.ldqgt = qgt.stride(0), c.sgt = sgt.mutable_data_ptr<float>();
      if (!qat.defined()) {
        qat = empty_fp8(K, padded, o), sat = at::empty({K, 1}, o.dtype(at::kFloat));
        c.a = ra.p, c.lda = ra.ld, c.a_col = a_col_in.const_data_ptr<float>();
        c.qat = qat.mutable_data_ptr(), c.ldqat = qat.stride(0), c.sat = sat.mutable_data_ptr<float>();
      }
      if (!qwt.defined()) {
        qwt = empty_fp8(K, N, o), swt = at::empty({1, 1}, o.dtype(at::kFloat));
        c.w = rw.p, c.ldw = rw.ld, c.amax_w = amax.const_data_ptr();
        c.qwt = qwt.mutable_data_ptr(), c.ldqwt = qwt.stride(0), c.swt = swt.mutable_data_ptr<float>();
      }
      c.workspace_bytes = lib.l8_cast_rowwise_workspace(M, N);
      const Space ws(g, c.workspace_bytes);
      c.workspace = ws.p();
      check(lib.l8_linear_bwd_casts(&c), "l8_linear_bwd_casts");
    }
    if (need_b && !together) g_col = at::empty({N}, o.dtype(at::kFloat));
    if (need_a && !together) {
      qg = empty_fp8(M, N, o), sg = at::empty({M, 1}, o.dtype(at::kFloat));
      const int64_t ws_bytes = need_b ? lib.l8_cast_rowwise_workspace(M, N) : 0;
      const Space ws(g, ws_bytes);
      check(lib.l8_cast_rowwise(rg.p, M, N, rg.ld, qg.mutable_data_ptr(), qg.stride(0), sg.mutable_data_ptr<float>(), nullptr,
                                need_b ? g_col.mutable_data_ptr<float>() : nullptr, ws.p(), ws_bytes, stream), "l8_cast_rowwise");
      if (!qwt.defined()) {
        qwt = empty_fp8(K, N, o);
        swt = at::empty({1, 1}, o.dtype(at::kFloat));
        if (N % 8 == 0 && N <= 16384 && (reinterpret_cast<uintptr_t>(amax.const_data_ptr()) % 16) == 0) {
          check(lib.l8_cast_tensorwise_t_rows(rw.p, N, K, rw.ld, amax.const_data_ptr(), N, qwt.mutable_data_ptr(), qwt.stride(0), swt.mutable_data_ptr<float>(), stream),
                "l8_cast_tensorwise_t_rows");
        } else {
          Tensor whole = at::empty({1, 1}, o);
          check(lib.l8_amax_reduce(amax.const_data_ptr(), N, whole.mutable_data_ptr(), stream), "l8_amax_reduce");
          check(lib.l8_cast_tensorwise(rw.p, N, K, rw.ld, whole.const_data_ptr(), L8_AMAX_BF16, 1, qwt.mutable_data_ptr(), qwt.stride(0), swt.mutable_data_ptr<float>(), stream),
                "l8_cast_tensorwise");
        }
      }
    }
    if (need_a) {
      ga = at::empty({M, K}, o);
      check(lib.l8_gemm_nt(qg.const_data_ptr(), qwt.const_data_ptr(), M, K, N, qg.stride(0), qwt.stride(0), sg.const_data_ptr<float>(), L8_SCALE_ROW, swt.const_data_ptr<float>(),
                           L8_SCALE_SCALAR, nullptr, ga.mutable_data_ptr(), K, algo, stream), "l8_gemm_nt");
    } else if (need_b) {
      check(lib.l8_col_amax(rg.p, M, N, rg.ld, g_col.mutable_data_ptr<float>(), stream), "l8_col_amax");
    }
    if (need_b) {
      if (together) {   // made above
      } else if (qat.defined()) {
        cast_colwise_t(g, rg, g_col, true, qgt, sgt, stream);
      } else {
        Tensor a_col = a_col_in;
        if (!a_col.defined()) {
          a_col = at::empty({K}, o.dtype(at::kFloat));
          check(lib.l8_col_amax(ra.p, M, K, ra.ld, a_col.mutable_data_ptr<float>(), stream), "l8_col_amax");
        }
        qgt = empty_fp8(N, padded, o), sgt = at::empty({N, 1}, o.dtype(at::kFloat));
        qat = empty_fp8(K, padded, o), sat = at::empty({K, 1}, o.dtype(at::kFloat));
        const l8_cast_transposed_item both[2] = {
            {rg.p, M, N, rg.ld, g_col.const_data_ptr<float>(), nullptr, 0, qgt.mutable_data_ptr(), qgt.stride(0), padded, sgt.mutable_data_ptr<float>()},
            {ra.p, M, K, ra.ld, a_col.const_data_ptr<float>(), nullptr, 0, qat.mutable_data_ptr(), qat.stride(0), padded, sat.mutable_data_ptr<float>()}};
        check(lib.l8_cast_transposed_many(both, 2, stream), "l8_cast_transposed_many");
      }
      gb = at::empty({N, K}, o);
      check(lib.l8_gemm_nt(qgt.const_data_ptr(), qat.const_data_ptr(), N, K, padded, qgt.stride(0), qat.stride(0), sgt.const_data_ptr<float>(), L8_SCALE_ROW,
                           sat.const_data_ptr<float>(), L8_SCALE_ROW, nullptr, gb.mutable_data_ptr(), K, algo, stream), "l8_gemm_nt");
    }
    if (need_bias) {
      gbias = at::empty({N}, o);
      const int64_t ws_bytes = lib.l8_col_sum_workspace(M, N);
      const Space ws(g, ws_bytes);
      check(lib.l8_col_sum(rg.p, M, N, rg.ld, gbias.mutable_data_ptr(), ws.p(), ws_bytes, stream), "l8_col_sum");
    }
  }
  return tuple_of({ga, gb, gbias, qat, sat});
  END_HANDLE_TH_ERRORS
}

// cast_colwise_transposed(a, col amax, on_lines) -> (q, s) or None, as in lingua_amd.ops
PyObject *cast_colwise_transposed(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 3) throw std::runtime_error("cast_colwise_transposed: 3 arguments");
  if (!tensors(args, 2) || args[0] == Py_None || args[1] == Py_None) Py_RETURN_NONE;
  const Tensor &a = THPVariable_Unpack(args[0]), &col = THPVariable_Unpack(args[1]);
  if (!a.is_cuda()) Py_RETURN_NONE;
  const int device = a.get_device();
  Rows ra;
  if (a.dim() != 2 || !as_rows(a, device, ra) || !dense(col, at::kFloat, ra.cols, device) || c10::hip::current_device() != device) Py_RETURN_NONE;
  const bool on_lines = truth(args[2]);
  Tensor q, s;
  {
    pybind11::gil_scoped_release no_gil;
    cast_colwise_t(a, ra, col, on_lines, q, s, c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream());
  }
  return tuple_of({q, s});
  END_HANDLE_TH_ERRORS
}

// key(tensor) -> bytes: equal for two tensors of the same memory, shape, strides, type, device and version, seen from the
// same current stream.
PyObject *key(PyObject *, PyObject *o) {
  HANDLE_TH_ERRORS
  const Tensor &t = THPVariable_Unpack(o);
  const int64_t dim = t.dim();
  c10::SmallVector<int64_t, 16> v;
  v.push_back(reinterpret_cast<int64_t>(t.const_data_ptr()));
  v.push_back((int64_t)t._version());
  v.push_back(((int64_t)t.scalar_type() << 32) | ((int64_t)t.device().type() << 16) | (uint16_t)t.device().index());
  v.push_back(t.is_cuda() ? reinterpret_cast<int64_t>(c10::hip::getCurrentHIPStream((c10::DeviceIndex)t.get_device()).stream()) : 0);
  for (int64_t i = 0; i < dim; ++i) {
    v.push_back(t.size(i));
    v.push_back(t.stride(i));
  }
  return PyBytes_FromStringAndSize(reinterpret_cast<const char *>(v.data()), (Py_ssize_t)(v.size() * sizeof(int64_t)));
  END_HANDLE_TH_ERRORS
}

// bind(handle of the loaded library, as ctypes holds it)
PyObject *bind(PyObject *, PyObject *o) {
  HANDLE_TH_ERRORS
  void *h = PyLong_AsVoidPtr(o);
  if (!h && PyErr_Occurred()) throw python_error();
#define L8_LOOK_UP(name)                                                   \
  lib.name = reinterpret_cast<decltype(lib.name)>(dlsym(h, #name));        \
  if (!lib.name) throw std::runtime_error("the library has no entry " #name);
  L8_ENTRIES(L8_LOOK_UP)
#undef L8_LOOK_UP
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"bind", bind, METH_O, nullptr},
    {"key", key, METH_O, nullptr},
    {"linear_fwd", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(linear_fwd)), METH_FASTCALL, nullptr},
    {"linear_bwd", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(linear_bwd)), METH_FASTCALL, nullptr},
    {"cast_colwise_transposed", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(cast_colwise_transposed)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native() { return PyModule_Create(&module_def); }

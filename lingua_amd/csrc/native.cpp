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
  X(l8_cast_tensorwise) X(l8_cast_tensorwise_t_rows) X(l8_amax_reduce) X(l8_cast_colwise_transposed_pad) X(l8_cast_transposed_many) X(l8_col_amax) X(l8_col_sum) X(l8_col_sum_workspace) X(l8_gemm_nt) X(l8_linear_bwd_casts_bias) X(l8_linear_bwd_casts_pays)  \
  X(l8_cast_rowwise_many) X(l8_cast_rowwise_cols_many) X(l8_gemm_nt_multi) X(l8_gemm_nt_sum) X(l8_rmsnorm_cast_rowwise)            \
  X(l8_rmsnorm_workspace) X(l8_rmsnorm_bwd_as) X(l8_rmsnorm_bwd_workspace) X(l8_swiglu_cast_rowwise) X(l8_swiglu_workspace)        \
  X(l8_swiglu_bwd_cast_rowwise_q) X(l8_swiglu_bwd_cast_transposed)
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
      if (need_bias) gbias = at::empty({N}, o);
      check(lib.l8_linear_bwd_casts_bias(&c, need_bias ? gbias.mutable_data_ptr() : nullptr), "l8_linear_bwd_casts");
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
    if (need_bias && !together) {
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

// ---- fused blocks ----
// Attention projections, gated MLP and norm: one call per pass where the Python form (lingua_amd/qkv.py, swiglu.py, norm.py,
// float8.shared_input_backward) makes ten to fifteen and twice as many allocations.  us per pass, forward + backward, bound by
// the host, before / now: norm and projections [337,2624] 517 / 160, norm and MLP [400,1328] with 2688 hidden 554 / 234.

// Temporaries of one phase of a pass, in one allocation that is freed into the caching allocator behind the phase.
struct Arena {
  int64_t bytes = 0;
  Tensor t;
  int64_t add(int64_t n) {
    const int64_t at = bytes;
    bytes += (n + 255) / 256 * 256;
    return at;
  }
  void make(const Tensor &like) { t = at::empty({bytes > 0 ? bytes : 1}, like.options().dtype(at::kByte)); }
  uint8_t *p(int64_t at) const { return static_cast<uint8_t *>(t.mutable_data_ptr()) + at; }
  float *f(int64_t at) const { return reinterpret_cast<float *>(p(at)); }
};

int64_t on_lines(int64_t cols) { return (cols + 127) / 128 * 128; }

// A quantised operand in an arena: rows on 128-byte lines, and its scales.
struct Quantised {
  int64_t rows, cols, ld, q, s;
  Quantised(Arena &a, int64_t rows_, int64_t cols_, int64_t scales) : rows(rows_), cols(cols_), ld(on_lines(cols_)), q(a.add(rows_ * on_lines(cols_))), s(a.add(scales * 4)) {}
};

// Can a weight with these row amaxes be quantised tensor-wise from the list (as lingua_amd.ops asks)?
bool listed(const Tensor &amax, int64_t rows, int device) {
  return dense(amax, at::kBFloat16, rows, device) && rows % 8 == 0 && rows <= 16384 && reinterpret_cast<uintptr_t>(amax.const_data_ptr()) % 16 == 0;
}
l8_cast_transposed_item by_columns(const Rows &m, const float *col, const Arena &a, const Quantised &q) {
  return {m.p, m.rows, m.cols, m.ld, col, nullptr, 0, a.p(q.q), q.ld, q.cols, a.f(q.s)};
}
l8_cast_transposed_item by_tensor(const Rows &w, const Tensor &amax, const Arena &a, const Quantised &q) {
  return {w.p, w.rows, w.cols, w.ld, nullptr, amax.const_data_ptr(), w.rows, a.p(q.q), q.ld, w.rows, a.f(q.s)};
}
bool weight(const Tensor &w, int device, Rows &m) { return w.defined() && w.dim() == 2 && as_rows(w, device, m) && m.rows % 16 == 0 && m.cols % 16 == 0; }
void *stream_of(int device) { return c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream(); }
// the activation of a block: plain, on the current device
bool activation(const Tensor &x, Rows &m) {
  return x.defined() && x.is_cuda() && x.dim() == 2 && as_rows(x, x.get_device(), m) && m.cols % 16 == 0 && c10::hip::current_device() == x.get_device();
}

// rmsnorm_fwd(x, weight, eps, want_col) -> (y, q, scale, rstd, col amax) or None
PyObject *rmsnorm_fwd(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 4) throw std::runtime_error("rmsnorm_fwd: 4 arguments");
  if (!tensors(args, 2) || args[0] == Py_None || args[1] == Py_None) Py_RETURN_NONE;
  const Tensor &x = THPVariable_Unpack(args[0]), &w = THPVariable_Unpack(args[1]);
  const double eps = PyFloat_AsDouble(args[2]);
  if (eps == -1.0 && PyErr_Occurred()) throw python_error();
  const bool want_col = truth(args[3]);
  Rows rx;
  if (!activation(x, rx)) Py_RETURN_NONE;
  const int device = x.get_device();
  const int64_t R = rx.rows, C = rx.cols;
  const bool f32 = w.scalar_type() == at::kFloat;
  if (!dense(w, f32 ? at::kFloat : at::kBFloat16, C, device)) Py_RETURN_NONE;
  Tensor y, q, s, rstd, col;
  {
    pybind11::gil_scoped_release no_gil;
    const auto o = x.options();
    y = at::empty({R, C}, o);
    q = empty_fp8(R, C, o);
    s = at::empty({R, 1}, o.dtype(at::kFloat));
    rstd = at::empty({R, 1}, o.dtype(at::kFloat));
    if (want_col) col = at::empty({C}, o.dtype(at::kFloat));
    const int64_t ws_bytes = want_col ? lib.l8_rmsnorm_workspace(R, C) : 0;
    const Space ws(x, ws_bytes);
    check(lib.l8_rmsnorm_cast_rowwise(rx.p, w.const_data_ptr(), f32, R, C, rx.ld, (float)eps, y.mutable_data_ptr(), C, q.mutable_data_ptr(), q.stride(0),
                                      s.mutable_data_ptr<float>(), rstd.mutable_data_ptr<float>(), want_col ? col.mutable_data_ptr<float>() : nullptr, ws.p(),
                                      ws_bytes, stream_of(device)), "l8_rmsnorm_cast_rowwise");
  }
  return tuple_of({y, q, s, rstd, col});
  END_HANDLE_TH_ERRORS
}

// rmsnorm_bwd(gy, x, weight, rstd) -> (gx, gw of the weight's type) or None
PyObject *rmsnorm_bwd(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 4) throw std::runtime_error("rmsnorm_bwd: 4 arguments");
  if (!tensors(args, 4)) Py_RETURN_NONE;
  const Tensor gy = arg(args[0]), x = arg(args[1]), w = arg(args[2]), rstd = arg(args[3]);
  Rows rx, rg;
  if (!activation(x, rx) || !activation(gy, rg) || gy.get_device() != x.get_device() || rg.rows != rx.rows || rg.cols != rx.cols) Py_RETURN_NONE;
  const int device = x.get_device();
  const int64_t R = rx.rows, C = rx.cols;
  const bool f32 = w.defined() && w.scalar_type() == at::kFloat;
  if (!dense(w, f32 ? at::kFloat : at::kBFloat16, C, device) || !dense(rstd, at::kFloat, R, device)) Py_RETURN_NONE;
  Tensor gx, gw;
  {
    pybind11::gil_scoped_release no_gil;
    gx = at::empty({R, C}, x.options());
    gw = at::empty({C}, w.options());
    const int64_t ws_bytes = lib.l8_rmsnorm_bwd_workspace(R, C);
    const Space ws(x, ws_bytes > 16 ? ws_bytes : 16);
    check(lib.l8_rmsnorm_bwd_as(rg.p, rx.p, w.const_data_ptr(), f32, rstd.const_data_ptr<float>(), R, C, rg.ld, rx.ld, gx.mutable_data_ptr(), C,
                                gw.mutable_data_ptr(), f32, ws.p(), ws_bytes, stream_of(device)), "l8_rmsnorm_bwd");
  }
  return tuple_of({gx, gw});
  END_HANDLE_TH_ERRORS
}

// The activation quantised, if it is not yet, for a block's forward pass.
void cast_activation(const Tensor &x, const Rows &rx, bool want_col, void *q, int64_t ldq, float *s, Tensor &col, void *stream) {
  if (want_col) col = at::empty({rx.cols}, x.options().dtype(at::kFloat));
  const int64_t ws_bytes = want_col ? lib.l8_cast_rowwise_workspace(rx.rows, rx.cols) : 0;
  const Space ws(x, ws_bytes);
  check(lib.l8_cast_rowwise(rx.p, rx.rows, rx.cols, rx.ld, q, ldq, s, nullptr, want_col ? col.mutable_data_ptr<float>() : nullptr, ws.p(), ws_bytes, stream),
        "l8_cast_rowwise");
}

// qkv_fwd(x, wq, wk, wv, qx, sx, want_col, algo) -> (y, row amax of wq, of wk, of wv, qx, sx, col amax of x) or None.
// qx / sx: x already quantised (then want_col is not looked at).
PyObject *qkv_fwd(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 8) throw std::runtime_error("qkv_fwd: 8 arguments");
  if (!tensors(args, 6)) Py_RETURN_NONE;
  const Tensor x = arg(args[0]), w[3] = {arg(args[1]), arg(args[2]), arg(args[3])}, qx_in = arg(args[4]), sx_in = arg(args[5]);
  const bool want_col = truth(args[6]);
  const int algo = (int)PyLong_AsLongLong(args[7]);
  Rows rx, rw[3];
  if (!activation(x, rx)) Py_RETURN_NONE;
  const int device = x.get_device();
  const int64_t M = rx.rows, K = rx.cols;
  int64_t N = 0;
  for (int i = 0; i < 3; ++i) {
    if (!weight(w[i], device, rw[i]) || rw[i].cols != K) Py_RETURN_NONE;
    N += rw[i].rows;
  }
  int64_t ldqx = qx_in.defined() ? fp8_rows(qx_in, M, K, device) : on_lines(K);
  if (!ldqx || (qx_in.defined() && !dense(sx_in, at::kFloat, M, device))) Py_RETURN_NONE;
  Tensor y, qx = qx_in, sx = sx_in, col, amax[3];
  {
    pybind11::gil_scoped_release no_gil;
    const auto o = x.options();
    void *stream = stream_of(device);
    if (!qx.defined()) {
      qx = empty_fp8(M, K, o), sx = at::empty({M, 1}, o.dtype(at::kFloat));
      cast_activation(x, rx, want_col, qx.mutable_data_ptr(), ldqx, sx.mutable_data_ptr<float>(), col, stream);
    }
    Arena a;
    const Quantised qw(a, N, K, N);
    a.make(x);
    l8_cast_rowwise_item items[3];
    for (int64_t i = 0, row = 0; i < 3; row += rw[i++].rows) {
      amax[i] = at::empty({rw[i].rows, 1}, o);
      items[i] = {rw[i].p, rw[i].rows, rw[i].ld, a.p(qw.q) + row * qw.ld, qw.ld, a.f(qw.s) + row, amax[i].mutable_data_ptr()};
    }
    check(lib.l8_cast_rowwise_many(items, 3, K, stream), "l8_cast_rowwise_many");
    y = at::empty({M, N}, o);
    check(lib.l8_gemm_nt(qx.const_data_ptr(), a.p(qw.q), M, N, K, ldqx, qw.ld, sx.const_data_ptr<float>(), L8_SCALE_ROW, a.f(qw.s), L8_SCALE_ROW, nullptr,
                         y.mutable_data_ptr(), N, algo, stream), "l8_gemm_nt");
  }
  return tuple_of({y, amax[0], amax[1], amax[2], qx, sx, col});
  END_HANDLE_TH_ERRORS
}

// shared_bwd((grad ...), x, (w ...), (row amax of w ...), col amax of x, qxt, sxt, algo) -> (grad x, qxt, sxt, grad w ...) or None:
// float8.shared_input_backward of up to three linears that all learn.  qxt / sxt: x already quantised along the tokens.
PyObject *shared_bwd(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 8) throw std::runtime_error("shared_bwd: 8 arguments");
  constexpr int kMost = 3;
  const Py_ssize_t k = PyTuple_Check(args[0]) ? PyTuple_GET_SIZE(args[0]) : 0;
  if (k < 1 || k > kMost || !PyTuple_Check(args[2]) || !PyTuple_Check(args[3]) || PyTuple_GET_SIZE(args[2]) != k || PyTuple_GET_SIZE(args[3]) != k) Py_RETURN_NONE;
  for (int i : {0, 2, 3})
    if (!tensors(&PyTuple_GET_ITEM(args[i], 0), (int)k)) Py_RETURN_NONE;
  if (!tensors(args + 1, 1) || !tensors(args + 4, 3)) Py_RETURN_NONE;
  const Tensor x = arg(args[1]), x_col = arg(args[4]), qxt_in = arg(args[5]), sxt_in = arg(args[6]);
  const int algo = (int)PyLong_AsLongLong(args[7]);
  Rows rx, rg[kMost], rw[kMost];
  Tensor g[kMost], w[kMost], amax[kMost];
  if (!activation(x, rx)) Py_RETURN_NONE;
  const int device = x.get_device();
  const int64_t M = rx.rows, K = rx.cols, padded = (M + 15) / 16 * 16;
  for (Py_ssize_t i = 0; i < k; ++i) {
    g[i] = arg(PyTuple_GET_ITEM(args[0], i)), w[i] = arg(PyTuple_GET_ITEM(args[2], i)), amax[i] = arg(PyTuple_GET_ITEM(args[3], i));
    if (!activation(g[i], rg[i]) || g[i].get_device() != device || !weight(w[i], device, rw[i]) || rg[i].rows != M || rw[i].cols != K ||
        rw[i].rows != rg[i].cols || !amax[i].defined() || !listed(amax[i], rw[i].rows, device))
      Py_RETURN_NONE;
  }
  if (qxt_in.defined() ? !(fp8_rows(qxt_in, K, padded, device) && dense(sxt_in, at::kFloat, K, device)) : !(x_col.defined() && dense(x_col, at::kFloat, K, device)))
    Py_RETURN_NONE;
  Tensor gx, gw[kMost], qxt = qxt_in, sxt = sxt_in;
  {
    pybind11::gil_scoped_release no_gil;
    const auto o = x.options();
    void *stream = stream_of(device);
    Arena cols;  // column amaxes of the gradients: from the first phase to the second
    int64_t col[kMost];
    for (int i = 0; i < k; ++i) col[i] = cols.add(rg[i].cols * 4);
    cols.make(x);
    {
      Arena a;
      std::vector<Quantised> qg, qw;
      int64_t ws[kMost], ws_bytes[kMost];
      for (int i = 0; i < k; ++i) {
        qg.emplace_back(a, M, rg[i].cols, M);
        qw.emplace_back(a, K, rw[i].rows, 1);
        ws_bytes[i] = lib.l8_cast_rowwise_workspace(M, rg[i].cols);
        ws[i] = a.add(ws_bytes[i]);
      }
      a.make(x);
      l8_cast_rowwise_cols_item casts[kMost];
      l8_cast_transposed_item weights[kMost];
      l8_gemm_term terms[kMost];
      for (int i = 0; i < k; ++i) {
        casts[i] = {rg[i].p, M, rg[i].cols, rg[i].ld, a.p(qg[i].q), qg[i].ld, a.f(qg[i].s), nullptr, cols.f(col[i]), a.p(ws[i]), ws_bytes[i]};
        weights[i] = by_tensor(rw[i], amax[i], a, qw[i]);
        terms[i] = {a.p(qg[i].q), a.p(qw[i].q), rg[i].cols, qg[i].ld, qw[i].ld, a.f(qg[i].s), a.f(qw[i].s)};
      }
      check(lib.l8_cast_rowwise_cols_many(casts, k, stream), "l8_cast_rowwise_cols_many");
      check(lib.l8_cast_transposed_many(weights, k, stream), "l8_cast_transposed_many");
      gx = at::empty({M, K}, o);
      check(lib.l8_gemm_nt_sum(terms, k, M, K, gx.mutable_data_ptr(), K, algo, stream), "l8_gemm_nt_sum");
    }
    Arena a;
    std::vector<Quantised> qt;
    for (int i = 0; i < k; ++i) qt.emplace_back(a, rg[i].cols, padded, rg[i].cols);
    a.make(x);
    l8_cast_transposed_item casts[kMost + 1];
    l8_gemm_part parts[kMost];
    for (int i = 0; i < k; ++i) {
      gw[i] = at::empty({rw[i].rows, K}, o);
      casts[i] = by_columns(rg[i], cols.f(col[i]), a, qt[i]);
      parts[i] = {a.p(qt[i].q), rw[i].rows, a.f(qt[i].s), gw[i].mutable_data_ptr()};
    }
    int64_t n_casts = k;
    if (!qxt.defined()) {
      qxt = empty_fp8(K, padded, o), sxt = at::empty({K, 1}, o.dtype(at::kFloat));
      casts[n_casts++] = {rx.p, M, K, rx.ld, x_col.const_data_ptr<float>(), nullptr, 0, qxt.mutable_data_ptr(), qxt.stride(0), padded, sxt.mutable_data_ptr<float>()};
    }
    check(lib.l8_cast_transposed_many(casts, n_casts, stream), "l8_cast_transposed_many");
    check(lib.l8_gemm_nt_multi(parts, k, qxt.const_data_ptr(), K, padded, on_lines(padded), qxt.stride(0), sxt.const_data_ptr<float>(), L8_SCALE_ROW, K, algo, stream),
          "l8_gemm_nt_multi");
  }
  PyObject *out = PyTuple_New(3 + k);
  if (!out) throw python_error();
  PyTuple_SET_ITEM(out, 0, wrap(gx));
  PyTuple_SET_ITEM(out, 1, wrap(qxt));
  PyTuple_SET_ITEM(out, 2, wrap(sxt));
  for (Py_ssize_t i = 0; i < k; ++i) PyTuple_SET_ITEM(out, 3 + i, wrap(gw[i]));
  return out;
  END_HANDLE_TH_ERRORS
}

// swiglu_fwd(x, w1, w3, w2, qx, sx, want_x_col, want_h_col, want_h, algo)
//   -> (y, h1, h3, row amax of w1, of w3, of w2, h, col amax of x, of h) or None.  qx / sx: x already quantised (no col amax then).
PyObject *swiglu_fwd(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 10) throw std::runtime_error("swiglu_fwd: 10 arguments");
  if (!tensors(args, 6)) Py_RETURN_NONE;
  const Tensor x = arg(args[0]), w1 = arg(args[1]), w3 = arg(args[2]), w2 = arg(args[3]), qx = arg(args[4]), sx = arg(args[5]);
  const bool want_x_col = truth(args[6]), want_h_col = truth(args[7]), want_h = truth(args[8]);
  const int algo = (int)PyLong_AsLongLong(args[9]);
  Rows rx, r1, r3, r2;
  if (!activation(x, rx)) Py_RETURN_NONE;
  const int device = x.get_device();
  if (!weight(w1, device, r1) || !weight(w3, device, r3) || !weight(w2, device, r2)) Py_RETURN_NONE;
  const int64_t M = rx.rows, K = rx.cols, F = r1.rows, D = r2.rows;
  if (r1.cols != K || r3.cols != K || r3.rows != F || r2.cols != F) Py_RETURN_NONE;
  const int64_t ldqx = qx.defined() ? fp8_rows(qx, M, K, device) : on_lines(K);
  if (!ldqx || (qx.defined() && !dense(sx, at::kFloat, M, device))) Py_RETURN_NONE;
  Tensor y, h1, h3, h, amax1, amax3, amax2, x_col, h_col;
  {
    pybind11::gil_scoped_release no_gil;
    const auto o = x.options();
    void *stream = stream_of(device);
    amax1 = at::empty({F, 1}, o), amax3 = at::empty({F, 1}, o), amax2 = at::empty({D, 1}, o);
    {
      Arena a;
      const Quantised q1(a, F, K, F), q3(a, F, K, F), q(a, qx.defined() ? 0 : M, K, M);
      a.make(x);
      if (!qx.defined()) cast_activation(x, rx, want_x_col, a.p(q.q), q.ld, a.f(q.s), x_col, stream);
      const void *at_x = qx.defined() ? qx.const_data_ptr() : a.p(q.q);
      const float *scale_x = qx.defined() ? sx.const_data_ptr<float>() : a.f(q.s);
      const l8_cast_rowwise_item items[2] = {{r1.p, F, r1.ld, a.p(q1.q), q1.ld, a.f(q1.s), amax1.mutable_data_ptr()},
                                             {r3.p, F, r3.ld, a.p(q3.q), q3.ld, a.f(q3.s), amax3.mutable_data_ptr()}};
      check(lib.l8_cast_rowwise_many(items, 2, K, stream), "l8_cast_rowwise_many");
      h1 = at::empty({M, F}, o), h3 = at::empty({M, F}, o);
      check(lib.l8_gemm_nt(at_x, a.p(q1.q), M, F, K, ldqx, q1.ld, scale_x, L8_SCALE_ROW, a.f(q1.s), L8_SCALE_ROW, nullptr, h1.mutable_data_ptr(), F, algo, stream), "l8_gemm_nt");
      check(lib.l8_gemm_nt(at_x, a.p(q3.q), M, F, K, ldqx, q3.ld, scale_x, L8_SCALE_ROW, a.f(q3.s), L8_SCALE_ROW, nullptr, h3.mutable_data_ptr(), F, algo, stream), "l8_gemm_nt");
    }
    if (want_h) h = at::empty({M, F}, o);
    if (want_h_col) h_col = at::empty({F}, o.dtype(at::kFloat));
    Arena a;
    const Quantised qh(a, M, F, M), q2(a, D, F, D);
    const int64_t amax_h = a.add(M * 2), ws_bytes = want_h_col ? lib.l8_swiglu_workspace(M, F) / 2 : 0, ws = a.add(ws_bytes);
    a.make(x);
    check(lib.l8_swiglu_cast_rowwise(h1.const_data_ptr(), h3.const_data_ptr(), M, F, F, F, want_h ? h.mutable_data_ptr() : nullptr, F, a.p(qh.q), qh.ld, a.f(qh.s),
                                     a.p(amax_h), want_h_col ? h_col.mutable_data_ptr<float>() : nullptr, ws_bytes ? a.p(ws) : nullptr, ws_bytes, stream), "l8_swiglu_cast_rowwise");
    check(lib.l8_cast_rowwise(r2.p, D, F, r2.ld, a.p(q2.q), q2.ld, a.f(q2.s), amax2.mutable_data_ptr(), nullptr, nullptr, 0, stream), "l8_cast_rowwise");
    y = at::empty({M, D}, o);
    check(lib.l8_gemm_nt(a.p(qh.q), a.p(q2.q), M, D, F, qh.ld, q2.ld, a.f(qh.s), L8_SCALE_ROW, a.f(q2.s), L8_SCALE_ROW, nullptr, y.mutable_data_ptr(), D, algo, stream), "l8_gemm_nt");
  }
  return tuple_of({y, h1, h3, amax1, amax3, amax2, h, x_col, h_col});
  END_HANDLE_TH_ERRORS
}

// swiglu_bwd(gy, x, w1, w3, w2, h1, h3, row amax of w1, of w3, of w2, col amax of x, of h, algo) -> (grad x, grad w1, grad w3, grad w2)
// or None: every weight and x learn, the operands of the weight gradients are made from the gate's inputs.
PyObject *swiglu_bwd(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 13) throw std::runtime_error("swiglu_bwd: 13 arguments");
  if (!tensors(args, 12)) Py_RETURN_NONE;
  const Tensor gy = arg(args[0]), x = arg(args[1]), w1 = arg(args[2]), w3 = arg(args[3]), w2 = arg(args[4]), h1 = arg(args[5]), h3 = arg(args[6]), amax1 = arg(args[7]),
               amax3 = arg(args[8]), amax2 = arg(args[9]), x_col = arg(args[10]), h_col = arg(args[11]);
  const int algo = (int)PyLong_AsLongLong(args[12]);
  Rows rx, rg, r1, r3, r2, rh1, rh3;
  if (!activation(x, rx) || !activation(gy, rg) || !activation(h1, rh1) || !activation(h3, rh3)) Py_RETURN_NONE;
  const int device = x.get_device();
  if (gy.get_device() != device || h1.get_device() != device || h3.get_device() != device || !weight(w1, device, r1) || !weight(w3, device, r3) || !weight(w2, device, r2))
    Py_RETURN_NONE;
  const int64_t M = rx.rows, K = rx.cols, F = r1.rows, D = r2.rows, padded = (M + 15) / 16 * 16;
  if (rg.rows != M || rg.cols != D || rh1.rows != M || rh1.cols != F || rh3.rows != M || rh3.cols != F || r1.cols != K || r3.cols != K || r3.rows != F || r2.cols != F ||
      !amax1.defined() || !amax3.defined() || !amax2.defined() || !listed(amax1, F, device) || !listed(amax3, F, device) || !listed(amax2, D, device) ||
      !dense(x_col, at::kFloat, K, device) || !dense(h_col, at::kFloat, F, device))
    Py_RETURN_NONE;
  Tensor gx, gw1, gw3, gw2;
  {
    pybind11::gil_scoped_release no_gil;
    const auto o = x.options();
    void *stream = stream_of(device);
    Arena cols, hidden;  // column amaxes and the gradient of h: kept through the phases
    const int64_t gy_col = cols.add(D * 4), g1_col = cols.add(F * 4), g3_col = cols.add(F * 4), dh = hidden.add(M * F * 2);
    cols.make(x);
    hidden.make(x);
    {
      Arena a;
      const Quantised qgy(a, M, D, M), qw2(a, F, D, 1);
      const int64_t ws_bytes = lib.l8_cast_rowwise_workspace(M, D), ws = a.add(ws_bytes);
      a.make(x);
      check(lib.l8_cast_rowwise(rg.p, M, D, rg.ld, a.p(qgy.q), qgy.ld, a.f(qgy.s), nullptr, cols.f(gy_col), a.p(ws), ws_bytes, stream), "l8_cast_rowwise");
      check(lib.l8_cast_tensorwise_t_rows(r2.p, D, F, r2.ld, amax2.const_data_ptr(), D, a.p(qw2.q), qw2.ld, a.f(qw2.s), stream), "l8_cast_tensorwise_t_rows");
      check(lib.l8_gemm_nt(a.p(qgy.q), a.p(qw2.q), M, F, D, qgy.ld, qw2.ld, a.f(qgy.s), L8_SCALE_ROW, a.f(qw2.s), L8_SCALE_SCALAR, nullptr, hidden.p(dh), F, algo, stream),
            "l8_gemm_nt");
    }
    {
      Arena a;
      const Quantised q1(a, M, F, M), q3(a, M, F, M), qw1(a, K, F, 1), qw3(a, K, F, 1);
      const int64_t ws_bytes = lib.l8_swiglu_workspace(M, F), ws = a.add(ws_bytes);
      a.make(x);
      check(lib.l8_swiglu_bwd_cast_rowwise_q(hidden.p(dh), rh1.p, rh3.p, M, F, F, rh1.ld, rh3.ld, a.p(q1.q), a.p(q3.q), q1.ld, a.f(q1.s), a.f(q3.s), cols.f(g1_col),
                                             cols.f(g3_col), a.p(ws), ws_bytes, stream), "l8_swiglu_bwd_cast_rowwise");
      const l8_cast_transposed_item weights[2] = {by_tensor(r1, amax1, a, qw1), by_tensor(r3, amax3, a, qw3)};
      check(lib.l8_cast_transposed_many(weights, 2, stream), "l8_cast_transposed_many");
      gx = at::empty({M, K}, o);
      const l8_gemm_term terms[2] = {{a.p(q1.q), a.p(qw1.q), F, q1.ld, qw1.ld, a.f(q1.s), a.f(qw1.s)}, {a.p(q3.q), a.p(qw3.q), F, q3.ld, qw3.ld, a.f(q3.s), a.f(qw3.s)}};
      check(lib.l8_gemm_nt_sum(terms, 2, M, K, gx.mutable_data_ptr(), K, algo, stream), "l8_gemm_nt_sum");
    }
    Arena a;
    const Quantised qx(a, K, padded, K), qgy(a, D, padded, D), q1(a, F, padded, F), q3(a, F, padded, F), qh(a, F, padded, F);
    a.make(x);
    const l8_cast_transposed_item casts[2] = {by_columns(rx, x_col.const_data_ptr<float>(), a, qx), by_columns(rg, cols.f(gy_col), a, qgy)};
    check(lib.l8_cast_transposed_many(casts, 2, stream), "l8_cast_transposed_many");
    check(lib.l8_swiglu_bwd_cast_transposed(hidden.p(dh), rh1.p, rh3.p, M, F, F, rh1.ld, rh3.ld, cols.f(g1_col), cols.f(g3_col), h_col.const_data_ptr<float>(), a.p(q1.q),
                                            a.p(q3.q), a.p(qh.q), q1.ld, padded, a.f(q1.s), a.f(q3.s), a.f(qh.s), stream), "l8_swiglu_bwd_cast_transposed");
    hidden.t = Tensor();
    gw1 = at::empty({F, K}, o), gw3 = at::empty({F, K}, o), gw2 = at::empty({D, F}, o);
    const l8_gemm_part parts[2] = {{a.p(q1.q), F, a.f(q1.s), gw1.mutable_data_ptr()}, {a.p(q3.q), F, a.f(q3.s), gw3.mutable_data_ptr()}};
    check(lib.l8_gemm_nt_multi(parts, 2, a.p(qx.q), K, padded, q1.ld, qx.ld, a.f(qx.s), L8_SCALE_ROW, K, algo, stream), "l8_gemm_nt_multi");
    check(lib.l8_gemm_nt(a.p(qgy.q), a.p(qh.q), D, F, padded, qgy.ld, qh.ld, a.f(qgy.s), L8_SCALE_ROW, a.f(qh.s), L8_SCALE_ROW, nullptr, gw2.mutable_data_ptr(), F, algo, stream),
          "l8_gemm_nt");
  }
  return tuple_of({gx, gw1, gw3, gw2});
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
    {"rmsnorm_fwd", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(rmsnorm_fwd)), METH_FASTCALL, nullptr},
    {"rmsnorm_bwd", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(rmsnorm_bwd)), METH_FASTCALL, nullptr},
    {"qkv_fwd", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(qkv_fwd)), METH_FASTCALL, nullptr},
    {"shared_bwd", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(shared_bwd)), METH_FASTCALL, nullptr},
    {"swiglu_fwd", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(swiglu_fwd)), METH_FASTCALL, nullptr},
    {"swiglu_bwd", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(swiglu_bwd)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native() { return PyModule_Create(&module_def); }

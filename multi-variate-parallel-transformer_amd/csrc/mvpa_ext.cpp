// Python binding of the launch-bound paths: tensors in, launches of libmvpa_hip.so out.
//
// A call through ctypes takes apart its tensors in the interpreter, one attribute at a time (about 18 us
// for the attention operator, and 100 us per block of a stack); here it costs a few.  Nothing is
// computed in this file: every function fills an argument block of the C ABI (include/mvpa_hip.h),
// allocates the results with torch's caching allocator and enqueues on torch's current stream.
// Functions return an int status where the library refused, for the Python layer to raise on.
#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <c10/util/accumulate.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/grad_mode.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "mvpa_hip.h"

namespace {

using at::Tensor;

void* current_stream() { return (void*)c10::hip::getCurrentHIPStream().stream(); }

bool is_none(PyObject* o) { return o == nullptr || o == Py_None; }

const Tensor& tensor_of(PyObject* o) {
  TORCH_CHECK_TYPE(THPVariable_Check(o), "expected a tensor");
  return THPVariable_Unpack(o);
}

int dtype_code(at::ScalarType t) {
  if (t == at::kFloat) return MVPA_F32;
  if (t == at::kBFloat16) return MVPA_BF16;
  TORCH_CHECK_TYPE(t == at::kHalf, "libmvpa_hip supports float32, bfloat16 and float16");
  return MVPA_F16;
}

void on_gpu(const Tensor& t) {
  TORCH_CHECK(t.is_cuda(), "libmvpa_hip ops need tensors in GPU memory (there is no CPU path)");
}

// t itself where it already has the type and is contiguous
Tensor as_operand(const Tensor& t, at::ScalarType dt) {
  on_gpu(t);
  if (t.scalar_type() == dt && t.is_contiguous()) return t;
  return t.to(dt).contiguous();
}

// false, with an AssertionError set, where a shape is refused
bool require(bool ok, const char* what) {
  if (!ok) PyErr_SetString(PyExc_AssertionError, what);
  return ok;
}

// ---- the attention operator -----------------------------------------------------------------
// forward(q, k, v, u, vb, z, k_time, k_chan, out, chan_valid, key_bias, sm_scale, window, flags,
//         kernel, return_lse) -> out | (out, lse) | status
PyObject* py_forward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n == 16, "forward takes 16 arguments");
  const Tensor &q = tensor_of(args[0]), &k = tensor_of(args[1]), &v = tensor_of(args[2]);
  on_gpu(q);
  on_gpu(k);
  on_gpu(v);
  TORCH_CHECK(q.dim() == 4 && k.dim() == 4 && v.dim() == 4, "q, k and v have four dimensions");
  const Tensor &kt0 = tensor_of(args[6]), &kc0 = tensor_of(args[7]);
  TORCH_CHECK(kt0.dim() >= 2 && kc0.dim() >= 2, "k_time and k_chan are [.., T, Dh] and [.., C, Dh]");
  const int64_t rows = kt0.size(-2) * kc0.size(-2), hkv = k.size(1), dh = q.size(3);
  if (!require(k.size(3) == dh && v.size(3) == dh, "head dims of q, k, v differ") ||
      !require(k.size(2) == rows && v.size(2) == rows, "k and v must hold T*C rows") ||
      !require(q.size(2) == rows, "q must hold T*C rows (C with last_step_only)") ||
      !require(v.size(1) == hkv && k.size(0) == q.size(0) && v.size(0) == q.size(0), "q, k, v disagree on B or Hkv") ||
      !require(kt0.numel() == hkv * kt0.size(-2) * dh && kc0.numel() == hkv * kc0.size(-2) * dh,
               "k_time and k_chan must hold Hkv tables of Dh columns"))
    return nullptr;
  for (int i = 3; i < 6; ++i)
    if (!require(tensor_of(args[i]).numel() == hkv * dh, "u, vb, z must hold Hkv rows of Dh")) return nullptr;
  if (!is_none(args[8])) {
    const Tensor& o = tensor_of(args[8]);
    on_gpu(o);
    if (!require(o.dim() == 4 && o.sizes() == q.sizes() && o.scalar_type() == q.scalar_type(), "out must match q")) return nullptr;
  }
  if (!is_none(args[9]) &&
      !require(tensor_of(args[9]).dim() == 2 && tensor_of(args[9]).size(0) == q.size(0) && tensor_of(args[9]).size(1) == kc0.size(-2),
               "chan_valid is [B, C]"))
    return nullptr;
  if (!is_none(args[10]) &&
      !require(tensor_of(args[10]).dim() == 2 && tensor_of(args[10]).size(0) == q.size(0) && tensor_of(args[10]).size(1) == rows,
               "key_bias is [B, N]"))
    return nullptr;
  const auto dt = q.scalar_type();
  at::AutoDispatchBelowADInplaceOrView guard;
  const Tensor u = as_operand(tensor_of(args[3]), dt), vb = as_operand(tensor_of(args[4]), dt),
               z = as_operand(tensor_of(args[5]), dt), kt = as_operand(tensor_of(args[6]), dt),
               kc = as_operand(tensor_of(args[7]), dt);
  mvpa_fwd_args a;
  std::memset(&a, 0, sizeof(a));
  a.struct_size = sizeof(a);
  a.dtype = dtype_code(dt);
  a.window = (int32_t)PyLong_AsLong(args[12]);
  a.flags = (uint32_t)PyLong_AsUnsignedLong(args[13]);
  a.kernel = (int32_t)PyLong_AsLong(args[14]);
  a.sm_scale = (float)PyFloat_AsDouble(args[11]);
  if (PyErr_Occurred()) return nullptr;
  a.B = (int32_t)q.size(0);
  a.H = (int32_t)q.size(1);
  a.Dh = (int32_t)q.size(3);
  a.Hkv = (int32_t)k.size(1);
  a.T = (int32_t)kt.size(-2);
  a.C = (int32_t)kc.size(-2);
  Tensor out = is_none(args[8]) ? at::empty(q.sizes(), q.options(), at::MemoryFormat::Contiguous) : tensor_of(args[8]);
  TORCH_CHECK_VALUE(q.stride(3) == 1 && k.stride(3) == 1 && v.stride(3) == 1 && out.stride(3) == 1,
                    "q, k, v, out: last dim must be contiguous");
  a.q = q.data_ptr();
  a.k = k.data_ptr();
  a.v = v.data_ptr();
  a.o = out.data_ptr();
  a.q_stride_b = q.stride(0); a.q_stride_h = q.stride(1); a.q_stride_n = q.stride(2);
  a.k_stride_b = k.stride(0); a.k_stride_h = k.stride(1); a.k_stride_n = k.stride(2);
  a.v_stride_b = v.stride(0); a.v_stride_h = v.stride(1); a.v_stride_n = v.stride(2);
  a.o_stride_b = out.stride(0); a.o_stride_h = out.stride(1); a.o_stride_n = out.stride(2);
  a.bias_u = u.data_ptr();
  a.bias_v = vb.data_ptr();
  a.bias_z = z.data_ptr();
  a.k_time = kt.data_ptr();
  a.k_chan = kc.data_ptr();
  Tensor cv, kb, lse;
  if (!is_none(args[9])) {
    cv = as_operand(tensor_of(args[9]), tensor_of(args[9]).scalar_type() == at::kBool ? at::kBool : at::kByte);
    a.chan_valid = (const uint8_t*)cv.data_ptr();
  }
  if (!is_none(args[10])) {
    kb = as_operand(tensor_of(args[10]), at::kFloat);
    a.key_bias = (const float*)kb.data_ptr();
  }
  const bool want_lse = args[15] == Py_True;
  if (want_lse) {
    lse = at::empty({q.size(0), q.size(1), q.size(2)}, q.options().dtype(at::kFloat));
    a.lse = (float*)lse.data_ptr();
  }
  const int st = mvpa_forward(&a, current_stream());
  if (st != MVPA_OK) return PyLong_FromLong(st);
  if (!want_lse) return THPVariable_Wrap(out);
  PyObject* r = PyTuple_New(2);
  PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(out));
  PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(lse));
  return r;
  END_HANDLE_TH_ERRORS
}

// backward(q, k, v, o, d_o, lse, u, vb, z, k_time, k_chan, chan_valid, sm_scale, window, flags[, dq, dk, dv])
//   -> (dq, du, dvb, dz, dk, dk_time, dk_chan, dv) in bf16 | status.  dq, dk, dv: views that receive the gradients
PyObject* py_backward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n == 15 || n == 18, "backward takes 15 or 18 arguments");
  at::AutoDispatchBelowADInplaceOrView guard;
  const auto dt = at::kBFloat16;
  const Tensor &q = tensor_of(args[0]), &k = tensor_of(args[1]), &v = tensor_of(args[2]), &o = tensor_of(args[3]);
  Tensor d_o = tensor_of(args[4]);
  for (const Tensor* t : {&q, &k, &v, &o, (const Tensor*)&d_o}) {
    on_gpu(*t);
    TORCH_CHECK(t->dim() == 4 && t->scalar_type() == dt, "backward: q, k, v, o, d_o are bf16 with four dimensions");
  }
  TORCH_CHECK(o.sizes() == q.sizes() && d_o.sizes() == q.sizes() && k.sizes() == v.sizes(), "backward: shapes differ");
  if (d_o.stride(3) != 1 || ((d_o.stride(0) | d_o.stride(1) | d_o.stride(2)) & 7)) d_o = d_o.contiguous();
  const Tensor lse = as_operand(tensor_of(args[5]), at::kFloat);
  const Tensor u = as_operand(tensor_of(args[6]), dt), vb = as_operand(tensor_of(args[7]), dt),
               z = as_operand(tensor_of(args[8]), dt), kt = as_operand(tensor_of(args[9]), dt),
               kc = as_operand(tensor_of(args[10]), dt);
  mvpa_bwd_args a;
  std::memset(&a, 0, sizeof(a));
  a.struct_size = sizeof(a);
  a.dtype = MVPA_BF16;
  a.sm_scale = (float)PyFloat_AsDouble(args[12]);
  a.window = (int32_t)PyLong_AsLong(args[13]);
  a.flags = (uint32_t)PyLong_AsUnsignedLong(args[14]);
  if (PyErr_Occurred()) return nullptr;
  a.B = (int32_t)q.size(0);
  a.H = (int32_t)q.size(1);
  a.Dh = (int32_t)q.size(3);
  a.Hkv = (int32_t)k.size(1);
  a.T = (int32_t)kt.size(-2);
  a.C = (int32_t)kc.size(-2);
  TORCH_CHECK(q.size(2) == (int64_t)a.T * a.C && k.size(2) == q.size(2) && lse.numel() == q.numel() / a.Dh &&
                  u.numel() == (int64_t)a.Hkv * a.Dh && kt.numel() == (int64_t)a.Hkv * a.T * a.Dh &&
                  kc.numel() == (int64_t)a.Hkv * a.C * a.Dh,
              "backward: shapes differ");
  TORCH_CHECK_VALUE(q.stride(3) == 1 && k.stride(3) == 1 && v.stride(3) == 1 && o.stride(3) == 1,
                    "q, k, v, o: last dim must be contiguous");
  a.q = q.data_ptr(); a.k = k.data_ptr(); a.v = v.data_ptr(); a.o = o.data_ptr(); a.d_o = d_o.data_ptr();
  a.q_stride_b = q.stride(0); a.q_stride_h = q.stride(1); a.q_stride_n = q.stride(2);
  a.k_stride_b = k.stride(0); a.k_stride_h = k.stride(1); a.k_stride_n = k.stride(2);
  a.v_stride_b = v.stride(0); a.v_stride_h = v.stride(1); a.v_stride_n = v.stride(2);
  a.o_stride_b = o.stride(0); a.o_stride_h = o.stride(1); a.o_stride_n = o.stride(2);
  a.do_stride_b = d_o.stride(0); a.do_stride_h = d_o.stride(1); a.do_stride_n = d_o.stride(2);
  a.bias_u = u.data_ptr(); a.bias_v = vb.data_ptr(); a.bias_z = z.data_ptr();
  a.k_time = kt.data_ptr(); a.k_chan = kc.data_ptr();
  a.lse = (const float*)lse.data_ptr();
  Tensor cv;
  if (!is_none(args[11])) {
    cv = as_operand(tensor_of(args[11]), tensor_of(args[11]).scalar_type() == at::kBool ? at::kBool : at::kByte);
    a.chan_valid = (const uint8_t*)cv.data_ptr();
  }
  const auto opt = q.options();
  Tensor dq, dk, dv;
  if (n == 18) {
    dq = tensor_of(args[15]); dk = tensor_of(args[16]); dv = tensor_of(args[17]);
    for (const Tensor* t : {(const Tensor*)&dq, (const Tensor*)&dk, (const Tensor*)&dv}) {
      on_gpu(*t);
      TORCH_CHECK(t->scalar_type() == dt && t->dim() == 4 && t->stride(3) == 1, "backward: dq, dk, dv are bf16 with unit last stride");
    }
    TORCH_CHECK(dq.sizes() == q.sizes() && dk.sizes() == k.sizes() && dv.sizes() == k.sizes(), "backward: shapes differ");
  } else {
    dq = at::empty(q.sizes(), opt, at::MemoryFormat::Contiguous);
    dk = at::empty(k.sizes(), opt, at::MemoryFormat::Contiguous);
    dv = at::empty(v.sizes(), opt, at::MemoryFormat::Contiguous);
  }
  Tensor du = at::empty(u.sizes(), opt), dvb = at::empty(vb.sizes(), opt), dz = at::empty(z.sizes(), opt),
         dkt = at::empty(kt.sizes(), opt), dkc = at::empty(kc.sizes(), opt);
  mvpa_bwd_grads g;
  std::memset(&g, 0, sizeof(g));
  g.struct_size = sizeof(g);
  g.dq = dq.data_ptr(); g.dk = dk.data_ptr(); g.dv = dv.data_ptr();
  g.dq_stride_b = dq.stride(0); g.dq_stride_h = dq.stride(1); g.dq_stride_n = dq.stride(2);
  g.dk_stride_b = dk.stride(0); g.dk_stride_h = dk.stride(1); g.dk_stride_n = dk.stride(2);
  g.dv_stride_b = dv.stride(0); g.dv_stride_h = dv.stride(1); g.dv_stride_n = dv.stride(2);
  g.dbias_u = du.data_ptr(); g.dbias_v = dvb.data_ptr(); g.dbias_z = dz.data_ptr();
  g.dk_time = dkt.data_ptr(); g.dk_chan = dkc.data_ptr();
  const int64_t bytes = (int64_t)mvpa_backward_full_ws_bytes(&a);
  Tensor ws = at::empty({bytes}, opt.dtype(at::kByte));
  const int st = mvpa_backward_full(&a, &g, ws.data_ptr(), (size_t)bytes, current_stream());
  if (st != MVPA_OK) return PyLong_FromLong(st);
  PyObject* r = PyTuple_New(8);
  int i = 0;
  for (Tensor* t : {&dq, &du, &dvb, &dz, &dk, &dkt, &dkc, &dv}) PyTuple_SET_ITEM(r, i++, THPVariable_Wrap(*t));
  return r;
  END_HANDLE_TH_ERRORS
}

// ---- dense ops ------------------------------------------------------------------------------
// linear(x, w) -> x @ w^T, bf16, plain product | status
PyObject* py_linear(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n == 2, "linear takes x and w");
  Tensor x = tensor_of(args[0]);
  const Tensor& w = tensor_of(args[1]);
  on_gpu(x);
  on_gpu(w);
  TORCH_CHECK_TYPE(x.scalar_type() == at::kBFloat16 && w.scalar_type() == at::kBFloat16, "linear: bf16 only");
  at::AutoDispatchBelowADInplaceOrView guard;
  const int64_t K = x.size(-1), N = w.size(0);
  if (!require(w.dim() == 2 && w.size(1) == K && w.stride(1) == 1, "linear: w is [N, K] with unit last stride")) return nullptr;
  std::vector<int64_t> shape(x.sizes().begin(), x.sizes().end());
  shape.back() = N;
  if (!(x.dim() == 2 && x.stride(1) == 1)) x = x.contiguous();
  const int64_t M = c10::multiply_integers(x.sizes().slice(0, x.dim() - 1)), ldx = x.dim() == 2 ? x.stride(0) : K;
  Tensor y = at::empty(shape, x.options());
  int st;
  if (M <= 128 && K >= 1536 && N <= 4096) {
    Tensor ws = at::empty({(int64_t)mvpa_linear_splitk_ws_bytes(M, N, K, 0)}, x.options().dtype(at::kByte));
    st = mvpa_linear_bf16_splitk(x.data_ptr(), w.data_ptr(), y.data_ptr(), M, N, K, ldx, w.stride(0), N, 0,
                                 ws.data_ptr(), (size_t)ws.numel(), current_stream());
  } else {
    st = mvpa_linear_bf16(x.data_ptr(), w.data_ptr(), y.data_ptr(), M, N, K, ldx, w.stride(0), N, 0, current_stream());
  }
  return st == MVPA_OK ? THPVariable_Wrap(y) : PyLong_FromLong(st);
  END_HANDLE_TH_ERRORS
}

// linear_wgrad(dy [M, N], x [M, K]) -> dy^T x | status
PyObject* py_linear_wgrad(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n == 2, "linear_wgrad takes dy and x");
  const Tensor &dy = tensor_of(args[0]), &x = tensor_of(args[1]);
  on_gpu(dy);
  on_gpu(x);
  TORCH_CHECK(dy.dim() == 2 && x.dim() == 2 && dy.size(0) == x.size(0) && dy.scalar_type() == at::kBFloat16 &&
                  x.scalar_type() == at::kBFloat16,
              "linear_wgrad: bf16 rows");
  TORCH_CHECK(dy.device() == x.device(), "linear_wgrad: dy and x on one GPU");
  const int64_t M = dy.size(0), N = dy.size(1), K = x.size(1);
  if (dy.stride(1) != 1 || x.stride(1) != 1 || M == 0) return PyLong_FromLong(MVPA_ERR_UNSUPPORTED);
  at::AutoDispatchBelowADInplaceOrView guard;
  Tensor dw = at::empty({N, K}, x.options()), ws;
  const size_t bytes = mvpa_linear_wgrad_ws_bytes(M, N, K);
  if (bytes) ws = at::empty({(int64_t)bytes}, x.options().dtype(at::kByte));
  const int st = mvpa_linear_wgrad_bf16(dy.data_ptr(), x.data_ptr(), dw.data_ptr(), M, N, K, dy.stride(0), x.stride(0), K,
                                        bytes ? ws.data_ptr() : nullptr, bytes, current_stream());
  return st == MVPA_OK ? THPVariable_Wrap(dw) : PyLong_FromLong(st);
  END_HANDLE_TH_ERRORS
}

// linear_nn(dy [M, K], w [K, N]) -> dy w | status
PyObject* py_linear_nn(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n == 2, "linear_nn takes dy and w");
  const Tensor &dy = tensor_of(args[0]), &w = tensor_of(args[1]);
  on_gpu(dy);
  on_gpu(w);
  TORCH_CHECK(dy.dim() == 2 && w.dim() == 2 && dy.size(1) == w.size(0) && dy.scalar_type() == at::kBFloat16 &&
                  w.scalar_type() == at::kBFloat16,
              "linear_nn: bf16 matrices");
  TORCH_CHECK(dy.device() == w.device(), "linear_nn: dy and w on one GPU");
  const int64_t M = dy.size(0), K = dy.size(1), N = w.size(1);
  if (dy.stride(1) != 1 || w.stride(1) != 1 || M == 0) return PyLong_FromLong(MVPA_ERR_UNSUPPORTED);
  at::AutoDispatchBelowADInplaceOrView guard;
  Tensor dx = at::empty({M, N}, dy.options());
  const int st = mvpa_linear_bf16_nn(dy.data_ptr(), w.data_ptr(), dx.data_ptr(), M, N, K, dy.stride(0), w.stride(0), N, current_stream());
  return st == MVPA_OK ? THPVariable_Wrap(dx) : PyLong_FromLong(st);
  END_HANDLE_TH_ERRORS
}

// linear_nn2(dy [M, K0 + K1], w0 [K0, N], w1 [K1, N]) -> dy [w0; w1] | status
PyObject* py_linear_nn2(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n == 3, "linear_nn2 takes dy and the two halves of w");
  const Tensor &dy = tensor_of(args[0]), &w0 = tensor_of(args[1]), &w1 = tensor_of(args[2]);
  on_gpu(dy);
  TORCH_CHECK(dy.dim() == 2 && w0.dim() == 2 && w1.dim() == 2 && w0.size(1) == w1.size(1) && dy.size(1) == w0.size(0) + w1.size(0) &&
                  dy.scalar_type() == at::kBFloat16 && w0.scalar_type() == at::kBFloat16 && w1.scalar_type() == at::kBFloat16,
              "linear_nn2: bf16 matrices");
  TORCH_CHECK(dy.device() == w0.device() && dy.device() == w1.device(), "linear_nn2: operands on one GPU");
  const int64_t M = dy.size(0), N = w0.size(1);
  if (dy.stride(1) != 1 || w0.stride(1) != 1 || w1.stride(1) != 1 || w0.stride(0) != w1.stride(0) || M == 0)
    return PyLong_FromLong(MVPA_ERR_UNSUPPORTED);
  at::AutoDispatchBelowADInplaceOrView guard;
  Tensor dx = at::empty({M, N}, dy.options());
  const int st = mvpa_linear_bf16_nn2(dy.data_ptr(), w0.data_ptr(), w1.data_ptr(), dx.data_ptr(), M, N, w0.size(0), w1.size(0),
                                      dy.stride(0), w0.stride(0), N, current_stream());
  return st == MVPA_OK ? THPVariable_Wrap(dx) : PyLong_FromLong(st);
  END_HANDLE_TH_ERRORS
}

// gated_rows(x [M, K], gate [N, K], up [N, K]) -> (x [gate; up]^T, silu(gate) up) | status
PyObject* py_gated_rows(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n == 3, "gated_rows takes x and two weights");
  const Tensor &x = tensor_of(args[0]), &g = tensor_of(args[1]), &u = tensor_of(args[2]);
  on_gpu(x);
  TORCH_CHECK(x.dim() == 2 && g.dim() == 2 && g.sizes() == u.sizes() && g.size(1) == x.size(1) && x.scalar_type() == at::kBFloat16 &&
                  g.scalar_type() == at::kBFloat16 && u.scalar_type() == at::kBFloat16 && x.device() == g.device() && x.device() == u.device(),
              "gated_rows: bf16 matrices on one GPU");
  const int64_t M = x.size(0), N = g.size(0);
  if (x.stride(1) != 1 || g.stride(1) != 1 || u.stride(1) != 1 || g.stride(0) != u.stride(0) || M == 0) return PyLong_FromLong(MVPA_ERR_UNSUPPORTED);
  at::AutoDispatchBelowADInplaceOrView guard;
  Tensor gu = at::empty({M, 2 * N}, x.options()), mid = at::empty({M, N}, x.options());
  const int st = mvpa_gated_rows_bf16(x.data_ptr(), g.data_ptr(), u.data_ptr(), gu.data_ptr(), mid.data_ptr(), M, N, x.size(1), x.stride(0),
                                      g.stride(0), current_stream());
  if (st != MVPA_OK) return PyLong_FromLong(st);
  PyObject* r = PyTuple_New(2);
  PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(gu));
  PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(mid));
  return r;
  END_HANDLE_TH_ERRORS
}

// gated_rows_backward(dy [M, K], down [K, N], gu [M, 2 N]) -> the gradient of gu | status
PyObject* py_gated_rows_backward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n == 3, "gated_rows_backward takes dy, the weight and the rows");
  const Tensor &dy = tensor_of(args[0]), &w = tensor_of(args[1]), &gu = tensor_of(args[2]);
  on_gpu(dy);
  TORCH_CHECK(dy.dim() == 2 && w.dim() == 2 && gu.dim() == 2 && dy.size(1) == w.size(0) && gu.size(0) == dy.size(0) &&
                  gu.size(1) == 2 * w.size(1) && gu.is_contiguous() && dy.scalar_type() == at::kBFloat16 &&
                  w.scalar_type() == at::kBFloat16 && gu.scalar_type() == at::kBFloat16 && dy.device() == w.device() && dy.device() == gu.device(),
              "gated_rows_backward: bf16 matrices on one GPU");
  const int64_t M = dy.size(0);
  if (dy.stride(1) != 1 || w.stride(1) != 1 || M == 0) return PyLong_FromLong(MVPA_ERR_UNSUPPORTED);
  at::AutoDispatchBelowADInplaceOrView guard;
  Tensor dgu = at::empty_like(gu);
  const int st = mvpa_gated_rows_backward_bf16(dy.data_ptr(), w.data_ptr(), gu.data_ptr(), dgu.data_ptr(), M, w.size(1), dy.size(1),
                                               dy.stride(0), w.stride(0), current_stream());
  return st == MVPA_OK ? THPVariable_Wrap(dgu) : PyLong_FromLong(st);
  END_HANDLE_TH_ERRORS
}

// as_operand, starting at a 16-byte boundary
Tensor aligned_operand(const Tensor& t, at::ScalarType dt) {
  Tensor r = as_operand(t, dt);
  return (uintptr_t)r.const_data_ptr() & 15 ? r.clone() : r;
}

bool f32_or_bf16(const Tensor& t) { return t.scalar_type() == at::kFloat || t.scalar_type() == at::kBFloat16; }

// encode(x [M, L] fp32, norm weight fp32, levels, dwt_size, pitch, eps) -> [M, pitch] bf16 | status
PyObject* py_encode(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n == 6, "encode takes 6 arguments");
  at::AutoDispatchBelowADInplaceOrView guard;
  const Tensor x = as_operand(tensor_of(args[0]), at::kFloat), w = as_operand(tensor_of(args[1]), at::kFloat);
  const long levels = PyLong_AsLong(args[2]), dwt = PyLong_AsLong(args[3]), pitch = PyLong_AsLong(args[4]);
  const double eps = PyFloat_AsDouble(args[5]);
  if (PyErr_Occurred()) return nullptr;
  Tensor y = at::empty({x.size(0), pitch}, x.options().dtype(at::kBFloat16));
  const int st = mvpa_wavedec_db4_rmsnorm((const float*)x.data_ptr(), (const float*)w.data_ptr(), y.data_ptr(), x.size(0),
                                          (int32_t)x.size(1), (int32_t)levels, (int32_t)dwt, pitch, (float)eps,
                                          current_stream());
  return st == MVPA_OK ? THPVariable_Wrap(y) : PyLong_FromLong(st);
  END_HANDLE_TH_ERRORS
}

// encode_saved(as encode) -> ([M, pitch] bf16, the coefficients [M, pitch] fp32, the row factors [M]) | status
PyObject* py_encode_saved(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n == 6, "encode_saved takes 6 arguments");
  at::AutoDispatchBelowADInplaceOrView guard;
  const Tensor x = as_operand(tensor_of(args[0]), at::kFloat), w = as_operand(tensor_of(args[1]), at::kFloat);
  const long levels = PyLong_AsLong(args[2]), dwt = PyLong_AsLong(args[3]), pitch = PyLong_AsLong(args[4]);
  const double eps = PyFloat_AsDouble(args[5]);
  if (PyErr_Occurred()) return nullptr;
  TORCH_CHECK(x.dim() == 2 && w.numel() == dwt && w.device() == x.device(), "encode_saved: rows of samples, a weight per coefficient on their GPU");
  Tensor y = at::empty({x.size(0), pitch}, x.options().dtype(at::kBFloat16));
  Tensor coeffs = at::empty({x.size(0), pitch}, x.options()), inv = at::empty({x.size(0)}, x.options());
  const int st = mvpa_wavedec_db4_rmsnorm_saved((const float*)x.data_ptr(), (const float*)w.data_ptr(), y.data_ptr(),
                                                (float*)coeffs.data_ptr(), (float*)inv.data_ptr(), x.size(0), (int32_t)x.size(1),
                                                (int32_t)levels, (int32_t)dwt, pitch, (float)eps, current_stream());
  if (st != MVPA_OK) return PyLong_FromLong(st);
  PyObject* r = PyTuple_New(3);
  PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(y));
  PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(coeffs));
  PyTuple_SET_ITEM(r, 2, THPVariable_Wrap(inv));
  return r;
  END_HANDLE_TH_ERRORS
}

// norm_dw(x [M, pitch] fp32, inv [M] fp32, dy [M, pitch] bf16, weight) -> the weight's gradient | status
PyObject* py_norm_dw(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n == 4, "norm_dw takes 4 arguments");
  at::AutoDispatchBelowADInplaceOrView guard;
  const Tensor x = aligned_operand(tensor_of(args[0]), at::kFloat), inv = as_operand(tensor_of(args[1]), at::kFloat);
  const Tensor dy = aligned_operand(tensor_of(args[2]), at::kBFloat16);
  const Tensor& w = tensor_of(args[3]);
  TORCH_CHECK_TYPE(f32_or_bf16(w), "norm_dw: fp32 or bf16");
  TORCH_CHECK(x.dim() == 2 && dy.sizes() == x.sizes() && inv.numel() == x.size(0) && w.numel() <= x.size(1) &&
              dy.device() == x.device() && inv.device() == x.device() && w.device() == x.device(), "norm_dw: operands differ");
  const int64_t rows = x.size(0);
  const int32_t cols = (int32_t)w.numel();
  Tensor dw = at::empty(w.sizes(), w.options());
  Tensor ws = at::empty({(int64_t)mvpa_norm_dw_ws_bytes(rows, cols)}, x.options().dtype(at::kByte));
  const int st = mvpa_norm_dw((const float*)x.data_ptr(), (const float*)inv.data_ptr(), dy.data_ptr(), dw.data_ptr(), ws.data_ptr(),
                              rows, cols, x.size(1), x.size(1), w.scalar_type() == at::kFloat, current_stream());   // (one row may have any stride)
  return st == MVPA_OK ? THPVariable_Wrap(dw) : PyLong_FromLong(st);
  END_HANDLE_TH_ERRORS
}

// mean_rows(x [G, R, E] bf16, unit last stride) -> [G, E] | status
PyObject* py_mean_rows(PyObject*, PyObject* arg) {
  HANDLE_TH_ERRORS
  const Tensor& x = tensor_of(arg);
  on_gpu(x);
  TORCH_CHECK(x.dim() == 3 && x.stride(2) == 1 && x.scalar_type() == at::kBFloat16, "mean_rows: bf16 [G, R, E]");
  at::AutoDispatchBelowADInplaceOrView guard;
  Tensor y = at::empty({x.size(0), x.size(2)}, x.options());
  const int st = mvpa_mean_rows_bf16(x.data_ptr(), y.data_ptr(), x.size(0), x.size(1), (int32_t)x.size(2), x.stride(1),
                                     x.stride(0), current_stream());
  return st == MVPA_OK ? THPVariable_Wrap(y) : PyLong_FromLong(st);
  END_HANDLE_TH_ERRORS
}

// ---- row operations of the training path -------------------------------------------------------
// norm_backward(x, weight, dy, res | None, eps, need_dx, need_dw) -> (dx | None, dw | None) | status
PyObject* py_norm_backward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n == 7, "norm_backward takes 7 arguments");
  at::AutoDispatchBelowADInplaceOrView guard;
  const Tensor x = as_operand(tensor_of(args[0]), tensor_of(args[0]).scalar_type());
  const Tensor w = as_operand(tensor_of(args[1]), tensor_of(args[1]).scalar_type());
  const Tensor dy = as_operand(tensor_of(args[2]), at::kBFloat16);
  TORCH_CHECK_TYPE(f32_or_bf16(x) && f32_or_bf16(w), "norm_backward: fp32 or bf16");
  const int64_t cols = x.size(-1), rows = x.numel() / std::max<int64_t>(cols, 1);
  Tensor res, dx, dw, ws;
  if (!is_none(args[3])) res = as_operand(tensor_of(args[3]), x.scalar_type());
  TORCH_CHECK(dy.sizes() == x.sizes() && w.numel() == cols && (!res.defined() || res.sizes() == x.sizes()),
              "norm_backward: shapes differ");
  const double eps = PyFloat_AsDouble(args[4]);
  if (PyErr_Occurred()) return nullptr;
  if (args[5] == Py_True) dx = at::empty_like(x);
  if (args[6] == Py_True) {
    dw = at::empty(w.sizes(), w.options());
    ws = at::empty({(int64_t)mvpa_rmsnorm_backward_ws_bytes(rows, (int32_t)cols)}, x.options().dtype(at::kByte));
  }
  const int st = mvpa_rmsnorm_backward(x.data_ptr(), w.data_ptr(), dy.data_ptr(), res.defined() ? res.data_ptr() : nullptr,
                                       dx.defined() ? dx.data_ptr() : nullptr, dw.defined() ? dw.data_ptr() : nullptr,
                                       ws.defined() ? ws.data_ptr() : nullptr, rows, (int32_t)cols, (float)eps,
                                       x.scalar_type() == at::kFloat, w.scalar_type() == at::kFloat, current_stream());
  if (st != MVPA_OK) return PyLong_FromLong(st);
  PyObject* r = PyTuple_New(2);
  PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(dx));           // an undefined tensor comes out as None
  PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(dw));
  return r;
  END_HANDLE_TH_ERRORS
}

// silu_gate(gu [.., 2n]) -> [.., n];  silu_gate(gu, d [.., n]) -> the gradient of gu | status
PyObject* py_silu_gate(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n == 1 || n == 2, "silu_gate takes gu and, for the backward, the gradient");
  at::AutoDispatchBelowADInplaceOrView guard;
  const Tensor gu = aligned_operand(tensor_of(args[0]), at::kBFloat16);
  TORCH_CHECK(gu.dim() >= 1 && gu.size(-1) % 2 == 0 && gu.numel() > 0, "silu_gate: rows of gate and up");
  const int64_t cols = gu.size(-1) / 2, rows = gu.numel() / (2 * cols);
  std::vector<int64_t> shape(gu.sizes().begin(), gu.sizes().end());
  shape.back() = cols;
  Tensor y;
  int st;
  if (n == 1) {
    y = at::empty(shape, gu.options());
    st = mvpa_silu_gate_bf16(gu.data_ptr(), y.data_ptr(), rows, (int32_t)cols, current_stream());
  } else {
    const Tensor d = aligned_operand(tensor_of(args[1]), at::kBFloat16);
    TORCH_CHECK(d.sizes() == at::IntArrayRef(shape), "silu_gate: shapes differ");
    y = at::empty_like(gu);
    st = mvpa_silu_gate_backward_bf16(gu.data_ptr(), d.data_ptr(), y.data_ptr(), rows, (int32_t)cols, current_stream());
  }
  return st == MVPA_OK ? THPVariable_Wrap(y) : PyLong_FromLong(st);
  END_HANDLE_TH_ERRORS
}

// cosine_steps_backward(nxt [B,T,C,E], pred, d [B,T-1,C], eps, need_nxt, need_pred) -> (d_nxt | None, d_pred | None) | status
PyObject* py_cosine_steps_backward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n == 6, "cosine_steps_backward takes 6 arguments");
  at::AutoDispatchBelowADInplaceOrView guard;
  const Tensor a = aligned_operand(tensor_of(args[0]), at::kBFloat16), b = aligned_operand(tensor_of(args[1]), at::kBFloat16);
  const Tensor d = as_operand(tensor_of(args[2]), at::kFloat);
  const double eps = PyFloat_AsDouble(args[3]);
  if (PyErr_Occurred()) return nullptr;
  TORCH_CHECK(a.dim() == 4 && b.sizes() == a.sizes() && d.dim() == 3 && d.size(0) == a.size(0) && d.size(1) == a.size(1) - 1 &&
              d.size(2) == a.size(2) && b.device() == a.device() && d.device() == a.device(), "cosine_steps_backward: operands differ");
  Tensor da, db;
  if (args[4] == Py_True) da = at::empty_like(a);
  if (args[5] == Py_True) db = at::empty_like(b);
  const int st = mvpa_cosine_steps_backward_bf16(a.data_ptr(), b.data_ptr(), (const float*)d.data_ptr(), da.defined() ? da.data_ptr() : nullptr,
                                                 db.defined() ? db.data_ptr() : nullptr, a.size(0), a.size(1), a.size(2),
                                                 (int32_t)a.size(3), (float)eps, current_stream());
  if (st != MVPA_OK) return PyLong_FromLong(st);
  PyObject* r = PyTuple_New(2);
  PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(da));           // an undefined tensor comes out as None
  PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(db));
  return r;
  END_HANDLE_TH_ERRORS
}

// ---- the stack of blocks ----------------------------------------------------------------------
// What a model looked like when a plan was made from it: entries of modules' parameter and sub-module tables
// (identity), the storages and versions of the tensors found there, and the sizes of the tables that grow
// when a method is replaced on an object or a hook is registered.
struct Watch {
  struct Entry { PyObject *dict, *key, *value; };
  std::vector<Entry> entries;
  std::vector<Tensor> tensors;
  std::vector<std::pair<const void*, uint32_t>> seen;
  std::vector<std::pair<PyObject*, Py_ssize_t>> sized;

  bool unchanged() const {
    for (const auto& e : entries)
      if (PyDict_GetItem(e.dict, e.key) != e.value) return false;
    for (const auto& [dict, n] : sized)
      if (PyDict_Size(dict) != n) return false;
    for (size_t i = 0; i < tensors.size(); ++i)
      if (tensors[i].const_data_ptr() != seen[i].first || tensors[i]._version() != (int64_t)seen[i].second) return false;
    return true;
  }
  ~Watch() {
    for (auto& e : entries) {
      Py_DECREF(e.dict);
      Py_DECREF(e.key);
      Py_DECREF(e.value);
    }
    for (auto& [dict, n] : sized) Py_DECREF(dict);
  }
};

const char* kWatchName = "mvpa_stack_watch";

// watch(entries (dict, key, value), tensors, dicts watched by their size)
PyObject* py_watch(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n == 3, "watch takes 3 arguments");
  auto watch = std::make_unique<Watch>();
  for (Py_ssize_t i = 0; i < PyList_Size(args[0]); ++i) {
    PyObject* t = PyList_GetItem(args[0], i);
    TORCH_CHECK(PyTuple_Check(t) && PyTuple_Size(t) == 3 && PyDict_Check(PyTuple_GetItem(t, 0)), "watch: (dict, key, value)");
    watch->entries.push_back({Py_NewRef(PyTuple_GetItem(t, 0)), Py_NewRef(PyTuple_GetItem(t, 1)), Py_NewRef(PyTuple_GetItem(t, 2))});
  }
  for (Py_ssize_t i = 0; i < PyList_Size(args[1]); ++i) {
    const Tensor& t = tensor_of(PyList_GetItem(args[1], i));
    watch->tensors.push_back(t);
    watch->seen.emplace_back(t.const_data_ptr(), (uint32_t)t._version());
  }
  for (Py_ssize_t i = 0; i < PyList_Size(args[2]); ++i) {
    PyObject* d = PyList_GetItem(args[2], i);
    TORCH_CHECK(PyDict_Check(d), "watch: a dict");
    watch->sized.emplace_back(Py_NewRef(d), PyDict_Size(d));
  }
  if (PyErr_Occurred()) return nullptr;
  return PyCapsule_New(watch.release(), kWatchName, [](PyObject* o) { delete (Watch*)PyCapsule_GetPointer(o, kWatchName); });
  END_HANDLE_TH_ERRORS
}

PyObject* py_watch_current(PyObject*, PyObject* o) {
  const Watch* w = (const Watch*)PyCapsule_GetPointer(o, kWatchName);
  return w ? PyBool_FromLong(w->unchanged()) : nullptr;
}

struct Plan {
  std::vector<Tensor> keep;                  // every operand, alive as long as the plan
  std::vector<mvpa_stack_block> blocks;
  std::vector<char> honours_mask;
  long set = 0;                              // blocks whose operands are there
  mvpa_stack_args args;
};

const char* kPlanName = "mvpa_stack_plan";

Plan* plan_of(PyObject* o) { return (Plan*)PyCapsule_GetPointer(o, kPlanName); }

void free_plan(PyObject* o) { delete plan_of(o); }

// The pointer of a plan's operand, which the plan keeps; null for None
const void* operand(Plan* plan, PyObject* o, at::ScalarType dt) {
  if (is_none(o)) return nullptr;
  const Tensor& t = tensor_of(o);
  on_gpu(t);
  TORCH_CHECK(t.scalar_type() == dt && t.is_contiguous(), "plan: operands are contiguous and of the stack's type");
  plan->keep.push_back(t);
  return t.const_data_ptr();
}

// plan(dims (T, C, H, Hkv, Dh, E, inner), lnf_weight, lnf_eps, blocks): a block is what no tensor is needed for,
//   (ln_eps, sm_scale, flags, window, honours_mask)
PyObject* py_plan(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n == 4, "plan takes 4 arguments");
  auto plan = std::make_unique<Plan>();
  mvpa_stack_args& a = plan->args;
  std::memset(&a, 0, sizeof(a));
  a.struct_size = sizeof(a);
  int32_t* dims[7] = {&a.T, &a.C, &a.H, &a.Hkv, &a.Dh, &a.E, &a.inner};
  for (int i = 0; i < 7; ++i) *dims[i] = (int32_t)PyLong_AsLong(PyTuple_GetItem(args[0], i));
  a.lnf_weight = (const float*)operand(plan.get(), args[1], at::kFloat);
  a.lnf_eps = (float)PyFloat_AsDouble(args[2]);
  a.n_blocks = (int32_t)PyList_Size(args[3]);
  for (int32_t i = 0; i < a.n_blocks; ++i) {
    PyObject* t = PyList_GetItem(args[3], i);
    mvpa_stack_block b;
    std::memset(&b, 0, sizeof(b));
    b.ln_eps = (float)PyFloat_AsDouble(PyTuple_GetItem(t, 0));
    b.sm_scale = (float)PyFloat_AsDouble(PyTuple_GetItem(t, 1));
    b.flags = (uint32_t)PyLong_AsUnsignedLong(PyTuple_GetItem(t, 2));
    b.window = (int32_t)PyLong_AsLong(PyTuple_GetItem(t, 3));
    plan->honours_mask.push_back(PyTuple_GetItem(t, 4) == Py_True);
    plan->blocks.push_back(b);
  }
  if (PyErr_Occurred()) return nullptr;
  return PyCapsule_New(plan.release(), kPlanName, free_plan);
  END_HANDLE_TH_ERRORS
}

// set_block(plan, i, (w_qkv, w_gu, w_qkv_normed|None, w_gu_normed|None, w_tail, ln_weight, u, vb, z, k_time, k_chan),
//           ln_weight of the block behind it|None)
//   in the order of the blocks; once block 0 is set a pass can begin(), and every block that is set be enqueued
PyObject* py_set_block(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n == 4, "set_block takes 4 arguments");
  Plan* p = plan_of(args[0]);
  if (!p) return nullptr;
  const long at = PyLong_AsLong(args[1]);
  TORCH_CHECK(at >= 0 && at < (long)p->blocks.size() && at == p->set && PyTuple_Check(args[2]) && PyTuple_Size(args[2]) == 11,
              "set_block: the next block's operands");
  TORCH_CHECK(is_none(args[3]) == (at + 1 == (long)p->blocks.size()), "set_block: the norm of the block behind it");
  mvpa_stack_block& b = p->blocks[at];
  const void** ops[11] = {&b.w_qkv, &b.w_gate_up, &b.w_qkv_normed, &b.w_gate_up_normed, &b.w_tail,
                          (const void**)&b.ln_weight, &b.bias_u, &b.bias_v, &b.bias_z, &b.k_time, &b.k_chan};
  for (int j = 0; j < 11; ++j) *ops[j] = operand(p, PyTuple_GetItem(args[2], j), j == 5 ? at::kFloat : at::kBFloat16);
  if (!is_none(args[3])) p->blocks[at + 1].ln_weight = (const float*)operand(p, args[3], at::kFloat);
  ++p->set;
  if (at == 0)                                // sizes are asked for before the others are set: as many weights as here
    for (auto& other : p->blocks) {
      other.w_qkv_normed = b.w_qkv_normed;
      other.w_gate_up_normed = b.w_gate_up_normed;
    }
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

// plan_tensors(plan): every tensor it keeps
PyObject* py_plan_tensors(PyObject*, PyObject* o) {
  HANDLE_TH_ERRORS
  const Plan* p = plan_of(o);
  if (!p) return nullptr;
  PyObject* r = PyList_New(0);
  for (const Tensor& t : p->keep) {
    PyObject* w = THPVariable_Wrap(t);
    PyList_Append(r, w);
    Py_DECREF(w);
  }
  return r;
  END_HANDLE_TH_ERRORS
}

// One pass over the blocks of a plan: its arguments, checked, and every buffer it needs.
struct Run {
  std::vector<Tensor> keep;
  std::vector<mvpa_stack_block> blocks;
  mvpa_stack_args args;
  Tensor y;
  PyObject* plan = nullptr;
  long done = 0;                             // blocks enqueued
  ~Run() { Py_XDECREF(plan); }
};

const char* kRunName = "mvpa_stack_run";

// begin(plan, x [B, T|1, C, E] bf16 contiguous, chan_valid [B,C]|None, caches|None, ring_head|None, sumsq|None)
//   caches, one step: (k tensors, v tensors, first live steps), the tensors [B,Hkv,steps,C,Dh] contiguous.
//   Checks and allocates; nothing is enqueued.  Returns the pass | status
PyObject* py_begin(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n == 6, "begin takes 6 arguments");
  const Plan* p = plan_of(args[0]);
  if (!p) return nullptr;
  at::AutoDispatchBelowADInplaceOrView guard;
  auto run = std::make_unique<Run>();
  run->args = p->args;
  run->blocks = p->blocks;
  run->plan = Py_NewRef(args[0]);
  mvpa_stack_args& a = run->args;
  a.blocks = run->blocks.data();
  auto held = [&](const Tensor& t) -> const Tensor& { return run->keep.emplace_back(t); };
  const Tensor& x0 = tensor_of(args[1]);
  run->keep.reserve(5 + 2 * run->blocks.size());
  const Tensor& x = held(as_operand(x0, at::kBFloat16));
  TORCH_CHECK(x.dim() == 4 && x.size(3) == a.E && x.size(2) == a.C, "begin: x is [B, T, C, E]");
  a.B = (int32_t)x.size(0);
  a.step = is_none(args[3]) ? 0 : 1;
  TORCH_CHECK(x.size(1) == (a.step ? 1 : a.T), "begin: x and the plan disagree on T");
  if (!is_none(args[2]) && std::count(p->honours_mask.begin(), p->honours_mask.end(), 1)) {
    const Tensor& cv = held(as_operand(tensor_of(args[2]), at::kBool));
    if (!require(cv.dim() == 2 && cv.size(0) == a.B && cv.size(1) == a.C, "chan_valid is [B, C]")) return nullptr;
    for (size_t i = 0; i < run->blocks.size(); ++i)
      if (p->honours_mask[i]) run->blocks[i].chan_valid = (const uint8_t*)cv.const_data_ptr();
  }
  if (a.step) {
    PyObject *ks = PyTuple_GetItem(args[3], 0), *vs = PyTuple_GetItem(args[3], 1), *st = PyTuple_GetItem(args[3], 2);
    TORCH_CHECK(ks && vs && st && PyList_Size(ks) == (Py_ssize_t)run->blocks.size(), "begin: one cache per block");
    for (size_t i = 0; i < run->blocks.size(); ++i) {
      const Tensor &k = held(tensor_of(PyList_GetItem(ks, i))), &v = held(tensor_of(PyList_GetItem(vs, i)));
      const int64_t first = PyLong_AsLong(PyList_GetItem(st, i));
      TORCH_CHECK(k.dim() == 5 && k.sizes() == v.sizes() && k.is_cuda() && v.is_cuda() && k.is_contiguous() && v.is_contiguous() &&
                      k.scalar_type() == at::kBFloat16 && v.scalar_type() == at::kBFloat16 && k.size(0) == a.B &&
                      k.size(1) == a.Hkv && k.size(3) == a.C && k.size(4) == a.Dh && first >= 0 &&
                      first + a.T <= k.size(2),
                  "begin: caches are contiguous bf16 [B, Hkv, steps, C, Dh] with room for the step");
      mvpa_stack_block& b = run->blocks[i];
      const int64_t slot = (int64_t)a.C * a.Dh;
      b.k_cache = (char*)k.data_ptr() + first * slot * 2;
      b.v_cache = (char*)v.data_ptr() + first * slot * 2;
      b.cache_stride_b = k.stride(0);
      b.cache_stride_g = k.stride(1);
    }
    if (!is_none(args[4])) {
      const Tensor& h = held(tensor_of(args[4]));
      TORCH_CHECK(h.is_cuda() && h.scalar_type() == at::kInt && h.numel() == 1, "begin: ring_head is one int32 on the GPU");
      a.ring_head = (const int32_t*)h.data_ptr();
    }
  }
  if (!is_none(args[5])) {
    const Tensor& ss = held(tensor_of(args[5]));
    TORCH_CHECK(ss.is_cuda() && ss.scalar_type() == at::kFloat && ss.is_contiguous() && ss.numel() * a.E == x.numel(),
                "begin: sumsq holds one fp32 value per row");
    a.sumsq = (const float*)ss.data_ptr();
  }
  if (PyErr_Occurred()) return nullptr;
  const int64_t bytes = (int64_t)mvpa_stack_ws_bytes(&a);
  if (bytes == 0) return PyLong_FromLong(MVPA_ERR_UNSUPPORTED);
  run->y = at::empty(x.sizes(), x.options());
  const Tensor& ws = held(at::empty({bytes}, x.options().dtype(at::kByte)));
  a.x = x.data_ptr();
  a.y = run->y.data_ptr();
  a.ws = ws.data_ptr();
  a.ws_bytes = (size_t)bytes;
  return PyCapsule_New(run.release(), kRunName, [](PyObject* o) { delete (Run*)PyCapsule_GetPointer(o, kRunName); });
  END_HANDLE_TH_ERRORS
}

// enqueue(pass, first, end): blocks [first, end), which the parts of a pass take in order -> the normed output,
// shaped like x, with the last | None | status
PyObject* py_enqueue(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n == 3, "enqueue takes 3 arguments");
  Run* run = (Run*)PyCapsule_GetPointer(args[0], kRunName);
  if (!run) return nullptr;
  const Plan* p = plan_of(run->plan);
  const long first = PyLong_AsLong(args[1]), end = PyLong_AsLong(args[2]), blocks = (long)run->blocks.size();
  TORCH_CHECK(first == run->done && first < end && end <= blocks && end <= p->set, "enqueue: the next blocks, set");
  for (long i = first; i < std::min(end + 1, blocks); ++i) {       // operands set since begin()
    mvpa_stack_block b = p->blocks[i];
    const mvpa_stack_block& own = run->blocks[i];
    b.chan_valid = own.chan_valid;
    b.k_cache = own.k_cache;
    b.v_cache = own.v_cache;
    b.cache_stride_b = own.cache_stride_b;
    b.cache_stride_g = own.cache_stride_g;
    run->blocks[i] = b;
  }
  const int status = mvpa_stack_forward_blocks(&run->args, (int32_t)first, (int32_t)end, current_stream());
  if (status != MVPA_OK) return PyLong_FromLong(status);
  run->done = end;
  if (end < blocks) Py_RETURN_NONE;
  return THPVariable_Wrap(run->y);
  END_HANDLE_TH_ERRORS
}

// `mods`: a tuple of (enable, w, a | None, b | None) per module, enable a tuple of truth values
bool lora_modules(PyObject* mods) {
  if (!PyTuple_Check(mods) || PyTuple_GET_SIZE(mods) == 0) return false;
  for (Py_ssize_t m = 0; m < PyTuple_GET_SIZE(mods); ++m) {
    PyObject* mod = PyTuple_GET_ITEM(mods, m);
    if (!PyTuple_Check(mod) || PyTuple_GET_SIZE(mod) != 4 || !PyTuple_Check(PyTuple_GET_ITEM(mod, 0))) return false;
  }
  return true;
}

// The parts of stacked projections with adapters: equal row slices of a module, each with its share of a and b
// where enabled.  Operands as the kernels read them; the backward's come out of autograd's hands (a saved-tensor hook
// may return them in another layout).  Of w the backward takes the shape.
struct LoraParts {
  std::vector<mvpa_lora_part> parts;
  std::vector<Tensor> keep;
  int64_t rows = 0, K = 0, r = 0;
};
bool lora_parts(PyObject* mods, bool backward, LoraParts& l) {
  TORCH_CHECK(lora_modules(mods), "lora_stack: (enable, w, a, b) per module");
  auto held = [&](const Tensor& t) -> Tensor {
    l.keep.emplace_back(aligned_operand(t, at::kBFloat16));
    TORCH_CHECK(l.keep.back().device() == l.keep.front().device(), "lora_stack: operands on one GPU");
    return l.keep.back();
  };
  for (Py_ssize_t m = 0; m < PyTuple_GET_SIZE(mods); ++m) {
    PyObject* mod = PyTuple_GET_ITEM(mods, m);
    PyObject* enable = PyTuple_GET_ITEM(mod, 0);
    const Tensor& shape = tensor_of(PyTuple_GET_ITEM(mod, 1));
    const bool has = !is_none(PyTuple_GET_ITEM(mod, 2));
    const int64_t slices = has ? PyTuple_GET_SIZE(enable) : 1;
    TORCH_CHECK(shape.dim() == 2 && slices > 0 && shape.size(0) % slices == 0 && (l.K == 0 || shape.size(1) == l.K),
                "lora_stack: weights of one width, in equal slices");
    const int64_t rows = shape.size(0) / slices;
    l.K = shape.size(1);
    const Tensor w = backward ? Tensor() : held(shape);
    Tensor a, b;
    if (has) {
      a = held(tensor_of(PyTuple_GET_ITEM(mod, 2)));
      b = held(tensor_of(PyTuple_GET_ITEM(mod, 3)));
      TORCH_CHECK(a.dim() == 2 && b.dim() == 2 && a.size(1) == l.K && (l.r == 0 || b.size(1) == l.r),
                  "lora_stack: an adapter does not fit its weight");
      l.r = b.size(1);
    }
    int64_t j = 0;
    for (int64_t i = 0; i < slices; ++i) {
      mvpa_lora_part p{};
      if (!backward) p.w = (const char*)w.const_data_ptr() + i * rows * l.K * 2;
      p.rows = (int32_t)rows;
      if (has && PyTuple_GET_ITEM(enable, i) == Py_True) {
        TORCH_CHECK(a.size(0) >= (j + 1) * l.r && b.size(0) >= (j + 1) * rows, "lora_stack: an adapter does not fit its weight");
        p.a = (const char*)a.const_data_ptr() + j * l.r * l.K * 2;
        p.b = (const char*)b.const_data_ptr() + j * rows * l.r * 2;
        ++j;
      }
      l.rows += rows;
      l.parts.push_back(p);
    }
  }
  return l.parts.size() <= MVPA_LORA_PARTS && l.r > 0;
}

// lora_fits(mods): whether lora_stack takes them and is the faster way
PyObject* py_lora_fits(PyObject*, PyObject* mods) {
  HANDLE_TH_ERRORS
  int64_t K = -1, r = -1, parts = 0, most = 0;
  const Tensor* first = nullptr;
  auto bad = [&](PyObject* o) {
    if (!THPVariable_Check(o)) return true;
    const Tensor& t = THPVariable_Unpack(o);
    if (!first) first = &t;
    return !t.is_cuda() || t.device() != first->device() || t.scalar_type() != at::kBFloat16 || t.dim() != 2 || !t.is_contiguous() || t.numel() == 0 ||
           ((uintptr_t)t.const_data_ptr() & 15);
  };
  if (!lora_modules(mods)) Py_RETURN_FALSE;
  for (Py_ssize_t m = 0; m < PyTuple_GET_SIZE(mods); ++m) {
    PyObject* mod = PyTuple_GET_ITEM(mods, m);
    PyObject* enable = PyTuple_GET_ITEM(mod, 0);
    if (bad(PyTuple_GET_ITEM(mod, 1))) Py_RETURN_FALSE;
    const Tensor& w = THPVariable_Unpack(PyTuple_GET_ITEM(mod, 1));
    if (w.size(1) % 8 || (K >= 0 && w.size(1) != K)) Py_RETURN_FALSE;
    K = w.size(1);
    if (is_none(PyTuple_GET_ITEM(mod, 2))) {
      if (w.size(0) > MVPA_LORA_ROWS) Py_RETURN_FALSE;
      ++parts;
      continue;
    }
    if (bad(PyTuple_GET_ITEM(mod, 2)) || bad(PyTuple_GET_ITEM(mod, 3))) Py_RETURN_FALSE;
    const Tensor &a = THPVariable_Unpack(PyTuple_GET_ITEM(mod, 2)), &b = THPVariable_Unpack(PyTuple_GET_ITEM(mod, 3));
    const int64_t slices = PyTuple_GET_SIZE(enable);
    int64_t on = 0;
    for (int64_t i = 0; i < slices; ++i) on += PyTuple_GET_ITEM(enable, i) == Py_True;
    if (slices == 0 || on == 0 || w.size(0) % slices || a.size(1) != K || a.size(0) != on * b.size(1) ||
        b.size(0) != w.size(0) / slices * on || (r >= 0 && b.size(1) != r))
      Py_RETURN_FALSE;
    r = b.size(1);
    parts += slices;
    most = std::max(most, w.size(0) / slices);
  }
  // The kernel walks all rows of a part for every eight of its r terms, 64 columns a workgroup: beyond this tensor
  // operations are faster.  Both ways on the GPU, us, kernels / tensor operations, q and two slices of kv rows: 2048 +
  // 2 x 1024 rows of 2048 r 64 203 / 281, r 96 293 / 281; 4096 + 2 x 1024 of 4096 r 32 259 / 403, r 48 381 / 436, r 64
  // 506 / 434; 1024 + 2 x 512 of 1024 r 128 160 / 205; 768 + 2 x 256 of 768 r 8 18 / 164.
  if (r > 0 && parts <= MVPA_LORA_PARTS && r * most <= 160 * 1024) Py_RETURN_TRUE;
  Py_RETURN_FALSE;
  END_HANDLE_TH_ERRORS
}

// lora_stack(mods, scale) -> the stacked weight;  lora_stack(mods, scale, d) -> gradients of each module's a
// and b in turn (None without an adapter) | status
PyObject* py_lora_stack(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n == 2 || n == 3, "lora_stack takes the modules' weights, a scale and, for the backward, a gradient");
  const double scale = PyFloat_AsDouble(args[1]);
  if (PyErr_Occurred()) return nullptr;
  at::AutoDispatchBelowADInplaceOrView guard;
  LoraParts l;
  if (!lora_parts(args[0], n == 3, l)) return PyLong_FromLong(MVPA_ERR_UNSUPPORTED);
  const Tensor& first = tensor_of(PyTuple_GET_ITEM(PyTuple_GET_ITEM(args[0], 0), 1));
  if (n == 2) {
    Tensor out = at::empty({l.rows, l.K}, first.options());
    const int st = mvpa_lora_stack_bf16(l.parts.data(), (int32_t)l.parts.size(), (int32_t)l.K, (int32_t)l.r, (float)scale,
                                        out.data_ptr(), current_stream());
    return st == MVPA_OK ? THPVariable_Wrap(out) : PyLong_FromLong(st);
  }
  const Tensor d = aligned_operand(tensor_of(args[2]), at::kBFloat16);
  TORCH_CHECK(d.dim() == 2 && d.size(0) == l.rows && d.size(1) == l.K, "lora_stack: the gradient's shape differs");
  TORCH_CHECK(l.keep.empty() || d.device() == l.keep.front().device(), "lora_stack: operands on one GPU");
  const Py_ssize_t mods = PyTuple_GET_SIZE(args[0]);
  std::vector<Tensor> grads(2 * mods);
  size_t at = 0;
  for (Py_ssize_t m = 0; m < mods; ++m) {
    PyObject* mod = PyTuple_GET_ITEM(args[0], m);
    if (is_none(PyTuple_GET_ITEM(mod, 2))) {
      ++at;
      continue;
    }
    for (int i = 0; i < 2; ++i) grads[2 * m + i] = at::empty(tensor_of(PyTuple_GET_ITEM(mod, 2 + i)).sizes(), d.options());
    int64_t j = 0;
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(PyTuple_GET_ITEM(mod, 0)); ++i, ++at) {
      mvpa_lora_part& p = l.parts[at];
      if (!p.a) continue;
      p.da = (char*)grads[2 * m].data_ptr() + j * l.r * l.K * 2;
      p.db = (char*)grads[2 * m + 1].data_ptr() + j * (int64_t)p.rows * l.r * 2;
      ++j;
    }
  }
  const int st = mvpa_lora_stack_backward_bf16(l.parts.data(), (int32_t)l.parts.size(), (int32_t)l.K, (int32_t)l.r, (float)scale,
                                               d.data_ptr(), current_stream());
  if (st != MVPA_OK) return PyLong_FromLong(st);
  PyObject* res = PyTuple_New(2 * mods);
  for (Py_ssize_t i = 0; i < 2 * mods; ++i) PyTuple_SET_ITEM(res, i, THPVariable_Wrap(grads[i]));
  return res;
  END_HANDLE_TH_ERRORS
}

PyMethodDef kMethods[] = {
    {"forward", (PyCFunction)(void*)py_forward, METH_FASTCALL, "fused MVPA forward"},
    {"backward", (PyCFunction)(void*)py_backward, METH_FASTCALL, "backward of the fused MVPA forward, bf16"},
    {"linear", (PyCFunction)(void*)py_linear, METH_FASTCALL, "x @ w^T in bf16"},
    {"linear_wgrad", (PyCFunction)(void*)py_linear_wgrad, METH_FASTCALL, "dy^T @ x in bf16"},
    {"linear_nn", (PyCFunction)(void*)py_linear_nn, METH_FASTCALL, "dy @ w in bf16"},
    {"linear_nn2", (PyCFunction)(void*)py_linear_nn2, METH_FASTCALL, "dy @ [w0; w1] in bf16"},
    {"gated_rows", (PyCFunction)(void*)py_gated_rows, METH_FASTCALL, "gate and up rows and silu(gate) * up"},
    {"gated_rows_backward", (PyCFunction)(void*)py_gated_rows_backward, METH_FASTCALL, "the gradient of gate and up rows"},
    {"encode", (PyCFunction)(void*)py_encode, METH_FASTCALL, "db4 analysis + RMSNorm of signal rows"},
    {"mean_rows", (PyCFunction)py_mean_rows, METH_O, "means of groups of rows"},
    {"encode_saved", (PyCFunction)(void*)py_encode_saved, METH_FASTCALL, "encode, with what its backward needs"},
    {"norm_dw", (PyCFunction)(void*)py_norm_dw, METH_FASTCALL, "gradient of a norm's weight from saved row factors"},
    {"norm_backward", (PyCFunction)(void*)py_norm_backward, METH_FASTCALL, "backward of RMSNorm"},
    {"cosine_steps_backward", (PyCFunction)(void*)py_cosine_steps_backward, METH_FASTCALL, "gradients of the generative score"},
    {"silu_gate", (PyCFunction)(void*)py_silu_gate, METH_FASTCALL, "silu(gate) * up, or its backward"},
    {"lora_fits", (PyCFunction)py_lora_fits, METH_O, "whether lora_stack takes these"},
    {"lora_stack", (PyCFunction)(void*)py_lora_stack, METH_FASTCALL, "stacked weights with adapters, or the adapters' gradients"},
    {"plan", (PyCFunction)(void*)py_plan, METH_FASTCALL, "operands of a stack of blocks"},
    {"watch", (PyCFunction)(void*)py_watch, METH_FASTCALL, "what a model looks like now"},
    {"watch_current", (PyCFunction)py_watch_current, METH_O, "whether it still looks like that"},
    {"set_block", (PyCFunction)(void*)py_set_block, METH_FASTCALL, "operands of one block"},
    {"plan_tensors", (PyCFunction)py_plan_tensors, METH_O, "the tensors a plan keeps"},
    {"begin", (PyCFunction)(void*)py_begin, METH_FASTCALL, "a pass over a plan's blocks, checked"},
    {"enqueue", (PyCFunction)(void*)py_enqueue, METH_FASTCALL, "launch blocks of a pass"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_mvpa_ext", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__mvpa_ext(void) { return PyModule_Create(&kModule); }

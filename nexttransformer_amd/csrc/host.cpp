// The layer's host path in native code: one call each for the forward and the backward of a layer
// on packed bf16 weights, the check of the weight masters, and handing out the experts' gradients.
// Bound to Python as the module nt_moe_host (ops.py and moe.py call it).
//
// The layer is about ten launches forward and seventeen backward; issued from Python, with an
// allocation or three, argument checks and a ctypes call each, a small batch waits for the host
// (one token of 32 experts: 99 us per forward, 55 of them GPU work). Here the same C-ABI calls are
// made with the same buffers in the same order, without the GIL.
//
// forward() and backward() take plain GPU tensors only and look at every condition the ops check
// in Python; where one does not hold (a subclass, a dispatch mode, a functorch wrapper, another
// layout or device), they return None before doing anything and the caller goes through the ops,
// which refuse or handle it. A failing C-ABI call is returned as (status, what) for the caller to
// raise.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <vector>

#include "nt_moe.h"

namespace {

using at::Tensor;

const uint16_t* bf(const Tensor& t) { return static_cast<const uint16_t*>(t.data_ptr()); }
uint16_t* bfw(const Tensor& t) { return static_cast<uint16_t*>(t.data_ptr()); }
float* f32(const Tensor& t) { return t.defined() ? static_cast<float*>(t.data_ptr()) : nullptr; }
int32_t* i32(const Tensor& t) { return static_cast<int32_t*>(t.data_ptr()); }
nt_moe_stream_t as_stream(int64_t s) { return reinterpret_cast<nt_moe_stream_t>(s); }

// Reads positional arguments; `fine` turns false at the first one that the native path does not
// take. A Python error (a number expected) is left set.
struct Args {
  PyObject* const* at_;
  Py_ssize_t n, i = 0;
  bool fine = true;
  c10::Device device{c10::kCPU};

  bool next(PyObject*& o) {
    if (i >= n) {
      fine = false;
      return false;
    }
    o = at_[i++];
    return true;
  }
  // a plain tensor of the first tensor's GPU; undefined for None where `maybe`
  Tensor tensor(c10::ScalarType type, int64_t dim, bool maybe = false) {
    PyObject* o;
    if (!next(o)) return {};
    if (maybe && o == Py_None) return {};
    if (!THPVariable_CheckExact(o)) {
      fine = false;
      return {};
    }
    const Tensor& t = THPVariable_Unpack(o);
    if (!t.is_cuda() || !t.has_storage() || t.layout() != c10::kStrided ||
        t.key_set().has(c10::DispatchKey::Functionalize) || t.scalar_type() != type ||
        t.dim() != dim || t.is_neg() || t.is_conj()) {
      fine = false;
      return {};
    }
    if (device.is_cpu()) device = t.device();
    if (t.device() != device) fine = false;
    return t;
  }
  Tensor whole(c10::ScalarType type, int64_t dim, bool maybe = false) {  // contiguous
    Tensor t = tensor(type, dim, maybe);
    if (t.defined() && !t.is_contiguous()) fine = false;
    return t;
  }
  Tensor rows(c10::ScalarType type, bool maybe = false) {  // a matrix with contiguous rows
    Tensor t = tensor(type, 2, maybe);
    if (t.defined() && t.stride(1) != 1) fine = false;
    return t;
  }
  int64_t integer() {
    PyObject* o;
    if (!next(o)) return 0;
    const int64_t v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) {
      PyErr_Clear();
      fine = false;
    }
    return v;
  }
  double number() {
    PyObject* o;
    if (!next(o)) return 0;
    const double v = PyFloat_AsDouble(o);
    if (v == -1 && PyErr_Occurred()) {
      PyErr_Clear();
      fine = false;
    }
    return v;
  }
};

struct Failed {
  int status;
  const char* what;
};

void must(int status, const char* what) {
  if (status != NT_MOE_OK) throw Failed{status, what};
}

struct NoGil {
  PyThreadState* s = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(s); }
};

PyObject* wrap_all(const std::vector<Tensor>& v) {
  PyObject* r = PyTuple_New((Py_ssize_t)v.size());
  if (!r) return nullptr;
  for (size_t i = 0; i < v.size(); ++i) {
    PyObject* o;
    if (v[i].defined()) {
      o = THPVariable_Wrap(v[i]);
    } else {
      o = Py_None;
      Py_INCREF(o);
    }
    if (!o) {
      Py_DECREF(r);
      return nullptr;
    }
    PyTuple_SET_ITEM(r, (Py_ssize_t)i, o);
  }
  return r;
}

PyObject* failed(const Failed& f) { return Py_BuildValue("(is)", f.status, f.what); }

bool modes_active() { return c10::impl::TorchDispatchModeTLS::any_modes_set(); }

int64_t route_blocks(int64_t T) { return (T + NT_MOE_ROUTE_BLOCK - 1) / NT_MOE_ROUTE_BLOCK; }

// forward(x, w_router_t, bias | None, w1, w2, shared_w1 | None, shared_w2 | None, segment | None,
//         top_k, score_fn, up_epilogue, aux_coeff, z_coeff, want_logits, keep, stream)
// -> (out, aux, logits, ids, weights, counts, offsets, src_row, perm_w, combine_dest, combine_w,
//     load, h, fc1, shared_h, shared_fc1); the last four None without keep. load: counts as int64.
PyObject* forward(PyObject*, PyObject* const* argv, Py_ssize_t argc) {
  HANDLE_TH_ERRORS
  constexpr auto BF = at::kBFloat16, F = at::kFloat, I = at::kInt;
  Args a{argv, argc};
  const Tensor x = a.rows(BF), wr = a.whole(F, 2), bias = a.whole(F, 1, true);
  const Tensor w1 = a.whole(BF, 3), w2 = a.whole(BF, 3), s1 = a.whole(BF, 3, true),
               s2 = a.whole(BF, 3, true), seg = a.whole(I, 1, true);
  const int64_t k = a.integer(), score = a.integer(), epi = a.integer();
  const double aux_coeff = a.number(), z_coeff = a.number();
  const bool want_logits = a.integer() != 0, keep = a.integer() != 0;
  const int64_t stream = a.integer();
  if (!a.fine || a.i != argc || modes_active()) Py_RETURN_NONE;
  const int64_t T = x.size(0), d = x.size(1), E = wr.size(1);
  const int64_t halves = epi == NT_MOE_EPI_SWIGLU ? 2 : 1;
  const int64_t F1 = w1.size(1), H = F1 / halves, D = w2.size(1);
  const bool sh = s1.defined();
  if (T < 1 || k < 1 || wr.size(0) != d || (bias.defined() && bias.size(0) != E) ||
      w1.size(0) != E || w2.size(0) != E || w1.size(2) != d || w2.size(2) != H ||
      F1 % halves != 0 || sh != s2.defined() || T > INT32_MAX / k)
    Py_RETURN_NONE;
  int64_t Fs = 0, Hs = 0;
  if (sh) {
    Fs = s1.size(1);
    Hs = Fs / halves;
    if (!seg.defined() || seg.size(0) != 2 || s1.size(0) != 1 || s2.size(0) != 1 ||
        s1.size(2) != d || s2.size(1) != D || s2.size(2) != Hs || Fs % halves != 0)
      Py_RETURN_NONE;
  }
  std::vector<Tensor> r;
  try {
    NoGil no_gil;
    const int64_t A = T * k;
    const auto opt = x.options().requires_grad(false);
    auto mk = [&](at::IntArrayRef s, c10::ScalarType t) { return at::empty(s, opt.dtype(t)); };
    Tensor logits = want_logits ? mk({T, E}, F) : mk({0}, F);
    Tensor ids = mk({T, k}, I), w = mk({T, k}, F), pp = mk({route_blocks(T), E}, F),
           zp = mk({route_blocks(T)}, F), counts = mk({E}, I), offsets = mk({E + 1}, I),
           src = mk({A}, I), perm_w = mk({A}, F), cdest = mk({T, k}, I), cw = mk({T, k}, F);
    const size_t ws_bytes = nt_moe_router_plan_workspace_bytes(T, (int32_t)d, (int32_t)E, (int32_t)k);
    Tensor ws = mk({(int64_t)(ws_bytes ? ws_bytes : 1)}, at::kByte);
    const nt_moe_stream_t st = as_stream(stream);
    must(nt_moe_router_plan(bf(x), x.stride(0), f32(wr), f32(bias), T, (int32_t)d, (int32_t)E,
                            (int32_t)k, (int32_t)score, want_logits ? f32(logits) : nullptr,
                            i32(ids), f32(w), f32(pp), f32(zp), i32(counts), i32(offsets), i32(src),
                            f32(perm_w), i32(cdest), f32(cw), ws.data_ptr(), ws_bytes, st),
         "ntmoe::router_plan");
    Tensor h = mk({A, H}, BF), fc1, hs, fc1s, ys;
    if (keep) fc1 = mk({A, F1}, BF);
    if (sh) {
      hs = mk({T, Hs}, BF);
      if (keep) fc1s = mk({T, Fs}, BF);
      must(nt_moe_grouped_gemm_bf16_packed_shared(
               bf(x), x.stride(0), T, i32(src), i32(offsets), (int32_t)E, A, bf(w1), (int32_t)d,
               (int32_t)H, bfw(h), keep ? bfw(fc1) : nullptr, bf(x), x.stride(0), T, i32(seg),
               bf(s1), (int32_t)d, (int32_t)Hs, bfw(hs), keep ? bfw(fc1s) : nullptr, (int32_t)epi,
               st),
           "ntmoe::grouped_gemm_packed_shared");
    } else if (keep) {
      must(nt_moe_grouped_gemm_bf16_packed_keep(bf(x), x.stride(0), T, i32(src), i32(offsets),
                                                (int32_t)E, A, bf(w1), (int32_t)d, (int32_t)H,
                                                (int32_t)epi, bfw(h), bfw(fc1), st),
           "ntmoe::grouped_gemm_packed_keep");
    } else {
      must(nt_moe_grouped_gemm_bf16_packed(bf(x), x.stride(0), T, i32(src), i32(offsets),
                                           (int32_t)E, A, bf(w1), (int32_t)d, (int32_t)H,
                                           (int32_t)epi, bfw(h), st),
           "ntmoe::grouped_gemm_packed");
    }
    Tensor y = mk({A, D}, BF);
    if (sh) {
      ys = mk({T, D}, BF);
      must(nt_moe_grouped_gemm_bf16_packed_shared(
               bf(h), H, A, nullptr, i32(offsets), (int32_t)E, A, bf(w2), (int32_t)H, (int32_t)D,
               bfw(y), nullptr, bf(hs), Hs, T, i32(seg), bf(s2), (int32_t)Hs, (int32_t)D, bfw(ys),
               nullptr, NT_MOE_EPI_NONE, st),
           "ntmoe::grouped_gemm_packed_shared");
    } else {
      must(nt_moe_grouped_gemm_bf16_packed(bf(h), H, A, nullptr, i32(offsets), (int32_t)E, A,
                                           bf(w2), (int32_t)H, (int32_t)D, NT_MOE_EPI_NONE,
                                           bfw(y), st),
           "ntmoe::grouped_gemm_packed");
    }
    Tensor out = mk({T, D}, BF), aux = mk({3}, F), load = mk({E}, at::kLong);
    must(nt_moe_combine_aux_load(bf(y), i32(cdest), f32(cw), T, (int32_t)D, (int32_t)k,
                                 sh ? bf(ys) : nullptr, sh ? D : 0, bfw(out), D, f32(pp), f32(zp),
                                 i32(counts), (int32_t)E, (float)aux_coeff, (float)z_coeff,
                                 f32(aux), static_cast<int64_t*>(load.data_ptr()), st),
         "ntmoe::combine_aux");
    r = {out, aux, logits, ids, w, counts, offsets, src, perm_w, cdest, cw, load};
    if (keep) r.insert(r.end(), {h, fc1, hs, fc1s});
    else r.resize(16);
  } catch (const Failed& f) {
    return failed(f);
  }
  return wrap_all(r);
  END_HANDLE_TH_ERRORS
}

// backward(g, grad_aux | None, x, w1_t packed, w2_t packed, shared_w2_t packed | None, first,
//          fc1, h, perm_w, src_row, offsets, combine_dest, ids, weights, logits, counts,
//          shared_fc1 | None, shared_h | None, segment, Fs, Ep, activation, score_fn, aux_coeff,
//          z_coeff, splits of dW1, dW2, the router's and the shared expert's two, weight gradients
//          fp32, stream)
// -> (dx, d router, dW1, dW2, shared dW1 | None, shared dW2 | None)
PyObject* backward(PyObject*, PyObject* const* argv, Py_ssize_t argc) {
  HANDLE_TH_ERRORS
  constexpr auto BF = at::kBFloat16, F = at::kFloat, I = at::kInt;
  Args a{argv, argc};
  const Tensor g = a.whole(BF, 2), grad_aux = a.whole(F, 1, true), x = a.rows(BF);
  const Tensor w1t = a.whole(BF, 3), w2t = a.whole(BF, 3), sw2t = a.whole(BF, 3, true),
               first_w = a.whole(BF, 3);
  const Tensor fc1 = a.whole(BF, 2), h = a.whole(BF, 2), perm_w = a.whole(F, 1),
               src = a.whole(I, 1), offsets = a.whole(I, 1), cdest = a.whole(I, 2),
               ids = a.whole(I, 2), w = a.whole(F, 2), logits = a.whole(F, 2),
               counts = a.whole(I, 1);
  const Tensor fc1s = a.whole(BF, 2, true), hs = a.whole(BF, 2, true);
  const Tensor seg = a.whole(I, 1);
  const int64_t Fs = a.integer(), Ep = a.integer(), act = a.integer(), score = a.integer();
  const double aux_coeff = a.number(), z_coeff = a.number();
  const int64_t n1 = a.integer(), n2 = a.integer(), nr = a.integer(), ns1 = a.integer(),
                ns2 = a.integer();
  const bool wide = a.integer() != 0;
  const int64_t stream = a.integer();
  if (!a.fine || a.i != argc || modes_active()) Py_RETURN_NONE;
  const int64_t T = x.size(0), d = x.size(1), E = logits.size(1), k = ids.size(1), A = T * k;
  const int64_t F1 = fc1.size(1), H = h.size(1), Kc = first_w.size(2);
  const int64_t halves = act == NT_MOE_ACT_SWIGLU ? 2 : 1;
  const bool sh = sw2t.defined();
  auto is = [](const Tensor& t, at::IntArrayRef s) { return t.sizes() == s; };
  if (T < 1 || !is(g, {T, d}) || (grad_aux.defined() && !is(grad_aux, {3})) ||
      !is(w1t, {E, d, F1}) || !is(w2t, {E, H, d}) || F1 != halves * H || !is(fc1, {A, F1}) ||
      !is(h, {A, H}) || !is(perm_w, {A}) || !is(src, {A}) || !is(offsets, {E + 1}) ||
      !is(cdest, {T, k}) || !is(ids, {T, k}) || !is(w, {T, k}) || !is(logits, {T, E}) ||
      !is(counts, {E}) || !is(seg, {2}) || !is(first_w, {1, d, Kc}) || sh != fc1s.defined() ||
      sh != hs.defined() || Kc < Fs + 3 * Ep || Ep < E || n1 < 1 || n2 < 1 || nr < 1 || ns1 < 1 ||
      ns2 < 1)
    Py_RETURN_NONE;
  const int64_t Hs = sh ? hs.size(1) : 0;
  if (sh ? !(is(sw2t, {1, Hs, d}) && is(fc1s, {T, Fs}) && is(hs, {T, Hs}) && Fs == halves * Hs)
         : Fs != 0)
    Py_RETURN_NONE;
  std::vector<Tensor> r;
  try {
    NoGil no_gil;
    const auto opt = x.options().requires_grad(false);
    auto mk = [&](at::IntArrayRef s, c10::ScalarType t) { return at::empty(s, opt.dtype(t)); };
    const nt_moe_stream_t st = as_stream(stream);
    // the down dgrad on the gradient's rows, before the routing weight (and the shared expert's)
    Tensor u = mk({A, H}, BF), dhs;
    if (sh) {
      dhs = mk({T, Hs}, BF);
      must(nt_moe_grouped_gemm_bf16_packed_shared(
               bf(g), d, T, i32(src), i32(offsets), (int32_t)E, A, bf(w2t), (int32_t)d, (int32_t)H,
               bfw(u), nullptr, bf(g), d, T, i32(seg), bf(sw2t), (int32_t)d, (int32_t)Hs, bfw(dhs),
               nullptr, NT_MOE_EPI_NONE, st),
           "ntmoe::grouped_gemm_packed_shared");
    } else {
      must(nt_moe_grouped_gemm_bf16_packed(bf(g), d, T, i32(src), i32(offsets), (int32_t)E, A,
                                           bf(w2t), (int32_t)d, (int32_t)H, NT_MOE_EPI_NONE,
                                           bfw(u), st),
           "ntmoe::grouped_gemm_packed");
    }
    Tensor dfc1 = mk({A, F1}, BF), wh = mk({A, H}, BF), gw = mk({A}, F);
    must(nt_moe_act_bwd_rows(bf(fc1), bf(h), bf(u), f32(perm_w), A, (int32_t)H, (int32_t)act,
                             bfw(dfc1), bfw(wh), f32(gw), st),
         "ntmoe::act_bwd_rows");
    Tensor dxp = mk({A, d}, BF);
    must(nt_moe_grouped_gemm_bf16_packed(bf(dfc1), F1, A, nullptr, i32(offsets), (int32_t)E, A,
                                         bf(w1t), (int32_t)F1, (int32_t)d, NT_MOE_EPI_NONE,
                                         bfw(dxp), st),
         "ntmoe::grouped_gemm_packed");
    Tensor dfc1s;
    if (sh) {
      dfc1s = mk({T, Fs}, BF);
      must(nt_moe_act_bwd(bf(fc1s), bf(dhs), T, (int32_t)Hs, (int32_t)act, bfw(dfc1s), st),
           "ntmoe::act_bwd");
    }
    Tensor dl = mk({T, E}, F);
    must(nt_moe_router_bwd_rows(f32(logits), i32(ids), f32(w), f32(gw), i32(cdest), i32(counts), T,
                                (int32_t)E, (int32_t)k, (int32_t)score, f32(grad_aux),
                                (float)aux_coeff, (float)z_coeff, f32(dl), st),
         "ntmoe::router_bwd_rows");
    Tensor cat = mk({T, Kc}, BF), first = mk({T, d}, BF);
    must(nt_moe_backward_first_operand(f32(dl), (int32_t)E, sh ? bf(dfc1s) : nullptr, (int32_t)Fs,
                                       T, (int32_t)Ep, (int32_t)Kc, bfw(cat), st),
         "ntmoe::backward_first_operand");
    const size_t gemm_ws = nt_moe_grouped_gemm_workspace_bytes();
    Tensor ws = mk({(int64_t)gemm_ws}, at::kByte);
    must(nt_moe_grouped_gemm_bf16(bf(cat), Kc, T, nullptr, i32(seg), 1, T, bf(first_w), (int32_t)Kc,
                                  (int32_t)d, NT_MOE_EPI_NONE, bfw(first), ws.data_ptr(), gemm_ws,
                                  st),
         "ntmoe::grouped_gemm");
    auto wgrad = [&](const uint16_t* pa, int64_t lda, int64_t N, const Tensor& b, int64_t splits,
                     bool out_wide) {  // over all T rows
      const int64_t M = b.size(1);
      Tensor c = mk({1, N, M}, out_wide ? F : BF), partial;
      if (splits > 1) partial = mk({splits, 1, N, M}, F);
      must(nt_moe_grouped_wgrad_splitk(pa, lda, bf(b), b.stride(0), b.size(0), nullptr, i32(seg), 1,
                                       T, (int32_t)N, (int32_t)M, (int32_t)splits, f32(partial),
                                       partial.defined() ? partial.nbytes() : 0, out_wide, c.data_ptr(),
                                       st),
           "ntmoe::grouped_wgrad");
      return c;
    };
    Tensor wr = wgrad(bf(cat) + Fs + Ep, Kc, 2 * Ep, x, nr, true)[0];
    Tensor d_router = at::add(wr.narrow(0, 0, E), wr.narrow(0, Ep, E));
    Tensor dx = mk({T, d}, BF);
    must(nt_moe_sum_rows(bf(dxp), i32(cdest), T, (int32_t)d, (int32_t)k, bf(first), d, bfw(dx), d,
                         st),
         "ntmoe::sum_rows");
    const auto wt = wide ? F : BF;
    Tensor dw1 = mk({E, F1, d}, wt), dw2 = mk({E, d, H}, wt), partial;
    const int64_t p1 = n1 > 1 ? n1 * F1 : 0, p2 = n2 > 1 ? n2 * H : 0;
    if (p1 || p2) partial = mk({(p1 > p2 ? p1 : p2) * E * d}, F);
    must(nt_moe_expert_wgrads(bf(dfc1), F1, bf(x), x.stride(0), bf(g), d, T, bf(wh), H, i32(src),
                              i32(offsets), (int32_t)E, A, (int32_t)F1, (int32_t)d, (int32_t)H,
                              (int32_t)n1, (int32_t)n2, f32(partial),
                              partial.defined() ? partial.nbytes() : 0, wide, dw1.data_ptr(),
                              dw2.data_ptr(), st),
         "ntmoe::expert_wgrads");
    r = {dx, d_router, dw1, dw2, Tensor(), Tensor()};
    if (sh) {
      r[4] = wgrad(bf(dfc1s), Fs, Fs, x, ns1, wide);
      r[5] = wgrad(bf(g), d, d, hs, ns2, wide);
    }
  } catch (const Failed& f) {
    return failed(f);
  }
  return wrap_all(r);
  END_HANDLE_TH_ERRORS
}

// masters(tables): the addresses and the version counters of table["weight"] for each parameter
// table, as two bytes objects of int64; None where one is not a plain tensor.
PyObject* masters(PyObject*, PyObject* tables) {
  HANDLE_TH_ERRORS
  static PyObject* const key = PyUnicode_InternFromString("weight");
  if (!PyList_Check(tables)) Py_RETURN_NONE;
  const Py_ssize_t n = PyList_GET_SIZE(tables);
  PyObject* ptrs = PyBytes_FromStringAndSize(nullptr, n * 8);
  PyObject* vers = PyBytes_FromStringAndSize(nullptr, n * 8);
  if (!ptrs || !vers) {
    Py_XDECREF(ptrs);
    Py_XDECREF(vers);
    return nullptr;
  }
  auto* p = reinterpret_cast<int64_t*>(PyBytes_AS_STRING(ptrs));
  auto* v = reinterpret_cast<int64_t*>(PyBytes_AS_STRING(vers));
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* table = PyList_GET_ITEM(tables, i);
    PyObject* o = PyDict_Check(table) ? PyDict_GetItemWithError(table, key) : nullptr;
    if (!o || !THPVariable_CheckExact(o) || !THPVariable_Unpack(o).has_storage() ||
        THPVariable_Unpack(o).is_inference()) {
      if (PyErr_Occurred()) PyErr_Clear();
      Py_DECREF(ptrs);
      Py_DECREF(vers);
      Py_RETURN_NONE;
    }
    const Tensor& t = THPVariable_Unpack(o);
    p[i] = reinterpret_cast<int64_t>(t.data_ptr());
    v[i] = t._version();
  }
  return Py_BuildValue("(NN)", ptrs, vers);
  END_HANDLE_TH_ERRORS
}

// give_grads(params, stack): where no parameter has a gradient yet, each that requires one takes
// its slice of stack [n, ...] (True); else nothing is done (False).
PyObject* give_grads(PyObject*, PyObject* const* argv, Py_ssize_t argc) {
  HANDLE_TH_ERRORS
  if (argc != 2 || !PyList_Check(argv[0]) || !THPVariable_CheckExact(argv[1])) Py_RETURN_FALSE;
  const Py_ssize_t n = PyList_GET_SIZE(argv[0]);
  const Tensor& stack = THPVariable_Unpack(argv[1]);
  if (stack.dim() < 1 || stack.size(0) != n || stack.requires_grad()) Py_RETURN_FALSE;
  const auto shape = stack.sizes().slice(1);
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* o = PyList_GET_ITEM(argv[0], i);
    if (!THPVariable_CheckExact(o)) Py_RETURN_FALSE;
    const Tensor& t = THPVariable_Unpack(o);
    if (t.grad().defined() || !t.is_leaf() || t.scalar_type() != stack.scalar_type() ||
        t.device() != stack.device() || t.sizes() != shape)
      Py_RETURN_FALSE;
  }
  const std::vector<Tensor> slices = stack.unbind(0);
  for (Py_ssize_t i = 0; i < n; ++i) {
    const Tensor& t = THPVariable_Unpack(PyList_GET_ITEM(argv[0], i));
    if (t.requires_grad()) t.mutable_grad() = slices[i];
  }
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"forward", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(forward)), METH_FASTCALL,
     "One layer forward on packed bf16 weights, or None where the ops have to be taken."},
    {"backward", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(backward)), METH_FASTCALL,
     "The backward of such a forward, or None where the ops have to be taken."},
    {"masters", masters, METH_O, "Addresses and versions of the weights in parameter tables."},
    {"give_grads", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(give_grads)),
     METH_FASTCALL, "Hands each parameter its slice of a gradient stack."},
    {nullptr, nullptr, 0, nullptr}};

// Read from the file before it is loaded (_native.host).
__attribute__((used)) const char marker[] = NT_MOE_HOST_MARKER;

PyModuleDef module = {PyModuleDef_HEAD_INIT, "nt_moe_host",
                      "Native host path of the MoE layer", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit_nt_moe_host() { return PyModule_Create(&module); }

// The operators' host path for plain calls, as a CPython extension: checks of shapes and types,
// outputs and workspaces from torch's caching allocator, and the C ABI call, without the interpreter
// in between. quant/kernels.py and layers/norm.py try it first; anything it does not take as it stands
// (op-layout weights, strided or CPU tensors, tensor subclasses, invalid arguments) returns None before
// anything is allocated or launched, and the Python path serves or refuses it as it always did.
//
// A decode call is bound by the host: K=N=4096 M=1 in int4 takes 5.4 us on the GPU, and took 14 us per
// call when every shape check, allocation and ctypes argument was a Python step.
//
// Nothing is kept between calls. The GIL is released around the C ABI calls (a launch may wait for
// room in its queue), as ctypes does.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <stdlib.h>
#include <string.h>

#include <exception>

#include "../../include/w4a8_mi355x.h"

namespace {

constexpr int kBF16 = 0, kF16 = 1, kF32 = 2;
constexpr int kScaleF16 = 0, kScaleE8M0 = 1, kScaleE4M3 = 2;
constexpr int kDecode = 1, kPrefill = 2;
constexpr int kUnsupported = 2;  // the C ABI's status for a call it leaves to another path

// the C ABI entry points, handed over once by address (they live in the library that ctypes loaded)
struct Abi {
  decltype(&w4a8_last_error) last_error;
  decltype(&w4a8_linear) linear;
  decltype(&w4a8_linear_workspace_bytes_for) linear_ws;
  decltype(&w4a8_gemm) gemm;
  decltype(&w4a8_gemm_workspace_bytes) gemm_ws;
  decltype(&w4a8_rms_norm) rms_norm;
  decltype(&w4a8_moe_padded_capacity) moe_capacity;
  decltype(&w4a8_moe_route_gemm1) moe_route_gemm1;
  decltype(&w4a8_moe_route_slots) moe_route_slots;
  decltype(&w4a8_moe_route_align) moe_route_align;
  decltype(&w4a8_moe_gemm_workspace_bytes) moe_gemm_ws;
  decltype(&w4a8_moe_gemm) moe_gemm;
  decltype(&w4a8_moe_gemm2_combine_supported) moe_g2c_supported;
  decltype(&w4a8_moe_gemm2_combine) moe_g2c;
  decltype(&w4a8_moe_gemm_quant_workspace_bytes) moe_quant_ws;
  decltype(&w4a8_moe_gemm_quant) moe_quant;
  decltype(&w4a8_moe_combine) moe_combine;
};
Abi abi;
bool bound = false;

// A plain tensor argument on the GPU (torch.Tensor itself or a Parameter), or null
const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  return t.is_cuda() && t.layout() == at::kStrided && t.is_contiguous() ? &t : nullptr;
}
// an optional tensor: false when it is given and not plain
bool optional(PyObject* o, const at::Tensor*& t) {
  t = nullptr;
  if (o == Py_None) return true;
  t = plain(o);
  return t != nullptr;
}

int act_dtype(const at::Tensor& t) {
  return t.scalar_type() == at::kBFloat16 ? kBF16 : t.scalar_type() == at::kHalf ? kF16 : -1;
}
int any_dtype(const at::Tensor& t) { return t.scalar_type() == at::kFloat ? kF32 : act_dtype(t); }

// every tensor on x's device, which is the current one
template <typename... T>
bool same_device(const at::Tensor& x, const T*... t) {
  const auto d = x.get_device();
  return d == c10::hip::current_device() && (... && (!t || t->get_device() == d));
}

// scale format of (scales, zeros) for a weight with `n` channels, `g` groups and `lead` experts (0:
// dense), or -1 when the pair is not one that the operators take as it stands
int scale_format(const at::Tensor& s, const at::Tensor* z, bool e2m1, int64_t lead, int64_t g, int64_t n) {
  const int o = lead ? 1 : 0;
  auto dims = [&](const at::Tensor& t, int64_t a, int64_t b) {
    return t.dim() == 2 + o && (!o || t.size(0) == lead) && t.size(o) == a && t.size(o + 1) == b;
  };
  if (!dims(s, g, n)) return -1;
  const auto st = s.scalar_type();
  if (st == at::kHalf) {
    if (!z) return kScaleF16;
    return !e2m1 && z->scalar_type() == at::kInt && dims(*z, g, n / 8) ? kScaleF16 : -1;
  }
  if (!e2m1) return -1;
  if (st == at::kByte && !z) return kScaleE8M0;
  if (st != at::kByte && st != at::kFloat8_e4m3fn) return -1;
  // NVFP4: the per-channel global as its int32 bits (dense: or as f32)
  if (!z || z->dim() != 1 + o || (o && z->size(0) != lead) || z->size(o) != n) return -1;
  return z->scalar_type() == at::kInt || (!o && z->scalar_type() == at::kFloat) ? kScaleE4M3 : -1;
}

at::Tensor empty(const at::Tensor& like, at::IntArrayRef sizes, at::ScalarType t) {
  return at::empty(sizes, like.options().dtype(t));
}

void* stream_of(const at::Tensor& x) { return c10::hip::getCurrentHIPStream(x.get_device()).stream(); }

PyObject* failed(int rc, const char* what) {
  const char* m = abi.last_error();
  if (m && *m) PyErr_Format(PyExc_RuntimeError, "%s: %s", what, m);
  else PyErr_Format(PyExc_RuntimeError, "%s: status %d", what, rc);
  return nullptr;
}

template <typename F>
int unlocked(F f) {
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = f();
  Py_END_ALLOW_THREADS
  return rc;
}

// C++ exceptions (an allocator out of memory) as torch's own bindings report them
template <typename F>
PyObject* guarded(F f) {
  try {
    return f();
  } catch (...) {
    torch::translate_exception_to_python(std::current_exception());
  }
  return nullptr;
}

// linear(x, w, scales, zeros, group, e2m1, x_fp8, act_scales, silu, arm) -> (out, arm) or None.
// arm 0: the decode kernels for up to 16 rows of a K that is a multiple of 32, else the tiled ones, which
// MINISGL_FORCE_TILED_LINEARS=1 takes always.
PyObject* linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 10 || !bound) {
    PyErr_SetString(PyExc_TypeError, "linear: 10 arguments, after bind()");
    return nullptr;
  }
  return guarded([&]() -> PyObject* {
    const at::Tensor *x = plain(a[0]), *w = plain(a[1]), *s = plain(a[2]), *z, *xq, *xs;
    if (!x || !w || !s || !optional(a[3], z) || !optional(a[6], xq) || !optional(a[7], xs) || !xq != !xs) Py_RETURN_NONE;
    if (!PyLong_Check(a[4])) Py_RETURN_NONE;
    const int64_t group = PyLong_AsLongLong(a[4]);
    const bool e2m1 = PyObject_IsTrue(a[5]) == 1, silu = PyObject_IsTrue(a[8]) == 1;
    int arm = (int)PyLong_AsLong(a[9]);
    if (PyErr_Occurred()) return nullptr;
    const int dt = act_dtype(*x);
    if (x->dim() != 2 || dt < 0 || w->scalar_type() != at::kByte || w->dim() != 3 || w->size(2) != 1024) Py_RETURN_NONE;
    const int64_t M = x->size(0), K = x->size(1), N = w->size(0) * 16;
    if (M <= 0 || K <= 0 || w->size(1) != (K + 127) / 128 || group <= 0 || K % group) Py_RETURN_NONE;
    if (z && z->numel() == 0) z = nullptr;
    if (silu && N % 32) Py_RETURN_NONE;
    const int sfmt = scale_format(*s, z, e2m1, 0, K / group, N);
    if (sfmt < 0 || !same_device(*x, w, s, z, xq, xs)) Py_RETURN_NONE;
    if (xq && ((xq->scalar_type() != at::kByte && xq->scalar_type() != at::kFloat8_e4m3fn) || xq->dim() != 2 ||
               xq->size(0) != M || xq->size(1) != K || xs->scalar_type() != at::kFloat || xs->dim() != 1 || xs->size(0) != M))
      Py_RETURN_NONE;
    if (arm == 0) {
      const char* f = getenv("MINISGL_FORCE_TILED_LINEARS");
      arm = !(f && !strcmp(f, "1")) && M <= 16 && K % 32 == 0 ? kDecode : kPrefill;
    }
    const int64_t nout = silu ? N / 2 : N;
    at::Tensor out = empty(*x, {M, nout}, x->scalar_type());
    const int wfmt = e2m1 ? 1 : 0;
    const int64_t wsb = xq ? abi.gemm_ws(M, N, K, arm) : abi.linear_ws(M, N, K, sfmt, z != nullptr, wfmt, group, silu, arm);
    at::Tensor ws;
    if (wsb > 0) ws = empty(*x, {wsb}, at::kByte);
    void* wp = ws.defined() ? ws.data_ptr() : nullptr;
    const int32_t* zp = z ? static_cast<const int32_t*>(z->data_ptr()) : nullptr;
    void* st = stream_of(*x);
    const int rc = unlocked([&] {
      return xq ? abi.gemm(static_cast<const uint8_t*>(xq->data_ptr()), K, static_cast<const float*>(xs->data_ptr()), M,
                           w->data_ptr(), N, K, s->data_ptr(), sfmt, zp, wfmt, group, out.data_ptr(), dt, nout, silu, wp,
                           wsb > 0 ? wsb : 0, arm, st)
                : abi.linear(x->data_ptr(), dt, M, K, K, w->data_ptr(), N, s->data_ptr(), sfmt, zp, wfmt, group,
                             out.data_ptr(), dt, nout, silu, wp, wsb, arm, st);
    });
    if (rc) return failed(rc, silu ? "w4a8_linear_silu" : "w4a8_linear");
    return Py_BuildValue("(Ni)", THPVariable_Wrap(std::move(out)), arm);
  });
}

// rms_norm(x, weight, eps, plus_one, residual, quant) -> out, (out, x_fp8, act_scales) or None
PyObject* rms_norm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 6 || !bound) {
    PyErr_SetString(PyExc_TypeError, "rms_norm: 6 arguments, after bind()");
    return nullptr;
  }
  return guarded([&]() -> PyObject* {
    const at::Tensor *x = plain(a[0]), *w, *r;
    if (!x || !optional(a[1], w) || !optional(a[4], r)) Py_RETURN_NONE;
    const double eps = PyFloat_AsDouble(a[2]);
    const bool plus_one = PyObject_IsTrue(a[3]) == 1, quant = PyObject_IsTrue(a[5]) == 1;
    if (PyErr_Occurred()) return nullptr;
    const int dt = act_dtype(*x);
    if (dt < 0 || x->dim() < 1 || x->numel() == 0) Py_RETURN_NONE;
    const int64_t K = x->size(-1), M = x->numel() / K;
    if ((w && (w->scalar_type() != x->scalar_type() || w->numel() != K)) ||
        (r && (r->scalar_type() != x->scalar_type() || r->sizes() != x->sizes())) || !same_device(*x, w, r))
      Py_RETURN_NONE;
    at::Tensor out = empty(*x, x->sizes(), x->scalar_type()), q, s;
    if (quant) {
      q = empty(*x, x->sizes(), at::kByte);
      s = empty(*x, {M}, at::kFloat);
    }
    void* st = stream_of(*x);
    const int rc = unlocked([&] {
      return abi.rms_norm(x->data_ptr(), dt, M, K, K, r ? r->data_ptr() : nullptr, K, w ? w->data_ptr() : nullptr,
                          plus_one, (float)eps, out.data_ptr(), K, quant ? static_cast<uint8_t*>(q.data_ptr()) : nullptr, K,
                          quant ? static_cast<float*>(s.data_ptr()) : nullptr, st);
    });
    if (rc) return failed(rc, "rms_norm");
    if (!quant) return THPVariable_Wrap(std::move(out));
    return Py_BuildValue("(NNN)", THPVariable_Wrap(std::move(out)), THPVariable_Wrap(std::move(q)),
                         THPVariable_Wrap(std::move(s)));
  });
}

struct Experts {
  const at::Tensor *w, *s, *z;
  int64_t N, K, group;
  int fmt;
};
// one expert weight (E, N/16, K tiles, 1024) with its scales; false when it is not a plain one
bool experts(PyObject* w, PyObject* s, PyObject* z, bool e2m1, int64_t E, int64_t K, Experts& e) {
  e.w = plain(w);
  e.s = plain(s);
  if (!e.w || !e.s || !optional(z, e.z)) return false;
  if (e.w->scalar_type() != at::kByte || e.w->dim() != 4 || e.w->size(3) != 1024 || e.w->size(0) != E ||
      e.w->size(2) != (K + 127) / 128 || e.s->dim() != 3 || e.s->size(1) <= 0 || K % e.s->size(1))
    return false;
  e.N = e.w->size(1) * 16;
  e.K = K;
  e.group = K / e.s->size(1);
  e.fmt = scale_format(*e.s, e.z, e2m1, E, e.s->size(1), e.N);
  return e.fmt >= 0;
}

// moe(x, w13, s13, z13, w2, s2, z2, gating, top_k, renormalize, e2m1, block_m, slots, routed, g2fuse, g2c)
// -> (out, took) or None: the silu forward of quant/kernels.py `_moe_forward` with the route computed
// here. slots: one block per slot; routed / g2fuse / g2c: the module's switches (g2c already bounded by
// the token count). took: 1 route + gemm1 in one launch, 2 gemm2 + combine in one launch.
PyObject* moe(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 16 || !bound) {
    PyErr_SetString(PyExc_TypeError, "moe: 16 arguments, after bind()");
    return nullptr;
  }
  return guarded([&]() -> PyObject* {
    const at::Tensor *x = plain(a[0]), *gate = plain(a[7]);
    if (!x || !gate || x->dim() != 2 || gate->dim() != 2) Py_RETURN_NONE;
    const long top_k = PyLong_AsLong(a[8]), bm = PyLong_AsLong(a[11]);
    const bool renorm = PyObject_IsTrue(a[9]) == 1, e2m1 = PyObject_IsTrue(a[10]) == 1;
    bool slots = PyObject_IsTrue(a[12]) == 1;
    const bool routed = PyObject_IsTrue(a[13]) == 1, g2fuse = PyObject_IsTrue(a[14]) == 1, g2c = PyObject_IsTrue(a[15]) == 1;
    if (PyErr_Occurred()) return nullptr;
    const int64_t T = x->size(0), K = x->size(1), E = gate->size(1);
    const int dt = act_dtype(*x), gdt = any_dtype(*gate);
    if (dt < 0 || gdt < 0 || T <= 0 || K <= 0 || gate->size(0) != T || top_k <= 0 || top_k > E || bm <= 0) Py_RETURN_NONE;
    Experts e1, e2;
    if (!experts(a[1], a[2], a[3], e2m1, E, K, e1) || e1.N % 32) Py_RETURN_NONE;
    if (e1.group != 16 && e1.group != 32 && e1.group != 64 && e1.group != 128) Py_RETURN_NONE;
    const int64_t I = e1.N / 2;
    if (!experts(a[4], a[5], a[6], e2m1, E, I, e2) || e2.N != K) Py_RETURN_NONE;
    if (!same_device(*x, gate, e1.w, e1.s, e1.z, e2.w, e2.s, e2.z)) Py_RETURN_NONE;

    const int arm = bm < 64 ? kDecode : kPrefill, wfmt = e2m1 ? 1 : 0;
    const int64_t numel = T * top_k, P = abi.moe_capacity(numel, E, (int)bm);
    // rows enter the combine unrounded where the reference runs its fused decode gemm2 + gather-reduce
    const bool round_y2 = !(g2fuse && e2.fmt != kScaleE4M3 && e1.fmt != kScaleE4M3 && T <= 32 && bm != 128);
    const int row_dt = round_y2 ? dt : kF32;
    const bool fuse2 = g2fuse && g2c && arm == kDecode &&
                       abi.moe_g2c_supported(I, e2.fmt, e2.z != nullptr, wfmt, e2.group, (int)top_k) == 1;
    const int64_t ws1 = abi.moe_gemm_ws(numel, E, (int)bm, P, e1.N, K, arm);
    const int64_t ws2 = fuse2 ? 0 : abi.moe_quant_ws(P, I);
    // every intermediate in one allocation, each 256-byte aligned
    int64_t at = 0;
    auto take = [&](int64_t bytes) {
      const int64_t o = at;
      at += (bytes + 255) / 256 * 256;
      return o;
    };
    const int64_t o_tw = take(numel * 4), o_ids = take(numel * 4), o_sorted = take(P * 4),
                  o_eid = take((P + bm - 1) / bm * 4), o_ntp = take(4), o_inv = take(numel * 4), o_xq = take(T * K),
                  o_xs = take(T * 4), o_b2 = take(P * I * 2), o_ws1 = take(ws1 > 0 ? ws1 : 0),
                  o_ws2 = take(ws2 > 0 ? ws2 : 0), o_y2 = take(fuse2 ? 0 : P * K * (row_dt == kF32 ? 4 : 2));
    at::Tensor out = empty(*x, {T, K}, x->scalar_type()), mem = empty(*x, {at}, at::kByte);
    uint8_t* m = static_cast<uint8_t*>(mem.data_ptr());
    auto f32 = [&](int64_t o) { return reinterpret_cast<float*>(m + o); };
    auto i32 = [&](int64_t o) { return reinterpret_cast<int32_t*>(m + o); };
    auto zp = [](const Experts& e) { return e.z ? static_cast<const int32_t*>(e.z->data_ptr()) : nullptr; };
    void* st = stream_of(*x);
    int took = 0;
    const char* what = "";
    const int rc = unlocked([&]() -> int {
      int r = kUnsupported;
      if (slots && routed && numel <= E && numel * bm <= P) {
        what = "w4a8_moe route_gemm1";
        r = abi.moe_route_gemm1(gate->data_ptr(), gdt, T, E, (int)top_k, renorm, x->data_ptr(), dt, K, (int)bm, P,
                                e1.w->data_ptr(), e1.N, K, e1.s->data_ptr(), e1.fmt, zp(e1), wfmt, e1.group, f32(o_tw),
                                i32(o_ids), i32(o_sorted), i32(o_eid), i32(o_ntp), i32(o_inv), m + o_b2, dt, I, st);
        if (r == 0) took |= 1;
        else if (r != kUnsupported) return r;
      }
      if (r) {
        // the grouped GEMMs size their grids for at most numel / block + min(E, numel) blocks
        const bool sl = slots && numel <= E && numel * bm <= P;
        what = sl ? "moe_route_slots" : "moe_route_align";
        r = (sl ? abi.moe_route_slots : abi.moe_route_align)(
            gate->data_ptr(), gdt, T, E, (int)top_k, renorm, (int)bm, P, f32(o_tw), i32(o_ids), i32(o_sorted),
            i32(o_eid), i32(o_ntp), i32(o_inv), x->data_ptr(), dt, K, K, m + o_xq, K, f32(o_xs), st);
        if (r) return r;
        what = "w4a8_moe gemm1";
        r = abi.moe_gemm(m + o_xq, K, f32(o_xs), 1, i32(o_sorted), i32(o_eid), i32(o_ntp), numel, (int)top_k, (int)bm, P,
                         e1.w->data_ptr(), E, e1.N, K, e1.s->data_ptr(), e1.fmt, zp(e1), wfmt, e1.group, m + o_b2, dt, I,
                         1, ws1 > 0 ? m + o_ws1 : nullptr, ws1, arm, st);
        if (r) return r;
      }
      if (fuse2) {
        took |= 2;
        what = "w4a8_moe gemm2+combine";
        return abi.moe_g2c(m + o_b2, dt, I, i32(o_ids), f32(o_tw), i32(o_inv), T, (int)top_k, (int)bm, P,
                           e2.w->data_ptr(), E, K, I, e2.s->data_ptr(), e2.fmt, zp(e2), wfmt, e2.group, out.data_ptr(), dt,
                           K, row_dt, st);
      }
      what = "w4a8_moe gemm2";
      r = abi.moe_quant(m + o_b2, dt, I, i32(o_sorted), i32(o_eid), i32(o_ntp), numel, (int)bm, P, e2.w->data_ptr(), E, K,
                        I, e2.s->data_ptr(), e2.fmt, zp(e2), wfmt, e2.group, m + o_y2, row_dt, K, m + o_ws2, ws2, arm, st);
      if (r) return r;
      what = "w4a8_moe combine";
      return abi.moe_combine(m + o_y2, row_dt, K, i32(o_inv), f32(o_tw), T, (int)top_k, K, out.data_ptr(), dt, st);
    });
    if (rc) return failed(rc, what);
    return Py_BuildValue("(Ni)", THPVariable_Wrap(std::move(out)), took);
  });
}

// bind(address of each entry point in Abi's order)
PyObject* bind(PyObject*, PyObject* args) {
  constexpr Py_ssize_t kCount = sizeof(Abi) / sizeof(void*);
  if (PyTuple_GET_SIZE(args) != kCount) {
    PyErr_Format(PyExc_TypeError, "bind: %zd addresses", kCount);
    return nullptr;
  }
  void* p[kCount];
  for (Py_ssize_t i = 0; i < kCount; ++i) {
    p[i] = PyLong_AsVoidPtr(PyTuple_GET_ITEM(args, i));
    if (!p[i]) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "bind: a null address");
      return nullptr;
    }
  }
  memcpy(&abi, p, sizeof abi);
  bound = true;
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, nullptr},
    {"linear", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(linear)), METH_FASTCALL, nullptr},
    {"rms_norm", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(rms_norm)), METH_FASTCALL, nullptr},
    {"moe", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(moe)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "w4a8_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_w4a8_host() {
  PyObject* m = PyModule_Create(&module_def);
  if (m && PyModule_AddStringConstant(m, "built_for", W4A8_BUILT_FOR) < 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}

// Native call path of ferret_amd.ops: argument checks, output and workspace
// allocation, and the C-ABI call in one CPython function per operator.
//
// A decode-sized kernel takes 5 - 15 us; the checks, torch.empty calls and the
// ctypes call in Python took about 15 us per operator, so a step made of such
// calls ran at the host's pace (an FP8 projection of 8 tokens: 5.6 us of kernel,
// 15 us a call).  Here an operator costs about 5 us (a linear of one token 4.6).
//
// Every function takes the operator's tensors (None where optional) and returns
// its result, or None whenever anything is not the plain case: an argument that
// is no exact torch.Tensor (or Parameter), not a contiguous GPU tensor of the
// expected type and shape, wrapped by a transform, under a dispatch or function
// mode, or a rejected argument (a negative return code).  The caller (ops.py) then
// takes its Python path, which names the error or handles the case.  A HIP error
// (a positive code) is raised at once (native_run.hpp).
#include <Python.h>
#include <ATen/ATen.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/PythonTorchFunctionTLS.h>

#include <climits>

#include "../../include/ferret_hip.h"
#include "native_run.hpp"

namespace {

using ferret::native::declined;
using ferret::native::run;

constexpr auto kBf16 = at::kBFloat16;
constexpr auto kF32 = at::kFloat;
constexpr auto kI32 = at::kInt;
constexpr auto kFp8 = at::kFloat8_e4m3fn;

// Transform wrappers (vmap, grad, functionalization): left to Python.
const c10::DispatchKeySet kWrapped({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                    c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize,
                                    c10::DispatchKey::BatchedNestedTensor, c10::DispatchKey::Batched});

// The tensors of one call.  ok() turns false at the first argument outside the
// plain case; a device is taken from the first tensor and asked of all others.
class Call {
 public:
  Call() : ok_(!c10::impl::TorchDispatchModeTLS::any_modes_set() && !at::impl::torch_function_mode_enabled()) {}

  bool ok() const { return ok_; }
  void require(bool c) { ok_ = ok_ && c; }

  // A required tensor of `ndim` dimensions (0: any) and one of up to two types.
  const at::Tensor* in(PyObject* o, int ndim, at::ScalarType type, at::ScalarType or_type) {
    if (!ok_ || !THPVariable_CheckExact(o)) {
      ok_ = false;
      return nullptr;
    }
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.key_set().has_any(kWrapped) ||
        (ndim != 0 && t.dim() != ndim) || (t.scalar_type() != type && t.scalar_type() != or_type) ||
        !t.is_contiguous()) {
      ok_ = false;
      return nullptr;
    }
    for (const int64_t s : t.sizes()) require(s <= INT_MAX);
    if (!has_device_) {
      device_ = t.device();
      has_device_ = true;
    }
    require(t.device() == device_);
    return &t;
  }
  const at::Tensor* in(PyObject* o, int ndim, at::ScalarType type) { return in(o, ndim, type, type); }

  // A caller's output of exactly this shape, or a new one.
  at::Tensor out(PyObject* o, at::IntArrayRef shape, at::ScalarType type, at::ScalarType or_type) {
    if (o == Py_None) return ok_ ? fresh(shape, type) : at::Tensor();
    const at::Tensor* t = in(o, 0, type, or_type);
    require(t != nullptr && t->sizes() == shape);
    return ok_ ? *t : at::Tensor();
  }
  at::Tensor out(PyObject* o, at::IntArrayRef shape, at::ScalarType type) { return out(o, shape, type, type); }

  at::Tensor fresh(at::IntArrayRef shape, at::ScalarType type) {
    return at::empty(shape, at::TensorOptions().dtype(type).device(device_));
  }

  // The caller's workspace if it holds `need` bytes, else a new one; undefined
  // for need == 0.
  at::Tensor workspace(PyObject* o, size_t need) {
    if (o != Py_None) {
      // any type; its device counts even where it is too small or not needed
      if (!ok_ || !THPVariable_CheckExact(o)) {
        ok_ = false;
        return at::Tensor();
      }
      const at::Tensor& t = THPVariable_Unpack(o);
      require(t.defined() && t.is_cuda() && t.device() == device_ && t.layout() == at::kStrided &&
              !t.key_set().has_any(kWrapped) && t.is_contiguous());
      if (!ok_) return at::Tensor();
      if (need != 0 && t.nbytes() >= need) return t;
    }
    return ok_ && need != 0 ? fresh({(int64_t)need}, at::kByte) : at::Tensor();
  }

 private:
  bool ok_;
  bool has_device_ = false;
  at::Device device_ = at::Device(at::kCUDA);
};

void* ptr(const at::Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
void* ptr(const at::Tensor* t) { return t->data_ptr(); }
template <typename T>
T* ptr_as(const at::Tensor& t) { return static_cast<T*>(ptr(t)); }
template <typename T>
T* ptr_as(const at::Tensor* t) { return static_cast<T*>(t->data_ptr()); }

void* stream() { return c10::hip::getCurrentHIPStream().stream(); }

bool as_int(PyObject* o, int* v) {
  const long x = PyLong_CheckExact(o) ? PyLong_AsLong(o) : -1;
  if (PyErr_Occurred() != nullptr) PyErr_Clear();
  *v = (int)x;
  return x >= 0 && x <= INT_MAX;
}

PyObject* wrap(const at::Tensor& t) { return THPVariable_Wrap(t); }

#define NATIVE(name, nargs)                                                                    \
  PyObject* name##_body(PyObject* const* a);                                                   \
  PyObject* name(PyObject*, PyObject* const* a, Py_ssize_t n) {                                \
    HANDLE_TH_ERRORS                                                                           \
    if (n != (nargs)) {                                                                        \
      PyErr_Format(PyExc_TypeError, #name " takes %d arguments, got %zd", (int)(nargs), n);    \
      return nullptr;                                                                          \
    }                                                                                          \
    return name##_body(a);                                                                     \
    END_HANDLE_TH_ERRORS                                                                       \
  }                                                                                            \
  PyObject* name##_body(PyObject* const* a)

// The bounds of ferret_workspace_bytes(6, ...).
bool on_bounds(const void* x, const void* w, const void* residual, const void* y) {
  const auto bits = [](const void* p) { return reinterpret_cast<uintptr_t>(p); };
  return ((bits(x) | bits(w)) & 15) == 0 && ((bits(residual) | bits(y)) & 7) == 0;
}

// x, w, residual, out, workspace
NATIVE(linear_bf16, 5) {
  Call c;
  const auto* x = c.in(a[0], 2, kBf16);
  const auto* w = c.in(a[1], 2, kBf16);
  if (!c.ok()) Py_RETURN_NONE;
  const int M = x->size(0), K = x->size(1), N = w->size(0);
  c.require(w->size(1) == K && M >= 1 && N >= 16);
  const at::Tensor* r = a[2] == Py_None ? nullptr : c.in(a[2], 2, kBf16);
  if (!c.ok() || (r != nullptr && (r->size(0) != M || r->size(1) != N))) Py_RETURN_NONE;
  const at::Tensor y = c.out(a[3], {M, N}, kBf16);
  if (!c.ok()) Py_RETURN_NONE;
  void *xp = ptr(x), *wp = ptr(w), *rp = r ? ptr(r) : nullptr, *yp = ptr(y);
  const size_t need = ferret_workspace_bytes(on_bounds(xp, wp, rp, yp) ? 6 : 0, M, N, K, 0);
  const at::Tensor ws = c.workspace(a[4], need);
  if (!c.ok()) Py_RETURN_NONE;
  void* st = stream();
  const size_t have = ws.defined() ? ws.nbytes() : 0;
  if (!run("ferret_linear_bf16", [&] { return ferret_linear_bf16(xp, wp, rp, yp, M, N, K, ptr(ws), have, st); }))
    return declined();
  return wrap(y);
}

// a, sa, b, sb, out, workspace, flags
NATIVE(fp8_gemm_blockscale, 7) {
  Call c;
  int flags;
  const auto* x = c.in(a[0], 2, kFp8, at::kByte);
  const auto* sx = c.in(a[1], 2, kF32);
  const auto* w = c.in(a[2], 2, kFp8, at::kByte);
  const auto* sw = c.in(a[3], 2, kF32);
  if (!c.ok() || !as_int(a[6], &flags)) Py_RETURN_NONE;
  const int M = x->size(0), K = x->size(1), N = w->size(0);
  c.require(w->size(1) == K && M >= 1 && N >= 16 && sx->size(0) == M && sx->size(1) == K / 128 &&
            sw->size(0) == (N + 127) / 128 && sw->size(1) == K / 128);
  const at::Tensor y = c.out(a[4], {M, N}, kBf16);
  if (!c.ok()) Py_RETURN_NONE;
  const size_t need = ferret_workspace_bytes(1, M, N, K, 0);
  const at::Tensor ws = c.workspace(a[5], need);
  if (!c.ok()) Py_RETURN_NONE;
  void* st = stream();
  if (!run("ferret_fp8_gemm_blockscale", [&] {
        return ferret_fp8_gemm_blockscale_ex(ptr(x), ptr_as<float>(sx), ptr(w), ptr_as<float>(sw), ptr(y), M, N, K,
                                             ptr(ws), need, flags, st);
      }))
    return declined();
  return wrap(y);
}

// a, sfa, b, sfb, out, workspace
NATIVE(fp8_gemm_ue8m0, 6) {
  Call c;
  const auto* x = c.in(a[0], 2, kFp8, at::kByte);
  const auto* sx = c.in(a[1], 2, kI32);
  const auto* w = c.in(a[2], 2, kFp8, at::kByte);
  const auto* sw = c.in(a[3], 2, kI32);
  if (!c.ok()) Py_RETURN_NONE;
  const int M = x->size(0), K = x->size(1), N = w->size(0), nsk = (K / 128 + 3) / 4;
  c.require(w->size(1) == K && sx->size(0) == nsk && sx->size(1) == M && sw->size(0) == nsk && sw->size(1) == N);
  const at::Tensor y = c.out(a[4], {M, N}, kBf16);
  if (!c.ok()) Py_RETURN_NONE;
  const size_t need = ferret_workspace_bytes(5, M, N, K, 0);
  if (need == 0) Py_RETURN_NONE;
  const at::Tensor ws = c.workspace(a[5], need);
  if (!c.ok()) Py_RETURN_NONE;
  void* st = stream();
  if (!run("ferret_fp8_gemm_ue8m0", [&] {
        return ferret_fp8_gemm_ue8m0(ptr(x), ptr_as<uint32_t>(sx), ptr(w), ptr_as<uint32_t>(sw), ptr(y), M, N, K,
                                     ptr(ws), ws.nbytes(), st);
      }))
    return declined();
  return wrap(y);
}

// logits, topk, with_weights -> (ids, weights or None)
NATIVE(moe_route_topk, 3) {
  Call c;
  int topk;
  const auto* x = c.in(a[0], 2, kF32);
  if (!c.ok() || !as_int(a[1], &topk)) Py_RETURN_NONE;
  const int T = x->size(0), E = x->size(1);
  if (topk < 1 || topk > E) Py_RETURN_NONE;
  const int with_weights = PyObject_IsTrue(a[2]);
  if (with_weights < 0) return nullptr;
  const at::Tensor ids = c.fresh({T, topk}, kI32);
  const at::Tensor w = with_weights ? c.fresh({T, topk}, kF32) : at::Tensor();
  void* st = stream();
  if (!run("ferret_moe_route_topk", [&] {
        return ferret_moe_route_topk(ptr_as<float>(x), T, E, topk, ptr_as<int32_t>(ids), ptr_as<float>(w), st);
      }))
    return declined();
  PyObject* pw = Py_None;
  if (with_weights) pw = wrap(w);
  else Py_INCREF(pw);
  return Py_BuildValue("(NN)", wrap(ids), pw);
}

// ids, num_experts, tile_m (or None), workspace -> (counts, offsets, sorted_pair, tiles, ntiles, tile_m, max_tiles,
// topk, T)
NATIVE(moe_permute, 4) {
  Call c;
  int E, tile_m;
  const auto* ids = c.in(a[0], 2, kI32);
  if (!c.ok() || !as_int(a[1], &E) || E < 1) Py_RETURN_NONE;
  const int T = ids->size(0), topk = ids->size(1);
  const int64_t P = (int64_t)T * topk;
  if (P > (1 << 22)) Py_RETURN_NONE;
  if (a[2] == Py_None) tile_m = ferret_moe_tile_m((int)P, E);
  else if (!as_int(a[2], &tile_m) || tile_m < 1) Py_RETURN_NONE;
  const size_t need = ferret_workspace_bytes(4, (int)P, 0, 0, E);
  const at::Tensor ws = c.workspace(a[3], need);
  if (!c.ok()) Py_RETURN_NONE;
  const int max_tiles = std::max(1, ferret_moe_max_tiles((int)P, E, tile_m));
  const at::Tensor counts = c.fresh({E}, kI32), offsets = c.fresh({E + 1}, kI32),
                   sorted_pair = c.fresh({std::max<int64_t>(P, 1)}, kI32), tiles = c.fresh({max_tiles, 3}, kI32),
                   ntiles = c.fresh({1}, kI32);
  void* st = stream();
  if (!run("ferret_moe_permute", [&] {
        return ferret_moe_permute(ptr_as<int32_t>(ids), T, topk, E, tile_m, ptr_as<int32_t>(counts),
                                  ptr_as<int32_t>(offsets), ptr_as<int32_t>(sorted_pair), ptr_as<int32_t>(tiles),
                                  max_tiles, ptr_as<int32_t>(ntiles), ptr(ws), need, st);
      }))
    return declined();
  return Py_BuildValue("(NNNNNiiii)", wrap(counts), wrap(offsets), wrap(sorted_pair), wrap(tiles), wrap(ntiles),
                       tile_m, max_tiles, topk, T);
}

// The routing arguments of the grouped products: sorted_pair, tiles, ntiles,
// max_tiles, tile_m, topk, num_experts, num_tokens.
struct Routing {
  const at::Tensor *sorted_pair, *tiles, *ntiles;
  int max_tiles, tile_m, topk, E, T;
  bool read(Call& c, PyObject* const* a) {
    sorted_pair = c.in(a[0], 1, kI32);
    tiles = c.in(a[1], 2, kI32);
    ntiles = c.in(a[2], 1, kI32);
    return c.ok() && as_int(a[3], &max_tiles) && as_int(a[4], &tile_m) && as_int(a[5], &topk) && as_int(a[6], &E) &&
           as_int(a[7], &T) && (int64_t)T * topk <= INT_MAX;
  }
};

// x, sx, w, sw, routing (8), out, flags
NATIVE(moe_w13_fp8, 14) {
  Call c;
  Routing rt;
  int flags;
  const auto* x = c.in(a[0], 2, kFp8, at::kByte);
  const auto* sx = c.in(a[1], 2, kF32);
  const auto* w = c.in(a[2], 3, kFp8, at::kByte);
  const auto* sw = c.in(a[3], 3, kF32);
  if (!c.ok() || !rt.read(c, a + 4) || !as_int(a[13], &flags)) Py_RETURN_NONE;
  const int T = x->size(0), K = x->size(1), E = w->size(0), N = w->size(1), P = T * rt.topk;
  c.require(w->size(2) == K && E == rt.E && T == rt.T && sx->size(0) == T && sx->size(1) == K / 128 &&
            sw->size(0) == E && sw->size(1) == N / 128 && sw->size(2) == K / 128);
  const at::Tensor y = c.out(a[12], {P, N / 2}, kBf16);
  if (!c.ok()) Py_RETURN_NONE;
  void* st = stream();
  if (!run("ferret_moe_w13_fp8", [&] {
        return ferret_moe_w13_fp8_ex(ptr(x), ptr_as<float>(sx), ptr(w), ptr_as<float>(sw),
                                     ptr_as<int32_t>(rt.sorted_pair), ptr_as<int32_t>(rt.tiles),
                                     ptr_as<int32_t>(rt.ntiles), rt.max_tiles, rt.tile_m, T, rt.topk, E, N, K, ptr(y),
                                     flags, st);
      }))
    return declined();
  return wrap(y);
}

// h, sh, w, sw, routing (8), out, flags
NATIVE(moe_w2_fp8, 14) {
  Call c;
  Routing rt;
  int flags;
  const auto* h = c.in(a[0], 2, kFp8, at::kByte);
  const auto* sh = c.in(a[1], 2, kF32);
  const auto* w = c.in(a[2], 3, kFp8, at::kByte);
  const auto* sw = c.in(a[3], 3, kF32);
  if (!c.ok() || !rt.read(c, a + 4) || !as_int(a[13], &flags)) Py_RETURN_NONE;
  const int P = h->size(0), K = h->size(1), E = w->size(0), N = w->size(1);
  c.require(w->size(2) == K && E == rt.E && P == (int64_t)rt.T * rt.topk && sh->size(0) == P &&
            sh->size(1) == K / 128 && sw->size(0) == E && sw->size(1) == N / 128 && sw->size(2) == K / 128);
  const at::Tensor y = c.out(a[12], {P, N}, kBf16);
  if (!c.ok()) Py_RETURN_NONE;
  void* st = stream();
  if (!run("ferret_moe_w2_fp8", [&] {
        return ferret_moe_w2_fp8_ex(ptr(h), ptr_as<float>(sh), ptr(w), ptr_as<float>(sw),
                                    ptr_as<int32_t>(rt.sorted_pair), ptr_as<int32_t>(rt.tiles),
                                    ptr_as<int32_t>(rt.ntiles), rt.max_tiles, rt.tile_m, P, E, N, K, ptr(y), flags, st);
      }))
    return declined();
  return wrap(y);
}

// x, wq (3-D words or 5-D tiles), ws, routing (8), out
NATIVE(moe_w13_w4a16, 12) {
  Call c;
  Routing rt;
  const auto* x = c.in(a[0], 2, kBf16);
  const auto* wq = c.in(a[1], 0, kI32);
  const auto* ws = c.in(a[2], 3, kBf16);
  if (!c.ok() || !rt.read(c, a + 3) || (wq->dim() != 3 && wq->dim() != 5)) Py_RETURN_NONE;
  const bool tiled = wq->dim() == 5;
  const int T = x->size(0), K = x->size(1), E = wq->size(0), P = T * rt.topk;
  const int64_t rows = tiled ? wq->size(1) * 16 : wq->size(1);
  c.require(rows <= INT_MAX && (tiled ? wq->size(3) == 16 && wq->size(4) == 16 && wq->size(2) * 128 == K
                                      : wq->size(2) * 8 == K));
  const int N = (int)rows;
  c.require(E == rt.E && T == rt.T && ws->size(0) == E && ws->size(1) == N && ws->size(2) == K / 32);
  const at::Tensor y = c.out(a[11], {P, N / 2}, kBf16);
  if (!c.ok()) Py_RETURN_NONE;
  void* st = stream();
  if (!run(tiled ? "ferret_moe_w13_w4a16_tiled" : "ferret_moe_w13_w4a16", [&] {
        if (tiled)
          return ferret_moe_w13_w4a16_tiled(ptr(x), ptr(wq), ptr(ws), ptr_as<int32_t>(rt.sorted_pair),
                                            ptr_as<int32_t>(rt.tiles), ptr_as<int32_t>(rt.ntiles), rt.max_tiles,
                                            rt.tile_m, T, rt.topk, E, N, K, ptr(y), st);
        return ferret_moe_w13_w4a16(ptr(x), ptr_as<int32_t>(wq), ptr(ws), ptr_as<int32_t>(rt.sorted_pair),
                                    ptr_as<int32_t>(rt.tiles), ptr_as<int32_t>(rt.ntiles), rt.max_tiles, rt.tile_m, T,
                                    rt.topk, E, N, K, ptr(y), st);
      }))
    return declined();
  return wrap(y);
}

// x, q, scale -> (q, scale)
NATIVE(quant_act_e4m3, 3) {
  Call c;
  const auto* x = c.in(a[0], 2, kBf16);
  if (!c.ok()) Py_RETURN_NONE;
  const int M = x->size(0), K = x->size(1);
  const at::Tensor q = c.out(a[1], {M, K}, kFp8, at::kByte);
  const at::Tensor s = c.out(a[2], {M, K / 128}, kF32);
  if (!c.ok()) Py_RETURN_NONE;
  void* st = stream();
  if (!run("ferret_quant_act_e4m3",
           [&] { return ferret_quant_act_e4m3(ptr(x), ptr(q), ptr_as<float>(s), M, K, st); }))
    return declined();
  return Py_BuildValue("(NN)", wrap(q), wrap(s));
}

// o, weights, out
NATIVE(moe_combine, 3) {
  Call c;
  const auto* o = c.in(a[0], 2, kBf16);
  const auto* w = c.in(a[1], 2, kF32);
  if (!c.ok()) Py_RETURN_NONE;
  const int T = w->size(0), topk = w->size(1), N = o->size(1);
  c.require(o->size(0) == (int64_t)T * topk);
  const at::Tensor y = c.out(a[2], {T, N}, kBf16);
  if (!c.ok()) Py_RETURN_NONE;
  void* st = stream();
  if (!run("ferret_moe_combine",
           [&] { return ferret_moe_combine(ptr(o), ptr_as<float>(w), T, topk, N, ptr(y), st); }))
    return declined();
  return wrap(y);
}

#define METHOD(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {METHOD(linear_bf16),   METHOD(fp8_gemm_blockscale), METHOD(fp8_gemm_ue8m0),
                          METHOD(moe_route_topk), METHOD(moe_permute),         METHOD(moe_w13_fp8),
                          METHOD(moe_w2_fp8),     METHOD(moe_w13_w4a16),       METHOD(quant_act_e4m3),
                          METHOD(moe_combine),    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_native", "Native call path of ferret_amd.ops.", -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&kModule); }

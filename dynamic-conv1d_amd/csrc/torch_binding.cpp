// Native autograd binding of the C ABI (include/dynconv.h) for PyTorch: the
// operators' autograd Functions as C++ nodes, called from dynconv/*.py.
//
// A small or medium call is bound by its host path.  Through Python's
// autograd.Function and ctypes a forward takes 11-15 us and a backward 70-100 us
// of host time (the engine's thread has to take the GIL, and every argument
// passes through Python), against 5-20 us of kernels; here the checks, the
// allocations and the launches are native and the backward runs without the GIL.
//
// Each entry point returns None for every call it does not take (another type,
// layout, device or dtype than the plain one, function transforms, forward-mode
// derivatives, tracing, dispatch modes, failed preconditions): the Python
// Functions then take the call, and raise what they raise.  So this file holds
// no second copy of the operators' error behaviour.  What a taken call computes,
// saves and launches is what those Functions do (headwise.py:218-309,
// lowrank.py:214-299); kernel errors surface as the same RuntimeError.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <dlfcn.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/utils/pybind.h>

#include "dynconv.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;

// The C ABI, from the library that dynconv._capi loaded.
struct Abi {
  decltype(&dc_status_string) status_string;
  decltype(&dc_headwise_fwd) headwise_fwd;
  decltype(&dc_headwise_bwd_ws_bytes) headwise_bwd_ws_bytes;
  decltype(&dc_headwise_bwd) headwise_bwd;
  decltype(&dc_lowrank_zeff_bytes) lowrank_zeff_bytes;
  decltype(&dc_lowrank_fwd) lowrank_fwd;
  decltype(&dc_lowrank_bwd_ws_bytes) lowrank_bwd_ws_bytes;
  decltype(&dc_lowrank_bwd) lowrank_bwd;
  decltype(&dc_lowrank_fwd_grouped) lowrank_fwd_grouped;
  decltype(&dc_lowrank_bwd_grouped_ws_bytes) lowrank_bwd_grouped_ws_bytes;
  decltype(&dc_lowrank_bwd_grouped) lowrank_bwd_grouped;
  decltype(&dc_proj_in_fwd) proj_in_fwd;
  decltype(&dc_proj_in_bwd_ws_bytes) proj_in_bwd_ws_bytes;
  decltype(&dc_proj_in_bwd) proj_in_bwd;
};
Abi abi{};
bool ready = false;

void check(int64_t status, const char* what) {
  TORCH_CHECK(status >= 0, "dynconv ", what, " failed: ", abi.status_string((int)status), " (status ", status, ")");
}

int dtype_code(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kBFloat16: return DC_DTYPE_BF16;
    case at::kHalf: return DC_DTYPE_FP16;
    case at::kFloat: return DC_DTYPE_FP32;
    default: return -1;
  }
}

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }
void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

// n bytes of device memory beside t (n == 0: none).
Tensor bytes_like(const Tensor& t, int64_t n) {
  return n > 0 ? at::empty({n}, t.options().dtype(at::kByte)) : Tensor();
}
// A gradient as the kernels read it: contiguous, in x's dtype.
Tensor grad_in(const Tensor& dy, at::ScalarType dtype) { return dy.contiguous().to(dtype); }

// ---------------------------------------------------------------- headwise
Tensor headwise_forward(const Tensor& x, const Tensor& w, const Tensor& sw, bool residual) {
  Tensor y = at::empty_like(x);
  check(abi.headwise_fwd(ptr(x), ptr(w), ptr(sw), ptr(y), x.size(0), x.size(1), x.size(2), w.size(2), w.size(3),
                         dtype_code(x), residual, stream_of(x)),
        "headwise forward");
  return y;
}

struct HeadwiseFn : public Function<HeadwiseFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w, const std::optional<Tensor>& sw,
                        bool residual) {
    const Tensor s = sw.value_or(Tensor());
    Tensor y = headwise_forward(x, w, s, residual);
    ctx->save_for_backward({x, w, s});
    ctx->saved_data["residual"] = residual;
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list saved = ctx->get_saved_variables();
    const Tensor &x = saved[0], &w = saved[1], &sw = saved[2];
    const c10::DeviceGuard guard(x.device());
    const Tensor dy = grad_in(grads[0], x.scalar_type());
    Tensor dx = at::empty_like(x), dw = at::empty_like(w), dsw = sw.defined() ? at::empty_like(sw) : Tensor();
    const int64_t B = x.size(0), T = x.size(1), D = x.size(2), H = w.size(2), W = w.size(3);
    const int dt = dtype_code(x);
    const int64_t n = abi.headwise_bwd_ws_bytes(B, T, D, H, W, dt, sw.defined());
    check(n, "headwise backward workspace query");
    const Tensor ws = bytes_like(x, n);
    check(abi.headwise_bwd(ptr(x), ptr(w), ptr(sw), ptr(dy), ptr(dx), ptr(dw), ptr(dsw), ptr(ws), n, B, T, D, H, W, dt,
                           ctx->saved_data["residual"].toBool(), stream_of(x)),
          "headwise backward");
    return {dx, dw, dsw, Tensor()};
  }
};

// ----------------------------------------------------------------- lowrank
struct LowrankFn : public Function<LowrankFn> {
  // zeff: the padded z copy that the forward keeps for the backward (null: none)
  static Tensor run(const Tensor& x, const Tensor& z, const Tensor& U, const Tensor& sw, const Tensor& zeff,
                    int64_t nzeff, bool residual) {
    Tensor y = at::empty_like(x);
    const int64_t D = x.size(2);
    check(abi.lowrank_fwd(ptr(x), ptr(z), ptr(U), ptr(sw), ptr(y), ptr(zeff), nzeff, x.size(0), x.size(1), D, z.size(2),
                          U.size(1) / D, dtype_code(x), residual, stream_of(x)),
          "lowrank forward");
    return y;
  }
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& z, const Tensor& U,
                        const std::optional<Tensor>& sw, bool residual) {
    const Tensor s = sw.value_or(Tensor());
    const int64_t D = x.size(2);
    const int64_t nz = abi.lowrank_zeff_bytes(x.size(0), x.size(1), D, z.size(2), U.size(1) / D, dtype_code(x), s.defined());
    check(nz, "lowrank z_eff size query");
    const Tensor zeff = bytes_like(x, nz);
    Tensor y = run(x, z, U, s, zeff, nz, residual);
    ctx->save_for_backward({x, z, U, s});
    ctx->saved_data["residual"] = residual;
    if (zeff.defined()) ctx->saved_data["zeff"] = zeff;  // internal buffer, a function of z
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list saved = ctx->get_saved_variables();
    const Tensor &x = saved[0], &z = saved[1], &U = saved[2], &sw = saved[3];
    const c10::DeviceGuard guard(x.device());
    const Tensor dy = grad_in(grads[0], x.scalar_type());
    Tensor dx = at::empty_like(x), dz = at::empty_like(z), dU = at::empty_like(U);
    Tensor dsw = sw.defined() ? at::empty_like(sw) : Tensor();
    const int64_t B = x.size(0), T = x.size(1), D = x.size(2), R = z.size(2), W = U.size(1) / D;
    const int dt = dtype_code(x);
    const int64_t n = abi.lowrank_bwd_ws_bytes(B, T, D, R, W, dt, sw.defined());
    check(n, "lowrank backward workspace query");
    const Tensor ws = bytes_like(x, n);
    const auto it = ctx->saved_data.find("zeff");
    const Tensor zeff = it != ctx->saved_data.end() ? it->second.toTensor() : Tensor();
    check(abi.lowrank_bwd(ptr(x), ptr(z), ptr(U), ptr(sw), ptr(zeff), zeff.defined() ? zeff.numel() : 0, ptr(dy),
                          ptr(dx), ptr(dz), ptr(dU), ptr(dsw), ptr(ws), n, B, T, D, R, W, dt,
                          ctx->saved_data["residual"].toBool(), stream_of(x)),
          "lowrank backward");
    return {dx, dz, dU, dsw, Tensor()};
  }
};

// ------------------------------------------------- grouped lowrank, with proj_in
// G device pointers, `stride` bytes apart from base (base null: all null).
struct Ptrs {
  void* p[DC_MAX_GROUPS] = {};
  Ptrs() = default;
  Ptrs(void* base, int64_t stride, int64_t G) {
    for (int64_t g = 0; g < G && base; ++g) p[g] = static_cast<char*>(base) + g * stride;
  }
  const void* const* in() const { return p; }
  void* const* out() const { return p; }
};

constexpr int64_t round256(int64_t n) { return (n + 255) / 256 * 256; }

// The sizes of a grouped module call: x [B, T, G*D], pre_z [B, T, K], w_in [G*R, K],
// U [G, R, W*D], sw [G, W, D].
struct GroupedShape {
  int64_t G, B, T, D, R, W, K, zbytes, es;
  int dt;
  GroupedShape(const Tensor& x, const Tensor& pre, const Tensor& U)
      : G(U.size(0)), B(x.size(0)), T(x.size(1)), D(x.size(2) / U.size(0)), R(U.size(1)), W(U.size(2) / D),
        K(pre.size(2)), es(x.element_size()), dt(dtype_code(x)) {
    zbytes = round256(B * T * R * es);  // one group's z (or dz), on its own aligned range of one buffer
  }
};

// GroupedLowRankDynamicShortConvolution: z = proj_in(pre_z), then the grouped
// operator, as one node: the parameters' gradients are written as the whole
// tensors they belong to (slicing them per group costs a fill, a copy and an
// add per slice in the backward: 16 launches, 85 us of 864 at B2 T8192 D4096).
struct GroupedModuleFn : public Function<GroupedModuleFn> {
  static variable_list run(const Tensor& x, const Tensor& pre, const Tensor& w_in, const Tensor& U, const Tensor& sw,
                           int64_t hd, const GroupedShape& s, const Tensor& z, const Tensor& zeff, int64_t nzeff) {
    void* st = stream_of(x);
    const Ptrs zs(ptr(z), s.zbytes, s.G);
    check(abi.proj_in_fwd(ptr(pre), ptr(w_in), zs.out(), s.G, s.B * s.T, s.K, s.R, s.dt, st), "proj_in forward");
    variable_list ys;
    Ptrs yp;
    for (int64_t g = 0; g < s.G; ++g) {
      ys.push_back(hd ? at::empty({s.B, s.D / hd, s.T, hd}, x.options()) : at::empty({s.B, s.T, s.D}, x.options()));
      yp.p[g] = ptr(ys.back());
    }
    const Ptrs Us(ptr(U), s.R * s.W * s.D * s.es, s.G), sws(ptr(sw), s.W * s.D * s.es, s.G);
    const Ptrs ze(ptr(zeff), round256(nzeff), s.G);
    check(abi.lowrank_fwd_grouped(s.G, ptr(x), x.stride(1), zs.in(), Us.in(), sws.in(), yp.out(),
                                  zeff.defined() ? ze.out() : nullptr, nzeff, hd, s.B, s.T, s.D, s.R, s.W, s.dt, 1, st),
          "grouped lowrank forward");
    return ys;
  }
  static Tensor z_buffer(const Tensor& x, const GroupedShape& s) {
    return at::empty({s.G * s.zbytes / s.es}, x.options());
  }
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& pre, const Tensor& w_in,
                               const Tensor& U, const Tensor& sw, int64_t hd) {
    const GroupedShape s(x, pre, U);
    const int64_t nz = abi.lowrank_zeff_bytes(s.B, s.T, s.D, s.R, s.W, s.dt, 1);
    check(nz, "lowrank z_eff size query");
    const Tensor z = z_buffer(x, s), zeff = bytes_like(x, s.G * round256(nz));
    variable_list ys = run(x, pre, w_in, U, sw, hd, s, z, zeff, nz);
    ctx->save_for_backward({x, pre, w_in, U, sw, z});
    ctx->saved_data["hd"] = hd;
    if (zeff.defined()) ctx->saved_data["zeff"] = zeff;
    return ys;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list saved = ctx->get_saved_variables();
    const Tensor &x = saved[0], &pre = saved[1], &w_in = saved[2], &U = saved[3], &sw = saved[4], &z = saved[5];
    const c10::DeviceGuard guard(x.device());
    const GroupedShape s(x, pre, U);
    const int64_t hd = ctx->saved_data["hd"].toInt(), C = s.G * s.D;
    void* st = stream_of(x);
    variable_list dys;
    Ptrs dyp;
    for (int64_t g = 0; g < s.G; ++g) {
      dys.push_back(grad_in(grads[g], x.scalar_type()));
      dyp.p[g] = ptr(dys.back());
    }
    // pre_z or proj_in.weight wanted (inputs 1, 2): a frozen projection has no backward
    const bool proj = ctx->needs_input_grad(1) || ctx->needs_input_grad(2);
    Tensor dx = at::empty({s.B, s.T, C}, x.options()), dpre, dw;
    if (proj) {
      dpre = at::empty_like(pre);
      dw = at::empty_like(w_in);
    }
    Tensor dU = at::empty_like(U), dsw = at::empty_like(sw);
    const Tensor dz = z_buffer(x, s);
    const auto it = ctx->saved_data.find("zeff");
    const Tensor zeff = it != ctx->saved_data.end() ? it->second.toTensor() : Tensor();
    const int64_t nz = zeff.defined() ? abi.lowrank_zeff_bytes(s.B, s.T, s.D, s.R, s.W, s.dt, 1) : 0;
    const int64_t n1 = abi.lowrank_bwd_grouped_ws_bytes(s.G, s.B, s.T, s.D, s.R, s.W, s.dt, 1);
    check(n1, "grouped lowrank backward workspace query");
    const int64_t n2 = proj ? abi.proj_in_bwd_ws_bytes(s.G, s.B * s.T, s.K, s.R, s.dt) : 0;
    check(n2, "proj_in backward workspace query");
    // one workspace: proj_in's backward runs after the convolutions' on the same stream
    const Tensor ws = bytes_like(x, std::max<int64_t>(std::max(n1, n2), 1));
    const Ptrs zs(ptr(z), s.zbytes, s.G), dzs(ptr(dz), s.zbytes, s.G), ze(ptr(zeff), round256(nz), s.G);
    const int64_t ub = s.R * s.W * s.D * s.es, sb = s.W * s.D * s.es;
    const Ptrs Us(ptr(U), ub, s.G), sws(ptr(sw), sb, s.G), dUs(ptr(dU), ub, s.G), dsws(ptr(dsw), sb, s.G);
    check(abi.lowrank_bwd_grouped(s.G, ptr(x), x.stride(1), zs.in(), Us.in(), sws.in(),
                                  zeff.defined() ? ze.in() : nullptr, nz, dyp.in(), hd, ptr(dx), C, dzs.out(),
                                  dUs.out(), dsws.out(), ptr(ws), n1, s.B, s.T, s.D, s.R, s.W, s.dt, 1, st),
          "grouped lowrank backward");
    if (proj)
      check(abi.proj_in_bwd(ptr(pre), ptr(w_in), dzs.in(), ptr(dpre), ptr(dw), ptr(ws), n2, s.G, s.B * s.T, s.K, s.R,
                            s.dt, st),
            "proj_in backward");
    return {dx, dpre, dw, dU, dsw, Tensor()};
  }
};

// ------------------------------------------------------------ entry points
// No function transform, dispatch mode or tracer is looking at this call.
bool plain_call() {
  using c10::DispatchKey;
  return ready && !c10::impl::tls_is_dispatch_key_included(DispatchKey::FuncTorchDynamicLayerFrontMode) &&
         !c10::impl::tls_is_dispatch_key_included(DispatchKey::Python) &&
         !c10::impl::TorchDispatchModeTLS::any_modes_set() && !torch::jit::tracer::isTracing();
}

// A torch.Tensor or Parameter (no subclass) in dense device memory, of x's dtype
// and device when given, without a forward-mode tangent.
bool plain_tensor(PyObject* o, Tensor* out, const Tensor* like = nullptr) {
  if (!THPVariable_CheckExact(o)) return false;
  const Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.numel() == 0 || !t.has_storage()) return false;
  if (t.key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                               c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Negative,
                                               c10::DispatchKey::Functionalize})))
    return false;
  if (t._fw_grad(/*level=*/0).defined()) return false;
  if (like && (t.scalar_type() != like->scalar_type() || t.device() != like->device())) return false;
  *out = t;
  return true;
}

bool any_requires_grad(std::initializer_list<const Tensor*> ts) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor* t : ts)
    if (t->defined() && t->requires_grad()) return true;
  return false;
}

#define DC_DECLINE_UNLESS(cond) \
  if (!(cond)) Py_RETURN_NONE

std::optional<Tensor> opt(const Tensor& t) { return t.defined() ? std::optional<Tensor>(t) : std::nullopt; }

// headwise(x, weight, static_w or None, residual) -> y, or None (not taken)
PyObject* py_headwise(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  Tensor x, w, sw;
  DC_DECLINE_UNLESS(nargs == 4 && plain_call() && plain_tensor(args[0], &x) && plain_tensor(args[1], &w, &x));
  DC_DECLINE_UNLESS(args[2] == Py_None || plain_tensor(args[2], &sw, &x));
  DC_DECLINE_UNLESS(dtype_code(x) >= 0 && x.dim() == 3 && w.dim() == 4 && x.is_contiguous() && w.is_contiguous());
  DC_DECLINE_UNLESS(w.size(0) == x.size(0) && w.size(1) == x.size(1) && x.size(2) % w.size(2) == 0);
  DC_DECLINE_UNLESS(!sw.defined() || (sw.dim() == 2 && sw.size(0) == w.size(3) && sw.size(1) == x.size(2) &&
                                      sw.is_contiguous()));
  const int residual = PyObject_IsTrue(args[3]);
  if (residual < 0) return nullptr;
  Tensor y;
  {
    pybind11::gil_scoped_release no_gil;
    const c10::DeviceGuard guard(x.device());
    y = any_requires_grad({&x, &w, &sw}) ? HeadwiseFn::apply(x, w, opt(sw), residual != 0)
                                         : headwise_forward(x, w, sw, residual != 0);
  }
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// lowrank(x, z, U, static_w or None, residual) -> y, or None (not taken)
PyObject* py_lowrank(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  Tensor x, z, U, sw;
  DC_DECLINE_UNLESS(nargs == 5 && plain_call() && plain_tensor(args[0], &x) && plain_tensor(args[1], &z, &x) &&
                    plain_tensor(args[2], &U, &x));
  DC_DECLINE_UNLESS(args[3] == Py_None || plain_tensor(args[3], &sw, &x));
  DC_DECLINE_UNLESS(dtype_code(x) >= 0 && x.dim() == 3 && z.dim() == 3 && U.dim() == 2);
  DC_DECLINE_UNLESS(x.is_contiguous() && z.is_contiguous() && U.is_contiguous());
  const int64_t D = x.size(2), R = z.size(2), rank = R + (sw.defined() ? 1 : 0);
  DC_DECLINE_UNLESS((rank & (rank - 1)) == 0 && z.size(0) == x.size(0) && z.size(1) == x.size(1));
  DC_DECLINE_UNLESS(U.size(0) == R && U.size(1) % D == 0);
  DC_DECLINE_UNLESS(!sw.defined() || (sw.dim() == 2 && sw.size(0) == U.size(1) / D && sw.size(1) == D &&
                                      sw.is_contiguous()));
  const int residual = PyObject_IsTrue(args[4]);
  if (residual < 0) return nullptr;
  Tensor y;
  {
    pybind11::gil_scoped_release no_gil;
    const c10::DeviceGuard guard(x.device());
    y = any_requires_grad({&x, &z, &U, &sw}) ? LowrankFn::apply(x, z, U, opt(sw), residual != 0)
                                             : LowrankFn::run(x, z, U, sw, Tensor(), 0, residual != 0);
  }
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

bool aligned16(const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }

// grouped_module(x, pre_z, w_in, proj_out, proj_out_bias, head_dim) -> tuple of G outputs, or None (not taken)
PyObject* py_grouped_module(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  Tensor x, pre, w_in, U, sw;
  DC_DECLINE_UNLESS(nargs == 6 && plain_call() && plain_tensor(args[0], &x) && plain_tensor(args[1], &pre, &x) &&
                    plain_tensor(args[2], &w_in, &x) && plain_tensor(args[3], &U, &x) && plain_tensor(args[4], &sw, &x));
  DC_DECLINE_UNLESS(x.scalar_type() == at::kBFloat16 || x.scalar_type() == at::kHalf);
  DC_DECLINE_UNLESS(x.dim() == 3 && pre.dim() == 3 && w_in.dim() == 2 && U.dim() == 3 && sw.dim() == 3);
  const int64_t G = U.size(0), B = x.size(0), T = x.size(1), R = U.size(1), K = pre.size(2);
  DC_DECLINE_UNLESS(G >= 1 && G <= DC_MAX_GROUPS && x.size(2) % G == 0);
  const int64_t D = x.size(2) / G;
  DC_DECLINE_UNLESS(((R + 1) & R) == 0 && U.size(2) % D == 0 && sw.size(0) == G && sw.size(1) == U.size(2) / D &&
                    sw.size(2) == D);
  DC_DECLINE_UNLESS(pre.size(0) == B && pre.size(1) == T && w_in.size(0) == G * R && w_in.size(1) == K);
  DC_DECLINE_UNLESS(x.stride(2) == 1 && x.stride(0) == T * x.stride(1));
  DC_DECLINE_UNLESS(pre.is_contiguous() && w_in.is_contiguous() && U.is_contiguous() && sw.is_contiguous());
  // proj_in on the library's kernels (modules._proj_in_native)
  DC_DECLINE_UNLESS(G * R <= 128 && K % 8 == 0 && aligned16(pre) && aligned16(w_in));
  int64_t hd = 0;
  if (args[5] != Py_None) {
    hd = PyLong_AsLongLong(args[5]);
    if (hd == -1 && PyErr_Occurred()) return nullptr;
    DC_DECLINE_UNLESS(hd > 0 && hd <= D && D % hd == 0);
  }
  variable_list ys;
  {
    pybind11::gil_scoped_release no_gil;
    const c10::DeviceGuard guard(x.device());
    if (any_requires_grad({&x, &pre, &w_in, &U, &sw})) {
      ys = GroupedModuleFn::apply(x, pre, w_in, U, sw, hd);
    } else {
      const GroupedShape s(x, pre, U);
      ys = GroupedModuleFn::run(x, pre, w_in, U, sw, hd, s, GroupedModuleFn::z_buffer(x, s), Tensor(), 0);
    }
  }
  PyObject* out = PyTuple_New((Py_ssize_t)ys.size());
  if (!out) return nullptr;
  for (size_t g = 0; g < ys.size(); ++g) {
    PyObject* o = THPVariable_Wrap(std::move(ys[g]));
    if (!o) {
      Py_DECREF(out);
      return nullptr;
    }
    PyTuple_SET_ITEM(out, (Py_ssize_t)g, o);
  }
  return out;
  END_HANDLE_TH_ERRORS
}

// init(path): take the C ABI from the library at path (loaded already by dynconv._capi).
PyObject* py_init(PyObject*, PyObject* path) {
  HANDLE_TH_ERRORS
  const char* p = PyUnicode_AsUTF8(path);
  if (!p) return nullptr;
  void* lib = dlopen(p, RTLD_NOW | RTLD_LOCAL);
  TORCH_CHECK(lib != nullptr, "cannot load ", p, ": ", dlerror());
  auto sym = [&](auto& f, const char* name) {
    f = reinterpret_cast<std::decay_t<decltype(f)>>(dlsym(lib, name));
    TORCH_CHECK(f != nullptr, p, " has no symbol ", name);
  };
  sym(abi.status_string, "dc_status_string");
  sym(abi.headwise_fwd, "dc_headwise_fwd");
  sym(abi.headwise_bwd_ws_bytes, "dc_headwise_bwd_ws_bytes");
  sym(abi.headwise_bwd, "dc_headwise_bwd");
  sym(abi.lowrank_zeff_bytes, "dc_lowrank_zeff_bytes");
  sym(abi.lowrank_fwd, "dc_lowrank_fwd");
  sym(abi.lowrank_bwd_ws_bytes, "dc_lowrank_bwd_ws_bytes");
  sym(abi.lowrank_bwd, "dc_lowrank_bwd");
  sym(abi.lowrank_fwd_grouped, "dc_lowrank_fwd_grouped");
  sym(abi.lowrank_bwd_grouped_ws_bytes, "dc_lowrank_bwd_grouped_ws_bytes");
  sym(abi.lowrank_bwd_grouped, "dc_lowrank_bwd_grouped");
  sym(abi.proj_in_fwd, "dc_proj_in_fwd");
  sym(abi.proj_in_bwd_ws_bytes, "dc_proj_in_bwd_ws_bytes");
  sym(abi.proj_in_bwd, "dc_proj_in_bwd");
  ready = true;
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"init", py_init, METH_O, "Take the C ABI from the library at a path."},
    {"headwise", (PyCFunction)(void*)py_headwise, METH_FASTCALL, "headwise(x, weight, static_w, residual)"},
    {"lowrank", (PyCFunction)(void*)py_lowrank, METH_FASTCALL, "lowrank(x, z, U, static_w, residual)"},
    {"grouped_module", (PyCFunction)(void*)py_grouped_module, METH_FASTCALL,
     "grouped_module(x, pre_z, w_in, proj_out, proj_out_bias, head_dim)"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_binding", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__binding(void) {
  PyObject* m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION_BUILT) < 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}

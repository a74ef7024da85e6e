// Torch operator module of fast_rnnt_amd: fast_rnnt_amd/_C*.so.
//
// The counterpart of the reference's pybind module (fast_rnnt/python/csrc/fast_rnnt.cu:24,
// fast_rnnt/python/csrc/mutual_information.cu:27-75): plain C++ with no kernels in it.  It
// takes torch tensors, checks them, allocates the outputs with torch, takes the stream from
// c10::hip::getCurrentHIPStream and the device guard from c10::hip, and calls the C
// ABI of libfast_rnnt_amd.so (include/fast_rnnt_amd.h).  Besides the reference's three
// functions it holds the autograd nodes of the loss functions that are called once per
// training step, so that a loss call costs the host a few microseconds of C++ instead of a
// Python autograd Function and a ctypes call each way.  Everything is also registered with
// the dispatcher as torch.ops.fast_rnnt_amd.*.
//
// Built by fast_rnnt_amd/csrc/Makefile (g++ against the installed torch and pybind11
// headers; no hipify pass, no torch.utils.cpp_extension).
#include <torch/extension.h>
#include <torch/library.h>

#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>

#include <array>
#include <cstring>
#include <mutex>
#include <stdexcept>
#include <string>
#include <tuple>
#include <vector>

#include "fast_rnnt_amd.h"

namespace {

using at::Tensor;
// PyTorch-ROCm labels the MI355X's tensors with device type "cuda"; this is its device guard
// for them (the counterpart of the reference's DeviceGuard, fast_rnnt/csrc/device_guard.h:31-90)
using DeviceGuard = c10::hip::HIPGuardMasqueradingAsCUDA;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// ---- the C ABI, overloaded on the element type -------------------------------------------
inline int abi_mi_forward(const float *px, const float *py, const int64_t *bnd, float *p,
                          float *ans, int B, int S, int T, int modified, int checks,
                          int32_t *status, void *stream) {
  return frnnt_mi_forward_checked_f32(px, py, bnd, p, ans, B, S, T, modified, checks, status,
                                      stream);
}
inline int abi_mi_forward(const double *px, const double *py, const int64_t *bnd, double *p,
                          double *ans, int B, int S, int T, int modified, int checks,
                          int32_t *status, void *stream) {
  return frnnt_mi_forward_checked_f64(px, py, bnd, p, ans, B, S, T, modified, checks, status,
                                      stream);
}
inline int abi_mi_backward(const float *px, const float *py, const int64_t *bnd, const float *p,
                           float *ans_grad, float *gx, float *gy, int B, int S, int T,
                           int modified, int overwrite, void *stream) {
  return frnnt_mi_backward_f32(px, py, bnd, p, ans_grad, gx, gy, B, S, T, modified, overwrite,
                               stream);
}
inline int abi_mi_backward(const double *px, const double *py, const int64_t *bnd,
                           const double *p, double *ans_grad, double *gx, double *gy, int B,
                           int S, int T, int modified, int overwrite, void *stream) {
  return frnnt_mi_backward_f64(px, py, bnd, p, ans_grad, gx, gy, B, S, T, modified, overwrite,
                               stream);
}
#define FRNNT_BOTH(NAME, PARAMS_F, PARAMS_D, ARGS)                       \
  inline int abi_##NAME PARAMS_F { return frnnt_##NAME##_f32 ARGS; }     \
  inline int abi_##NAME PARAMS_D { return frnnt_##NAME##_f64 ARGS; }

FRNNT_BOTH(mi_loss_fwd,
           (const float *px, const float *py, const int64_t *bnd, float *p, float *sc, float *gx,
            float *gy, float *loss, int B, int S, int T, int modified, int red, int checks,
            int32_t *status, void *st),
           (const double *px, const double *py, const int64_t *bnd, double *p, double *sc,
            double *gx, double *gy, double *loss, int B, int S, int T, int modified, int red,
            int checks, int32_t *status, void *st),
           (px, py, bnd, p, sc, gx, gy, loss, B, S, T, modified, red, checks | FRNNT_SCRATCH_P, status,
            st))
FRNNT_BOTH(mi_scale_grads,
           (float *gx, float *gy, const float *g, int gstride, double gscale, int B, int S, int T,
            int modified, void *st),
           (double *gx, double *gy, const double *g, int gstride, double gscale, int B, int S,
            int T, int modified, void *st),
           (gx, gy, g, gstride, gscale, B, S, T, modified, st))
#undef FRNNT_BOTH

void check_rc(int rc, const char *what) {
  TORCH_CHECK(rc == FRNNT_OK, what, " failed (", rc, "): ", frnnt_last_error());
}

template <typename R>
R *ptr(const Tensor &t) {
  return t.defined() ? t.data_ptr<R>() : nullptr;
}
const int64_t *iptr(const Tensor &t) { return t.defined() ? t.data_ptr<int64_t>() : nullptr; }

void *stream_of(const Tensor &t) {
  return static_cast<void *>(c10::hip::getCurrentHIPStream(t.device().index()).stream());
}

Tensor or_undefined(const std::optional<Tensor> &t) { return t.has_value() ? *t : Tensor(); }

// ---- boundary rows that fail their tests: reported by the device, raised later -----------
// The reference's Python layer asserts every boundary row on the host
// (mutual_information.py:277-288, rnnt_loss.py:25-42) through boundary.tolist(), which makes
// every call wait for the device.  Here the forward kernel of the recursion tests the rows
// (it skips a bad one and makes its score NaN) and stores what failed in two words of pinned
// host memory, one pair per device; the host looks at them on entry to every later call of
// this module and in check_boundaries(), and raises the reference's AssertionError then.
// set_deferred_checks(false) makes the Python layer check on the host before the call, as
// the reference does.
struct BoundaryAssertion : public std::runtime_error {
  using std::runtime_error::runtime_error;
};

struct StatusWords {
  int32_t *host = nullptr;
  int32_t *device = nullptr;
};
std::array<StatusWords, 64> g_status;
std::mutex g_status_mutex;
bool g_deferred = true;

StatusWords status_of(int device) {
  TORCH_CHECK(device >= 0 && device < (int)g_status.size(), "device index out of range");
  std::lock_guard<std::mutex> lock(g_status_mutex);
  StatusWords &w = g_status[device];
  if (w.host == nullptr) {
    void *h = nullptr, *d = nullptr;
    TORCH_CHECK(hipHostMalloc(&h, 64, hipHostMallocDefault) == hipSuccess,
                "hipHostMalloc of the boundary status words failed");
    std::memset(h, 0, 64);
    TORCH_CHECK(hipHostGetDevicePointer(&d, h, 0) == hipSuccess,
                "hipHostGetDevicePointer of the boundary status words failed");
    w.host = static_cast<int32_t *>(h);
    w.device = static_cast<int32_t *>(d);
  }
  return w;
}

std::string describe(int code, int row) {
  std::string what;
  switch (code) {
    case FRNNT_STATUS_WINDOW:
      what = "0 <= s_begin <= s_end <= S and 0 <= t_begin <= t_end <= T";
      break;
    case FRNNT_STATUS_NO_SYMBOLS:
      what = "boundary[:, 2] >= 1";
      break;
    case FRNNT_STATUS_FEW_FRAMES:
      what = "T >= S for the modified transducer (boundary[:, 3] >= boundary[:, 2])";
      break;
    default:
      what = "unknown test " + std::to_string(code);
  }
  return "boundary row " + std::to_string(row) + " of an earlier call violates " + what +
         " (found on the device; that call's loss for the row is nan)";
}

// (code, row) of a failure the device has reported on `device`, or (0, 0); clears it.
std::pair<int, int> take_pending(int device) {
  if (device < 0 || device >= (int)g_status.size()) return {0, 0};
  int32_t *h = g_status[device].host;
  if (h == nullptr) return {0, 0};
  const int code = *reinterpret_cast<volatile int32_t *>(h);
  if (code == 0) return {0, 0};
  const int row = *reinterpret_cast<volatile int32_t *>(h + 1);
  h[0] = 0;
  h[1] = 0;
  return {code, row};
}

void raise_pending(int device) {
  const auto pending = take_pending(device);
  if (pending.first != 0) throw BoundaryAssertion(describe(pending.first, pending.second));
}

// Waits for the device, then raises what it has reported.
void check_boundaries(int64_t device) {
  DeviceGuard guard(static_cast<c10::DeviceIndex>(device));
  TORCH_CHECK(hipDeviceSynchronize() == hipSuccess, "hipDeviceSynchronize failed");
  raise_pending((int)device);
}

int32_t *status_for(const Tensor &like, const Tensor &boundary) {
  if (!g_deferred || !boundary.defined()) return nullptr;
  const int device = like.device().index();
  raise_pending(device);
  return status_of(device).device;
}

// ---- the reference's three operator functions -----------------------------------------
struct Dims {
  int B, S, T, modified;
};

Dims common_checks(const Tensor &px, const Tensor &py, const Tensor &boundary, const Tensor &p) {
  TORCH_CHECK(px.dim() == 3, "px must be 3-dimensional");
  TORCH_CHECK(py.dim() == 3, "py must be 3-dimensional.");
  TORCH_CHECK(p.dim() == 3, "p must be 3-dimensional.");
  TORCH_CHECK(px.is_cuda() && py.is_cuda() && p.is_cuda(),
              "inputs must be GPU tensors: fast_rnnt_amd has no CPU path");
  TORCH_CHECK(px.device() == py.device() && px.device() == p.device(),
              "px, py and p must share one device");
  TORCH_CHECK(px.scalar_type() == py.scalar_type() && px.scalar_type() == p.scalar_type(),
              "px, py and p must share one dtype");
  TORCH_CHECK(px.scalar_type() == at::kFloat || px.scalar_type() == at::kDouble,
              "fast_rnnt_amd supports float32 and float64 tensors here, got ", px.scalar_type());
  const int64_t B = px.size(0), S = px.size(1), T1 = px.size(2), T = py.size(2);
  const bool modified = T1 == T;
  TORCH_CHECK(T1 == (modified ? T : T + 1), "px.size(2) must be T or T + 1");
  TORCH_CHECK(py.size(0) == B && py.size(1) == S + 1, "py must have shape [B][S+1][T]");
  TORCH_CHECK(p.size(0) == B && p.size(1) == S + 1 && p.size(2) == T + 1,
              "p must have shape [B][S+1][T+1]");
  if (boundary.defined()) {
    TORCH_CHECK(boundary.dim() == 2, "boundary must be 2-dimensional.");
    TORCH_CHECK(boundary.size(0) == B && boundary.size(1) == 4, "boundary must have shape [B][4]");
    TORCH_CHECK(boundary.device() == px.device() && boundary.scalar_type() == at::kLong,
                "boundary must be an int64 tensor on the same device");
  }
  return Dims{(int)B, (int)S, (int)T, (int)modified};
}

template <typename R>
Tensor mi_forward_t(const Tensor &px, const Tensor &py, const Tensor &boundary, Tensor &p,
                    const Dims &d) {
  Tensor pxc = px.contiguous(), pyc = py.contiguous();
  Tensor bnd = boundary.defined() ? boundary.contiguous() : Tensor();
  Tensor pc = p.is_contiguous() ? p : at::empty(p.sizes(), p.options());
  Tensor ans = at::empty({d.B}, px.options());
  // a bad row also makes ans[b] NaN; the status words only add the AssertionError later
  int32_t *status = status_for(px, bnd);
  check_rc(abi_mi_forward(ptr<R>(pxc), ptr<R>(pyc), iptr(bnd), ptr<R>(pc), ptr<R>(ans), d.B, d.S,
                          d.T, d.modified, 0, status, stream_of(px)),
           "frnnt_mi_forward");
  if (!pc.is_same(p)) p.copy_(pc);
  return ans;
}

// fast_rnnt/python/csrc/mutual_information.cu:27-45
Tensor mutual_information_forward(const Tensor &px, const Tensor &py,
                                  const std::optional<Tensor> &boundary_, Tensor p) {
  const Tensor boundary = or_undefined(boundary_);
  const Dims d = common_checks(px, py, boundary, p);
  DeviceGuard guard(px.device());
  return px.scalar_type() == at::kFloat ? mi_forward_t<float>(px, py, boundary, p, d)
                                        : mi_forward_t<double>(px, py, boundary, p, d);
}

template <typename R>
std::vector<Tensor> mi_backward_t(const Tensor &px, const Tensor &py, const Tensor &boundary,
                                  const Tensor &p, Tensor &ans_grad, const Dims &d) {
  Tensor pxc = px.contiguous(), pyc = py.contiguous(), pc = p.contiguous();
  Tensor bnd = boundary.defined() ? boundary.contiguous() : Tensor();
  Tensor agc = ans_grad.contiguous();
  Tensor gx = at::empty(pxc.sizes(), pxc.options()), gy = at::empty(pyc.sizes(), pyc.options());
  check_rc(abi_mi_backward(ptr<R>(pxc), ptr<R>(pyc), iptr(bnd), ptr<R>(pc), ptr<R>(agc),
                           ptr<R>(gx), ptr<R>(gy), d.B, d.S, d.T, d.modified, 1, stream_of(px)),
           "frnnt_mi_backward");
  if (!agc.is_same(ans_grad)) ans_grad.copy_(agc);
  return {gx, gy};
}

// fast_rnnt/python/csrc/mutual_information.cu:47-67.  Like the reference's GPU path
// (mutual_information_cuda.cu:667-669) ans_grad is overwritten with the gradient that
// reaches the start of each lattice.
std::vector<Tensor> mutual_information_backward(const Tensor &px, const Tensor &py,
                                                const std::optional<Tensor> &boundary_,
                                                const Tensor &p, Tensor ans_grad) {
  const Tensor boundary = or_undefined(boundary_);
  const Dims d = common_checks(px, py, boundary, p);
  TORCH_CHECK(ans_grad.dim() == 1, "ans_grad must be 1-dimensional.");
  TORCH_CHECK(ans_grad.size(0) == d.B, "ans_grad must have B elements");
  TORCH_CHECK(ans_grad.device() == px.device() && ans_grad.scalar_type() == px.scalar_type(),
              "ans_grad must match px in device and dtype");
  DeviceGuard guard(px.device());
  return px.scalar_type() == at::kFloat ? mi_backward_t<float>(px, py, boundary, p, ans_grad, d)
                                        : mi_backward_t<double>(px, py, boundary, p, ans_grad, d);
}

// fast_rnnt/python/csrc/mutual_information.cu:69-75: PyTorch-ROCm shows the MI355X as
// device type "cuda".
bool with_cuda() { return true; }

// ---- the tail every loss shares: recursion, its eager backward, the reduction ------------
// One autograd node: forward = frnnt_mi_loss_fwd (recursion, its backward with a gradient of
// ones as mutual_information.py:159-168 does whenever gradients will be wanted, and the
// reduction rnnt_loss.py:326-340); backward = frnnt_mi_scale_grads, the in-place scaling of
// the occupation gradients by the gradient of the scores (mutual_information.py:173-181),
// with the reduction's sign and 1/B folded in.
constexpr int kRedNone = 0, kRedMean = 1;

// The occupation gradients of a node that has scaled them in place: a second backward through it
// (retain_graph=True) finds its saved tensors changed and raises, as after torch's own "*=" in
// mutual_information.py:179-180, instead of scaling them twice.
void count_as_changed(const Tensor &gx, const Tensor &gy) {
  gx.unsafeGetTensorImpl()->bump_version();
  gy.unsafeGetTensorImpl()->bump_version();
}

// element offsets of consecutive buffers, each 16-byte aligned for 4- and 8-byte elements
struct Carver {
  int64_t total = 0;
  int64_t take(int64_t n) {
    const int64_t at = total;
    total += (n + 3) & ~int64_t(3);
    return at;
  }
};

struct RecursionLossFn : public torch::autograd::Function<RecursionLossFn> {
  // (an absent boundary travels as an empty optional: the autograd machinery does not take
  // undefined tensors as inputs)
  static variable_list forward(AutogradContext *ctx, const Tensor &px, const Tensor &py,
                               const std::optional<Tensor> &boundary_, bool want_grads,
                               int64_t reduction, int64_t checks, bool need_grad) {
    const Tensor boundary = or_undefined(boundary_);
    return px.scalar_type() == at::kFloat
               ? run<float>(ctx, px, py, boundary, want_grads, reduction, checks, need_grad)
               : run<double>(ctx, px, py, boundary, want_grads, reduction, checks, need_grad);
  }

  template <typename R>
  static variable_list run(AutogradContext *ctx, const Tensor &px_, const Tensor &py_,
                           const Tensor &boundary, bool want_grads, int64_t reduction,
                           int64_t checks, bool need_grad) {
    const Tensor px = px_.contiguous(), py = py_.contiguous();
    const int64_t B = px.size(0), S = px.size(1), T1 = px.size(2), T = py.size(2);
    const Tensor bnd = boundary.defined() ? boundary.contiguous() : Tensor();
    ctx->set_materialize_grads(false);
    DeviceGuard guard(px.device());
    const auto opts = px.options();
    Tensor p = at::empty({B, S + 1, T + 1}, opts), scores = at::empty({B}, opts);
    Tensor gx, gy;
    if (want_grads || need_grad) {
      gx = at::empty({B, S, T1}, opts);
      gy = at::empty({B, S + 1, T}, opts);
    }
    Tensor loss = reduction == kRedNone ? at::empty({B}, opts) : at::empty({}, opts);
    check_rc(abi_mi_loss_fwd(ptr<R>(px), ptr<R>(py), iptr(bnd), ptr<R>(p), ptr<R>(scores),
                             ptr<R>(gx), ptr<R>(gy), ptr<R>(loss), (int)B, (int)S, (int)T,
                             (int)(T1 == T), (int)reduction, (int)checks, status_for(px, bnd),
                             stream_of(px)),
             "frnnt_mi_loss_fwd");
    if (need_grad) {
      ctx->save_for_backward({gx, gy});
      ctx->saved_data["reduction"] = reduction;
    }
    // (undefined tensors cannot be outputs of an autograd node)
    if (!gx.defined()) return {loss};
    ctx->mark_non_differentiable({gx, gy});
    return {loss, gx, gy};
  }

  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    variable_list out(7);
    const Tensor &g_loss = grads[0];
    if (!g_loss.defined()) return out;
    const auto saved = ctx->get_saved_variables();
    Tensor gx = saved[0], gy = saved[1];
    const int64_t reduction = ctx->saved_data["reduction"].toInt();
    const int64_t B = gx.size(0), S = gx.size(1), T1 = gx.size(2), T = gy.size(2);
    DeviceGuard guard(gx.device());
    const Tensor g = g_loss.contiguous();
    const int stride = reduction == kRedNone ? 1 : 0;
    const double scale = reduction == kRedMean ? -1.0 / (double)B : -1.0;
    int rc;
    if (gx.scalar_type() == at::kFloat)
      rc = abi_mi_scale_grads(ptr<float>(gx), ptr<float>(gy), ptr<float>(g), stride, scale,
                              (int)B, (int)S, (int)T, (int)(T1 == T), stream_of(gx));
    else
      rc = abi_mi_scale_grads(ptr<double>(gx), ptr<double>(gy), ptr<double>(g), stride, scale,
                              (int)B, (int)S, (int)T, (int)(T1 == T), stream_of(gx));
    check_rc(rc, "frnnt_mi_scale_grads");
    count_as_changed(gx, gy);
    out[0] = gx;
    out[1] = gy;
    return out;
  }
};

// mutual_information_recursion (mutual_information.py:24-181) behind one autograd node: the scores,
// the occupation gradients where they are handed out or a gradient may be wanted, and their
// in-place scaling in the backward.  Unless they are handed out nobody else holds them by then, so
// that px.grad and py.grad take them over without a copy; and in float32 they are formed then, from
// the gradient of the scores, instead of in the forward and scaled afterwards (a pass over both:
// 12 us of 144 at B 12, S 220, T 1500).  Kept until then are the shares, one lattice
// instead of two, and a copy of the boundary: the caller may write to its own.
struct RecursionFn : public torch::autograd::Function<RecursionFn> {
  static variable_list forward(AutogradContext *ctx, const Tensor &px_, const Tensor &py_,
                               const std::optional<Tensor> &boundary_, bool want_grads,
                               bool need_grad) {
    const Tensor boundary = or_undefined(boundary_);
    const Tensor px = px_.contiguous(), py = py_.contiguous();
    const Tensor bnd = boundary.defined() ? boundary.contiguous() : Tensor();
    const int64_t B = px.size(0), S = px.size(1), T1 = px.size(2), T = py.size(2);
    ctx->set_materialize_grads(false);
    DeviceGuard guard(px.device());
    const auto opts = px.options();
    Tensor scores = at::empty({B}, opts);
    if (need_grad && !want_grads && px.scalar_type() == at::kFloat) {
      const Tensor kept = at::empty({frnnt_mi_kept_size((int)B, (int)S, (int)T)}, opts);
      check_rc(frnnt_mi_kept_fwd_f32(ptr<float>(px), ptr<float>(py), iptr(bnd), ptr<float>(kept),
                                     ptr<float>(scores), (int)B, (int)S, (int)T, (int)(T1 == T), 0,
                                     status_for(px, bnd), stream_of(px)),
               "frnnt_mi_kept_fwd");
      ctx->save_for_backward({kept});
      ctx->saved_data["sizes"] = std::vector<int64_t>{B, S, T1, T, bnd.defined()};
      return {scores};
    }
    Tensor p = at::empty({B, S + 1, T + 1}, opts), gx, gy;
    if (want_grads || need_grad) {
      gx = at::empty({B, S, T1}, opts);
      gy = at::empty({B, S + 1, T}, opts);
    }
    auto run = [&](auto r) {
      using R = decltype(r);
      return abi_mi_loss_fwd(ptr<R>(px), ptr<R>(py), iptr(bnd), ptr<R>(p), ptr<R>(scores),
                             ptr<R>(gx), ptr<R>(gy), (R *)nullptr, (int)B, (int)S, (int)T,
                             (int)(T1 == T), 0, 0, status_for(px, bnd), stream_of(px));
    };
    check_rc(px.scalar_type() == at::kFloat ? run(float()) : run(double()), "frnnt_mi_loss_fwd");
    if (need_grad) ctx->save_for_backward({gx, gy});
    if (!want_grads) return {scores};
    ctx->mark_non_differentiable({gx, gy});
    return {scores, gx, gy};
  }

  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    if (!grads[0].defined()) return variable_list(5);
    const auto saved = ctx->get_saved_variables();
    const auto sizes = ctx->saved_data.find("sizes");
    const bool of_shares = sizes != ctx->saved_data.end();
    DeviceGuard guard(saved[0].device());
    Tensor gx, gy;
    int has_boundary = 0;
    if (of_shares) {
      const auto n = sizes->second.toIntVector();
      has_boundary = (int)n[4];
      gx = at::empty({n[0], n[1], n[2]}, saved[0].options());
      gy = at::empty({n[0], n[1] + 1, n[3]}, saved[0].options());
    } else {
      gx = saved[0];
      gy = saved[1];
    }
    const int64_t B = gx.size(0), S = gx.size(1), T1 = gx.size(2), T = gy.size(2);
    const bool one_for_all = B > 1 && grads[0].stride(0) == 0;  // (e.g. of a sum)
    const Tensor g = one_for_all ? grads[0] : grads[0].contiguous();
    const bool on_record = at::GradMode::is_enabled() && g.requires_grad();
    if (of_shares) {
      check_rc(frnnt_mi_kept_bwd_f32(ptr<float>(saved[0]), has_boundary, on_record ? nullptr : ptr<float>(g),
                                     one_for_all ? 0 : 1, ptr<float>(gx), ptr<float>(gy), (int)B, (int)S,
                                     (int)T, (int)(T1 == T), stream_of(gx)),
               "frnnt_mi_kept_bwd");
      // (a second backward is refused as where the gradients are scaled in place)
      saved[0].unsafeGetTensorImpl()->bump_version();
      if (!on_record) return {gx, gy, Tensor(), Tensor(), Tensor()};
    }
    if (on_record) {
      // (differentiated itself, e.g. with respect to weights of the scores: an operation on record)
      const Tensor f = g.view({B, 1, 1});
      return {gx.mul_(f), gy.mul_(f), Tensor(), Tensor(), Tensor()};
    }
    auto run = [&](auto r) {
      using R = decltype(r);
      return abi_mi_scale_grads(ptr<R>(gx), ptr<R>(gy), ptr<R>(g), one_for_all ? 0 : 1, 1.0, (int)B, (int)S, (int)T,
                                (int)(T1 == T), stream_of(gx));
    };
    check_rc(gx.scalar_type() == at::kFloat ? run(float()) : run(double()), "frnnt_mi_scale_grads");
    count_as_changed(gx, gy);
    return {gx, gy, Tensor(), Tensor(), Tensor()};
  }
};

void require_float_gpu(const Tensor &t, const char *name) {
  TORCH_CHECK(t.is_cuda(), "fast_rnnt_amd runs on GPU tensors only (no CPU path): ", name);
  TORCH_CHECK(t.scalar_type() == at::kFloat || t.scalar_type() == at::kDouble,
              "fast_rnnt_amd supports float32 and float64 tensors here, got ", t.scalar_type());
}

using LossResult = std::tuple<Tensor, std::optional<Tensor>, std::optional<Tensor>>;

LossResult as_result(const variable_list &out) {
  std::optional<Tensor> gx, gy;
  if (out.size() == 3) {
    gx = out[1];
    gy = out[2];
  }
  return LossResult(out[0], gx, gy);
}

LossResult recursion(const Tensor &px, const Tensor &py, const std::optional<Tensor> &boundary_,
                     bool return_grad) {
  const Tensor boundary = or_undefined(boundary_);
  require_float_gpu(px, "px");
  TORCH_CHECK(px.dim() == 3 && py.dim() == 3, "px and py must be 3-dimensional");
  const int64_t B = px.size(0), S = px.size(1), T1 = px.size(2), T = py.size(2);
  TORCH_CHECK((T1 == T || T1 == T + 1) && py.size(0) == B && py.size(1) == S + 1,
              "px must be [B][S][T or T+1], py [B][S+1][T]");
  TORCH_CHECK(px.device() == py.device() && px.scalar_type() == py.scalar_type(),
              "px and py must share one device and one dtype");
  if (boundary.defined())
    TORCH_CHECK(boundary.dim() == 2 && boundary.size(0) == B && boundary.size(1) == 4 &&
                    boundary.scalar_type() == at::kLong && boundary.device() == px.device(),
                "boundary must be an int64 [B][4] tensor on the same device");
  const bool need_grad = at::GradMode::is_enabled() && (px.requires_grad() || py.requires_grad());
  return as_result(RecursionFn::apply(px, py, boundary_, return_grad, need_grad));
}

LossResult recursion_loss(const Tensor &px, const Tensor &py,
                          const std::optional<Tensor> &boundary_, bool return_grad,
                          int64_t reduction, int64_t checks) {
  const Tensor boundary = or_undefined(boundary_);
  require_float_gpu(px, "px");
  TORCH_CHECK(px.dim() == 3 && py.dim() == 3, "px and py must be 3-dimensional");
  TORCH_CHECK(py.device() == px.device() && py.scalar_type() == px.scalar_type(),
              "px and py must share device and dtype");
  const int64_t B = px.size(0), S = px.size(1), T1 = px.size(2), T = py.size(2);
  TORCH_CHECK((T1 == T || T1 == T + 1) && py.size(0) == B && py.size(1) == S + 1,
              "px must be [B][S][T or T+1] and py [B][S+1][T]");
  TORCH_CHECK(reduction >= 0 && reduction <= 2, "reduction must be 0 (none), 1 (mean) or 2 (sum)");
  if (boundary.defined())
    TORCH_CHECK(boundary.dim() == 2 && boundary.size(0) == B && boundary.size(1) == 4 &&
                    boundary.scalar_type() == at::kLong && boundary.device() == px.device(),
                "boundary must be an int64 [B][4] tensor on the same device");
  const bool need_grad = at::GradMode::is_enabled() && (px.requires_grad() || py.requires_grad());
  return as_result(
      RecursionLossFn::apply(px, py, boundary_, return_grad, reduction, checks, need_grad));
}

// ---- rnnt_loss_simple behind one autograd node -------------------------------------------
// forward = frnnt_additive_loss_fwd: px / py (row maxima + MFMA contraction, rnnt_loss.py:66-227,
// the delay penalty :309-324), the recursion, its backward with a gradient of ones
// (mutual_information.py:159-168), the reduction (rnnt_loss.py:326-340);
// backward = frnnt_additive_loss_bwd: scales the occupation gradients in place by the
// gradient of the scores (mutual_information.py:173-181) and pushes them through the two
// gradient products to lm.grad and am.grad.  float16 / bfloat16 inputs are widened by the first
// kernel and their gradients written in their type; everything between is float32.
int dtype_code(at::ScalarType t) {
  return t == at::kFloat ? FRNNT_F32 : t == at::kDouble ? FRNNT_F64 : t == at::kHalf ? FRNNT_F16 : FRNNT_BF16;
}

struct SimpleLossFn : public torch::autograd::Function<SimpleLossFn> {
  static variable_list forward(AutogradContext *ctx, const Tensor &lm_, const Tensor &am_,
                               const Tensor &symbols, const std::optional<Tensor> &boundary_,
                               int64_t term, int64_t kind, double delay_penalty, bool want_grads,
                               int64_t reduction, int64_t checks, bool need_lm, bool need_am) {
    const Tensor boundary = or_undefined(boundary_);
    const Tensor lm = lm_.contiguous(), am = am_.contiguous(), sym = symbols.contiguous();
    const Tensor bnd = boundary.defined() ? boundary.contiguous() : Tensor();
    const int64_t B = am.size(0), T = am.size(1), C = am.size(2), S = lm.size(1) - 1;
    const int64_t T1 = kind == 0 ? T + 1 : T;
    const bool need_grad = need_lm || need_am;
    const int dtype = dtype_code(am.scalar_type());
    const bool narrow = dtype >= FRNNT_F16;
    ctx->set_materialize_grads(false);
    DeviceGuard guard(am.device());
    const auto opts = am.options().dtype(narrow ? at::kFloat : am.scalar_type());
    const int64_t item = dtype == FRNNT_F64 ? 8 : 4;
    // what the backward reads, in one allocation: lm_max | am_max | norm_raw | wide lm | wide am
    const int64_t n_py = B * (S + 1) * T;
    Carver keep;
    const int64_t o_lmx = keep.take(B * (S + 1)), o_amx = keep.take(B * T),
                  o_nr = keep.take(need_grad ? n_py : 0),
                  o_lmw = keep.take(narrow ? B * (S + 1) * C : 0),
                  o_amw = keep.take(narrow ? B * T * C : 0);
    Tensor kept = at::empty({keep.total}, opts);
    // what it does not: px | py | p | scores
    Carver carve;
    const int64_t n_p = dtype == FRNNT_F64 ? B * (S + 1) * (T + 1)
                                           : frnnt_loss_scratch((int)B, (int)S, (int)T, (int)C, bnd.defined());
    const int64_t o_px = carve.take(B * S * T1), o_py = carve.take(n_py), o_p = carve.take(n_p),
                  o_sc = carve.take(B);
    const Tensor work = at::empty({carve.total}, opts);
    char *k = static_cast<char *>(kept.data_ptr()), *w = static_cast<char *>(work.data_ptr());
    Tensor gx, gy;
    if (want_grads || need_grad) {
      gx = at::empty({B, S, T1}, opts);
      gy = at::empty({B, S + 1, T}, opts);
    }
    Tensor loss = reduction == kRedNone ? at::empty({B}, opts) : at::empty({}, opts);
    check_rc(frnnt_additive_loss_fwd(
                 dtype, lm.data_ptr(), am.data_ptr(), iptr(sym), iptr(bnd),
                 narrow ? k + o_lmw * item : nullptr, narrow ? k + o_amw * item : nullptr,
                 w + o_px * item, w + o_py * item, k + o_lmx * item, k + o_amx * item,
                 need_grad ? k + o_nr * item : nullptr, w + o_p * item, w + o_sc * item,
                 gx.defined() ? gx.data_ptr() : nullptr, gy.defined() ? gy.data_ptr() : nullptr,
                 loss.data_ptr(), (int)B, (int)S, (int)T, (int)C,
                 (int)term, (int)kind, delay_penalty, (int)reduction,
                 (int)checks | FRNNT_SCRATCH_P | FRNNT_LARGE_SCRATCH,
                 status_for(am, bnd), stream_of(am)),
             "frnnt_additive_loss_fwd");
    if (need_grad) {
      // (an absent boundary is not saved: saved tensors must be defined)
      variable_list save{lm, am, sym, kept, gx, gy};
      if (bnd.defined()) save.push_back(bnd);
      ctx->save_for_backward(std::move(save));
      ctx->saved_data["meta"] = std::vector<int64_t>{term, kind, reduction, need_lm, need_am};
    }
    // (undefined tensors cannot be outputs of an autograd node)
    if (!gx.defined()) return {loss};
    ctx->mark_non_differentiable({gx, gy});
    return {loss, gx, gy};
  }

  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    variable_list out(12);
    const Tensor &g_loss = grads[0];
    if (!g_loss.defined()) return out;
    const auto saved = ctx->get_saved_variables();
    const Tensor &lm = saved[0], &am = saved[1], &sym = saved[2], &kept = saved[3];
    Tensor gx = saved[4], gy = saved[5];
    const Tensor bnd = saved.size() > 6 ? saved[6] : Tensor();
    const std::vector<int64_t> meta = ctx->saved_data["meta"].toIntVector();
    const int64_t reduction = meta[2];
    const int64_t B = am.size(0), T = am.size(1), C = am.size(2), S = lm.size(1) - 1;
    const int dtype = dtype_code(am.scalar_type());
    const bool narrow = dtype >= FRNNT_F16;
    const int64_t item = dtype == FRNNT_F64 ? 8 : 4;
    DeviceGuard guard(am.device());
    // (the forward's layout)
    Carver keep;
    const int64_t o_lmx = keep.take(B * (S + 1)), o_amx = keep.take(B * T),
                  o_nr = keep.take(B * (S + 1) * T), o_lmw = keep.take(narrow ? B * (S + 1) * C : 0),
                  o_amw = keep.take(narrow ? B * T * C : 0);
    char *k = static_cast<char *>(kept.data_ptr());
    // d loss / d scores[b] = scale * g_loss[b * stride]
    const Tensor g = g_loss.contiguous();
    const int stride = reduction == kRedNone ? 1 : 0;
    const double scale = reduction == kRedMean ? -1.0 / (double)B : -1.0;
    const int64_t ldd = (T + 3) / 4 * 4;
    // scratch in one allocation: dmat | row_x | row_y | col_y
    Carver carve;
    const int64_t o_d = carve.take(B * (S + 1) * ldd), o_rx = carve.take(B * (S + 1)),
                  o_ry = carve.take(B * (S + 1)), o_cy = carve.take(B * T);
    const Tensor scratch = at::empty({carve.total}, kept.options());
    char *s = static_cast<char *>(scratch.data_ptr());
    if (meta[3]) out[0] = at::empty(lm.sizes(), lm.options());
    if (meta[4]) out[1] = at::empty(am.sizes(), am.options());
    // gx / gy are scaled in place by the scores' gradient, exactly as the recursion's autograd
    // node does to the tensors it handed out
    check_rc(frnnt_additive_loss_bwd(
                 dtype, narrow ? k + o_lmw * item : lm.data_ptr(),
                 narrow ? k + o_amw * item : am.data_ptr(), iptr(sym), iptr(bnd), k + o_lmx * item,
                 k + o_amx * item, k + o_nr * item, g.data_ptr(), stride, scale, gx.data_ptr(),
                 gy.data_ptr(), s + o_d * item, s + o_rx * item, s + o_ry * item, s + o_cy * item,
                 meta[3] ? out[0].data_ptr() : nullptr, meta[4] ? out[1].data_ptr() : nullptr,
                 (int)B, (int)S, (int)T, (int)C, (int)meta[0], (int)meta[1], stream_of(am)),
             "frnnt_additive_loss_bwd");
    count_as_changed(gx, gy);
    return out;
  }
};

void check_additive(const Tensor &lm, const Tensor &am, const Tensor &symbols,
                    const Tensor &boundary) {
  TORCH_CHECK(lm.dim() == 3 && am.dim() == 3 && symbols.dim() == 2,
              "lm and am must be 3-dimensional, symbols 2-dimensional");
  const int64_t B = am.size(0), S = lm.size(1) - 1;
  TORCH_CHECK(lm.size(0) == B && lm.size(2) == am.size(2) && symbols.size(0) == B &&
                  symbols.size(1) == S,
              "lm must be [B][S+1][C], am [B][T][C], symbols [B][S]");
  TORCH_CHECK(lm.device() == am.device() && symbols.device() == am.device(),
              "all tensors must be on the same device");
  TORCH_CHECK(lm.scalar_type() == am.scalar_type(),
              "floating-point tensors must share one dtype");
  TORCH_CHECK(symbols.scalar_type() == at::kLong, "symbols must be an int64 tensor, got ",
              symbols.scalar_type());
  if (boundary.defined())
    TORCH_CHECK(boundary.dim() == 2 && boundary.size(0) == B && boundary.size(1) == 4 &&
                    boundary.scalar_type() == at::kLong && boundary.device() == am.device(),
                "boundary must be an int64 [B][4] tensor on the same device");
}

LossResult simple_loss(const Tensor &lm, const Tensor &am, const Tensor &symbols,
                       const std::optional<Tensor> &boundary_, int64_t termination_symbol,
                       int64_t rnnt_type, double delay_penalty, bool return_grad,
                       int64_t reduction, int64_t checks) {
  const Tensor boundary = or_undefined(boundary_);
  if (am.scalar_type() != at::kHalf && am.scalar_type() != at::kBFloat16) require_float_gpu(am, "am");
  TORCH_CHECK(am.is_cuda(), "fast_rnnt_amd runs on GPU tensors only (no CPU path): am");
  check_additive(lm, am, symbols, boundary);
  TORCH_CHECK(rnnt_type >= 0 && rnnt_type <= 2, "rnnt_type must be 0, 1 or 2");
  TORCH_CHECK(reduction >= 0 && reduction <= 2, "reduction must be 0 (none), 1 (mean) or 2 (sum)");
  const bool grad_mode = at::GradMode::is_enabled();
  const bool need_lm = grad_mode && lm.requires_grad(), need_am = grad_mode && am.requires_grad();
  return as_result(SimpleLossFn::apply(lm, am, symbols, boundary_, termination_symbol, rnnt_type,
                                       delay_penalty, return_grad, reduction, checks, need_lm,
                                       need_am));
}

// ---- rnnt_loss_smoothed behind one autograd node (float32) -----------------------------------
// forward = frnnt_smoothed_loss_fwd, backward = frnnt_smoothed_loss_bwd: the joint model's node
// above with the lm-only and am-only models' terms folded into its kernels.
struct SmoothedLossFn : public torch::autograd::Function<SmoothedLossFn> {
  static variable_list forward(AutogradContext *ctx, const Tensor &lm_, const Tensor &am_,
                               const Tensor &symbols, const std::optional<Tensor> &boundary_,
                               int64_t term, int64_t kind, double lm_scale, double am_scale,
                               double delay_penalty, bool want_grads, int64_t reduction,
                               int64_t checks, bool need_grad) {
    const Tensor boundary = or_undefined(boundary_);
    const Tensor lm = lm_.contiguous(), am = am_.contiguous(), sym = symbols.contiguous();
    const Tensor bnd = boundary.defined() ? boundary.contiguous() : Tensor();
    const int64_t B = am.size(0), T = am.size(1), C = am.size(2), S = lm.size(1) - 1;
    const int64_t T1 = kind == 0 ? T + 1 : T;
    ctx->set_materialize_grads(false);
    DeviceGuard guard(am.device());
    const auto opts = am.options();
    Tensor kept = at::empty({frnnt_smoothed_loss_kept((int)B, (int)S, (int)T, (int)C)}, opts);
    const int64_t n_px = B * S * T1, n_py = B * (S + 1) * T;
    Carver carve;
    const int64_t o_px = carve.take(n_px),
                  o_py = carve.take(n_py),
                  o_p = carve.take(frnnt_loss_scratch((int)B, (int)S, (int)T, (int)C, bnd.defined())),
                  o_sc = carve.take(B), o_part = carve.take((B * (S + 1) + 15) / 16 * C);
    const Tensor work = at::empty({carve.total}, opts);
    float *w = work.data_ptr<float>();
    Tensor gx, gy;
    if (want_grads || need_grad) {
      gx = at::empty({B, S, T1}, opts);
      gy = at::empty({B, S + 1, T}, opts);
    }
    Tensor loss = reduction == kRedNone ? at::empty({B}, opts) : at::empty({}, opts);
    check_rc(frnnt_smoothed_loss_fwd_f32(
                 ptr<float>(lm), ptr<float>(am), iptr(sym), iptr(bnd), nullptr, nullptr, w + o_px,
                 w + o_py, ptr<float>(kept), w + o_part, w + o_p, w + o_sc, ptr<float>(gx),
                 ptr<float>(gy), ptr<float>(loss), (int)B, (int)S, (int)T, (int)C, (int)term,
                 (int)kind, lm_scale, am_scale, delay_penalty, (int)reduction,
                 (int)checks | FRNNT_LARGE_SCRATCH, status_for(am, bnd), stream_of(am)),
             "frnnt_smoothed_loss_fwd");
    if (need_grad) {
      // (the constrained lattice's backward reads the copy of the boundary in `kept`: its caller may write to the
      // tensor itself, as where the backward did not need it)
      variable_list save{lm, am, sym, kept, gx, gy};
      const bool copied = kind == 2 && bnd.defined();
      if (bnd.defined() && !copied) save.push_back(bnd);
      ctx->save_for_backward(std::move(save));
      ctx->saved_data["meta"] = std::vector<int64_t>{term, kind, reduction, copied};
      ctx->saved_data["scales"] = std::vector<double>{lm_scale, am_scale};
    }
    if (!gx.defined()) return {loss};
    ctx->mark_non_differentiable({gx, gy});
    return {loss, gx, gy};
  }

  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    variable_list out(13);
    const Tensor &g_loss = grads[0];
    if (!g_loss.defined()) return out;
    const auto saved = ctx->get_saved_variables();
    const Tensor &lm = saved[0], &am = saved[1], &sym = saved[2], &kept = saved[3];
    Tensor gx = saved[4], gy = saved[5];
    const Tensor bnd = saved.size() > 6 ? saved[6] : Tensor();
    const std::vector<int64_t> meta = ctx->saved_data["meta"].toIntVector();
    const std::vector<double> scales = ctx->saved_data["scales"].toDoubleVector();
    const int64_t reduction = meta[2];
    const int64_t B = am.size(0), T = am.size(1), C = am.size(2), S = lm.size(1) - 1;
    const int64_t *rows =
        meta[3] ? reinterpret_cast<const int64_t *>(ptr<float>(kept) + kept.numel() - 8 * B) : iptr(bnd);
    DeviceGuard guard(am.device());
    const Tensor g = g_loss.contiguous();
    const Tensor scratch =
        at::empty({B * (S + 1) * (4 + (T + 3) / 4 * 4) + 2 * B * T + C + (B * T + 15) / 16 * C + 40},
                  am.options());
    out[0] = at::empty(lm.sizes(), lm.options());
    out[1] = at::empty(am.sizes(), am.options());
    check_rc(frnnt_smoothed_loss_bwd_f32(
                 ptr<float>(lm), ptr<float>(am), iptr(sym), rows, ptr<float>(kept),
                 ptr<float>(g), reduction == kRedNone ? 1 : 0,
                 reduction == kRedMean ? -1.0 / (double)B : -1.0, ptr<float>(gx), ptr<float>(gy),
                 ptr<float>(scratch), ptr<float>(out[0]), ptr<float>(out[1]), (int)B, (int)S, (int)T,
                 (int)C, (int)meta[0], (int)meta[1], scales[0], scales[1], stream_of(am)),
             "frnnt_smoothed_loss_bwd");
    count_as_changed(gx, gy);
    return out;
  }
};

LossResult smoothed_loss(const Tensor &lm, const Tensor &am, const Tensor &symbols,
                         const std::optional<Tensor> &boundary_, int64_t termination_symbol,
                         int64_t rnnt_type, double lm_only_scale, double am_only_scale,
                         double delay_penalty, bool return_grad, int64_t reduction,
                         int64_t checks) {
  require_float_gpu(am, "am");
  TORCH_CHECK(am.scalar_type() == at::kFloat, "smoothed_loss takes float32 tensors");
  check_additive(lm, am, symbols, or_undefined(boundary_));
  TORCH_CHECK(rnnt_type >= 0 && rnnt_type <= 2, "rnnt_type must be 0, 1 or 2");
  TORCH_CHECK(reduction >= 0 && reduction <= 2, "reduction must be 0 (none), 1 (mean) or 2 (sum)");
  const bool need_grad = at::GradMode::is_enabled() && (lm.requires_grad() || am.requires_grad());
  return as_result(SmoothedLossFn::apply(lm, am, symbols, boundary_, termination_symbol, rnnt_type,
                                         lm_only_scale, am_only_scale, delay_penalty, return_grad,
                                         reduction, checks, need_grad));
}

// ---- rnnt_loss and rnnt_loss_pruned behind one autograd node ------------------------------
// forward = frnnt_lattice_loss_fwd: px / py from the logits (rnnt_loss.py:343-449, :856-1024), the
// recursion, its backward with a gradient of ones, the reduction; backward =
// frnnt_lattice_loss_bwd.  Occupation gradients that were handed out are scaled in place first
// (mutual_information.py:173-181); otherwise their scale is applied as they are read.
inline int abi_lattice_loss_fwd(at::ScalarType type, const void *logits, const int64_t *sym,
                                const int64_t *rng, const int64_t *bnd, float *px, float *py,
                                float *norm, float *xr, float *yr, float *p, float *sc, float *gx,
                                float *gy, float *loss, int B, int S, int T, int R, int C,
                                int term, int kind, double delay, int red, int checks,
                                int32_t *status, void *st) {
  if (type == at::kFloat)
    return frnnt_lattice_loss_fwd_f32(static_cast<const float *>(logits), sym, rng, bnd, px, py,
                                      norm, xr, yr, p, sc, gx, gy, loss, B, S, T, R, C, term, kind,
                                      delay, red, checks, status, st);
  return (type == at::kHalf ? frnnt_lattice_loss_fwd_f16 : frnnt_lattice_loss_fwd_bf16)(
      logits, sym, rng, bnd, px, py, norm, xr, yr, p, sc, gx, gy, loss, B, S, T, R, C, term, kind,
      delay, red, checks, status, st);
}
inline int abi_lattice_loss_fwd(at::ScalarType, const void *logits, const int64_t *sym,
                                const int64_t *rng, const int64_t *bnd, double *px, double *py,
                                double *norm, double *xr, double *yr, double *p, double *sc,
                                double *gx, double *gy, double *loss, int B, int S, int T, int R,
                                int C, int term, int kind, double delay, int red, int checks,
                                int32_t *status, void *st) {
  return frnnt_lattice_loss_fwd_f64(static_cast<const double *>(logits), sym, rng, bnd, px, py,
                                    norm, xr, yr, p, sc, gx, gy, loss, B, S, T, R, C, term, kind,
                                    delay, red, checks, status, st);
}
inline int abi_lattice_loss_bwd(at::ScalarType type, const void *logits, const int64_t *sym,
                                const int64_t *rng, const int64_t *bnd, const float *norm,
                                const float *g, int gstride, double gscale, const float *gx,
                                const float *gy, void *out, int B, int S, int T, int R, int C,
                                int term, int kind, void *st) {
  if (type == at::kFloat)
    return frnnt_lattice_loss_bwd_f32(static_cast<const float *>(logits), sym, rng, bnd, norm, g,
                                      gstride, gscale, gx, gy, static_cast<float *>(out), B, S, T,
                                      R, C, term, kind, st);
  return (type == at::kHalf ? frnnt_lattice_loss_bwd_f16 : frnnt_lattice_loss_bwd_bf16)(
      logits, sym, rng, bnd, norm, g, gstride, gscale, gx, gy, out, B, S, T, R, C, term, kind, st);
}
inline int abi_lattice_loss_bwd(at::ScalarType, const void *logits, const int64_t *sym,
                                const int64_t *rng, const int64_t *bnd, const double *norm,
                                const double *g, int gstride, double gscale, const double *gx,
                                const double *gy, void *out, int B, int S, int T, int R, int C,
                                int term, int kind, void *st) {
  return frnnt_lattice_loss_bwd_f64(static_cast<const double *>(logits), sym, rng, bnd, norm, g,
                                    gstride, gscale, gx, gy, static_cast<double *>(out), B, S, T,
                                    R, C, term, kind, st);
}

struct LatticeLossFn : public torch::autograd::Function<LatticeLossFn> {
  static variable_list forward(AutogradContext *ctx, const Tensor &logits, const Tensor &symbols,
                               const std::optional<Tensor> &ranges,
                               const std::optional<Tensor> &boundary, int64_t term, int64_t kind,
                               double delay_penalty, bool want_grads, int64_t reduction,
                               int64_t checks, bool need_grad) {
    return logits.scalar_type() == at::kDouble
               ? run<double>(ctx, logits, symbols, or_undefined(ranges), or_undefined(boundary),
                             term, kind, delay_penalty, want_grads, reduction, checks, need_grad)
               : run<float>(ctx, logits, symbols, or_undefined(ranges), or_undefined(boundary),
                            term, kind, delay_penalty, want_grads, reduction, checks, need_grad);
  }

  template <typename R>
  static variable_list run(AutogradContext *ctx, const Tensor &logits_, const Tensor &symbols,
                           const Tensor &ranges, const Tensor &boundary, int64_t term,
                           int64_t kind, double delay_penalty, bool want_grads, int64_t reduction,
                           int64_t checks, bool need_grad) {
    const Tensor logits = logits_.contiguous(), sym = symbols.contiguous();
    const Tensor rng = ranges.defined() ? ranges.contiguous() : Tensor();
    const Tensor bnd = boundary.defined() ? boundary.contiguous() : Tensor();
    const int64_t B = logits.size(0), T = logits.size(1), K = logits.size(2), C = logits.size(3),
                  S = sym.size(1);
    const int64_t T1 = kind == 0 ? T + 1 : T;
    ctx->set_materialize_grads(false);
    DeviceGuard guard(logits.device());
    const auto opts = logits.options().dtype(c10::CppTypeToScalarType<R>::value);
    const int64_t n_px = B * S * T1, n_py = B * (S + 1) * T;
    // what the backward reads besides its inputs, in one allocation: norm | px_grad | py_grad, the
    // latter two unless they are handed out
    Carver keep;
    const int64_t o_nr = keep.take(B * T * K), o_gx = keep.take(want_grads ? 0 : n_px),
                  o_gy = keep.take(want_grads ? 0 : n_py);
    const Tensor kept = need_grad ? at::empty({keep.total}, opts) : Tensor();
    // what it does not: px | py | xr | yr | p | scores (and norm, without a backward)
    Carver carve;
    const int64_t o_px = carve.take(n_px), o_py = carve.take(n_py), o_xr = carve.take(B * T * K),
                  o_yr = carve.take(B * T * K), o_p = carve.take(B * (S + 1) * (T + 1)),
                  o_sc = carve.take(B), o_unkept = carve.take(need_grad ? 0 : B * T * K);
    const Tensor work = at::empty({carve.total}, opts);
    R *w = work.data_ptr<R>(), *k = ptr<R>(kept);
    Tensor gx, gy;
    if (want_grads) {
      gx = at::empty({B, S, T1}, opts);
      gy = at::empty({B, S + 1, T}, opts);
    }
    R *p_gx = want_grads ? ptr<R>(gx) : need_grad ? k + o_gx : nullptr;
    R *p_gy = want_grads ? ptr<R>(gy) : need_grad ? k + o_gy : nullptr;
    Tensor loss = reduction == kRedNone ? at::empty({B}, opts) : at::empty({}, opts);
    check_rc(abi_lattice_loss_fwd(logits.scalar_type(), logits.data_ptr(), iptr(sym), iptr(rng),
                                  iptr(bnd), w + o_px, w + o_py, need_grad ? k + o_nr : w + o_unkept,
                                  w + o_xr, w + o_yr, w + o_p, w + o_sc, p_gx, p_gy, ptr<R>(loss),
                                  (int)B, (int)S, (int)T, (int)K, (int)C, (int)term, (int)kind,
                                  delay_penalty > 0.0 ? delay_penalty : 0.0, (int)reduction,
                                  (int)checks | FRNNT_SCRATCH_P, status_for(logits, bnd),
                                  stream_of(logits)),
             "frnnt_lattice_loss_fwd");
    if (need_grad) {
      // (absent tensors are not saved: saved tensors must be defined)
      variable_list save{logits, sym, kept};
      for (const Tensor &t : {rng, bnd, gx, gy})
        if (t.defined()) save.push_back(t);
      ctx->save_for_backward(std::move(save));
      ctx->saved_data["meta"] =
          std::vector<int64_t>{term, kind, reduction, rng.defined(), bnd.defined(), want_grads};
    }
    // (undefined tensors cannot be outputs of an autograd node)
    if (!want_grads) return {loss};
    ctx->mark_non_differentiable({gx, gy});
    return {loss, gx, gy};
  }

  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    variable_list out(11);
    const Tensor &g_loss = grads[0];
    if (!g_loss.defined()) return out;
    const auto saved = ctx->get_saved_variables();
    out[0] = saved[0].scalar_type() == at::kDouble ? run_backward<double>(ctx, saved, g_loss)
                                                   : run_backward<float>(ctx, saved, g_loss);
    return out;
  }

  template <typename R>
  static Tensor run_backward(AutogradContext *ctx, const variable_list &saved,
                             const Tensor &g_loss) {
    const Tensor &logits = saved[0], &sym = saved[1], &kept = saved[2];
    const std::vector<int64_t> meta = ctx->saved_data["meta"].toIntVector();
    const int64_t kind = meta[1], reduction = meta[2];
    const Tensor rng = meta[3] ? saved[3] : Tensor();
    const Tensor bnd = meta[4] ? saved[3 + meta[3]] : Tensor();
    const bool handed_out = meta[5] != 0;
    const int64_t B = logits.size(0), T = logits.size(1), K = logits.size(2), C = logits.size(3),
                  S = sym.size(1);
    DeviceGuard guard(logits.device());
    const Tensor g = g_loss.contiguous();
    const int stride = reduction == kRedNone ? 1 : 0;
    const double scale = reduction == kRedMean ? -1.0 / (double)B : -1.0;
    void *stream = stream_of(logits);
    // (the forward's layout)
    Carver keep;
    const int64_t o_nr = keep.take(B * T * K),
                  o_gx = keep.take(handed_out ? 0 : B * S * (kind == 0 ? T + 1 : T)),
                  o_gy = keep.take(handed_out ? 0 : B * (S + 1) * T);
    R *k = ptr<R>(kept), *gx = k + o_gx, *gy = k + o_gy;
    if (handed_out) {
      const Tensor &t_gx = saved[3 + meta[3] + meta[4]], &t_gy = saved[4 + meta[3] + meta[4]];
      gx = ptr<R>(t_gx), gy = ptr<R>(t_gy);
      check_rc(abi_mi_scale_grads(gx, gy, ptr<R>(g), stride, scale, (int)B, (int)S, (int)T,
                                  (int)(kind != 0), stream),
               "frnnt_mi_scale_grads");
      count_as_changed(t_gx, t_gy);
    }
    Tensor grad = at::empty(logits.sizes(), logits.options());
    check_rc(abi_lattice_loss_bwd(logits.scalar_type(), logits.data_ptr(), iptr(sym), iptr(rng),
                                  iptr(bnd), k + o_nr, handed_out ? (const R *)nullptr : ptr<R>(g),
                                  stride, scale, gx, gy, grad.data_ptr(), (int)B, (int)S, (int)T,
                                  (int)K, (int)C, (int)meta[0], (int)kind, stream),
             "frnnt_lattice_loss_bwd");
    return grad;
  }
};

LossResult lattice_loss(const Tensor &logits, const Tensor &symbols,
                        const std::optional<Tensor> &ranges_,
                        const std::optional<Tensor> &boundary_, int64_t termination_symbol,
                        int64_t rnnt_type, double delay_penalty, bool return_grad,
                        int64_t reduction, int64_t checks) {
  const Tensor ranges = or_undefined(ranges_), boundary = or_undefined(boundary_);
  TORCH_CHECK(logits.is_cuda(), "fast_rnnt_amd runs on GPU tensors only (no CPU path): logits");
  TORCH_CHECK(logits.scalar_type() == at::kFloat || logits.scalar_type() == at::kDouble ||
                  logits.scalar_type() == at::kHalf || logits.scalar_type() == at::kBFloat16,
              "fast_rnnt_amd supports float32, float64, float16 and bfloat16 logits, got ",
              logits.scalar_type());
  TORCH_CHECK(logits.dim() == 4 && symbols.dim() == 2 && symbols.size(0) == logits.size(0),
              "logits must be [B][T][S+1 or s_range][C], symbols [B][S]");
  const int64_t B = logits.size(0);
  auto check_index = [&](const Tensor &t, const char *name) {
    TORCH_CHECK(t.scalar_type() == at::kLong && t.device() == logits.device(), name,
                " must be an int64 tensor on the device of the logits");
  };
  check_index(symbols, "symbols");
  if (ranges.defined()) {
    check_index(ranges, "ranges");
    TORCH_CHECK(ranges.dim() == 3 && ranges.size(0) == B && ranges.size(1) == logits.size(1) &&
                    ranges.size(2) == logits.size(2),
                "ranges must have the first three sizes of the logits");
  } else {
    TORCH_CHECK(logits.size(2) == symbols.size(1) + 1, "logits must be [B][T][S+1][C]");
  }
  if (boundary.defined()) {
    check_index(boundary, "boundary");
    TORCH_CHECK(boundary.dim() == 2 && boundary.size(0) == B && boundary.size(1) == 4,
                "boundary must have shape [B][4]");
  }
  TORCH_CHECK(rnnt_type >= 0 && rnnt_type <= 2, "rnnt_type must be 0, 1 or 2");
  TORCH_CHECK(reduction >= 0 && reduction <= 2, "reduction must be 0 (none), 1 (mean) or 2 (sum)");
  const bool need_grad = at::GradMode::is_enabled() && logits.requires_grad();
  return as_result(LatticeLossFn::apply(logits, symbols, ranges_, boundary_, termination_symbol,
                                        rnnt_type, delay_penalty, return_grad, reduction, checks,
                                        need_grad));
}

// ---- get_rnnt_prune_ranges and do_rnnt_pruning ---------------------------------------------
// What get_rnnt_prune_ranges needs of the boundary rows (their copy on the host): the smallest
// s_end, the smallest t_end - s_end, whether a t_end is 0, and the largest
// trunc((s_end - 1) / t_end) + 2 (rnnt_loss.py:696-710).
std::tuple<int64_t, int64_t, bool, int64_t> boundary_summary(const Tensor &rows) {
  TORCH_CHECK(rows.device().is_cpu() && rows.scalar_type() == at::kLong && rows.dim() == 2 &&
                  rows.size(1) == 4 && rows.is_contiguous() && rows.size(0) > 0,
              "rows must be a contiguous int64 [B][4] tensor on the host");
  const int64_t *r = rows.data_ptr<int64_t>();
  int64_t least_s = r[2], least_slack = r[3] - r[2], most = INT64_MIN;
  bool empty = false;
  for (int64_t b = 0; b < rows.size(0); ++b, r += 4) {
    least_s = std::min(least_s, r[2]);
    least_slack = std::min(least_slack, r[3] - r[2]);
    if (r[3] == 0) empty = true;
    else most = std::max(most, (r[2] - 1) / r[3] + 2);
  }
  return {least_s, least_slack, empty, most};
}

Tensor prune_ranges(const Tensor &px_grad, const Tensor &py_grad, const Tensor &boundary,
                    int64_t s_range) {
  require_float_gpu(px_grad, "px_grad");
  TORCH_CHECK(px_grad.dim() == 3 && py_grad.dim() == 3, "px_grad and py_grad must be 3-dimensional");
  const int64_t B = px_grad.size(0), S = px_grad.size(1), T1 = px_grad.size(2), T = py_grad.size(2);
  TORCH_CHECK((T1 == T || T1 == T + 1) && py_grad.size(0) == B && py_grad.size(1) == S + 1 &&
                  py_grad.scalar_type() == px_grad.scalar_type() &&
                  py_grad.device() == px_grad.device(),
              "px_grad must be [B][S][T or T+1], py_grad [B][S+1][T] of the same type and device");
  TORCH_CHECK(boundary.dim() == 2 && boundary.size(0) == B && boundary.size(1) == 4 &&
                  boundary.scalar_type() == at::kLong && boundary.device() == px_grad.device(),
              "boundary must be an int64 [B][4] tensor on the same device");
  DeviceGuard guard(px_grad.device());
  const Tensor gx = px_grad.contiguous(), gy = py_grad.contiguous(), bnd = boundary.contiguous();
  Tensor ranges = at::empty({B, T, s_range}, bnd.options());
  const int modified = T1 == T;
  check_rc(gx.scalar_type() == at::kFloat
               ? frnnt_prune_ranges_f32(ptr<float>(gx), ptr<float>(gy), iptr(bnd),
                                        ranges.data_ptr<int64_t>(), (int)B, (int)S, (int)T,
                                        modified, (int)s_range, stream_of(gx))
               : frnnt_prune_ranges_f64(ptr<double>(gx), ptr<double>(gy), iptr(bnd),
                                        ranges.data_ptr<int64_t>(), (int)B, (int)S, (int)T,
                                        modified, (int)s_range, stream_of(gx)),
           "frnnt_prune_ranges");
  return ranges;
}

Tensor gather_rows(const Tensor &lm, const Tensor &rng) {
  const int B = (int)rng.size(0), T = (int)rng.size(1), R = (int)rng.size(2),
            S = (int)lm.size(1) - 1, C = (int)lm.size(2);
  Tensor out = at::empty({B, T, R, C}, lm.options());
  void *stream = stream_of(lm);
  int rc;
  switch (lm.scalar_type()) {
    case at::kFloat:
      rc = frnnt_prune_gather_f32(ptr<float>(lm), iptr(rng), ptr<float>(out), B, S, T, R, C, stream);
      break;
    case at::kDouble:
      rc = frnnt_prune_gather_f64(ptr<double>(lm), iptr(rng), ptr<double>(out), B, S, T, R, C, stream);
      break;
    case at::kHalf:
      rc = frnnt_prune_gather_f16(lm.data_ptr(), iptr(rng), out.data_ptr(), B, S, T, R, C, stream);
      break;
    default:
      rc = frnnt_prune_gather_bf16(lm.data_ptr(), iptr(rng), out.data_ptr(), B, S, T, R, C, stream);
  }
  check_rc(rc, "frnnt_prune_gather");
  return out;
}

// the adjoint of gather_rows: [B][T][R][C] -> [B][rows][C]
Tensor scatter_rows(const Tensor &grad, const Tensor &rng, int64_t rows) {
  const Tensor g = grad.contiguous();
  const int64_t B = rng.size(0), T = rng.size(1), R = rng.size(2), C = g.size(3);
  Tensor out = at::empty({B, rows, C}, g.options());
  check_rc(frnnt_pruning_bwd(dtype_code(g.scalar_type()), nullptr, g.data_ptr(), iptr(rng), nullptr,
                             out.data_ptr(), (int)B, (int)rows - 1, (int)T, (int)R, (int)C,
                             stream_of(g)),
           "frnnt_pruning_bwd");
  return out;
}

// gather_rows and its adjoint as autograd nodes, each the other's derivative: both can be
// differentiated as often as the caller likes (create_graph=True).
struct GatherRowsFn : public torch::autograd::Function<GatherRowsFn> {
  static Tensor forward(AutogradContext *ctx, const Tensor &lm_, const Tensor &ranges);
  static variable_list backward(AutogradContext *ctx, variable_list grads);
};
struct ScatterRowsFn : public torch::autograd::Function<ScatterRowsFn> {
  static Tensor forward(AutogradContext *ctx, const Tensor &grad, const Tensor &rng, int64_t rows) {
    DeviceGuard guard(grad.device());
    ctx->save_for_backward({rng});
    return scatter_rows(grad, rng, rows);
  }
  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    return {GatherRowsFn::apply(grads[0], ctx->get_saved_variables()[0]), Tensor(), Tensor()};
  }
};
Tensor GatherRowsFn::forward(AutogradContext *ctx, const Tensor &lm_, const Tensor &ranges) {
  DeviceGuard guard(lm_.device());
  const Tensor lm = lm_.contiguous(), rng = ranges.contiguous();
  ctx->save_for_backward({rng});
  ctx->saved_data["rows"] = lm.size(1);
  return gather_rows(lm, rng);
}
variable_list GatherRowsFn::backward(AutogradContext *ctx, variable_list grads) {
  const Tensor rng = ctx->get_saved_variables()[0];
  const int64_t rows = ctx->saved_data["rows"].toInt();
  if (at::GradMode::is_enabled()) return {ScatterRowsFn::apply(grads[0], rng, rows), Tensor()};
  DeviceGuard guard(grads[0].device());
  return {scatter_rows(grads[0], rng, rows), Tensor()};
}

// do_rnnt_pruning as one autograd node (rnnt_loss.py:780-818): am_pruned is a view of am, lm_pruned
// a gathered copy; backward = frnnt_pruning_bwd, which reads a gradient that both share -- the
// joiner that follows adds the two -- once.  A backward that is to be differentiated itself takes
// the two adjoints as nodes of their own.
struct PruningFn : public torch::autograd::Function<PruningFn> {
  static variable_list forward(AutogradContext *ctx, const Tensor &, const Tensor &lm_,
                               const Tensor &ranges) {
    DeviceGuard guard(lm_.device());
    const Tensor lm = lm_.contiguous(), rng = ranges.contiguous();
    ctx->set_materialize_grads(false);
    ctx->save_for_backward({rng});
    ctx->saved_data["rows"] = lm.size(1);
    const Tensor rows = gather_rows(lm, rng);
    // (the first output stands for am_pruned: its sizes and type, not its values -- see pruning)
    return {rows.detach(), rows};
  }

  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    variable_list out(3);
    const Tensor rng = ctx->get_saved_variables()[0];
    const int64_t B = rng.size(0), T = rng.size(1), R = rng.size(2),
                  S1 = ctx->saved_data["rows"].toInt();
    const Tensor &any = grads[0].defined() ? grads[0] : grads[1];
    if (!any.defined()) return out;
    const int64_t C = any.size(3);
    if (at::GradMode::is_enabled()) {
      if (grads[0].defined()) out[0] = grads[0].sum(2);
      if (grads[1].defined()) out[1] = ScatterRowsFn::apply(grads[1], rng, S1);
      return out;
    }
    DeviceGuard guard(any.device());
    const Tensor ga = grads[0].defined() ? grads[0].contiguous() : Tensor();
    // (one tensor stays one, also where a copy of it has to be made)
    const Tensor gl = !grads[1].defined()                                ? Tensor()
                      : ga.defined() && grads[1].is_same(grads[0]) ? ga
                                                                         : grads[1].contiguous();
    if (ga.defined()) out[0] = at::empty({B, T, C}, any.options());
    if (gl.defined()) out[1] = at::empty({B, S1, C}, any.options());
    auto at_ = [](const Tensor &t) { return t.defined() ? t.data_ptr() : nullptr; };
    check_rc(frnnt_pruning_bwd(dtype_code(any.scalar_type()), at_(ga), at_(gl), iptr(rng),
                               at_(out[0]), at_(out[1]), (int)B, (int)S1 - 1, (int)T, (int)R,
                               (int)C, stream_of(any)),
             "frnnt_pruning_bwd");
    return out;
  }
};

std::tuple<Tensor, Tensor> pruning(const Tensor &am, const Tensor &lm, const Tensor &ranges) {
  TORCH_CHECK(lm.is_cuda(), "fast_rnnt_amd runs on GPU tensors only (no CPU path): lm");
  TORCH_CHECK(lm.scalar_type() == at::kFloat || lm.scalar_type() == at::kDouble ||
                  lm.scalar_type() == at::kHalf || lm.scalar_type() == at::kBFloat16,
              "fast_rnnt_amd supports float32, float64, float16 and bfloat16 tensors here, got ",
              lm.scalar_type());
  TORCH_CHECK(am.dim() == 3 && lm.dim() == 3 && ranges.dim() == 3 && am.size(0) == lm.size(0) &&
                  ranges.size(0) == lm.size(0) && am.size(1) == ranges.size(1),
              "am must be [B][T][C], lm [B][S+1][C], ranges [B][T][s_range]");
  TORCH_CHECK(am.device() == lm.device() && ranges.device() == lm.device() &&
                  am.scalar_type() == lm.scalar_type() && ranges.scalar_type() == at::kLong,
              "am and lm must share a device and a type, ranges be int64 on that device");
  const Tensor am_pruned =
      am.unsqueeze(2).expand({am.size(0), am.size(1), ranges.size(2), lm.size(2)});
  // (a tangent of am passes through the view and would be refused by the node)
  if (!at::GradMode::is_enabled() || !am.requires_grad() || !lm.requires_grad() ||
      am.size(2) != lm.size(2) || am._fw_grad(/*level=*/0).defined())
    return {am_pruned, GatherRowsFn::apply(lm, ranges)};
  // The view stays the plain one, which autograd follows when am or the view itself is written to
  // (a view that a node returns is refused then); only its gradient goes to the node.
  const variable_list out = PruningFn::apply(am, lm, ranges);
  torch::autograd::impl::set_gradient_edge(
      am_pruned, {out[0].grad_fn(), static_cast<uint32_t>(out[0].output_nr())});
  return {am_pruned, out[1]};
}

void set_deferred_checks(bool on) { g_deferred = on; }
bool deferred_checks() { return g_deferred; }

}  // namespace

// ---- dispatcher registration: torch.ops.fast_rnnt_amd.* -----------------------------------
TORCH_LIBRARY(fast_rnnt_amd, m) {
  m.def("mutual_information_forward(Tensor px, Tensor py, Tensor? boundary, Tensor(a!) p) -> Tensor");
  m.def(
      "mutual_information_backward(Tensor px, Tensor py, Tensor? boundary, Tensor p, "
      "Tensor(a!) ans_grad) -> Tensor[]");
  m.def(
      "recursion(Tensor px, Tensor py, Tensor? boundary, bool return_grad) -> "
      "(Tensor, Tensor?, Tensor?)");
  m.def(
      "recursion_loss(Tensor px, Tensor py, Tensor? boundary, bool return_grad, int reduction, "
      "int checks) -> (Tensor, Tensor?, Tensor?)");
  m.def(
      "simple_loss(Tensor lm, Tensor am, Tensor symbols, Tensor? boundary, int termination_symbol, "
      "int rnnt_type, float delay_penalty, bool return_grad, int reduction, int checks) -> "
      "(Tensor, Tensor?, Tensor?)");
  m.def(
      "smoothed_loss(Tensor lm, Tensor am, Tensor symbols, Tensor? boundary, "
      "int termination_symbol, int rnnt_type, float lm_only_scale, float am_only_scale, "
      "float delay_penalty, bool return_grad, int reduction, int checks) -> "
      "(Tensor, Tensor?, Tensor?)");
  m.def(
      "lattice_loss(Tensor logits, Tensor symbols, Tensor? ranges, Tensor? boundary, "
      "int termination_symbol, int rnnt_type, float delay_penalty, bool return_grad, "
      "int reduction, int checks) -> (Tensor, Tensor?, Tensor?)");
  m.def("prune_ranges(Tensor px_grad, Tensor py_grad, Tensor boundary, int s_range) -> Tensor");
  m.def("pruning(Tensor am, Tensor lm, Tensor ranges) -> (Tensor, Tensor)");
}
// (PyTorch-ROCm keeps the dispatch key name CUDA for the MI355X)
TORCH_LIBRARY_IMPL(fast_rnnt_amd, CUDA, m) {
  m.impl("mutual_information_forward", &mutual_information_forward);
  m.impl("mutual_information_backward", &mutual_information_backward);
  m.impl("recursion", &recursion);
  m.impl("recursion_loss", &recursion_loss);
  m.impl("simple_loss", &simple_loss);
  m.impl("smoothed_loss", &smoothed_loss);
  m.impl("lattice_loss", &lattice_loss);
  m.impl("prune_ranges", &prune_ranges);
  m.impl("pruning", &pruning);
}
// The loss ops carry their own autograd nodes: the same functions serve the Autograd key
// (they call the C ABI themselves and never re-dispatch).
TORCH_LIBRARY_IMPL(fast_rnnt_amd, Autograd, m) {
  m.impl("recursion", &recursion);
  m.impl("recursion_loss", &recursion_loss);
  m.impl("simple_loss", &simple_loss);
  m.impl("smoothed_loss", &smoothed_loss);
  m.impl("lattice_loss", &lattice_loss);
  m.impl("pruning", &pruning);
}

PYBIND11_MODULE(_C, m) {
  m.doc() = "fast_rnnt_amd operator module (torch tensors -> C ABI of libfast_rnnt_amd.so)";
  py::register_exception<BoundaryAssertion>(m, "BoundaryAssertionError", PyExc_AssertionError);
  m.def("mutual_information_forward", &mutual_information_forward, py::arg("px"), py::arg("py"),
        py::arg("boundary"), py::arg("p"));
  m.def("mutual_information_backward", &mutual_information_backward, py::arg("px"),
        py::arg("py"), py::arg("boundary"), py::arg("p"), py::arg("ans_grad"));
  m.def("with_cuda", &with_cuda);
  m.def("recursion", &recursion, py::arg("px"), py::arg("py"), py::arg("boundary"),
        py::arg("return_grad"));
  m.def("recursion_loss", &recursion_loss, py::arg("px"), py::arg("py"), py::arg("boundary"),
        py::arg("return_grad"), py::arg("reduction"), py::arg("checks") = 0);
  m.def("simple_loss", &simple_loss, py::arg("lm"), py::arg("am"), py::arg("symbols"),
        py::arg("boundary"), py::arg("termination_symbol"), py::arg("rnnt_type"),
        py::arg("delay_penalty"), py::arg("return_grad"), py::arg("reduction"),
        py::arg("checks") = 0);
  m.def("smoothed_loss", &smoothed_loss, py::arg("lm"), py::arg("am"), py::arg("symbols"),
        py::arg("boundary"), py::arg("termination_symbol"), py::arg("rnnt_type"),
        py::arg("lm_only_scale"), py::arg("am_only_scale"), py::arg("delay_penalty"),
        py::arg("return_grad"), py::arg("reduction"), py::arg("checks") = 0);
  m.def("lattice_loss", &lattice_loss, py::arg("logits"), py::arg("symbols"), py::arg("ranges"),
        py::arg("boundary"), py::arg("termination_symbol"), py::arg("rnnt_type"),
        py::arg("delay_penalty"), py::arg("return_grad"), py::arg("reduction"),
        py::arg("checks") = 0);
  m.def("boundary_summary", &boundary_summary, py::arg("rows"));
  m.def("prune_ranges", &prune_ranges, py::arg("px_grad"), py::arg("py_grad"), py::arg("boundary"),
        py::arg("s_range"));
  m.def("pruning", &pruning, py::arg("am"), py::arg("lm"), py::arg("ranges"));
  m.def("set_deferred_checks", &set_deferred_checks, py::arg("on"));
  m.def("deferred_checks", &deferred_checks);
  m.def("check_boundaries", &check_boundaries, py::arg("device"));
  m.def("take_pending", &take_pending, py::arg("device"));
}

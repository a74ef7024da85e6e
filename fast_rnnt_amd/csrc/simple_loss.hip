// rnnt_loss_simple's forward pipeline behind one call (rnnt_loss.py:230-340):
// px/py from lm and am, the lattice recursion, optionally its backward with a
// gradient of ones (the occupation probabilities), and the reduction of the scores.
// It only chains the entry points of the other files on one stream; what it saves
// is host time, which matters once a whole call takes ~100 us on the GPU.
#include <type_traits>

#include "simple_shared.hip.h"

namespace frnnt {
namespace {

// The tail every loss function shares (e.g. rnnt_loss.py:326-340): the recursion, its
// backward with a gradient of ones when the occupation gradients are wanted, the reduction.
template <typename R, typename Reduce>
int mi_loss_fwd(Reduce reduce, const R *px, const R *py,
                const int64_t *boundary, R *p, R *scores, R *px_grad, R *py_grad, R *loss, int B,
                int S, int T, int modified, int reduction, int checks, int32_t *status,
                int *arrived, void *stream) {
  if ((px_grad == nullptr) != (py_grad == nullptr))
    return fail(FRNNT_EINVAL, "mi_loss_fwd: px_grad and py_grad go together");
  const bool p_wanted = (checks & FRNNT_SCRATCH_P) == 0;
  checks &= ~(FRNNT_SCRATCH_P | FRNNT_LARGE_SCRATCH);
  if constexpr (std::is_same<R, float>::value) {
    if (px_grad && !p_wanted && mi_shares_pay(B, S, T)) {
      int rc = mi_forward_shares(px, py, boundary, p, scores, B, S, T, modified, checks, status, px_grad,
                                 py_grad, stream);
      if (rc != FRNNT_OK) return rc;
      rc = mi_backward_shares(boundary, p, px_grad, py_grad, scores, loss, B, S, T, modified, reduction,
                              stream);
      if (rc != FRNNT_OK || B > 0) return rc;
      return loss ? reduce(scores, loss, B, reduction, stream) : rc;
    }
  }
  LossOf<R> formed{loss, reduction, arrived, false};
  int rc = mi_forward(px, py, boundary, p, scores, B, S, T, modified, checks, status, px_grad,
                      px_grad ? nullptr : &formed, stream);
  if (rc != FRNNT_OK || formed.formed) return rc;
  if (px_grad) {
    // with a loss to form, the backward kernel reduces the scores on its way
    rc = mi_backward_and_loss(px, boundary, p, px_grad, py_grad, scores, loss, B, S, T, modified,
                              reduction, stream);
    if (rc != FRNNT_OK || B > 0) return rc;
  }
  if (loss) rc = reduce(scores, loss, B, reduction, stream);
  return rc;
}

template <typename R, typename Reduce>
int simple_loss_fwd(Reduce reduce,
                    const R *lm, const R *am, const int64_t *symbols, const int64_t *boundary,
                    R *px, R *py, R *lm_max, R *am_max, R *norm_raw, R *p, R *scores, R *px_grad,
                    R *py_grad, R *loss, int B, int S, int T, int C, int term,
                    int rnnt_type, double delay_penalty, int reduction, int checks,
                    int32_t *status, void *stream) {
  if ((px_grad == nullptr) != (py_grad == nullptr))
    return fail(FRNNT_EINVAL, "simple_loss_fwd: px_grad and py_grad go together");
  // px / py only feed the recursion below, with the same boundary: what lies outside an
  // utterance's window need not be computed
  int rc;
  if constexpr (std::is_same<R, float>::value)
    rc = simple_logprobs_fwd(lm, am, symbols, boundary, px, py, lm_max, am_max, norm_raw, delay_penalty, B,
                             S, T, C, term, rnnt_type, boundary != nullptr, stream, nullptr,
                             checks & FRNNT_LARGE_SCRATCH ? p : nullptr);
  else
    rc = simple_logprobs_fwd(lm, am, symbols, boundary, px, py, lm_max, am_max, norm_raw, delay_penalty, B,
                             S, T, C, term, rnnt_type, boundary != nullptr, stream);
  if (rc != FRNNT_OK) return rc;
  return mi_loss_fwd<R>(reduce, px, py, boundary, p, scores, px_grad, py_grad,
                        loss, B, S, T, rnnt_type != kRegular, reduction, checks, status, nullptr, stream);
}

}  // namespace

int mi_loss(const float *px, const float *py, const int64_t *boundary, float *p, float *scores,
            float *px_grad, float *py_grad, float *loss, int B, int S, int T, int modified, int reduction,
            int checks, int32_t *status, int *arrived, void *stream) {
  return mi_loss_fwd<float>(frnnt_loss_reduce_f32, px, py, boundary, p, scores, px_grad, py_grad, loss, B,
                            S, T, modified, reduction, checks, status, arrived, stream);
}
int mi_loss(const double *px, const double *py, const int64_t *boundary, double *p, double *scores,
            double *px_grad, double *py_grad, double *loss, int B, int S, int T, int modified,
            int reduction, int checks, int32_t *status, int *arrived, void *stream) {
  return mi_loss_fwd<double>(frnnt_loss_reduce_f64, px, py, boundary, p, scores, px_grad, py_grad, loss,
                             B, S, T, modified, reduction, checks, status, arrived, stream);
}

}  // namespace frnnt

extern "C" {

int frnnt_mi_loss_fwd_f32(const float *px, const float *py, const int64_t *boundary, float *p,
                          float *scores, float *px_grad, float *py_grad, float *loss, int B, int S,
                          int T, int modified, int reduction, int checks, int32_t *status,
                          void *stream) {
  return frnnt::mi_loss(px, py, boundary, p, scores, px_grad, py_grad, loss, B, S, T, modified, reduction,
                        checks, status, nullptr, stream);
}
int frnnt_mi_loss_fwd_f64(const double *px, const double *py, const int64_t *boundary, double *p,
                          double *scores, double *px_grad, double *py_grad, double *loss, int B,
                          int S, int T, int modified, int reduction, int checks, int32_t *status,
                          void *stream) {
  return frnnt::mi_loss(px, py, boundary, p, scores, px_grad, py_grad, loss, B, S, T, modified, reduction,
                        checks, status, nullptr, stream);
}

int frnnt_simple_loss_fwd_f32(const float *lm, const float *am, const int64_t *symbols,
                              const int64_t *boundary, float *px, float *py, float *lm_max,
                              float *am_max, float *norm_raw, float *p, float *scores,
                              float *px_grad, float *py_grad, float *loss, int B, int S, int T,
                              int C, int termination_symbol, int rnnt_type, int reduction,
                              int checks, int32_t *status, void *stream) {
  return frnnt::simple_loss_fwd<float>(                                       frnnt_loss_reduce_f32, lm, am,
                                       symbols, boundary, px, py, lm_max, am_max, norm_raw, p,
                                       scores, px_grad, py_grad, loss, B, S,
                                       T, C, termination_symbol, rnnt_type, 0.0, reduction, checks,
                                       status, stream);
}
int frnnt_simple_loss_fwd_f64(const double *lm, const double *am, const int64_t *symbols,
                              const int64_t *boundary, double *px, double *py, double *lm_max,
                              double *am_max, double *norm_raw, double *p, double *scores,
                              double *px_grad, double *py_grad, double *loss, int B, int S, int T,
                              int C, int termination_symbol, int rnnt_type, int reduction,
                              int checks, int32_t *status, void *stream) {
  return frnnt::simple_loss_fwd<double>(                                        frnnt_loss_reduce_f64, lm, am,
                                        symbols, boundary, px, py, lm_max, am_max, norm_raw, p,
                                        scores, px_grad, py_grad, loss, B, S,
                                        T, C, termination_symbol, rnnt_type, 0.0, reduction, checks,
                                        status, stream);
}

int frnnt_additive_loss_fwd(int dtype, const void *lm, const void *am, const int64_t *symbols,
                            const int64_t *boundary, void *lm_wide, void *am_wide, void *px,
                            void *py, void *lm_max, void *am_max, void *norm_raw, void *p,
                            void *scores, void *px_grad, void *py_grad, void *loss,
                            int B, int S, int T, int C, int termination_symbol,
                            int rnnt_type, double delay_penalty, int reduction, int checks,
                            int32_t *status, void *stream) {
  using frnnt::fail;
  if (dtype < FRNNT_F32 || dtype > FRNNT_BF16)
    return fail(FRNNT_EINVAL, "additive_loss_fwd: unknown dtype");
  if (dtype >= FRNNT_F16 && B > 0 && S >= 0 && T >= 0 && C > 0) {
    if (!lm || (!am && T > 0) || !lm_wide || !am_wide)
      return fail(FRNNT_EINVAL, "additive_loss_fwd: null pointer");
    frnnt::widen_inputs(dtype, lm, am, static_cast<float *>(lm_wide),
                        static_cast<float *>(am_wide), (long)B * (S + 1) * C, (long)B * T * C,
                        static_cast<hipStream_t>(stream));
    lm = lm_wide;
    am = am_wide;
  }
  auto call = [&](auto r, auto reduce) {
    using R = decltype(r);
    auto out = [](void *q) { return static_cast<R *>(q); };
    return frnnt::simple_loss_fwd<R>(
        reduce, static_cast<const R *>(lm), static_cast<const R *>(am), symbols,
        boundary, out(px), out(py), out(lm_max), out(am_max), out(norm_raw), out(p), out(scores),
        out(px_grad), out(py_grad), out(loss), B, S, T, C, termination_symbol,
        rnnt_type, delay_penalty > 0.0 ? delay_penalty : 0.0, reduction, checks, status, stream);
  };
  if (dtype == FRNNT_F64)
    return call(double(), frnnt_loss_reduce_f64);
  return call(float(), frnnt_loss_reduce_f32);
}

}  // extern "C"

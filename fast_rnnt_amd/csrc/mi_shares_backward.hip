// The lattice recursion's backward kernel in float32 after the forward kernel of mi_shares_forward.hip (a
// source file of its own: the two want different scheduling strategies).
#include "mi_recursion.hip.h"

namespace frnnt {

int mi_backward_shares(const int64_t *boundary, const float *shares, float *px_grad, float *py_grad,
                       const float *scores, float *loss, int B, int S, int T, int modified,
                       int reduction, void *stream) {
  return backward_impl<float, true>(nullptr, nullptr, boundary, shares, nullptr, px_grad, py_grad, B, S,
                                    T, modified, 0, stream, scores, loss, reduction, true);
}

}  // namespace frnnt

extern "C" int frnnt_mi_shares_bwd_f32(const int64_t *boundary, const float *shares,
                                       const float *score_grad, int score_grad_stride, float *px_grad,
                                       float *py_grad, int B, int S, int T, int modified, void *stream) {
  if (score_grad_stride != 0 && score_grad_stride != 1)
    return frnnt::fail(FRNNT_EINVAL, "mi_shares_bwd: score_grad_stride must be 0 or 1");
  return frnnt::backward_impl<float, true>(nullptr, nullptr, boundary, shares,
                                           const_cast<float *>(score_grad), px_grad, py_grad, B, S, T,
                                           modified, 0, stream, nullptr, nullptr, 0, false,
                                           score_grad_stride);
}

extern "C" int frnnt_mi_kept_bwd_f32(float *kept, int has_boundary, const float *score_grad,
                                     int score_grad_stride, float *px_grad, float *py_grad, int B, int S, int T,
                                     int modified, void *stream) {
  using namespace frnnt;
  if (score_grad_stride != 0 && score_grad_stride != 1)
    return fail(FRNNT_EINVAL, "mi_kept_bwd: score_grad_stride must be 0 or 1");
  const bool room = kept && B > 0 && S >= 0 && T >= 0;
  float *post = room ? kept + shares_floats(B, S, T) : nullptr;
  const int64_t *boundary =
      room && has_boundary ? reinterpret_cast<const int64_t *>(kept + rows_at(B, S, T)) : nullptr;
  return backward_impl<float, true>(nullptr, nullptr, boundary, kept, const_cast<float *>(score_grad), px_grad,
                                    py_grad, B, S, T, modified, 0, stream, nullptr, nullptr, 0, false,
                                    score_grad_stride, post);
}

// The lattice recursion in float32, and what both types share (the kernels: mi_recursion.hip.h).
#include "mi_recursion.hip.h"

namespace frnnt {

int mi_spin_limit = kSpinLimit;

int mi_forward(const float *px, const float *py, const int64_t *boundary, float *p, float *scores,
               int B, int S, int T, int modified, int checks, int32_t *status, float *px_grad,
               LossOf<float> *loss, void *stream) {
  return forward_impl<float>(px, py, boundary, p, scores, B, S, T, modified, stream, checks, status,
                             px_grad, nullptr, loss);
}
int mi_backward_and_loss(const float *px, const int64_t *boundary, const float *p, float *px_grad,
                         float *py_grad, const float *scores, float *loss, int B, int S, int T,
                         int modified, int reduction, void *stream) {
  return backward_impl<float>(px, nullptr, boundary, p, nullptr, px_grad, py_grad, B, S, T,
                              modified, 0, stream, scores, loss, reduction, true);
}

}  // namespace frnnt

extern "C" {

void frnnt_set_spin_limit(int polls) {
  frnnt::mi_spin_limit = polls > 0 ? polls : frnnt::kSpinLimit;
}

int frnnt_mi_forward_f32(const float *px, const float *py, const int64_t *boundary, float *p,
                         float *ans, int B, int S, int T, int modified, void *stream) {
  return frnnt::forward_impl<float>(px, py, boundary, p, ans, B, S, T, modified, stream);
}
int frnnt_mi_forward_checked_f32(const float *px, const float *py, const int64_t *boundary,
                                 float *p, float *ans, int B, int S, int T, int modified,
                                 int checks, int32_t *status, void *stream) {
  return frnnt::forward_impl<float>(px, py, boundary, p, ans, B, S, T, modified, stream, checks,
                                    status);
}
int frnnt_mi_backward_f32(const float *px, const float *py, const int64_t *boundary,
                          const float *p, float *ans_grad, float *px_grad, float *py_grad, int B,
                          int S, int T, int modified, int overwrite_ans_grad, void *stream) {
  return frnnt::backward_impl<float>(px, py, boundary, p, ans_grad, px_grad, py_grad, B, S, T,
                                     modified, overwrite_ans_grad, stream);
}

}  // extern "C"

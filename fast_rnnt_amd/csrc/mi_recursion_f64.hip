// The lattice recursion in double64 (the kernels: mi_recursion.hip.h).
#include "mi_recursion.hip.h"

namespace frnnt {

int mi_forward(const double *px, const double *py, const int64_t *boundary, double *p, double *scores,
               int B, int S, int T, int modified, int checks, int32_t *status, double *px_grad,
               LossOf<double> *loss, void *stream) {
  return forward_impl<double>(px, py, boundary, p, scores, B, S, T, modified, stream, checks, status,
                             px_grad, nullptr, loss);
}
int mi_backward_and_loss(const double *px, const int64_t *boundary, const double *p, double *px_grad,
                         double *py_grad, const double *scores, double *loss, int B, int S, int T,
                         int modified, int reduction, void *stream) {
  return backward_impl<double>(px, nullptr, boundary, p, nullptr, px_grad, py_grad, B, S, T,
                              modified, 0, stream, scores, loss, reduction, true);
}

}  // namespace frnnt

extern "C" {

int frnnt_mi_forward_f64(const double *px, const double *py, const int64_t *boundary, double *p,
                         double *ans, int B, int S, int T, int modified, void *stream) {
  return frnnt::forward_impl<double>(px, py, boundary, p, ans, B, S, T, modified, stream);
}
int frnnt_mi_forward_checked_f64(const double *px, const double *py, const int64_t *boundary,
                                 double *p, double *ans, int B, int S, int T, int modified,
                                 int checks, int32_t *status, void *stream) {
  return frnnt::forward_impl<double>(px, py, boundary, p, ans, B, S, T, modified, stream, checks,
                                    status);
}
int frnnt_mi_backward_f64(const double *px, const double *py, const int64_t *boundary,
                          const double *p, double *ans_grad, double *px_grad, double *py_grad, int B,
                          int S, int T, int modified, int overwrite_ans_grad, void *stream) {
  return frnnt::backward_impl<double>(px, py, boundary, p, ans_grad, px_grad, py_grad, B, S, T,
                                     modified, overwrite_ans_grad, stream);
}

}  // extern "C"

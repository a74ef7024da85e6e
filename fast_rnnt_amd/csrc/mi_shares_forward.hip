// The lattice recursion's forward kernel in float32 for callers that want the scores and the occupation
// gradients and not the table of p: it leaves in p's place what the backward kernel needs (kShares in
// mi_recursion.hip.h; mi_shares_backward.hip).
#include "mi_recursion.hip.h"

namespace frnnt {

int mi_forward_shares(const float *px, const float *py, const int64_t *boundary, float *shares,
                      float *scores, int B, int S, int T, int modified, int checks, int32_t *status,
                      float *px_grad, float *py_grad, void *stream) {
  return forward_impl<float, true>(px, py, boundary, shares, scores, B, S, T, modified, stream, checks,
                                   status, px_grad, py_grad);
}

}  // namespace frnnt

extern "C" int frnnt_mi_shares_fwd_f32(const float *px, const float *py, const int64_t *boundary,
                                       float *shares, float *scores, float *px_grad, float *py_grad, int B,
                                       int S, int T, int modified, int checks, int32_t *status,
                                       void *stream) {
  if (B > 0 && (!px_grad || !py_grad)) return frnnt::fail(FRNNT_EINVAL, "mi_shares_fwd: null pointer");
  return frnnt::mi_forward_shares(px, py, boundary, shares, scores, B, S, T, modified, checks, status,
                                  px_grad, py_grad, stream);
}

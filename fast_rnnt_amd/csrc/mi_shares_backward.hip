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

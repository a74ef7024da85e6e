// The lattice recursion's forward kernel in float32 for callers that want the scores and the occupation
// gradients and not the table of p: it leaves in p's place what the backward kernel needs (kShares in
// mi_recursion.hip.h; mi_shares_backward.hip).
#include "mi_recursion.hip.h"

namespace frnnt {

// Whether a loss is faster with shares than with p (both kernels and the marks, p against shares).  With one sweep
// wave in the workgroup, always (S 40, B 32: T 100: 16.0 and 15.4 us; T 500: 39.5 and 35.1).  With two the forward
// kernel's staging waves, who have more to do, are what short lattices wait for, and the backward makes up for it from
// some 200 frames on (S 90, B 32, T 100: 22.9 and 24.3; T 200: 30.0 and 30.5; T 350: 41.2 and 40.5; S 120, B 100, T 500:
// 57.0 and 51.6); with three and four, which have three staging waves each, later (B 100, S 160, T 260: 53.2 and 60.1; T
// 450: 77.1 and 76.2; B 168, S 190, T 350: 93.2 and 90.1; T 900: 230 and 185).  Bands apart have the marks to make up
// for (B 4, S 130, T 100: 33.5 and 34.4; T 140: 36.8 and 35.0).  More than four bands, which a workgroup takes in
// turn, have the line of three and four together, between where large and small batches begin to gain (S 300: B 200,
// T 400: 211 and 181; B 64, T 350: 98.9 and 98.6, T 500: 121.5 and 118.5; B 16, T 400: 95.4 and 97.8, T 600: 133.6 and
// 129.6; B 2, T 400: 93.8 and 97.5, T 700: 139.1 and 139.2; B 16, S 500, T 400: 140 and 133).
bool mi_shares_pay(int B, int S, int T) {
  if (S < kWave) return true;
  if (S < 2 * kWave) return T >= 200;
  const bool apart = bands_apart<float, true>(B, S, T, false) && bands_apart<float, true>(B, S, T, true);
  return T >= (apart ? 120 : 400);
}

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
  (void)px_grad;  // (marked by the call that writes it)
  if (B > 0 && !py_grad) return frnnt::fail(FRNNT_EINVAL, "mi_shares_fwd: null pointer");
  return frnnt::mi_forward_shares(px, py, boundary, shares, scores, B, S, T, modified, checks, status,
                                  nullptr, py_grad, stream);
}

extern "C" int frnnt_mi_route(int B, int S, int T, int shares) {
  using namespace frnnt;
  if (B < 1 || S < 0 || T < 0) return fail(FRNNT_EINVAL, "mi_route: bad size");
  const bool forward = shares ? bands_apart<float, true>(B, S, T, false) : bands_apart<float, false>(B, S, T, false);
  const bool backward = shares ? bands_apart<float, true>(B, S, T, true) : bands_apart<float, false>(B, S, T, true);
  return (forward ? 1 : 0) | (backward ? 2 : 0) | (mi_shares_pay(B, S, T) ? 4 : 0);
}

extern "C" int64_t frnnt_mi_kept_size(int B, int S, int T) {
  if (B < 1 || S < 0 || T < 0) return 0;
  return frnnt::rows_at(B, S, T) + 8 * (int64_t)B;
}
extern "C" int frnnt_mi_kept_fwd_f32(const float *px, const float *py, const int64_t *boundary, float *kept,
                                     float *scores, int B, int S, int T, int modified, int checks,
                                     int32_t *status, void *stream) {
  using namespace frnnt;
  const bool room = kept && B > 0 && S >= 0 && T >= 0;
  float *post = room ? kept + shares_floats(B, S, T) : nullptr;
  int64_t *rows = room ? reinterpret_cast<int64_t *>(kept + rows_at(B, S, T)) : nullptr;
  if (reinterpret_cast<uintptr_t>(rows) & 7) return fail(FRNNT_EINVAL, "mi_kept_fwd: kept not aligned to 8 bytes");
  return forward_impl<float, true>(px, py, boundary, kept, scores, B, S, T, modified, stream, checks, status,
                                   nullptr, post, nullptr, true, rows);
}

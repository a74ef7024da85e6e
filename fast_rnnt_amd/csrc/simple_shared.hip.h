// What the kernels of the simple (additive-joiner) loss share between their two source
// files: simple_normalizer.hip (the forward's normalizer product, compiled with a scheduling
// strategy of its own) and simple_logprobs.hip (everything else).
#pragma once
#include <functional>

#include "xcd_grid.hip.h"

namespace frnnt {
namespace {

enum { kRegular = 0, kModified = 1, kConstrained = 2 };

// What the lattice recursion uses of utterance b: rows [s_begin, s_end] and frames
// [t_begin, t_end) of py, rows [s_begin, s_end) of px.  A caller that goes on to the
// recursion with the same boundary passes it as `window`: the kernels then leave px / py /
// the normalizers outside it undefined, and take the gradients to vanish there (the
// recursion writes exact zeros).  Without a window everything counts.
struct Limits {
  int s_begin, t_begin, s_end, t_end;
};
__device__ __forceinline__ Limits limits_of(const int64_t *window, int b, int S, int T) {
  Limits w{0, 0, S, T};
  if (window) {
    // clamped: a boundary row outside the lattice must not widen any loop
    w.s_begin = (int)max((int64_t)0, min(window[4 * b + 0], (int64_t)S));
    w.t_begin = (int)max((int64_t)0, min(window[4 * b + 1], (int64_t)T));
    w.s_end = (int)max((int64_t)0, min(window[4 * b + 2], (int64_t)S));
    w.t_end = (int)max((int64_t)0, min(window[4 * b + 3], (int64_t)T));
  }
  return w;
}

typedef float floatx4u __attribute__((ext_vector_type(4), aligned(4)));

// exp(x - m) as one fused multiply-add and one v_exp_f32: 2^(x log2(e) - m log2(e)),
// with shift2 = -m log2(e) prepared per row; x = -inf gives 0.
constexpr float kLog2e = 1.44269504088896341f;
__device__ __forceinline__ float exp_shifted(float x, float shift2) {
  return __builtin_amdgcn_exp2f(__builtin_fmaf(x, kLog2e, shift2));
}

// ---- float32 products on the bfloat16 matrix cores -----------------------------------------
// v_mfma_f32_32x32x16_bf16 does a multiply-add in a sixteenth of the cycles of
// v_mfma_f32_32x32x2_f32.  A float32 is the sum of three bfloat16 values to its last bit (8 + 8 +
// 8 bits, rounded to nearest, and bfloat16 has float32's range), so a product is
//   a b = a_lo b_hi + a_hi b_lo + a_mid b_mid + a_mid b_hi + a_hi b_mid + a_hi b_hi
// to 2^-26 of itself -- below the rounding of a float32 product -- in six matrix instructions,
// smallest terms first, accumulated in float32.  Measured against float64 on sums of 512 and
// 4992 products of exponentials: rms error 2.3e-7 and 6.7e-7 of the sum of magnitudes, where the
// float32 instruction leaves 3.3e-7 and 1.4e-6.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned uintx2 __attribute__((ext_vector_type(2)));
typedef unsigned uintx4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ unsigned pack_bf16(float a, float b) {  // v_cvt_pk_bf16_f32
  typedef float f2 __attribute__((ext_vector_type(2)));
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  const b2 h = __builtin_convertvector((f2{a, b}), b2);
  unsigned w;
  __builtin_memcpy(&w, &h, 4);
  return w;
}
// c minus the low (`high`: the high) half of w: v_dot2c_f32_bf16 with a unit vector, one instruction
// for the unpacking and the subtraction.  The difference of a float32 and its bfloat16 rounding is
// exact, and so are both products: the same bits as unpacking and subtracting (a million values over
// all normal exponents, small parts that are subnormal included: the instruction keeps those), in 7 instead
// of 11 instructions per split pair.  (Not finite: a NaN or an infinity also makes the other value of its
// pair NaN; the two belong to the same sums.)  What bounds the split itself is bfloat16's range: the last
// part of a value below 2^-110 ends at 2^-133, so a factor exp(x - max) of 2^-e has a relative error of
// 2^(e - 134) where e > 110 -- 76 nats below its row's maximum, 2e-6 at 80 nats.  Measured: none down to
// 2^-110, 3.0e-5 at 2^-119, 3.8e-3 at 2^-126, in products with a float32 beside it as well.
__device__ __forceinline__ float minus_half(float c, unsigned w, bool high) {
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  unsigned unit = high ? 0xbf800000u : 0x0000bf80u;
  asm("" : "+s"(unit));  // (the compiler's inline constant -1.0 is not this word)
  b2 values, units;
  __builtin_memcpy(&values, &w, 4);
  __builtin_memcpy(&units, &unit, 4);
  return __builtin_amdgcn_fdot2_f32_bf16(values, units, c, false);
}
// the three parts of a pair of floats, each part's two values in one word
__device__ __forceinline__ void split_pair(float a, float b, unsigned &hi, unsigned &mid,
                                           unsigned &lo) {
  hi = pack_bf16(a, b);
  const float ra = minus_half(a, hi, false), rb = minus_half(b, hi, true);
  mid = pack_bf16(ra, rb);
  lo = pack_bf16(minus_half(ra, mid, false), minus_half(rb, mid, true));
}
struct Split8 {  // eight consecutive k of one row: a lane's operand of a 32 x 32 x 16 product
  bf16x8 hi, mid, lo;
};
__device__ __forceinline__ dgemm::floatx16 multiply_add(const Split8 &a, const Split8 &b,
                                                        dgemm::floatx16 acc) {
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.lo, b.hi, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.hi, b.lo, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.mid, b.mid, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.mid, b.hi, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.hi, b.mid, acc, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.hi, b.hi, acc, 0, 0, 0);
}
// ---- memory without branches ---------------------------------------------------------------
// A load behind a branch ends, where the branch joins, in a wait for everything in flight; through
// a buffer resource "nothing to read or write here" is an offset outside it, which reads as 0 and
// moves no data.
constexpr int kNowhere = (int)0x80000000;  // an offset outside every resource
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const float *base, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(base), 0, bytes, 0x00020000);
}
// (`uniform`: a wave-uniform part of the offset, for the scalar register; it counts for the range)
__device__ __forceinline__ float get_float(__amdgpu_buffer_rsrc_t rs, bool there, int offset,
                                           int uniform = 0) {
  return __int_as_float(
      __builtin_amdgcn_raw_buffer_load_b32(rs, there ? offset : kNowhere, uniform, 0));
}
__device__ __forceinline__ void put_float(__amdgpu_buffer_rsrc_t rs, bool there, int offset, float x,
                                          int uniform = 0) {
  __builtin_amdgcn_raw_buffer_store_b32(__float_as_int(x), rs, there ? offset : kNowhere, uniform, 0);
}
// symbol s of an utterance (a resource over its int64 symbols): -1 outside [0, C) or not there
__device__ __forceinline__ int get_symbol(__amdgpu_buffer_rsrc_t rs, bool there, int s, int C) {
  typedef int intx2 __attribute__((ext_vector_type(2)));
  const intx2 w = __builtin_amdgcn_raw_buffer_load_b64(rs, there ? 8 * s : kNowhere, 0, 0);
  return there && w[1] == 0 && (unsigned)w[0] < (unsigned)C ? w[0] : -1;
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t symbols_of(const int64_t *symbols, int S) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<int64_t *>(symbols), 0, S * 8, 0x00020000);
}
// waits for this wave's LDS accesses only: loads into registers stay in flight over the barrier
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

}  // namespace

// What the smoothed loss mixes into px and py where they are formed: px = joint k_joint + lm_only k_lm +
// am_only k_am (py likewise), with the row statistics of the two models, max and sum of exp(x - max).
// k_am = 0: no am-only model; its three arrays are not read, but px and py still take the sum of
// `checks`, 0 or a NaN (the unigram of the am-only model is a mean over the whole batch, so that one bad
// row of lm reaches every utterance), which is also left in `check` for the backward.
struct SmoothMix {
  const float *lm_max, *lm_sum, *am_max, *am_z, *unigram, *checks;
  float *check;
  float k_joint, k_lm, k_am;
  int n_checks;
};
// The float32 normalizer product with px / py in its epilogue (simple_normalizer.hip).
void launch_normalizer_f32(const float *lm, const float *am, const int64_t *symbols,
                           const int64_t *boundary, float *lm_max, float *am_max, float *px,
                           float *py, float *norm_raw, const int64_t *window,
                           double delay_penalty, int B, int S, int T, int C, int term,
                           int rnnt_type, const SmoothMix *mix, float *workspace, hipStream_t stream);
// Floats of the workspace that it takes at this size, 0 if it needs none; without one it does without.
long normalizer_workspace(int B, int S, int T, int C, bool windowed);

// frnnt_simple_logprobs_fwd with the delay penalty (simple_logprobs.hip).
int simple_logprobs_fwd(const float *lm, const float *am, const int64_t *symbols,
                        const int64_t *boundary, float *px, float *py, float *lm_max,
                        float *am_max, float *norm_raw, double delay_penalty, int B, int S, int T, int C, int term, int rnnt_type, int window_only,
                        void *stream, const SmoothMix *mix = nullptr, float *workspace = nullptr);
int simple_logprobs_fwd(const double *lm, const double *am, const int64_t *symbols,
                        const int64_t *boundary, double *px, double *py, double *lm_max,
                        double *am_max, double *norm_raw, double delay_penalty, int B, int S, int T, int C, int term, int rnnt_type, int window_only,
                        void *stream);
// What the smoothed loss adds to the gradient products (smoothed_logprobs.hip): to lm's gradient
//   exp(lm[s,c] - lm_max[s]) / lm_sum[s] * ((g_unigram[c] - lm_dot[s]) / N - lm_scale (rx + ry))
//   + lm_scale (rx [c = sym] + ry [c = term]),
// rx and ry the row sums of px_grad and py_grad, and to am's
//   -exp(am[t,c] - max[t]) * am_scale * am_g[t] / am_z[t] * unigram[c];
// the joint model's terms count `joint` times and the per-symbol and termination terms of am symbol_scale
// times.  am_scale = 0: no am-only model; am_g, am_z, lm_dot and g_unigram are not read, and unigram is the
// check that the forward left (SmoothMix).
struct SmoothTerms {
  const float *am_g, *am_z, *unigram, *lm_max, *lm_sum, *lm_dot, *g_unigram;
  float am_scale, symbol_scale, joint, lm_scale, per_row;  // (1 / N)
};
// The backward of the joint model within the smoothed loss: simple_logprobs_bwd with these terms.
// px_grad and py_grad are scaled in place by score_grad (may be NULL); `between` is called when row_x and
// row_y (sums of the scaled gradients) are on their way and the products are not.
int simple_logprobs_bwd_smoothed(const float *lm, const float *am, const int64_t *symbols,
                                 const int64_t *boundary, const float *lm_max, const float *am_max,
                                 const float *norm_raw, const float *score_grad,
                                 int score_grad_stride, double score_grad_scale, float *px_grad,
                                 float *py_grad, float *dmat, float *row_x, float *row_y,
                                 const SmoothTerms &smooth, const std::function<void()> &between,
                                 float *lm_grad, float *am_grad, int B, int S, int T, int C, int term,
                                 int rnnt_type, void *stream);
// 2-byte lm and am (`dtype`: FRNNT_F16 or FRNNT_BF16) as float32, in one launch.
void widen_inputs(int dtype, const void *lm, const void *am, float *lm_wide, float *am_wide,
                  long n_lm, long n_am, hipStream_t stream);

}  // namespace frnnt

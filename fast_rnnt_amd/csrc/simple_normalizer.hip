// The normalizer product of the simple (additive-joiner) loss in float32, with px / py and
// log(P + tiny) written from its accumulators (rnnt_loss.py:66-227; the formulas are at the
// top of simple_logprobs.hip).
#include <algorithm>
#include <cmath>

#include "common.hip.h"
#include "simple_shared.hip.h"

namespace frnnt {
namespace {

// Normalizer GEMM, wave-private LDS slabs.  Both operands are k-contiguous ([rows][C]), the matrix
// cores want one row per lane.  A wave fetches a slab of (kS lattice rows + 32 frames) x 16 k with
// coalesced 16-byte loads (four lanes per row), applies exp(x - shift) in registers, writes the
// slab to its OWN LDS region and feeds the matrix cores from there; the next slab is requested
// between the LDS writes and the products.  k is dealt out to eight shares, slab by slab, a
// wave per share; the waves never wait for each other in the loop (a wave's LDS writes and reads
// are served in program order), only at the end, when the partial sums meet.
//
// The order in which a cell's products are summed -- slabs of 16 k, a slab's k in the order
// 0, 8, 1, 9, ..., eight shares, each with the shifts that its own slabs have set -- depends on C
// alone, not on tiles or workgroups: the lattice recursion sums these normalizers over hundreds of
// steps, and one rounding in a thousand cells moves the occupation probabilities of a long lattice
// by more than everything after it does.  (Splitting the operands into three bfloat16 parts for the
// faster bfloat16 instruction, as the gradient products do, is as accurate and took 70 us instead
// of 102 at B 64, S 120, T 600, C 500, but rounds differently: single occupation probabilities
// moved by up to 8e-3.)
//
// What bounds it: 32 matrix cycles per k and 32 x 32 cells (fp32 MFMA) plus what the wave issues
// for its operands (maximum, exp, LDS: about 14 cycles per 64 elements) -- on this part the two
// add up, also across the waves of a SIMD -- and the prologue and epilogue of a workgroup, which
// another one on the compute unit has to hide: with 32 or 64 lattice rows two share it, with 96 or
// 128, which convert less per cell, one fills it (launch_normalizer_f32 chooses; 96 or 128 rows
// always -> the choice: B 64, S 120, T 600, C 500: 102 -> 74 us; B 8, S 100, T 400, C 5000:
// 105 -> 64; B 2, S 53, T 343, C 4627: 56 -> 33; B 32, S 80, T 250, C 500: 18.6 -> 17.2).
constexpr int kNormK = 16;      // k per slab
constexpr int kNormWaves = 8;   // of a workgroup
constexpr int kNormT = 32;      // frames of a tile
template <int kS>
struct NormShape {
  static constexpr int kWaves = kNormWaves, kThreads = kWaves * kWave;
  static constexpr int kRows = kS + kNormT;      // rows of a slab: lm rows, then am rows
  static constexpr int kLoads = kRows / 16;      // 16-byte loads per lane and slab
  // Row pitch in LDS: 20 floats.  Rows start 16-byte aligned, so a lane's four values of a row go
  // in as one 16-byte write, and a lane reads its row's eight k of a slab half as two 16-byte reads:
  // sixteen lanes' reads (rows 20 floats apart) fall on all 64 banks.
  static constexpr int kPitch = kNormK + 4;
  static constexpr int kSlab = kRows * kPitch;   // floats
  // the partial sums of the waves meet in the slabs' space
  static constexpr int kSumPitch = kNormT + 4;
  static constexpr int kSums = kWaves * kS * kSumPitch;
  static constexpr size_t kLdsBytes = std::max(kWaves * kSlab, kSums) * 4;
  static constexpr int kItems =  // 16-byte outputs per thread
      (kS * kNormT / 4 + kThreads - 1) / kThreads;
  static constexpr size_t kFixedBytes = ((kWaves + 1) * kRows + 3 * kS + kNormT) * 4;  // (below)
  static constexpr int kPerCu = kS <= 64 ? 2 : 1;  // workgroups
  static_assert(kS % 32 == 0 && kS <= 128, "shape");
  static_assert(kPerCu * (kLdsBytes + kFixedBytes) <= 160 << 10, "LDS per CU");
};

// Which tile a workgroup takes.  A unit of placement is an utterance or, for batches of fewer than
// eight, a part of its frames (the parts share lm, the small operand): unit u runs on XCD u % 8,
// whose L2 then holds its operands.
struct NormPlan {
  int t_tiles, s_tiles, part_shift;
};
struct NormTile {
  int b, s_idx, t_idx;
};
__device__ __forceinline__ bool place_tile(int id, const NormPlan &plan, int B, NormTile &o) {
  using dgemm::kXcds;
  const int t_per = (plan.t_tiles + (1 << plan.part_shift) - 1) >> plan.part_shift;
  const int unit_tiles = t_per * plan.s_tiles;
  const int xcd = id % kXcds, slot = id / kXcds, round = slot / unit_tiles;
  const int within = slot - round * unit_tiles;
  const int unit = round * kXcds + xcd;
  o.b = unit >> plan.part_shift;
  o.s_idx = within / t_per;
  o.t_idx = (unit & ((1 << plan.part_shift) - 1)) * t_per + (within - o.s_idx * t_per);
  return o.b < B && o.t_idx < plan.t_tiles;
}

struct NormArgs {
  const float *lm, *am;
  const int64_t *symbols, *boundary, *window;
  float *lm_max, *am_max, *px, *py, *norm_raw;
  Delay<float> delay;
  int B, S, T, C, term, rnnt_type;
};

// f(a constant), the constant being min(max(n, 1), kMost)
template <int kMost, typename F>
__device__ __forceinline__ void with_tiles(int n, F &f) {
  if constexpr (kMost > 1) {
    if (n < kMost) return with_tiles<kMost - 1>(n, f);
  }
  f(std::integral_constant<int, kMost>{});
}

template <int kS>
__global__ void __launch_bounds__(kNormWaves *kWave, 2 * NormShape<kS>::kPerCu)
    simple_fwd_panel_kernel(NormArgs A, NormPlan plan) {
  using Shape = NormShape<kS>;
  constexpr int kT = kNormT, kWaves = kNormWaves;
  constexpr int kRows = Shape::kRows, kLoads = Shape::kLoads, kLmLoads = kS / 16;
  constexpr int kThreads = Shape::kThreads, kItems = Shape::kItems, kPitch = Shape::kPitch;
  using namespace dgemm;
  extern __shared__ __align__(16) float norm_lds[];
  __shared__ float factor[kWaves][kRows];      // scale factors for a wave's partial sums
  __shared__ float row_term[kS], row_sym[kS];  // lm[s,term], lm[s,sym[s]]
  __shared__ float slab_max[kRows];            // row maxima
  __shared__ int row_symbol[kS];
  __shared__ float col_term[kT];  // am[t,term]
  const int S = A.S, T = A.T, C = A.C, S1 = S + 1;
  NormTile tile;
  if (!place_tile((int)blockIdx.x, plan, A.B, tile)) return;
  const int b = tile.b, s_tile = tile.s_idx * kS, t_tile = tile.t_idx * kT;
  const int T1 = A.rnnt_type == kRegular ? T + 1 : T;
  // With a window only rows <= s_end and frames <= t_end are looked at afterwards (frame
  // t_end itself only for the -inf that closes the regular lattice): a tile past t_end has
  // nothing to do -- except the tiles of frame 0, which also store the row maxima of lm
  // and the lattice's last column -- and 32-row tiles past s_end are not computed.
  // (The window's words are looked at only after the first slab has been requested, so that
  // the two round trips to memory overlap; a tile that turns out to have nothing to do has
  // then requested a slab in vain, range-checked like all the others.)
  const float *lmb = A.lm + (long)b * S1 * C;
  const float *amb = A.am + (long)b * T * C;
  const int64_t *symb = A.symbols + (long)b * S;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5, r32 = lane & 31;
  const float ninf = -__builtin_huge_valf();

  // ---- the symbols come first: the gathers below depend on them
  const __amdgpu_buffer_rsrc_t sym_rs = symbols_of(symb, S);
  // threads 0 .. kS-1 own a lattice row each
  const int my_sym = get_symbol(sym_rs, tid < kS && s_tile + tid < S, s_tile + tid, C);

  // ---- what this lane fetches of every slab: rows sub + 16 j, k-offset kq
  const int sub = lane / 4, kq = 4 * (lane % 4);
  // row j of a fetch is lattice row s_tile + sub + 16 j while that stays below kS, a frame
  // after that.  The loads go through buffer resources that cover lm[b] and am[b]: one
  // instruction each, no branch, any alignment; a row past the last one lies past the
  // resource and reads as 0 -- such rows only feed outputs that are never written.
  // Columns at and past C (the last slab) belong to the next row and are replaced by
  // -inf, exp(-inf - shift) = 0 in the product.
  const __amdgpu_buffer_rsrc_t lm_rs =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(lmb), 0, S1 * C * 4, 0x00020000);
  const __amdgpu_buffer_rsrc_t am_rs =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(amb), 0, T * C * 4, 0x00020000);
  const int lm_off = ((s_tile + sub) * C + kq) * 4, am_off = ((t_tile + sub) * C + kq) * 4;  // bytes
  const int step = 16 * C * 4;
  typedef int intx4 __attribute__((ext_vector_type(4)));
  auto fetch = [&](auto live, floatx4 (&into)[kLoads], int k0) {
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      if (j >= 2 * live && j < kLmLoads) continue;
      // (the wave-uniform part of the offset rides in a scalar register)
      const intx4 raw = j < kLmLoads
                            ? __builtin_amdgcn_raw_buffer_load_b128(lm_rs, lm_off, j * step + k0 * 4, 0)
                            : __builtin_amdgcn_raw_buffer_load_b128(
                                  am_rs, am_off, (j - kLmLoads) * step + k0 * 4, 0);
      into[j] = floatx4{__int_as_float(raw[0]), __int_as_float(raw[1]), __int_as_float(raw[2]),
                        __int_as_float(raw[3])};
    }
    if (k0 + kNormK > C) {  // (wave-uniform) the slab that holds column C - 1
#pragma unroll
      for (int j = 0; j < kLoads; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (k0 + kq + i >= C) into[j][i] = ninf;
    }
  };
  const int chunks = (C + kNormK - 1) / kNormK;

  // ---- one pass over k.  The reference subtracts the row maxima before exp
  // (rnnt_loss.py:174-178); a maximum is known only after the whole row has been seen, so
  // each wave works with a SHIFT per row instead: the largest value of the row it had
  // seen when the shift was last set.  A value more than kMargin above the shift (always
  // the case for the first finite value of a row) makes the wave raise the row's shift and
  // scale its partial sums to match; anything closer stays representable, e^(2 kMargin)
  // per product.  Only rows that exceed their margin are touched: which rows share a tile
  // with them has no say in how a row rounds.  The running maxima are kept beside the shifts, and when the waves
  // meet their partial sums are brought to the true maxima, exp(shift - max) <= 1.
  constexpr float kMargin = 30.f;
  floatx4 slab[kLoads];
  if (wave < chunks) fetch(std::integral_constant<int, kS / 32>{}, slab, wave * kNormK);
  const Limits lim = limits_of(A.window, b, S, T);
  if (t_tile > lim.t_end && t_tile > 0) return;
  const int live_rows = min(S1, lim.s_end + 1) - s_tile;  // rows that count

  // ---- epilogue inputs, requested behind the first slab so that their latency hides under the
  // loop: the per-row / per-column terms
  const bool has_row = tid < kS && s_tile + tid < S1;
  const int my_row = (s_tile + tid) * C, my_frame = (t_tile + tid - 128) * C;
  const float my_symval = get_float(lm_rs, has_row && my_sym >= 0, (my_row + my_sym) * 4);
  const float row_value = get_float(lm_rs, has_row, (my_row + A.term) * 4);
  const float frame_value =
      get_float(am_rs, tid >= 128 && t_tile + tid - 128 < T, (my_frame + A.term) * 4);
  const float my_term = tid < kS ? row_value : frame_value;
  // ... and am[b, t, sym[b, s]] of this thread's outputs: 16-byte pieces (row item / 8, frames
  // 4 (item % 8) ..)
  float am_sym[kItems][4];
  auto item_row = [&](int j) { return (tid + kThreads * j) / (kT / 4); };
  const int out_t = 4 * (tid % (kT / 4));
#pragma unroll
  for (int j = 0; j < kItems; ++j) {
    const int m = item_row(j), sr = s_tile + m;
    const int y = get_symbol(sym_rs, m < kS && sr < S && m < live_rows, sr, C);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int tr = t_tile + out_t + i;
      am_sym[j][i] = get_float(am_rs, y >= 0 && tr < T, (tr * C + y) * 4);
    }
  }

  float seen[kLoads];     // largest value this lane has met in the row
  // -shift * log2(e), see exp_shifted; the lanes of a row agree on it.  kUnset while the
  // row has shown nothing finite: it sends -inf to exp2(-inf) = 0 and anything finite
  // above the margin.
  float shift2[kLoads];
  constexpr float kUnset = 3.0e38f;
#pragma unroll
  for (int j = 0; j < kLoads; ++j) seen[j] = ninf, shift2[j] = kUnset;
  const int live_tiles = max(1, min(kS / 32, (live_rows + 31) / 32));
  float *mine = norm_lds + wave * Shape::kSlab;
  floatx16 acc[kS / 32];
#pragma unroll
  for (int j = 0; j < kS / 32; ++j)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[j][v] = 0.f;

  auto across_row = [&](float v) {  // maximum over the four lanes that share a row
    v = fmaxf(v, __shfl_xor(v, 1, kWave));
    return fmaxf(v, __shfl_xor(v, 2, kWave));
  };
  // a row is above its margin exactly when its maximum is
  auto above_margin = [&](float top, float shift2_) {
    return __builtin_fmaf(top, kLog2e, shift2_) > kMargin * kLog2e;
  };
  // (the sums are brought along; -across_row(seen) is the new shift)
  auto raise_shifts = [&](auto live) {
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      if (j >= 2 * live && j < kLmLoads) continue;
      const float top = across_row(seen[j]);
      float f = 1.f;
      if (above_margin(top, shift2[j])) {
        const float now = fminf(shift2[j], -top * kLog2e);
        f = __builtin_amdgcn_exp2f(now - shift2[j]);  // exp(old shift - new shift)
        shift2[j] = now;
      }
      if (lane % 4 == 0) factor[wave][sub + 16 * j] = f;
    }
    __builtin_amdgcn_wave_barrier();
    const float ft = factor[wave][kS + r32];
#pragma unroll
    for (int j = 0; j < live; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v)
        acc[j][v] *= factor[wave][32 * j + 8 * (v / 4) + 4 * half + (v % 4)] * ft;
    __builtin_amdgcn_wave_barrier();
  };
  // where this lane's values of a slab row go, and where its operands lie
  float *put = mine + sub * kPitch + kq;
  const float *get = mine + r32 * kPitch + 8 * half;
  // This wave's share of k, with `live` 32-row tiles that hold lattice rows which count (a
  // constant: the code of a slab is one straight line, whose rows' chains of dependent
  // instructions the compiler interleaves -- with a test per row group a slab took 2.5 times as
  // long).
  auto look = [&](auto live) {  // maxima; true if a row exceeds its margin
    bool above = false;
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      if (j >= 2 * live && j < kLmLoads) continue;
      // two three-input maxima
      seen[j] = max3_raw(max3_raw(slab[j][0], slab[j][1], slab[j][2]), slab[j][3], seen[j]);
      above |= above_margin(seen[j], shift2[j]);
    }
    return above;
  };
  auto walk = [&](auto live) {
    int chunk = wave;
    if (chunk < chunks) {  // the first slab sets the shifts: there are no sums to bring along yet
      (void)look(live);
#pragma unroll
      for (int j = 0; j < kLoads; ++j)
        if (j < 2 * live || j >= kLmLoads)
          shift2[j] = fminf(shift2[j], -across_row(seen[j]) * kLog2e);
    }
    for (; chunk < chunks; chunk += kWaves) {
      // exp(x - shift) to LDS, the request for the slab that takes these registers next, then
      // the products
      if (__any(look(live))) raise_shifts(live);
#pragma unroll
      for (int j = 0; j < kLoads; ++j) {
        if (j >= 2 * live && j < kLmLoads) continue;
        floatx4 e;
#pragma unroll
        for (int i = 0; i < 4; ++i) e[i] = exp_shifted(slab[j][i], shift2[j]);
        *reinterpret_cast<floatx4 *>(put + j * 16 * kPitch) = e;
      }
      if (chunk + kWaves < chunks) fetch(live, slab, (chunk + kWaves) * kNormK);
      // MFMA i of the slab multiplies k = i (lanes 0..31) and k = i + 8 (lanes 32..63): a lane takes
      // its row's share of the slab with 16-byte reads
      floatx4 t_op[2], s_op[kS / 32][2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        t_op[h] = *reinterpret_cast<const floatx4 *>(get + kS * kPitch + 4 * h);
#pragma unroll
        for (int j = 0; j < live; ++j)
          s_op[j][h] = *reinterpret_cast<const floatx4 *>(get + 32 * j * kPitch + 4 * h);
      }
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < live; ++j)
            acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(s_op[j][h][i], t_op[h][i], acc[j], 0, 0, 0);
    }
  };
  with_tiles<kS / 32>(live_tiles, walk);

  // ---- the waves meet: maxima first (each wave's in what was its slab: the row maxima over its
  // share of k, then its final shifts) ...
#pragma unroll
  for (int j = 0; j < kLoads; ++j) {
    const float top = across_row(seen[j]);
    if (lane % 4 == 0) {
      mine[sub + 16 * j] = top;
      mine[kRows + sub + 16 * j] = shift2[j];
    }
  }
  if (tid < kS) {
    row_term[tid] = my_term;
    row_sym[tid] = my_symval;
    row_symbol[tid] = my_sym;
  } else if (tid >= 128 && tid < 128 + kT) {
    col_term[tid - 128] = my_term;
  }
  __syncthreads();
  float *lm_max = A.lm_max + (long)b * S1, *am_max = A.am_max + (long)b * T;
  if (tid < kRows) {
    const int row = tid;
    auto met_by = [&](int w, int i) { return norm_lds[w * Shape::kSlab + i]; };
    float r = met_by(0, row);
#pragma unroll
    for (int w = 1; w < kWaves; ++w) r = fmaxf(r, met_by(w, row));
    // saved for the backward pass; rows that do not exist get a harmless shift
    bool exists;
    if (row < kS) {
      exists = s_tile + row < S1 && row < 32 * live_tiles;
      if (s_tile + row < S1 && t_tile == 0) lm_max[s_tile + row] = exists ? r : 0.f;
    } else {
      exists = t_tile + row - kS < T;
      if (exists && s_tile == 0) am_max[t_tile + row - kS] = r;
    }
    slab_max[row] = exists ? r : 0.f;
    // what brings a wave's partial sums from its shift to the maximum (a wave that met
    // nothing finite in the row holds zeros there)
#pragma unroll
    for (int w = 0; w < kWaves; ++w)
      factor[w][row] = exists ? __builtin_amdgcn_exp2f(-__builtin_fmaf(r, kLog2e, met_by(w, kRows + row))) : 1.f;
  }
  __syncthreads();
  // ... then the partial sums: [wave][kS][kSumPitch] in the slab space
  constexpr int kSumPitch = Shape::kSumPitch;
  const int t_mask = (A.rnnt_type == kRegular && A.boundary) ? (int)A.boundary[4 * b + 3] : -1;
  float *pxb = A.px + (long)b * S * T1;
  float *pyb = A.py + (long)b * S1 * T;
  float *nrb = A.norm_raw ? A.norm_raw + (long)b * S1 * T : nullptr;
  {
    float *part = norm_lds + wave * kS * kSumPitch;
    const float ft = factor[wave][kS + r32];
#pragma unroll
    for (int j = 0; j < kS / 32; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int m = 32 * j + 8 * (v / 4) + 4 * half + (v % 4);
        part[m * kSumPitch + r32] = acc[j][v] * (factor[wave][m] * ft);
      }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kItems; ++j) {
    const int m = item_row(j), sr = s_tile + m, tr = t_tile + out_t;
    if (m >= kS || sr >= S1 || m >= live_rows) continue;
    floatx4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const floatx4 one =
          *reinterpret_cast<const floatx4 *>(norm_lds + (w * kS + m) * kSumPitch + out_t);
#pragma unroll
      for (int i = 0; i < 4; ++i) sum[i] += one[i];
    }
    floatx4 raw, yv, xv;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      raw[i] = logf(sum[i] + 1.17549435e-38f);
      const float norm = raw[i] + slab_max[m] + slab_max[kS + out_t + i];
      yv[i] = (col_term[out_t + i] + row_term[m]) - norm;
      xv[i] = (am_sym[j][i] + row_sym[m]) - norm;
      if (row_symbol[m] < 0) xv[i] = std::numeric_limits<float>::quiet_NaN();  // out-of-vocabulary
      if (tr + i == t_mask) xv[i] = ninf;
      xv[i] = A.delay.at(xv[i], A.boundary, b, tr + i, T);
    }
    if (tr + 4 <= T) {
      if (nrb)
        *reinterpret_cast<floatx4u *>(nrb + sr * T + tr) = floatx4u{raw[0], raw[1], raw[2], raw[3]};
      *reinterpret_cast<floatx4u *>(pyb + sr * T + tr) = floatx4u{yv[0], yv[1], yv[2], yv[3]};
      if (sr < S)
        *reinterpret_cast<floatx4u *>(pxb + sr * T1 + tr) = floatx4u{xv[0], xv[1], xv[2], xv[3]};
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (tr + i >= T) continue;
        if (nrb) nrb[sr * T + tr + i] = raw[i];
        pyb[sr * T + tr + i] = yv[i];
        if (sr < S) pxb[sr * T1 + tr + i] = xv[i];
      }
    }
  }
  // the extra column of the regular lattice: nothing can be emitted after the last frame
  if (A.rnnt_type == kRegular && t_tile == 0 && tid < kS && s_tile + tid < S)
    pxb[(s_tile + tid) * T1 + T] = ninf;
}

template <int kS>
void launch_fwd_panel(const NormArgs &args, const NormPlan &plan, hipStream_t stream) {
  auto kernel = simple_fwd_panel_kernel<kS>;
  constexpr size_t lds = NormShape<kS>::kLdsBytes;
  if (!allow_lds(reinterpret_cast<const void *>(kernel), lds)) return;
  const int t_per = (plan.t_tiles + (1 << plan.part_shift) - 1) >> plan.part_shift;
  const long units = (long)args.B << plan.part_shift;
  const unsigned grid = (unsigned)(dgemm::kXcds * ((units + dgemm::kXcds - 1) / dgemm::kXcds) *
                                   t_per * plan.s_tiles);
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(NormShape<kS>::kThreads), lds, stream, args, plan);
}

// The lattice rows of a workgroup's tile: what a model of the kernel's time says is fastest.  A
// workgroup takes a fixed time and one per round of its eight waves over k, both growing with the
// rows that count; two of 32 or 64 rows share a compute unit, where their loops take 1.76 times as
// long as one's, and their fixed parts overlap only once there is more than one round of
// workgroups.  The constants (microseconds) are fitted to 36 sizes, B 1 .. 128, C 50 .. 5000, that
// were timed with every row count; over these the choice is 0.4 % (geometric mean) from the best.
int rows_of_tile(int B, int S, int T, int C) {
  const int S1 = S + 1, t_tiles = (T + kNormT - 1) / kNormT;
  const int rounds_of_k = (C + kNormWaves * kNormK - 1) / (kNormWaves * kNormK);
  int best = 0;
  double best_us = 0;
  for (int rows : {32, 64, 96, 128}) {
    const int s_tiles = (S1 + rows - 1) / rows;
    const double live = 32.0 * ((S1 + 31) / 32) / s_tiles;  // rows of a tile that count
    const double fixed = 3.4 + 0.072 * live, loop = rounds_of_k * (0.35 + 0.0172 * live);
    // workgroups per compute unit (a ragged batch leaves about 0.85 of the tiles to compute)
    const double per_cu = 0.85 * B * s_tiles * (double)t_tiles / 256;
    double us;
    if (rows > 64) us = std::max(1.0, std::ceil(per_cu)) * (fixed + loop);
    else if (per_cu <= 1) us = fixed + loop;
    else if (per_cu <= 2) us = 1.58 * fixed + 1.76 * loop;
    else us = std::ceil(per_cu / 2) * (fixed + 1.76 * loop);
    if (best == 0 || us < best_us) best = rows, best_us = us;
  }
  return best;
}
}  // namespace

void launch_normalizer_f32(const float *lm, const float *am, const int64_t *symbols,
                           const int64_t *boundary, float *lm_max, float *am_max, float *px,
                           float *py, float *norm_raw, const int64_t *window,
                           double delay_penalty, int B, int S, int T, int C, int term,
                           int rnnt_type, hipStream_t stream) {
  const int rows = rows_of_tile(B, S, T, C);
  const NormArgs args{lm, am, symbols, boundary, window, lm_max, am_max, px, py, norm_raw,
                      Delay<float>{(float)delay_penalty}, B, S, T, C, term, rnnt_type};
  NormPlan plan;
  plan.t_tiles = T > 0 ? (T + kNormT - 1) / kNormT : 1;
  plan.s_tiles = (S + 1 + rows - 1) / rows;
  plan.part_shift = 0;
  while (((long)B << plan.part_shift) < dgemm::kXcds && (2 << plan.part_shift) <= plan.t_tiles)
    ++plan.part_shift;
  switch (rows) {
    case 32: launch_fwd_panel<32>(args, plan, stream); break;
    case 64: launch_fwd_panel<64>(args, plan, stream); break;
    case 96: launch_fwd_panel<96>(args, plan, stream); break;
    default: launch_fwd_panel<128>(args, plan, stream);
  }
}
}  // namespace frnnt

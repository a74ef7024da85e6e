// The normalizer product of the simple (additive-joiner) loss in float32, with px / py and
// log(P + tiny) written from its accumulators (rnnt_loss.py:66-227; the formulas are at the
// top of simple_logprobs.hip).
#include <algorithm>
#include <atomic>
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
// What bounds it: what its waves issue.  On this part the float32 matrix instruction, the VALU and the
// LDS accesses of a SIMD's waves add up (a slab of 32 x 32 cells takes a wave 512 cycles of the
// first, about 250 for maxima, conversions and a quarter-rate exp2, 100 for LDS, and 300 besides), so
// what counts is that every SIMD of the chip has its share of that, and that another workgroup's loop
// covers a workgroup's prologue and epilogue (4.5 and 5 us).  Hence small tiles -- taller ones convert
// less per cell, but leave compute units without any -- dealt out evenly (find_tile), and eight waves of
// one share each or four of two (choose_tile).  Measured within training steps on three batches in turn,
// against tiles chosen among 32 to 128 rows, a workgroup per tile whether it counted or not: B 64, S 120,
// T 600, C 500: 96 -> 89 us; B 32, S 80, T 250, C 500: 20.4 and 20.6; B 16, S 120, T 400, C 5000: 127 ->
// 122; B 10, S 137, T 817, C 500: 47 -> 26; B 5, S 224, T 743, C 2536: 131 -> 64; geometric mean over 64
// sizes, B 1 .. 128, C 50 .. 5000: 5.6 %.  Taller tiles dealt out the same way were the fastest at 12 of the
// 64, mostly by 1 to 5 %, and a choice among all of them, which cannot know how ragged a batch is, gained
// nothing; 64 and 96 rows are left where they have a compute unit each and, where no window makes a batch
// ragged, by the number of tiles of each height.  (128 rows there: 123 us instead of 129 at B 16, S 120,
// T 400, C 5000, and 68 instead of 70 at B 5, S 224, T 743, C 2536, the fastest at these two of 256 sizes.)
constexpr int kNormK = 16;      // k per slab
constexpr int kNormShares = 8;  // of k
constexpr int kNormT = 32;      // frames of a tile
constexpr int kComputeUnits = 256;
template <int kS, int kWaves_, int kParts_>
struct NormShape {
  static constexpr int kWaves = kWaves_, kParts = kParts_, kThreads = kWaves * kWave;
  static constexpr int kTurns = kNormShares / kParts / kWaves;  // shares of a wave, one after the other
  static constexpr int kRows = kS + kNormT;      // rows of a slab: lm rows, then am rows
  static constexpr int kLoads = kRows / 16;      // 16-byte loads per lane and slab
  // Row pitch in LDS: 20 floats.  Rows start 16-byte aligned, so a lane's four values of a row go
  // in as one 16-byte write, and a lane reads its row's eight k of a slab half as two 16-byte reads:
  // sixteen lanes' reads (rows 20 floats apart) fall on all 64 banks.  Sixteen lanes' writes, four rows of 16 floats,
  // span 76: the last row's end falls on the first one's banks (B 64, S 120, T 600, C 500: 4.0 M cycles of conflicts in
  // 2.2 M LDS instructions, the whole kernel's).
  static constexpr int kPitch = kNormK + 4;
  static constexpr int kSlab = kRows * kPitch;   // floats
  // the partial sums of the waves meet in the slabs' space
  static constexpr int kSumPitch = kNormT + 4;
  static constexpr int kSums = kParts > 1 ? 0 : kWaves * kS * kSumPitch;
  // of a tile, in the workspace: every share's partial sums, then its row maxima and final shifts
  static constexpr int kPartial = kS * kNormT + 2 * kRows;
  static constexpr size_t kLdsBytes = std::max(kWaves * kSlab, kSums) * 4;
  static constexpr int kItems =  // 16-byte outputs per thread
      (kS * kNormT / 4 + kThreads - 1) / kThreads;
  static constexpr size_t kFixedBytes = ((kNormShares + 1) * kRows + 3 * kS + kNormT) * 4;  // (below)
  static constexpr int kPerCu = kS <= 64 ? 16 / kWaves : 1;  // workgroups
  static_assert(kS % 32 == 0 && kS <= 96, "shape");
  static_assert(kPerCu * (kLdsBytes + kFixedBytes) <= 160 << 10, "LDS per CU");
};

// Which tile a workgroup takes.  Only tiles that hold a row <= s_end and a frame <= t_end count.  They
// are numbered utterance by utterance, the row tiles of a stretch of frames side by side, and dealt
// out in eight equal runs, one per XCD: every compute unit gets its share, and an utterance's operands
// lie in the L2 of one XCD or two.  (The grid has room for all tiles; the workgroups that are too
// many come last and end at once.  With utterance b on XCD b % 8 and a workgroup per tile whether it
// counts or not, ragged batches left the fullest XCD 15 to 50 % above the average, and workgroups
// that had nothing to do left holes between those that had.)  Every wave finds its tile itself, a lane
// per utterance.
struct NormPlan {
  int t_tiles, s_tiles;
  bool all;  // number all tiles: nothing to look up
};
struct NormTile {
  int b, s_idx, t_idx;
  Limits lim;
};
// Batches of few tiles, counting or not, number them all (choose_tile), and so do those without windows:
// a tile is then known without a look at the window, whose words arrive beside the first operands.
__device__ __forceinline__ bool number_tile(int id, const NormPlan &plan, int B, NormTile &o) {
  using dgemm::kXcds;
  const int of_utterance = plan.s_tiles * plan.t_tiles, total = B * of_utterance;
  const int per_xcd = (total + kXcds - 1) / kXcds, in_run = id / kXcds;
  const int n = id % kXcds * per_xcd + in_run;
  if (in_run >= per_xcd || n >= total) return false;
  o.b = n / of_utterance;
  const int within = n - o.b * of_utterance;
  o.t_idx = within / plan.s_tiles, o.s_idx = within - o.t_idx * plan.s_tiles;
  return true;
}
// inclusive sum over the lanes up to this one
__device__ __forceinline__ int sum_up_to_lane(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);   // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);   // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);   // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);   // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31
  return v;
}
// row tiles of an utterance that count
template <int kS>
__device__ __forceinline__ int row_tiles(const Limits &lim) {
  return lim.s_end / kS + 1;
}
template <int kS>
__device__ __forceinline__ bool find_tile(int id, const NormPlan &plan, const int64_t *window, int B,
                                          int S, int T, int lane, NormTile &o) {
  using dgemm::kXcds;
  struct {
    Limits lim;
    int tiles;
  } mine;
  auto look_up = [&](int b) {
    mine.lim = limits_of(window, min(b, B - 1), S, T);
    mine.tiles = b < B ? row_tiles<kS>(mine.lim) * min(plan.t_tiles, mine.lim.t_end / kNormT + 1) : 0;
  };
  look_up(lane);
  int sum = sum_up_to_lane(mine.tiles), total = __builtin_amdgcn_readlane(sum, kWave - 1);
  for (int b0 = kWave; b0 < B; b0 += kWave) {
    look_up(b0 + lane);
    total += __builtin_amdgcn_readlane(sum_up_to_lane(mine.tiles), kWave - 1);
  }
  const int per_xcd = (total + kXcds - 1) / kXcds, in_run = id / kXcds;
  int n = id % kXcds * per_xcd + in_run;
  if (in_run >= per_xcd || n >= total) return false;
  if (B > kWave) {
    look_up(lane);
    sum = sum_up_to_lane(mine.tiles);
  }
  int b0 = 0;
  for (int upto; n >= (upto = __builtin_amdgcn_readlane(sum, kWave - 1)); n -= upto) {
    b0 += kWave;
    look_up(b0 + lane);
    sum = sum_up_to_lane(mine.tiles);
  }
  const int at = __builtin_popcountll(__ballot(sum <= n));  // the first lane whose sum exceeds n
  n -= __builtin_amdgcn_readlane(sum - mine.tiles, at);
  o.b = b0 + at;
  o.lim.s_end = __builtin_amdgcn_readlane(mine.lim.s_end, at);
  o.lim.t_end = __builtin_amdgcn_readlane(mine.lim.t_end, at);
  const int s_tiles = row_tiles<kS>(o.lim);
  o.t_idx = n / s_tiles, o.s_idx = n - o.t_idx * s_tiles;
  return true;
}

struct NormArgs {
  const float *lm, *am;
  const int64_t *symbols, *boundary, *window;
  float *lm_max, *am_max, *px, *py, *norm_raw;
  Delay<float> delay;
  int B, S, T, C, term, rnnt_type;
  unsigned long long *met;    // (tiles in parts) a word per tile, holding anything
  float *partial;             // kNormShares * kPartial floats per tile
  unsigned long long ticket;  // an even number that no other call of this process has had (next_ticket)
};

// A joint model on its own
struct NoMix {};

// f(a constant), the constant being min(max(n, 1), kMost)
template <int kMost, typename F>
__device__ __forceinline__ void with_tiles(int n, F &f) {
  if constexpr (kMost > 1) {
    if (n < kMost) return with_tiles<kMost - 1>(n, f);
  }
  f(std::integral_constant<int, kMost>{});
}

// With a Mix (the smoothed loss) px and py leave interpolated with the lm-only and the am-only model:
// am[t,sym[s]] and what depends on a row or a frame alone are here already, and a launch of its own for
// the interpolation would read and write every cell again (B 32, S 80, T 250, C 500: 12.8 us).
//
// kParts = 2: two workgroups share a tile, four of k's shares each.  They leave their partial sums in a
// workspace; the one that comes second brings all together, in the one order that there is.
template <int kS, int kWaves, int kParts, typename Mix>
__global__ void __launch_bounds__(kWaves *kWave, (kWaves / 4 * NormShape<kS, kWaves, kParts>::kPerCu))
    simple_fwd_panel_kernel(NormArgs A, NormPlan plan, Mix mix) {
  constexpr bool kMix = !std::is_same_v<Mix, NoMix>;
  using Shape = NormShape<kS, kWaves, kParts>;
  constexpr int kT = kNormT, kShares = kNormShares, kTurns = Shape::kTurns;
  constexpr int kRows = Shape::kRows, kLoads = Shape::kLoads, kLmLoads = kS / 16;
  constexpr int kThreads = Shape::kThreads, kItems = Shape::kItems, kPitch = Shape::kPitch;
  using namespace dgemm;
  extern __shared__ __align__(16) float norm_lds[];
  __shared__ float factor[kShares][kRows];      // scale factors for a wave's partial sums
  __shared__ float row_term[kS], row_sym[kS];  // lm[s,term], lm[s,sym[s]]
  __shared__ float slab_max[kRows];            // row maxima
  __shared__ int row_symbol[kS];
  __shared__ float col_term[kT];  // am[t,term]
  // lm-only terms of a row (px, py), log-unigram of its symbol; am-only term (py) and normalizer of a frame
  constexpr int kMixRows = kMix ? kS : 1, kMixFrames = kMix ? kT : 1;
  __shared__ float mix_x[kMixRows], mix_y[kMixRows], mix_u[kMixRows], mix_n[kMixFrames], mix_t[kMixFrames];
  const int S = A.S, T = A.T, C = A.C, S1 = S + 1;
  NormTile tile;
  const int tid = threadIdx.x, lane = tid & 63;
  // (a tile's parts on one XCD, one after the other)
  const int part = kParts > 1 ? (int)blockIdx.x / kXcds % kParts : 0;
  const int id = kParts > 1 ? (int)blockIdx.x / (kXcds * kParts) * kXcds + (int)blockIdx.x % kXcds : (int)blockIdx.x;
  if (plan.all ? !number_tile(id, plan, A.B, tile)
               : !find_tile<kS>(id, plan, A.window, A.B, S, T, lane, tile))
    return;
  const int b = tile.b, s_tile = tile.s_idx * kS, t_tile = tile.t_idx * kT;
  const int T1 = A.rnnt_type == kRegular ? T + 1 : T;
  // With a window only rows <= s_end and frames <= t_end are looked at afterwards (frame
  // t_end itself only for the -inf that closes the regular lattice): other tiles are not
  // computed, nor 32-row tiles past s_end.
  const float *lmb = A.lm + (long)b * S1 * C;
  const float *amb = A.am + (long)b * T * C;
  const int64_t *symb = A.symbols + (long)b * S;
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
  const int first_share = part * kWaves + wave;
  if (first_share < chunks) fetch(std::integral_constant<int, kS / 32>{}, slab, first_share * kNormK);
  if (plan.all) {
    tile.lim = limits_of(A.window, b, S, T);
    if (t_tile > 0 && t_tile > tile.lim.t_end) return;
    if (tile.s_idx >= row_tiles<kS>(tile.lim)) return;
  }
  const int live_rows = min(S1, tile.lim.s_end + 1) - s_tile;  // rows that count

  // ---- epilogue inputs, requested behind the first slab so that their latency hides under the
  // loop: the per-row / per-column terms
  const bool has_row = tid < kS && s_tile + tid < S1;
  const int my_row = (s_tile + tid) * C, my_frame = (t_tile + tid - 128) * C;
  const float my_symval = get_float(lm_rs, has_row && my_sym >= 0, (my_row + my_sym) * 4);
  const float row_value = get_float(lm_rs, has_row, (my_row + A.term) * 4);
  const float frame_value =
      get_float(am_rs, tid >= 128 && t_tile + tid - 128 < T, (my_frame + A.term) * 4);
  const float my_term = tid < kS ? row_value : frame_value;
  // (of a row: maximum and sum of the lm-only model, unigram of its symbol; of a frame: maximum and sum
  // of the am-only model, unigram of the termination symbol)
  float mix_max = 0.f, mix_sum = 1.f, mix_unigram = 1.f;
  if constexpr (kMix) {
    const bool is_row = tid < kS, has_frame = tid >= 128 && t_tile + tid - 128 < T;
    const long rows = (long)b * S1, frames = (long)b * T;
    const int at = 4 * (is_row ? s_tile + tid : t_tile + tid - 128);
    mix_max = get_float(buffer_of(mix.lm_max + rows, S1 * 4), has_row, at);
    mix_sum = get_float(buffer_of(mix.lm_sum + rows, S1 * 4), has_row, at);
    if (mix.k_am != 0.f) {  // (uniform)
      const float am_max = get_float(buffer_of(mix.am_max + frames, T * 4), has_frame, at);
      const float am_z = get_float(buffer_of(mix.am_z + frames, T * 4), has_frame, at);
      mix_unigram = get_float(buffer_of(mix.unigram, C * 4), true, 4 * (is_row ? max(my_sym, 0) : A.term));
      mix_max = is_row ? mix_max : am_max, mix_sum = is_row ? mix_sum : am_z;
    } else if (!is_row) {
      for (int i = lane; i < mix.n_checks; i += 4 * kWave)
#pragma unroll
        for (int u = 0; u < 4; ++u) mix_max += mix.checks[min(i + kWave * u, mix.n_checks - 1)];
    }
  }
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

  float seen[kTurns][kLoads];     // largest value this lane has met in the row, per share
  // -shift * log2(e), see exp_shifted; the lanes of a row agree on it.  kUnset while the
  // row has shown nothing finite: it sends -inf to exp2(-inf) = 0 and anything finite
  // above the margin.
  float shift2[kTurns][kLoads];
  constexpr float kUnset = 3.0e38f;
#pragma unroll
  for (int q = 0; q < kTurns; ++q)
#pragma unroll
    for (int j = 0; j < kLoads; ++j) seen[q][j] = ninf, shift2[q][j] = kUnset;
  const int live_tiles = min(kS / 32, (live_rows + 31) / 32);
  float *mine = norm_lds + wave * Shape::kSlab;
  floatx16 acc[kTurns][kS / 32];
#pragma unroll
  for (int q = 0; q < kTurns; ++q)
#pragma unroll
    for (int j = 0; j < kS / 32; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[q][j][v] = 0.f;

  auto across_row = [&](float v) {  // maximum over the four lanes that share a row
    v = fmaxf(v, __shfl_xor(v, 1, kWave));
    return fmaxf(v, __shfl_xor(v, 2, kWave));
  };
  // a row is above its margin exactly when its maximum is
  auto above_margin = [&](float top, float shift2_) {
    return __builtin_fmaf(top, kLog2e, shift2_) > kMargin * kLog2e;
  };
  // (the sums are brought along; -across_row(seen) is the new shift)
  auto raise_shifts = [&](auto live, auto q) {
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      if (j >= 2 * live && j < kLmLoads) continue;
      const float top = across_row(seen[q][j]);
      float f = 1.f;
      if (above_margin(top, shift2[q][j])) {
        const float now = fminf(shift2[q][j], -top * kLog2e);
        f = __builtin_amdgcn_exp2f(now - shift2[q][j]);  // exp(old shift - new shift)
        shift2[q][j] = now;
      }
      if (lane % 4 == 0) factor[wave][sub + 16 * j] = f;
    }
    __builtin_amdgcn_wave_barrier();
    const float ft = factor[wave][kS + r32];
#pragma unroll
    for (int j = 0; j < live; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v)
        acc[q][j][v] *= factor[wave][32 * j + 8 * (v / 4) + 4 * half + (v % 4)] * ft;
    __builtin_amdgcn_wave_barrier();
  };
  // where this lane's values of a slab row go, and where its operands lie
  float *put = mine + sub * kPitch + kq;
  const float *get = mine + r32 * kPitch + 8 * half;
  // This wave's share of k, with `live` 32-row tiles that hold lattice rows which count (a
  // constant: the code of a slab is one straight line, whose rows' chains of dependent
  // instructions the compiler interleaves -- with a test per row group a slab took 2.5 times as
  // long).
  auto look = [&](auto live, auto q) {  // maxima; true if a row exceeds its margin
    bool above = false;
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      if (j >= 2 * live && j < kLmLoads) continue;
      // two three-input maxima
      seen[q][j] = max3_raw(max3_raw(slab[j][0], slab[j][1], slab[j][2]), slab[j][3], seen[q][j]);
      above |= above_margin(seen[q][j], shift2[q][j]);
    }
    return above;
  };
  auto walk_share = [&](auto live, auto q) {
    const int share = first_share + kWaves * q;
    int chunk = share;
    if (chunk < chunks) {  // the first slab sets the shifts: there are no sums to bring along yet
      (void)look(live, q);
#pragma unroll
      for (int j = 0; j < kLoads; ++j)
        if (j < 2 * live || j >= kLmLoads)
          shift2[q][j] = fminf(shift2[q][j], -across_row(seen[q][j]) * kLog2e);
    }
    for (; chunk < chunks; chunk += kShares) {
      // exp(x - shift) to LDS, the request for the slab that takes these registers next, then
      // the products
      if (__any(look(live, q))) raise_shifts(live, q);
#pragma unroll
      for (int j = 0; j < kLoads; ++j) {
        if (j >= 2 * live && j < kLmLoads) continue;
        floatx4 e;
#pragma unroll
        for (int i = 0; i < 4; ++i) e[i] = exp_shifted(slab[j][i], shift2[q][j]);
        *reinterpret_cast<floatx4 *>(put + j * 16 * kPitch) = e;
      }
      int next = chunk + kShares;
      if (q + 1 < kTurns && next >= chunks) next = share + kWaves;  // (the next share's first)
      if (next < chunks) fetch(live, slab, next * kNormK);
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
            acc[q][j] =
                __builtin_amdgcn_mfma_f32_32x32x2f32(s_op[j][h][i], t_op[h][i], acc[q][j], 0, 0, 0);
    }
  };
  auto walk = [&](auto live) {
    walk_share(live, std::integral_constant<int, 0>{});
    if constexpr (kTurns > 1) walk_share(live, std::integral_constant<int, 1>{});
  };
  with_tiles<kS / 32>(live_tiles, walk);

  // ---- the waves meet: maxima first (each wave's in what was its slab: the row maxima over its
  // share of k, then its final shifts) ...
  // (tiles in parts) Both parts' sums go through the workspace, past the XCDs' own L2: a share's cells, then
  // what follows; a part that finds the other's ticket in the tile's word comes second.  (What the word held
  // before is no ticket of this call: a call's ticket is its own, and a replay of a recorded call finds the 0
  // that the second part leaves, or what the recursion, whose scratch the workspace is next, has computed since.)
  const long tile_id = ((long)b * plan.t_tiles + tile.t_idx) * plan.s_tiles + tile.s_idx;
  float *const met = kParts > 1 ? A.partial + tile_id * (kNormShares * Shape::kPartial) : nullptr;
  const __amdgpu_buffer_rsrc_t met_rs = buffer_of(met, kNormShares * Shape::kPartial * 4);
  constexpr int kAgent = 16;  // sc1: device scope
  if constexpr (kParts > 1) {
    const int at = first_share * Shape::kPartial;
#pragma unroll
    for (int j = 0; j < kS / 32; ++j) {
      if (j >= live_tiles) break;  // (uniform)
#pragma unroll
      for (int v = 0; v < 16; ++v)
        __builtin_amdgcn_raw_buffer_store_b32(
            __float_as_int(acc[0][j][v]), met_rs,
            4 * (at + (32 * j + 8 * (v / 4) + 4 * half + (v % 4)) * kT + r32), 0, kAgent);
    }
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      const float top = across_row(seen[0][j]);
      const int to = lane % 4 == 0 ? 4 * (at + kS * kT + sub + 16 * j) : kNowhere;
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_int(top), met_rs, to, 0, kAgent);
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_int(shift2[0][j]), met_rs, to, 4 * kRows, kAgent);
    }
    __shared__ int second;
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): they have arrived
    asm volatile("" ::: "memory");
    __syncthreads();
    if (tid == 0) {
      unsigned long long *word = A.met + tile_id;
      second = __hip_atomic_exchange(word, A.ticket + part, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
               A.ticket + (1 - part);
      if (second) __hip_atomic_store(word, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!second) return;
  } else {
#pragma unroll
    for (int q = 0; q < kTurns; ++q)
#pragma unroll
      for (int j = 0; j < kLoads; ++j) {
        const float top = across_row(seen[q][j]);
        if (lane % 4 == 0) {
          mine[2 * kRows * q + sub + 16 * j] = top;
          mine[2 * kRows * q + kRows + sub + 16 * j] = shift2[q][j];
        }
      }
  }
  // (all of wave 2, whose first lanes own the frames)
  const float check = kMix && __any(mix_max != mix_max) ? std::numeric_limits<float>::quiet_NaN() : 0.f;
  if (tid < kS) {
    row_term[tid] = my_term;
    row_sym[tid] = my_symval;
    row_symbol[tid] = my_sym;
    if constexpr (kMix) {
      const float ln = logf(mix_sum) + mix_max;
      mix_x[tid] = my_symval - ln;
      mix_y[tid] = my_term - ln;
      mix_u[tid] = logf(mix_unigram);
    }
  } else if (tid >= 128 && tid < 128 + kT) {
    col_term[tid - 128] = my_term;
    if constexpr (kMix) {
      if (mix.k_am == 0.f && tid == 128 && b == 0 && t_tile == 0 && s_tile == 0) *mix.check = check;
      const float an = logf(mix_sum) + mix_max;
      mix_n[tid - 128] = mix.k_am != 0.f ? an : check;
      mix_t[tid - 128] = mix.k_am != 0.f ? ((my_term + logf(mix_unigram)) - an) * mix.k_am : check;
    }
  }
  __syncthreads();
  float *lm_max = A.lm_max + (long)b * S1, *am_max = A.am_max + (long)b * T;
  if (tid < kRows) {
    const int row = tid;
    float tops[kShares], shifts[kShares];
#pragma unroll
    for (int w = 0; w < kShares; ++w) {
      if constexpr (kParts > 1) {
        const int at = 4 * (w * Shape::kPartial + kS * kT + row);
        tops[w] = __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(met_rs, at, 0, kAgent));
        shifts[w] = __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(met_rs, at, 4 * kRows, kAgent));
      } else {
        const float *met_by = norm_lds + w % kWaves * Shape::kSlab + w / kWaves * 2 * kRows + row;
        tops[w] = met_by[0], shifts[w] = met_by[kRows];
      }
    }
    float r = tops[0];
#pragma unroll
    for (int w = 1; w < kShares; ++w) r = fmaxf(r, tops[w]);
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
    for (int w = 0; w < kShares; ++w)
      factor[w][row] = exists ? __builtin_amdgcn_exp2f(-__builtin_fmaf(r, kLog2e, shifts[w])) : 1.f;
  }
  __syncthreads();
  // ... then the partial sums: [wave][kS][kSumPitch] in the slab space, a share of every wave at a time
  constexpr int kSumPitch = Shape::kSumPitch;
  const int t_mask = (A.rnnt_type == kRegular && A.boundary) ? (int)A.boundary[4 * b + 3] : -1;
  float *pxb = A.px + (long)b * S * T1;
  float *pyb = A.py + (long)b * S1 * T;
  float *nrb = A.norm_raw ? A.norm_raw + (long)b * S1 * T : nullptr;
  floatx4 sums[kItems];
#pragma unroll
  for (int j = 0; j < kItems; ++j) sums[j] = floatx4{0.f, 0.f, 0.f, 0.f};
  if constexpr (kParts > 1) {
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      const int m = item_row(j);
      if (m >= kS) continue;
      intx4 one[kShares];
#pragma unroll
      for (int w = 0; w < kShares; ++w)
        one[w] = __builtin_amdgcn_raw_buffer_load_b128(met_rs, 4 * (m * kT + out_t), 4 * w * Shape::kPartial,
                                                       kAgent);
#pragma unroll
      for (int w = 0; w < kShares; ++w)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          sums[j][i] += __int_as_float(one[w][i]) * (factor[w][m] * factor[w][kS + out_t + i]);
    }
  } else {
#pragma unroll
    for (int q = 0; q < kTurns; ++q) {
      if (q > 0) __syncthreads();
      float *part = norm_lds + wave * kS * kSumPitch;
      const float *my_factor = factor[wave + kWaves * q];
      const float ft = my_factor[kS + r32];
#pragma unroll
      for (int j = 0; j < kS / 32; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int m = 32 * j + 8 * (v / 4) + 4 * half + (v % 4);
          part[m * kSumPitch + r32] = acc[q][j][v] * (my_factor[m] * ft);
        }
      __syncthreads();
#pragma unroll
      for (int j = 0; j < kItems; ++j) {
        const int m = item_row(j);
        if (m >= kS) continue;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
          const floatx4 one =
              *reinterpret_cast<const floatx4 *>(norm_lds + (w * kS + m) * kSumPitch + out_t);
#pragma unroll
          for (int i = 0; i < 4; ++i) sums[j][i] += one[i];
        }
      }
    }
  }
#pragma unroll
  for (int j = 0; j < kItems; ++j) {
    const int m = item_row(j), sr = s_tile + m, tr = t_tile + out_t;
    if (m >= kS || sr >= S1 || m >= live_rows) continue;
    const floatx4 sum = sums[j];
    floatx4 raw, yv, xv;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      raw[i] = logf(sum[i] + 1.17549435e-38f);
      const float norm = raw[i] + slab_max[m] + slab_max[kS + out_t + i];
      yv[i] = (col_term[out_t + i] + row_term[m]) - norm;
      xv[i] = (am_sym[j][i] + row_sym[m]) - norm;
      if constexpr (kMix) {
        // (left to right, as rnnt_loss.py:1338-1362)
        float am_only = mix_n[out_t + i];
        if (mix.k_am != 0.f) am_only = ((am_sym[j][i] + mix_u[m]) - am_only) * mix.k_am;  // (uniform)
        yv[i] = yv[i] * mix.k_joint + mix_y[m] * mix.k_lm + mix_t[out_t + i];
        xv[i] = xv[i] * mix.k_joint + mix_x[m] * mix.k_lm + am_only;
      }
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
  // (and what the row tiles that do not count would have left)
  if (t_tile == 0 && tile.s_idx == row_tiles<kS>(tile.lim) - 1) {
    for (int s = s_tile + kS + tid; s < S1; s += kThreads) {
      lm_max[s] = 0.f;
      if (A.rnnt_type == kRegular && s < S) pxb[s * T1 + T] = ninf;
    }
  }
}

// A ticket for a call's shared tiles, whichever of the kernels it takes.  The memory may hold anything, also small whole
// numbers: above a count of the calls, a ticket has the bits of a signalling NaN that no arithmetic forms.
unsigned long long next_ticket() {
  static std::atomic<unsigned long long> calls{0};
  return 0xffa5c3ull << 40 | (2 * calls.fetch_add(1, std::memory_order_relaxed) & ((1ull << 40) - 1));
}

template <int kS, int kWaves, int kParts, typename Mix>
void launch_fwd_panel(NormArgs args, const NormPlan &plan, const Mix &mix, float *workspace, hipStream_t stream) {
  using Shape = NormShape<kS, kWaves, kParts>;
  auto kernel = simple_fwd_panel_kernel<kS, kWaves, kParts, Mix>;
  constexpr size_t lds = Shape::kLdsBytes;
  if (!allow_lds(reinterpret_cast<const void *>(kernel), lds)) return;
  const long tiles = (long)args.B * plan.t_tiles * plan.s_tiles;
  const unsigned grid = (unsigned)((tiles + dgemm::kXcds - 1) / dgemm::kXcds * dgemm::kXcds * kParts);
  if (kParts > 1) {
    args.ticket = next_ticket();
    args.met = reinterpret_cast<unsigned long long *>(workspace);
    args.partial = workspace + (2 * tiles + 3) / 4 * 4;
  }
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(Shape::kThreads), lds, stream, args, plan, mix);
}

struct NormChoice {
  int rows, waves;  // of a tile
  bool all;         // its numbering: see number_tile
  int parts = 1;    // workgroups that share it
};
// The tile that a call takes.  `windowed`: what lies outside an utterance's window does not count.
NormChoice choose_tile(int B, int S, int T, int C, bool windowed, bool workspace) {
  const long t_tiles = T > 0 ? (T + kNormT - 1) / kNormT : 1;
  const int s_tiles = (S + 32) / 32;
  const long tiles = B * t_tiles * s_tiles;
  const int rounds = (C + kNormShares * kNormK - 1) / (kNormShares * kNormK);
  auto taller = [&](int rows) { return B * t_tiles * ((S + rows) / rows); };
  // Batches that leave half of the compute units without a tile, and loops of some length: two workgroups
  // share a tile, which moves half of its waves to an idle unit (B 2, S 44, T 287, C 5194, 36 tiles: 35.7 -> 27.9
  // us; B 4, S 28, T 186, C 3806, 24: 28.1 -> 21.9; B 2, S 114, T 463, C 3713, 120: 29.7 -> 24.1; B 8, S 15, T 84,
  // C 1961, 24: 17.4 -> 15.1; B 1, S 90, T 299, C 838, 30: 11.6 -> 10.1).  With shorter loops, or as many tiles as
  // there are units, the way through the workspace costs more than it gives (B 49, S 8, T 51, C 654, 98
  // tiles: 9.8 -> 11.3; B 49, S 17, T 130, C 1219, 245: 16.3 -> 17.3; B 53, S 24, T 116, C 2485, 212: 23.4 -> 27.1;
  // B 6, S 152, T 415, C 2803, 390: 42.9 -> 51.2).
  if (workspace && 2 * tiles <= kComputeUnits && rounds >= 7) return {32, 4, true, 2};
  // Four waves of two shares let four workgroups share a compute unit, whose prologues and epilogues
  // hide under each other's loops; eight of one share end a workgroup sooner.  The former pay where
  // a compute unit has several workgroups in turn and their loops are short (B 64, S 120, T 600,
  // C 500: 89 against 98 us; B 13, S 125, T 451, C 60: 12.1 against 14.7; B 10, S 137, T 817, C 500: 26.2
  // against 28.5), the latter elsewhere (B 23, S 41, T 444, C 444: 15.5 against 16.4; B 98, S 65,
  // T 209, C 722: 55.7 against 57.3; B 4, S 15, T 47, C 4482: 32 against 42).
  const int waves = tiles > 3 * kComputeUnits && rounds <= 5 ? 4 : 8;
  if (!windowed) {
    // Every tile counts and none is looked up.  The compute units take them in turn, so that a launch
    // lasts as long as the fullest unit: its tiles times what one takes, 1 : 1.8 : 2.35 for 32, 64 and 96
    // rows (C 5000: 35, 64 and 81 us).  32 rows against taller ones: 64 rows, B 16, S 120, T 400, C 5000:
    // 142 us against 129; B 64, S 40, T 200, C 1000: 44 against 39; B 5, S 224, T 743, C 2536: 77 against 70; 96
    // rows, B 32, S 80, T 250, C 500: 24.6 against 20.4, C 2500: 82 against 61; B 2, S 250, T 1320, C 4606: 103
    // against 87.  Prologue and epilogue of a tall tile show where loops are short (64 rows, B 128, S 60, T 250,
    // C 100: 23.1 against 23.7), and those of 96 rows, which have a unit to themselves, wherever
    // they come in turn (B 70, S 78, T 565, C 461: 83 against 95).  Three tiles of 32 to a unit are all there at
    // once with four waves, not with eight (B 47, S 53, T 243, C 1246: 45 against 53; B 45, S 33, T 240,
    // C 892: 29.7 against 34.0; B 15, S 58, T 568, C 120: 12.8 against 14.7).  Over 256 sizes, B 1 .. 128, C 50 ..
    // 5000, the choice is 0.2 % (geometric mean) from the best, 32 rows by the rule above 1.8 %.
    auto of_a_unit = [&](int rows) { return (taller(rows) + kComputeUnits - 1) / kComputeUnits; };
    NormChoice best{32, of_a_unit(32) == 3 ? 4 : waves, true};
    double least = (double)of_a_unit(32);
    if (rounds >= 4 && 1.8 * of_a_unit(64) < least) least = 1.8 * of_a_unit(64), best = {64, 8, true};
    if ((rounds >= 4 || best.waves == 8) && of_a_unit(96) == 1 && 2.35 < least) best = {96, 8, true};
    return best;
  }
  // A compute unit for each tile, or two to a unit that soon end or belong to lattices of a single row of
  // tiles, of which only the frames are ragged: the look-up would cost more than it gains.  (B 70, S 13,
  // T 149, C 80: 9.3 us with it, 8.0 without; one row of 384 to 500 tiles, B 96, S 14, T 114, C 854: 20.2 and
  // 19.2; B 128, S 10, T 100, C 500: 16.1 and 14.6; B 110, S 28, T 128, C 640: 18.7 and 17.4.  Two rows of
  // them, B 25, S 50, T 258, C 1400: 26.7 and 37.8; one row of more than two to a unit, B 80, S 12, T 250,
  // C 1500: 45 and 53; B 128, S 20, T 300, C 500: 30.5 and 34.5.)
  const bool two = rounds <= 2 || s_tiles == 1;
  if (tiles <= (two ? 2 : 1) * kComputeUnits) return {32, waves, true};
  // Where tiles of 64 or 96 rows all but fill the compute units, one to each, those of 32 would leave many
  // units with one more than the rest, and the taller ones are faster: 64 rows, B 60, S 50, T 110, C 2500
  // (240 tiles): 41.3 us against 49.5; B 8, S 100, T 400, C 5000 (208): 68.3 against 69.3; B 21, S 47, T 333,
  // C 503 (231): 14.8 against 15.5; B 64, S 40, T 100, C 800 (256): 18.3 against 19.3; 96 rows, B 32, S 80,
  // T 250 (256), C 500: 19.5 against 20.1, C 2500: 54.7 against 58.5; B 14, S 95, T 570, C 2000 (252): 46.6
  // against 49.1; B 64, S 85, T 110, C 150 (256): 12.9 against 15.0.  With fewer of them (of a ragged
  // batch some 0.7 of the small tiles count, and they come to one each as well) the small ones are: 64 rows,
  // B 40, S 60, T 100, C 600 (160): 15.8 against 12.2; B 40, S 33, T 150, C 400 (200): 12.2 against 10.3;
  // 96 rows, B 30, S 70, T 250, C 500 (240): 18.9 against 16.2; B 23, S 73, T 202, C 4093 (161): 78 against 75.
  auto fills = [&](int rows) {
    return taller(rows) <= kComputeUnits && 20 * taller(rows) > (rows == 64 ? 16 : 19) * kComputeUnits;
  };
  if (fills(64)) return {64, 8, true};
  if (fills(96)) return {96, 8, true};
  return {32, waves, false};
}
}  // namespace

void launch_normalizer_f32(const float *lm, const float *am, const int64_t *symbols,
                           const int64_t *boundary, float *lm_max, float *am_max, float *px,
                           float *py, float *norm_raw, const int64_t *window,
                           double delay_penalty, int B, int S, int T, int C, int term,
                           int rnnt_type, const SmoothMix *mix, float *workspace, hipStream_t stream) {
  if (reinterpret_cast<uintptr_t>(workspace) & 15) workspace = nullptr;  // (words of 8 bytes, pieces of 16)
  const NormArgs args{lm, am, symbols, boundary, window, lm_max, am_max, px, py, norm_raw,
                      Delay<float>{(float)delay_penalty}, B, S, T, C, term, rnnt_type, nullptr, nullptr, 0};
  const NormChoice choice = choose_tile(B, S, T, C, window != nullptr, workspace != nullptr);
  const NormPlan plan{T > 0 ? (T + kNormT - 1) / kNormT : 1, (S + choice.rows) / choice.rows, choice.all};
  auto launch = [&](const auto &m) {
    if (choice.parts > 1)
      launch_fwd_panel<32, 4, 2>(args, plan, m, workspace, stream);
    else if (choice.rows == 96)
      launch_fwd_panel<96, 8, 1>(args, plan, m, nullptr, stream);
    else if (choice.rows == 64)
      launch_fwd_panel<64, 8, 1>(args, plan, m, nullptr, stream);
    else if (choice.waves == 4)
      launch_fwd_panel<32, 4, 1>(args, plan, m, nullptr, stream);
    else
      launch_fwd_panel<32, 8, 1>(args, plan, m, nullptr, stream);
  };
  if (mix)
    launch(*mix);
  else
    launch(NoMix{});
}
long normalizer_workspace(int B, int S, int T, int C, bool windowed) {
  const NormChoice choice = choose_tile(B, S, T, C, windowed, true);
  if (choice.parts == 1) return 0;
  const long tiles = (long)B * (T > 0 ? (T + kNormT - 1) / kNormT : 1) * ((S + choice.rows) / choice.rows);
  return (2 * tiles + 3) / 4 * 4 +
         tiles * kNormShares * ((long)choice.rows * kNormT + 2 * (choice.rows + kNormT));
}
}  // namespace frnnt

extern "C" int frnnt_simple_logprobs_tile(int B, int S, int T, int C, int window_only, int *waves) {
  using namespace frnnt;
  if (B < 1 || S < 0 || T < 0 || C < 1) return fail(FRNNT_EINVAL, "simple_logprobs_tile: bad size");
  const NormChoice choice = choose_tile(B, S, T, C, window_only != 0, false);
  if (waves) *waves = choice.waves;
  return choice.rows;
}

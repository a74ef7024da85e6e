// The normalizer product of the simple (additive-joiner) loss in float32, with px / py and
// log(P + tiny) written from its accumulators (rnnt_loss.py:66-227; the formulas are at the
// top of simple_logprobs.hip).
#include <algorithm>
#include <cmath>

#include "common.hip.h"
#include "simple_shared.hip.h"

namespace frnnt {
namespace {

// Normalizer GEMM, wave-private LDS slabs.  Both operands are k-contiguous ([rows][C]); the matrix
// cores want eight k of one row per lane, in three bfloat16 parts (Split8).  A wave fetches a slab
// of (kS lattice rows + kT frames) x 16 k with coalesced 16-byte loads (four lanes per row),
// applies exp(x - shift), splits the values and writes the parts to its OWN LDS region, from
// where they are read back as operands; the next slab is requested between the LDS writes and
// the products.  The waves of a workgroup split k; they never wait for each other in the loop (a
// wave's LDS writes and reads are served in program order), only at the end, when the partial
// sums meet.
//
// What bounds it: the VALU work per operand element (maximum, exp, split: about 26 cycles per
// wave and element of its 64) against the products' 12 matrix cycles per k and 32 x 32 cells,
// which another wave of the SIMD runs beside it (unlike the fp32 matrix instruction, whose cycles
// add to the VALU's).  So a tile wants to be large: elements per cell and k are
// (kS + kT) / (kS kT).  Measured: B 32, S 80, T 250, C 500: 18.6 us with the float32 matrix
// instruction, 17.4 here; B 21, S 47, T 333, C 503: 13.7 and 11.7; B 4, S 10, T 50, C 50: 7.0 and 5.6.
constexpr int kNormK = 16;  // k per slab: one matrix instruction deep
constexpr int kNormWaves = 8;
constexpr int kPanelFrames = 32;  // of a workgroup
template <int kS, int kT>
struct NormShape {
  static constexpr int kWaves = kNormWaves;
  static constexpr int kThreads = kWaves * kWave;
  static constexpr int kRows = kS + kT;          // rows of a slab: lm rows, then am rows
  static constexpr int kLoads = kRows / 16;      // 16-byte loads per lane and slab
  // A row of a slab: three parts x 16 k x 2 bytes.  Rows whose bit 3 is set have the two halves
  // of each part swapped: the 16-byte reads of 16 consecutive rows then fall on all 64 banks
  // (rows are 24 words apart, which alone would put rows r and r + 8 on the same ones).
  static constexpr int kRowBytes = 96;
  static constexpr int kSlabBytes = kRows * kRowBytes;
  // the partial sums meet in rounds of kRound lattice rows that fit into the slabs' space
  static constexpr int kPitch = kT + 4;
  static constexpr int sums_bytes(int rows) { return kWaves * rows * kPitch * 4; }
  static constexpr int kSpace = 128 << 10;
  static constexpr int kRound = sums_bytes(kS) <= kSpace                    ? kS
                                : kS % 64 == 0 && sums_bytes(64) <= kSpace ? 64
                                                                           : 32;
  static constexpr int kRounds = kS / kRound;
  static constexpr size_t kLdsBytes =
      std::max(kWaves * kSlabBytes, sums_bytes(kRound));
  static constexpr int kItems =  // 16-byte outputs per thread and round
      (kRound * kT / 4 + kThreads - 1) / kThreads;
  static constexpr size_t kFixedBytes = ((kWaves + 1) * kRows + 3 * kS + kT) * 4;  // (below)
  static_assert(kS % 32 == 0 && kT % 32 == 0 && kS % kRound == 0, "shape");
  static_assert(kLdsBytes + kFixedBytes <= 160 << 10, "one workgroup per CU");
};

// Which tile a workgroup takes.  A unit of placement is an utterance, or one stretch of its
// vocabulary when k is cut into stretches (they share no operand), or, for batches of fewer
// than eight units, a part of the frames (the parts share lm, the small operand): unit u runs on
// XCD u % 8, whose L2 then holds its operands.
constexpr int kMostSplits = 8;
struct NormPlan {
  int t_tiles, s_tiles, splits, part_shift, chunks_per_split;
};
struct NormTile {
  int b, split, s_idx, t_idx;
};
__device__ __forceinline__ bool place_tile(int id, const NormPlan &plan, int B, NormTile &o) {
  using dgemm::kXcds;
  const int t_per = (plan.t_tiles + (1 << plan.part_shift) - 1) >> plan.part_shift;
  const int unit_tiles = t_per * plan.s_tiles;
  const int xcd = id % kXcds, slot = id / kXcds, round = slot / unit_tiles;
  const int within = slot - round * unit_tiles;
  const int unit = round * kXcds + xcd;
  const int whole = unit >> plan.part_shift;
  o.b = whole / plan.splits;
  o.split = whole - o.b * plan.splits;
  o.s_idx = within / t_per;
  o.t_idx = (unit & ((1 << plan.part_shift) - 1)) * t_per + (within - o.s_idx * t_per);
  return o.b < B && o.t_idx < plan.t_tiles;
}

// Where the stretches of k leave their sums: [split][B][S1][T] sums relative to the maxima of
// the stretch, [split][B][S1] and [split][B][T] maxima.
struct NormScratch {
  float *sums, *lm_max, *am_max;
};

struct NormArgs {
  const float *lm, *am;
  const int64_t *symbols, *boundary, *window;
  float *lm_max, *am_max, *px, *py, *norm_raw;
  NormScratch scratch;
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

template <int kS, int kT>
__global__ void __launch_bounds__(kNormWaves *kWave)
    simple_fwd_panel_kernel(NormArgs A, NormPlan plan) {
  using Shape = NormShape<kS, kT>;
  constexpr int kWaves = kNormWaves;
  constexpr int kRows = Shape::kRows, kLoads = Shape::kLoads, kLmLoads = kS / 16;
  constexpr int kThreads = Shape::kThreads, kItems = Shape::kItems, kRound = Shape::kRound;
  constexpr int kPitch = Shape::kPitch;
  using namespace dgemm;
  extern __shared__ __align__(16) char norm_lds[];
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
  const int first_chunk = tile.split * plan.chunks_per_split;
  const int chunks = min(first_chunk + plan.chunks_per_split, (C + kNormK - 1) / kNormK);

  // ---- one pass over k.  The reference subtracts the row maxima before exp
  // (rnnt_loss.py:174-178); a maximum is known only after the whole row has been seen, so
  // each wave works with a SHIFT per row instead: the largest value of the row it had
  // seen when the shift was last set.  A value more than kMargin above the shift (always
  // the case for the first finite value of a row) makes the wave raise its shifts and
  // scale its partial sums to match; anything closer stays representable, e^(2 kMargin)
  // per product.  The running maxima are kept beside the shifts, and when the waves
  // meet their partial sums are brought to the true maxima, exp(shift - max) <= 1.
  constexpr float kMargin = 30.f;
  floatx4 slab[kLoads];
  if (first_chunk + wave < chunks) fetch(std::integral_constant<int, kS / 32>{}, slab, (first_chunk + wave) * kNormK);
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
  // ... and am[b, t, sym[b, s]] of this thread's outputs in a round: 16-byte pieces (row
  // item / (kT / 4), frames 4 (item % (kT / 4)) ..).  The stretches of k share them out by rows.
  float am_sym[kItems][4];
  auto item_row = [&](int round, int j) { return round * kRound + (tid + kThreads * j) / (kT / 4); };
  auto item_t = [&](int j) { return 4 * ((tid + kThreads * j) % (kT / 4)); };
  auto gather = [&](int round) {
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      const int m = item_row(round, j), sr = s_tile + m;
      const int y = get_symbol(sym_rs,
                               (tid + kThreads * j) < kRound * kT / 4 && sr < S && m < live_rows &&
                                   (plan.splits == 1 || sr % plan.splits == tile.split),
                               sr, C);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int tr = t_tile + item_t(j) + i;
        am_sym[j][i] = get_float(am_rs, y >= 0 && tr < T, (tr * C + y) * 4);
      }
    }
  };
  if (Shape::kRounds == 1) gather(0);

  float seen[kLoads];     // largest value this lane has met in the row
  // -shift * log2(e), see exp_shifted; the lanes of a row agree on it.  kUnset while the
  // row has shown nothing finite: it sends -inf to exp2(-inf) = 0 and anything finite
  // above the margin.
  float shift2[kLoads];
  constexpr float kUnset = 3.0e38f;
#pragma unroll
  for (int j = 0; j < kLoads; ++j) seen[j] = ninf, shift2[j] = kUnset;
  const int live_tiles = max(1, min(kS / 32, (live_rows + 31) / 32));
  char *mine = norm_lds + wave * Shape::kSlabBytes;
  floatx16 acc[kS / 32][kT / 32];
#pragma unroll
  for (int j = 0; j < kS / 32; ++j)
#pragma unroll
    for (int n = 0; n < kT / 32; ++n)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[j][n][v] = 0.f;

  auto across_row = [&](float v) {  // maximum over the four lanes that share a row
    v = fmaxf(v, __shfl_xor(v, 1, kWave));
    return fmaxf(v, __shfl_xor(v, 2, kWave));
  };
  // (the sums are brought along; -across_row(seen) is the new shift)
  auto raise_shifts = [&](auto live) {
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      if (j >= 2 * live && j < kLmLoads) continue;
      const float now = fminf(shift2[j], -across_row(seen[j]) * kLog2e);
      const float f = __builtin_amdgcn_exp2f(now - shift2[j]);  // exp(old shift - new shift)
      shift2[j] = now;
      if (lane % 4 == 0) factor[wave][sub + 16 * j] = f;
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int n = 0; n < kT / 32; ++n) {
      const float ft = factor[wave][kS + 32 * n + r32];
#pragma unroll
      for (int j = 0; j < live; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          acc[j][n][v] *= factor[wave][32 * j + 8 * (v / 4) + 4 * half + (v % 4)] * ft;
    }
    __builtin_amdgcn_wave_barrier();
  };
  // where this lane's values of a slab row go, and where its operands lie
  char *put = mine + sub * Shape::kRowBytes + 16 * ((kq / 8) ^ ((sub >> 3) & 1)) + 2 * (kq % 8);
  const char *get = mine + r32 * Shape::kRowBytes + 16 * (half ^ ((r32 >> 3) & 1));
  auto operand = [&](int row) {
    Split8 o;
    o.hi = *reinterpret_cast<const bf16x8 *>(get + row * Shape::kRowBytes);
    o.mid = *reinterpret_cast<const bf16x8 *>(get + row * Shape::kRowBytes + 32);
    o.lo = *reinterpret_cast<const bf16x8 *>(get + row * Shape::kRowBytes + 64);
    return o;
  };
  // This wave's share of k, with `live` 32-row tiles that hold lattice rows which count (a
  // constant: the code of a slab is one straight line, whose rows' chains of dependent
  // instructions the compiler interleaves -- with a test per row group a slab took 2.5 times as
  // long).
  auto look = [&](auto live) {  // maxima; true if a row exceeds its margin
    bool above = false;
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      if (j >= 2 * live && j < kLmLoads) continue;
      // two three-input maxima; a row is above its margin exactly when its maximum is
      seen[j] = max3_raw(max3_raw(slab[j][0], slab[j][1], slab[j][2]), slab[j][3], seen[j]);
      above |= __builtin_fmaf(seen[j], kLog2e, shift2[j]) > kMargin * kLog2e;
    }
    return above;
  };
  auto walk = [&](auto live) {
    int chunk = first_chunk + wave;
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
        float e[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) e[i] = exp_shifted(slab[j][i], shift2[j]);
        unsigned h0, h1, m0, m1, l0, l1;
        split_pair(e[0], e[1], h0, m0, l0);
        split_pair(e[2], e[3], h1, m1, l1);
        char *to = put + j * 16 * Shape::kRowBytes;
        *reinterpret_cast<uintx2 *>(to) = uintx2{h0, h1};
        *reinterpret_cast<uintx2 *>(to + 32) = uintx2{m0, m1};
        *reinterpret_cast<uintx2 *>(to + 64) = uintx2{l0, l1};
      }
      if (chunk + kWaves < chunks) fetch(live, slab, (chunk + kWaves) * kNormK);
#pragma unroll
      for (int n = 0; n < kT / 32; ++n) {
        const Split8 t_op = operand(kS + 32 * n);
#pragma unroll
        for (int j = 0; j < live; ++j) acc[j][n] = multiply_add(operand(32 * j), t_op, acc[j][n]);
      }
    }
  };
  with_tiles<kS / 32>(live_tiles, walk);

  // ---- the waves meet: maxima first (each wave's in what was its slab: the row maxima over its
  // share of k, then its final shifts) ...
  float *met = reinterpret_cast<float *>(mine);
#pragma unroll
  for (int j = 0; j < kLoads; ++j) {
    const float top = across_row(seen[j]);
    if (lane % 4 == 0) {
      met[sub + 16 * j] = top;
      met[kRows + sub + 16 * j] = shift2[j];
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
  // (the stretches of k keep their own maxima)
  const long slot = (long)tile.split * A.B + b;
  float *lm_max = plan.splits == 1 ? A.lm_max + (long)b * S1 : A.scratch.lm_max + slot * S1;
  float *am_max = plan.splits == 1 ? A.am_max + (long)b * T : A.scratch.am_max + slot * T;
  for (int row = tid; row < kRows; row += kThreads) {
    auto met_by = [&](int w, int i) {
      return reinterpret_cast<const float *>(norm_lds + w * Shape::kSlabBytes)[i];
    };
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
  // ... then the partial sums, kRound rows at a time: [wave][kRound][kPitch] in the slab space
  float *sums = reinterpret_cast<float *>(norm_lds);
  const int t_mask = (A.rnnt_type == kRegular && A.boundary) ? (int)A.boundary[4 * b + 3] : -1;
  float *pxb = A.px + (long)b * S * T1;
  float *pyb = A.py + (long)b * S1 * T;
  float *nrb = A.norm_raw ? A.norm_raw + (long)b * S1 * T : nullptr;
  float *sumb = plan.splits == 1 ? nullptr : A.scratch.sums + slot * S1 * T;
#pragma unroll
  for (int round = 0; round < Shape::kRounds; ++round) {
    if (round * kRound >= live_rows && round > 0) break;  // (uniform)
    if (Shape::kRounds > 1) gather(round);
    if (round > 0) __syncthreads();  // the previous round's readers are done
    float *part = sums + wave * kRound * kPitch;
#pragma unroll
    for (int n = 0; n < kT / 32; ++n) {
      const float ft = factor[wave][kS + 32 * n + r32];
#pragma unroll
      for (int j = 0; j < kRound / 32; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int m = 32 * j + 8 * (v / 4) + 4 * half + (v % 4);
          part[m * kPitch + 32 * n + r32] =
              acc[round * (kRound / 32) + j][n][v] * (factor[wave][round * kRound + m] * ft);
        }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      const int item = tid + kThreads * j, m = item_row(round, j), out_t = item_t(j);
      const int sr = s_tile + m, tr = t_tile + out_t;
      if (item >= kRound * kT / 4 || sr >= S1 || m >= live_rows) continue;
      floatx4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        const floatx4 one = *reinterpret_cast<const floatx4 *>(
            sums + (w * kRound + m - round * kRound) * kPitch + out_t);
#pragma unroll
        for (int i = 0; i < 4; ++i) sum[i] += one[i];
      }
      floatx4 raw, yv, xv;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        yv[i] = col_term[out_t + i] + row_term[m];
        xv[i] = am_sym[j][i] + row_sym[m];
        if (plan.splits == 1) {
          raw[i] = logf(sum[i] + 1.17549435e-38f);
          const float norm = raw[i] + slab_max[m] + slab_max[kS + out_t + i];
          yv[i] -= norm;
          xv[i] -= norm;
        } else {
          raw[i] = sum[i];
        }
        if (row_symbol[m] < 0) xv[i] = std::numeric_limits<float>::quiet_NaN();  // out-of-vocabulary
        if (tr + i == t_mask) xv[i] = ninf;
        if (plan.splits == 1) xv[i] = A.delay.at(xv[i], A.boundary, b, tr + i, T);
      }
      float *raw_to = plan.splits == 1 ? nrb : sumb;
      const bool mine_here = plan.splits == 1 || sr % plan.splits == tile.split;
      if (tr + 4 <= T) {
        if (raw_to)
          *reinterpret_cast<floatx4u *>(raw_to + sr * T + tr) = floatx4u{raw[0], raw[1], raw[2], raw[3]};
        if (!mine_here) continue;
        *reinterpret_cast<floatx4u *>(pyb + sr * T + tr) = floatx4u{yv[0], yv[1], yv[2], yv[3]};
        if (sr < S)
          *reinterpret_cast<floatx4u *>(pxb + sr * T1 + tr) = floatx4u{xv[0], xv[1], xv[2], xv[3]};
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (tr + i >= T) continue;
          if (raw_to) raw_to[sr * T + tr + i] = raw[i];
          if (!mine_here) continue;
          pyb[sr * T + tr + i] = yv[i];
          if (sr < S) pxb[sr * T1 + tr + i] = xv[i];
        }
      }
    }
  }
  // the extra column of the regular lattice: nothing can be emitted after the last frame
  if (A.rnnt_type == kRegular && t_tile == 0 && tile.split == 0)
    for (int m = tid; m < kS; m += kThreads)
      if (s_tile + m < S) pxb[(s_tile + m) * T1 + T] = ninf;
}

// ---- the same with the operands shared by a small workgroup ------------------------------------
// kS lattice rows x kT frames, four waves, 40 KB of LDS and 128 registers: four workgroups share a
// compute unit, and while one waits for memory or at a barrier the others convert or multiply
// (a wave issues an instruction every five cycles at best, so it takes four waves on a SIMD to
// keep its VALU busy; the matrix cycles run beside).  The 256 threads fetch a chunk of 32 k
// together, apply exp, split the values and write the parts to LDS; after a barrier wave (m, n)
// multiplies kMTiles 32-row tiles by the 32 frames n.  Per cell that is (kS + kT) / (kS kT)
// operand elements.  (Tiles of 128 x 64, 64 x 128 and 32 x 128, which convert less per cell, are all
// slower: the matrix cycles are not what is short.)
constexpr int kTileThreads = 256;
constexpr int kTileSide = 64;                        // lattice rows and frames of a workgroup
constexpr int kTileChunk = 32;                       // k per chunk: two k-steps
constexpr int kTileRowLanes = kTileChunk / 4;        // lanes that share a row of a fetch
constexpr int kTileRowsPerLoad = kTileThreads / kTileRowLanes;
template <int kS, int kT>
struct TileShape {
  static constexpr int kRows = kS + kT;
  static constexpr int kLoads = kRows / kTileRowsPerLoad, kLmLoads = kS / kTileRowsPerLoad;
  // A row's operands in LDS: three parts x 16 k x 2 bytes; rows whose bit 3 is set have the
  // halves of each part swapped, so that the 16-byte reads of 16 consecutive rows fall on all 64
  // banks (rows are 24 words apart, which alone would put rows r and r + 8 on the same ones).
  static constexpr int kRowBytes = 96;
  static constexpr int kBufBytes = 2 * kRows * kRowBytes;
  static constexpr int kWavesN = std::min(4, kT / 32), kWavesM = 4 / kWavesN;
  static constexpr int kMTiles = kS / 32 / kWavesM;  // 32-row tiles per wave
  static constexpr int kPitch = kT + 4;
  static constexpr int kSumBytes = kS * kPitch * 4;
  static constexpr int kItems = kS * kT / 4 / kTileThreads;
  static constexpr size_t kLdsBytes = std::max(kBufBytes, kSumBytes + 2 * kRows * 4);
  static constexpr size_t kFixedBytes = (kRows + 3 * kS + kT + 4) * 4;
  static_assert(kMTiles >= 1 && kWavesN * 32 == kT, "a wave has one column of tiles");
  static_assert(kLdsBytes + kFixedBytes <= 40 << 10, "four workgroups per CU");
};

template <int kS, int kT>
__global__ void __launch_bounds__(kTileThreads, 4)
    simple_fwd_tile_kernel(NormArgs A, NormPlan plan) {
  using Shape = TileShape<kS, kT>;
  constexpr int kRows = Shape::kRows, kLoads = Shape::kLoads, kLmLoads = Shape::kLmLoads;
  constexpr int kPer = kTileRowsPerLoad, kRowLanes = kTileRowLanes, kChunk = kTileChunk;
  constexpr int kRowBytes = Shape::kRowBytes, kPitch = Shape::kPitch, kItems = Shape::kItems;
  constexpr int kMTiles = Shape::kMTiles;
  using namespace dgemm;
  extern __shared__ __align__(16) char norm_lds[];
  __shared__ float factor[kRows];              // what raised shifts scale the sums by
  __shared__ float row_term[kS], row_sym[kS];  // lm[s,term], lm[s,sym[s]]
  __shared__ int row_symbol[kS];
  __shared__ float col_term[kT];  // am[t,term]
  __shared__ int raised_at;       // the last chunk that raised a shift
  const int S = A.S, T = A.T, C = A.C, S1 = S + 1;
  NormTile tile;
  if (!place_tile((int)blockIdx.x, plan, A.B, tile)) return;
  const int b = tile.b, s_tile = tile.s_idx * kS, t_tile = tile.t_idx * kT;
  const int T1 = A.rnnt_type == kRegular ? T + 1 : T;
  const float *lmb = A.lm + (long)b * S1 * C;
  const float *amb = A.am + (long)b * T * C;
  const int64_t *symb = A.symbols + (long)b * S;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wave_n = wave % Shape::kWavesN, wave_m = wave / Shape::kWavesN;
  const int half = lane >> 5, r32 = lane & 31;
  const float ninf = -__builtin_huge_valf();
  // what this thread fetches of every chunk: rows sub + kPer j at k-offset kq (buffer resources as
  // in the kernel above)
  const int sub = tid / kRowLanes, kq = 4 * (tid % kRowLanes);
  const __amdgpu_buffer_rsrc_t lm_rs =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(lmb), 0, S1 * C * 4, 0x00020000);
  const __amdgpu_buffer_rsrc_t am_rs =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(amb), 0, T * C * 4, 0x00020000);
  const int lm_off = ((s_tile + sub) * C + kq) * 4, am_off = ((t_tile + sub) * C + kq) * 4;  // bytes
  const int step = kPer * C * 4;
  typedef int intx4 __attribute__((ext_vector_type(4)));
  floatx4 slab[kLoads];
  auto fetch = [&](int chunk) {
    const int k0 = chunk * kChunk;
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      const intx4 raw = j < kLmLoads
                            ? __builtin_amdgcn_raw_buffer_load_b128(lm_rs, lm_off, j * step + k0 * 4, 0)
                            : __builtin_amdgcn_raw_buffer_load_b128(
                                  am_rs, am_off, (j - kLmLoads) * step + k0 * 4, 0);
      slab[j] = floatx4{__int_as_float(raw[0]), __int_as_float(raw[1]), __int_as_float(raw[2]),
                        __int_as_float(raw[3])};
    }
    if (k0 + kChunk > C) {  // (uniform) the chunk that holds column C - 1
#pragma unroll
      for (int j = 0; j < kLoads; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (k0 + kq + i >= C) slab[j][i] = ninf;
    }
  };
  const int first_chunk = tile.split * plan.chunks_per_split;
  const int chunks = min(first_chunk + plan.chunks_per_split, (C + kChunk - 1) / kChunk);
  if (first_chunk < chunks) fetch(first_chunk);
  const __amdgpu_buffer_rsrc_t sym_rs = symbols_of(symb, S);
  // threads 0 .. kS-1 own a lattice row each
  const int my_sym = get_symbol(sym_rs, tid < kS && s_tile + tid < S, s_tile + tid, C);
  const Limits lim = limits_of(A.window, b, S, T);
  const int live_rows = min(S1, lim.s_end + 1) - s_tile;  // rows that count
  if ((t_tile > lim.t_end || live_rows <= 0) && t_tile > 0) return;
  const int live_tiles = max(1, min(kS / 32, (live_rows + 31) / 32));

  {
    const bool has_row = tid < kS && s_tile + tid < S1;
    const int my_row = (s_tile + tid) * C, my_frame = (t_tile + tid - 128) * C;
    const float at_sym = get_float(lm_rs, has_row && my_sym >= 0, (my_row + my_sym) * 4);
    const float at_term = get_float(lm_rs, has_row, (my_row + A.term) * 4);
    const float frame_term =
        get_float(am_rs, tid >= 128 && t_tile + tid - 128 < T, (my_frame + A.term) * 4);
    if (tid < kS) {
      row_symbol[tid] = my_sym;
      row_term[tid] = at_term;
      row_sym[tid] = at_sym;
    } else if (tid >= 128 && tid < 128 + kT) {
      col_term[tid - 128] = frame_term;
    }
  }
  for (int r = tid; r < kRows; r += kTileThreads) factor[r] = 1.f;
  if (tid == 0) raised_at = -1;
  lds_barrier();

  constexpr float kMargin = 30.f, kUnset = 3.0e38f;  // (see the kernel above)
  float seen[kLoads], shift2[kLoads];
#pragma unroll
  for (int j = 0; j < kLoads; ++j) seen[j] = ninf, shift2[j] = kUnset;
  floatx16 acc[kMTiles];
#pragma unroll
  for (int j = 0; j < kMTiles; ++j)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[j][v] = 0.f;
  auto across_row = [&](float v) {  // maximum over the lanes that share a row
#pragma unroll
    for (int off = 1; off < kRowLanes; off <<= 1) v = fmaxf(v, __shfl_xor(v, off, kWave));
    return v;
  };
  // where this thread's values go, and where this wave's operands lie
  char *put = norm_lds + ((kq / 16) * kRows + sub) * kRowBytes +
              16 * (((kq % 16) / 8) ^ ((sub >> 3) & 1)) + 2 * (kq % 8);
  const char *get = norm_lds + r32 * kRowBytes + 16 * (half ^ ((r32 >> 3) & 1));
  const char *get_t = get + (kS + 32 * wave_n) * kRowBytes;
  const char *get_s = get + 32 * kMTiles * wave_m * kRowBytes;
  auto operand = [&](const char *at) {
    Split8 o;
    o.hi = *reinterpret_cast<const bf16x8 *>(at);
    o.mid = *reinterpret_cast<const bf16x8 *>(at + 32);
    o.lo = *reinterpret_cast<const bf16x8 *>(at + 64);
    return o;
  };
  // (32-row tiles past the last row that counts are neither converted nor multiplied; a fetch is
  // one such tile)
  static_assert(kPer == 32, "a fetch is a 32-row tile");
  const int my_tiles = min(kMTiles, live_tiles - kMTiles * wave_m);
  for (int chunk = first_chunk; chunk < chunks; ++chunk) {
    // maxima; the first chunk sets the shifts, later ones raise them when a value exceeds its
    // margin, and leave the factor for the sums so far beside the chunk
    bool above = false;
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      seen[j] = max3_raw(max3_raw(slab[j][0], slab[j][1], slab[j][2]), slab[j][3], seen[j]);
      above |= __builtin_fmaf(seen[j], kLog2e, shift2[j]) > kMargin * kLog2e;
    }
    if (chunk == first_chunk || __any(above)) {
#pragma unroll
      for (int j = 0; j < kLoads; ++j) {
        const float now = fminf(shift2[j], -across_row(seen[j]) * kLog2e);
        if (chunk != first_chunk && tid % kRowLanes == 0)
          factor[sub + kPer * j] = __builtin_amdgcn_exp2f(now - shift2[j]);
        shift2[j] = now;
      }
      if (chunk != first_chunk) raised_at = chunk;
    }
    auto convert = [&](int j) {
      float e[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) e[i] = exp_shifted(slab[j][i], shift2[j]);
      unsigned h0, h1, m0, m1, l0, l1;
      split_pair(e[0], e[1], h0, m0, l0);
      split_pair(e[2], e[3], h1, m1, l1);
      char *to = put + j * kPer * kRowBytes;
      *reinterpret_cast<uintx2 *>(to) = uintx2{h0, h1};
      *reinterpret_cast<uintx2 *>(to + 32) = uintx2{m0, m1};
      *reinterpret_cast<uintx2 *>(to + 64) = uintx2{l0, l1};
    };
#pragma unroll
    for (int j = kLmLoads; j < kLoads; ++j) convert(j);
    convert(0);
#pragma unroll
    for (int j = 1; j < kLmLoads; ++j)
      if (j < live_tiles) convert(j);
    if (chunk + 1 < chunks) fetch(chunk + 1);
    lds_barrier();
    if (raised_at == chunk && my_tiles > 0) {  // (uniform)
      const float ft = factor[kS + 32 * wave_n + r32];
#pragma unroll
      for (int j = 0; j < kMTiles; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          acc[j][v] *= factor[32 * (kMTiles * wave_m + j) + 8 * (v / 4) + 4 * half + (v % 4)] * ft;
    }
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      constexpr int kStep = kRows * kRowBytes;
      if (my_tiles > 0) {
        const Split8 t_op = operand(get_t + g * kStep);
#pragma unroll
        for (int j = 0; j < kMTiles; ++j)
          if (j == 0 || j < my_tiles)
            acc[j] = multiply_add(operand(get_s + g * kStep + 32 * j * kRowBytes), t_op, acc[j]);
      }
    }
    lds_barrier();  // the operands have been read
    if (raised_at == chunk)  // (rare: the factors are 1 again for the next chunk)
      for (int r = tid; r < kRows; r += kTileThreads) factor[r] = 1.f;
  }

  // ---- am[b, t, sym[b, s]] of this thread's outputs; the stretches of k share them out by rows
  auto item_row = [&](int j) { return (tid + kTileThreads * j) / (kT / 4); };
  const int out_t = 4 * (tid % (kT / 4));
  constexpr int kAhead = std::min(kItems, 4);  // items whose values are requested together
  floatx4 am_sym[kAhead];
  auto gather = [&](int first) {
#pragma unroll
    for (int j = 0; j < kAhead; ++j) {
      const int m = item_row(first + j), sr = s_tile + m;
      int y = -1;
      if (m < live_rows && (plan.splits == 1 || sr % plan.splits == tile.split)) y = row_symbol[m];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int tr = t_tile + out_t + i;
        am_sym[j][i] = get_float(am_rs, y >= 0 && tr < T, (tr * C + y) * 4);
      }
    }
  };
  gather(0);
  // ---- maxima, and what brings the sums from the shifts to them, beside the sums
  float *sums = reinterpret_cast<float *>(norm_lds);
  float *final_factor = sums + kS * kPitch, *slab_max = final_factor + kRows;
  const long slot = (long)tile.split * A.B + b;
  float *lm_max = plan.splits == 1 ? A.lm_max + (long)b * S1 : A.scratch.lm_max + slot * S1;
  float *am_max = plan.splits == 1 ? A.am_max + (long)b * T : A.scratch.am_max + slot * T;
#pragma unroll
  for (int j = 0; j < kLoads; ++j) {
    const float r = across_row(seen[j]);
    const int row = sub + kPer * j;
    if (tid % kRowLanes != 0) continue;
    bool exists;
    if (j < kLmLoads) {
      exists = s_tile + row < S1;
      if (exists && t_tile == 0) lm_max[s_tile + row] = r;
    } else {
      exists = t_tile + row - kS < T;
      if (exists && s_tile == 0) am_max[t_tile + row - kS] = r;
    }
    slab_max[row] = exists ? r : 0.f;
    final_factor[row] = exists ? __builtin_amdgcn_exp2f(-__builtin_fmaf(r, kLog2e, shift2[j])) : 1.f;
  }
  lds_barrier();
  {
    const float ft = final_factor[kS + 32 * wave_n + r32];
    float *part = sums + 32 * wave_n + r32;
#pragma unroll
    for (int j = 0; j < kMTiles; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int m = 32 * (kMTiles * wave_m + j) + 8 * (v / 4) + 4 * half + (v % 4);
        part[m * kPitch] = acc[j][v] * (final_factor[m] * ft);
      }
  }
  lds_barrier();
  const int t_mask = (A.rnnt_type == kRegular && A.boundary) ? (int)A.boundary[4 * b + 3] : -1;
  float *pxb = A.px + (long)b * S * T1;
  float *pyb = A.py + (long)b * S1 * T;
  float *nrb = A.norm_raw ? A.norm_raw + (long)b * S1 * T : nullptr;
  float *raw_to = plan.splits == 1 ? nrb : A.scratch.sums + slot * S1 * T;
  for (int first = 0; first < kItems; first += kAhead) {
    if (first > 0) gather(first);
#pragma unroll
    for (int j = 0; j < kAhead; ++j) {
      const int m = item_row(first + j), sr = s_tile + m, tr = t_tile + out_t;
      if (sr >= S1 || m >= live_rows) continue;
      const floatx4 sum = *reinterpret_cast<const floatx4 *>(sums + m * kPitch + out_t);
      floatx4 raw, yv, xv;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        yv[i] = col_term[out_t + i] + row_term[m];
        xv[i] = am_sym[j][i] + row_sym[m];
        if (plan.splits == 1) {
          raw[i] = logf(sum[i] + 1.17549435e-38f);
          const float norm = raw[i] + slab_max[m] + slab_max[kS + out_t + i];
          yv[i] -= norm;
          xv[i] -= norm;
        } else {
          raw[i] = sum[i];
        }
        if (row_symbol[m] < 0) xv[i] = std::numeric_limits<float>::quiet_NaN();  // out-of-vocabulary
        if (tr + i == t_mask) xv[i] = ninf;
        if (plan.splits == 1) xv[i] = A.delay.at(xv[i], A.boundary, b, tr + i, T);
      }
      const bool mine_here = plan.splits == 1 || sr % plan.splits == tile.split;
      if (tr + 4 <= T) {
        if (raw_to)
          *reinterpret_cast<floatx4u *>(raw_to + sr * T + tr) = floatx4u{raw[0], raw[1], raw[2], raw[3]};
        if (!mine_here) continue;
        *reinterpret_cast<floatx4u *>(pyb + sr * T + tr) = floatx4u{yv[0], yv[1], yv[2], yv[3]};
        if (sr < S)
          *reinterpret_cast<floatx4u *>(pxb + sr * T1 + tr) = floatx4u{xv[0], xv[1], xv[2], xv[3]};
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (tr + i >= T) continue;
          if (raw_to) raw_to[sr * T + tr + i] = raw[i];
          if (!mine_here) continue;
          pyb[sr * T + tr + i] = yv[i];
          if (sr < S) pxb[sr * T1 + tr + i] = xv[i];
        }
      }
    }
  }
  // the extra column of the regular lattice: nothing can be emitted after the last frame
  if (A.rnnt_type == kRegular && t_tile == 0 && tile.split == 0 && tid < kS && s_tile + tid < S)
    pxb[(s_tile + tid) * T1 + T] = ninf;
}

// The stretches of k meet: their sums, each relative to its own maxima, are brought to the common
// maxima and added in the order of the stretches; px and py hold their numerators.  A wave takes
// 64 frames of one lattice row; the waves of row 0 also store the maxima.
template <int kSplits>
__global__ void __launch_bounds__(256) normalizer_merge_kernel(NormArgs A) {
  const int S1 = A.S + 1, T = A.T;
  const int b = blockIdx.z, s = blockIdx.y * 4 + (threadIdx.x >> 6);
  const int t = blockIdx.x * 64 + (threadIdx.x & 63);
  if (s >= S1) return;
  const Limits lim = limits_of(A.window, b, A.S, T);
  const bool out = s > lim.s_end || (int)blockIdx.x * 64 > lim.t_end;
  if (out && blockIdx.x > 0 && s > 0) return;
  const bool in = t < T && !out;
  float rs[kSplits], rt[kSplits], part[kSplits];
#pragma unroll
  for (int i = 0; i < kSplits; ++i) {
    const long slot = (long)i * A.B + b;
    rs[i] = A.scratch.lm_max[slot * S1 + s];
    rt[i] = A.scratch.am_max[slot * T + min(t, T - 1)];
    part[i] = in ? A.scratch.sums[(slot * S1 + s) * T + t] : 0.f;
  }
  float ms = rs[0], mt = rt[0];
#pragma unroll
  for (int i = 1; i < kSplits; ++i) ms = fmaxf(ms, rs[i]), mt = fmaxf(mt, rt[i]);
  if (t == 0) A.lm_max[(long)b * S1 + s] = ms;
  if (s == 0 && t < T) A.am_max[(long)b * T + t] = mt;
  if (!in) return;
  // (a stretch without a finite value has a sum of 0; a row without one in any stretch keeps
  // exp(-inf - -inf) out of it)
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < kSplits; ++i) {
    const float f = __builtin_amdgcn_exp2f(((rs[i] - ms) + (rt[i] - mt)) * kLog2e);
    sum += part[i] != 0.f ? part[i] * f : 0.f;
  }
  const float raw = logf(sum + 1.17549435e-38f);
  const float norm = raw + ms + mt;
  const long at = ((long)b * S1 + s) * T + t;
  if (A.norm_raw) A.norm_raw[at] = raw;
  A.py[at] -= norm;
  if (s == A.S) return;
  float *x = A.px + ((long)b * A.S + s) * (A.rnnt_type == kRegular ? T + 1 : T) + t;
  // (nothing is emitted at t_end, whatever that frame holds)
  const bool closed = A.rnnt_type == kRegular && A.boundary && t == (int)A.boundary[4 * b + 3];
  *x = closed ? -__builtin_huge_valf() : A.delay.at(*x - norm, A.boundary, b, t, T);
}

unsigned grid_of(const NormPlan &plan, int B) {
  const int t_per = (plan.t_tiles + (1 << plan.part_shift) - 1) >> plan.part_shift;
  const long units = ((long)B * plan.splits) << plan.part_shift;
  return (unsigned)(dgemm::kXcds * ((units + dgemm::kXcds - 1) / dgemm::kXcds) * t_per *
                    plan.s_tiles);
}
template <int kS>
void launch_fwd_panel(const NormArgs &args, const NormPlan &plan, hipStream_t stream) {
  using Shape = NormShape<kS, kPanelFrames>;
  auto kernel = simple_fwd_panel_kernel<kS, kPanelFrames>;
  if (!allow_lds(reinterpret_cast<const void *>(kernel), Shape::kLdsBytes)) return;
  hipLaunchKernelGGL(kernel, dim3(grid_of(plan, args.B)), dim3(Shape::kThreads), Shape::kLdsBytes,
                     stream, args, plan);
}
void launch_fwd_tile(const NormArgs &args, const NormPlan &plan, hipStream_t stream) {
  hipLaunchKernelGGL((simple_fwd_tile_kernel<kTileSide, kTileSide>), dim3(grid_of(plan, args.B)),
                     dim3(kTileThreads), (TileShape<kTileSide, kTileSide>::kLdsBytes), stream, args,
                     plan);
}

// Which kernel, and into how many stretches k is cut: what a model of the two kernels' times
// says is fastest.  A workgroup of the panel kernel has a compute unit to itself and walks k
// with eight waves: little overhead, best while its workgroups are one round of the chip's 256
// compute units.  Four of the tile kernel's share one: slow alone (1 us per 32 k), but twice as fast
// as the panel once there are several hundred (B 64, S 120, T 600, C 500: 65 against 88 us).
// A vocabulary of thousands leaves either with few workgroups and much k: stretches fill the chip
// (B 2, S 53, T 343, C 4627: 50 -> 18 us; B 8, S 100, T 400, C 5000: 92 -> 52), at the price of
// the merge.  The constants are fitted to 26 sizes, B 1 .. 128, C 50 .. 5000, that were timed with
// every kernel and 1 .. 8 stretches; over these the choice is 2.4 % (geometric mean) from the best.
struct NormChoice {
  bool small;  // simple_fwd_tile_kernel, else simple_fwd_panel_kernel
  int rows, frames, splits, chunks_per_split;
};
NormChoice choose(int B, int S, int T, int C, bool may_split) {
  const int S1 = S + 1;
  // the panel's row count that leaves fewest padding rows; the larger one on a tie
  int panel_rows = 32;
  for (int r : {64, 96, 128})
    if ((S1 + r - 1) / r * r <= (S1 + panel_rows - 1) / panel_rows * panel_rows || S1 > r)
      panel_rows = r;
  NormChoice best{};
  double best_us = 0;
  for (bool small : {false, true})
    for (int want : {1, 2, 3, 4, 6, kMostSplits}) {
      if (want > 1 && !may_split) continue;
      NormChoice c;
      c.small = small;
      c.rows = small ? kTileSide : panel_rows;
      c.frames = small ? kTileSide : kPanelFrames;
      const int chunk = small ? kTileChunk : kNormK, chunks = (C + chunk - 1) / chunk;
      c.chunks_per_split = (chunks + want - 1) / want;
      // (every stretch holds a chunk: an empty one would have neither maxima nor sums)
      c.splits = (chunks + c.chunks_per_split - 1) / c.chunks_per_split;
      // (a ragged batch leaves about 0.85 of the tiles to compute)
      const double tiles = 0.85 * B * ((S1 + c.rows - 1) / c.rows) *
                           (double)((T + c.frames - 1) / c.frames) * c.splits;
      const double per_cu = std::max(1.0, tiles / 256);
      double us;
      if (small) {
        const double together = std::min(per_cu, 4.0);
        us = per_cu / together * (3.8 + 2.15 * together + c.chunks_per_split * (0.63 + 0.41 * together));
      } else {
        us = std::ceil(per_cu) * (1.5 + 0.055 * c.rows +
                                  (c.chunks_per_split + kNormWaves - 1) / kNormWaves * (0.31 + 0.016 * c.rows));
      }
      if (c.splits > 1) us = 1.05 * (us + 4.9 + 2.8e-7 * c.splits * B * S1 * (double)T);
      if (best_us == 0 || us < best_us) best = c, best_us = us;
    }
  return best;
}

template <int kSplits>
void launch_merge(const NormArgs &args, hipStream_t stream) {
  const dim3 grid((args.T + 63) / 64, (args.S + 4) / 4, args.B);
  hipLaunchKernelGGL(normalizer_merge_kernel<kSplits>, grid, dim3(256), 0, stream, args);
}
}  // namespace

size_t normalizer_workspace_floats(int B, int S, int T, int C) {
  const NormChoice c = choose(B, S, T, C, T > 0);
  if (c.splits == 1) return 0;
  return (size_t)c.splits * B * ((size_t)(S + 1) * T + (S + 1) + T);
}

void launch_normalizer_f32(const float *lm, const float *am, const int64_t *symbols,
                           const int64_t *boundary, float *lm_max, float *am_max, float *px,
                           float *py, float *norm_raw, const int64_t *window, float *workspace,
                           double delay_penalty, int B, int S, int T, int C, int term,
                           int rnnt_type, hipStream_t stream) {
  const NormChoice c = choose(B, S, T, C, workspace != nullptr && T > 0);
  NormArgs args{lm, am, symbols, boundary, window, lm_max, am_max, px, py, norm_raw, {},
                Delay<float>{(float)delay_penalty}, B, S, T, C, term, rnnt_type};
  if (c.splits > 1) {
    args.scratch.sums = workspace;
    args.scratch.lm_max = workspace + (size_t)c.splits * B * (S + 1) * T;
    args.scratch.am_max = args.scratch.lm_max + (size_t)c.splits * B * (S + 1);
  }
  NormPlan plan;
  plan.t_tiles = T > 0 ? (T + c.frames - 1) / c.frames : 1;
  plan.s_tiles = (S + 1 + c.rows - 1) / c.rows;
  plan.splits = c.splits;
  plan.chunks_per_split = c.chunks_per_split;
  plan.part_shift = 0;
  while ((((long)B * c.splits) << plan.part_shift) < dgemm::kXcds &&
         (2 << plan.part_shift) <= plan.t_tiles)
    ++plan.part_shift;
  if (c.small) launch_fwd_tile(args, plan, stream);
  else if (c.rows == 32) launch_fwd_panel<32>(args, plan, stream);
  else if (c.rows == 64) launch_fwd_panel<64>(args, plan, stream);
  else if (c.rows == 96) launch_fwd_panel<96>(args, plan, stream);
  else launch_fwd_panel<128>(args, plan, stream);
  switch (c.splits) {
    case 2: launch_merge<2>(args, stream); break;
    case 3: launch_merge<3>(args, stream); break;
    case 4: launch_merge<4>(args, stream); break;
    case 5: launch_merge<5>(args, stream); break;
    case 6: launch_merge<6>(args, stream); break;
    case 7: launch_merge<7>(args, stream); break;
    case 8: launch_merge<8>(args, stream); break;
    default: break;
  }
}
}  // namespace frnnt

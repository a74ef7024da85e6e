// px / py of the "simple" RNN-T loss (additive joiner) and their backward.
//
// Forward (fast_rnnt/python/fast_rnnt/rnnt_loss.py:66-227):
//   lm_max[b,s] = max_c lm[b,s,c]           am_max[b,t] = max_c am[b,t,c]
//   P[b,s,t]    = sum_c exp(lm - lm_max) * exp(am - am_max)      <- MFMA GEMM,
//                                                    exp fused into the tile loads
//   norm        = log(P + tiny) + lm_max + am_max
//   px[b,s,t]   = am[b,t,sym[b,s]] + lm[b,s,sym[b,s]] - norm[b,s,t]   (t < T)
//   py[b,s,t]   = am[b,t,term]     + lm[b,s,term]     - norm[b,s,t]
//   regular:     px[b,s,T] = -inf and, with a boundary, px[b,s,T_b] = -inf
//   constrained: px[b,s,t] += py[b,s+1,t]
// The epilogue of the GEMM writes px, py and log(P + tiny) straight from the
// accumulators; the normalizers never make a round trip through HBM.
//
// Backward: with gx = dL/dpx (masked like px), gy = dL/dpy (+ gx one row up for
// constrained), W = -(gx + gy) and D = W / (P + tiny):
//   dL/dlm[b,s,c] = exp(lm - lm_max) * sum_t D[s,t] exp(am[t,c] - am_max[t])
//                   + [c = sym[b,s]] sum_t gx[s,t] + [c = term] sum_t gy[s,t]
//   dL/dam[b,t,c] = exp(am - am_max) * sum_s D[s,t] exp(lm[s,c] - lm_max[s])
//                   + sum_s [c = sym[b,s]] gx[s,t] + [c = term] sum_s gy[s,t]
// i.e. two more GEMMs with the same fused-exp loaders (what autograd derives for
// rnnt_loss.py:174-220; the derivatives through the two max() cancel).
#include <mutex>

#include "simple_shared.hip.h"
#include "tile_gemm.hip.h"

namespace frnnt {
namespace {

// Which XCD works on which utterance in the gradient products.  Workgroup i runs on XCD
// i % 8 and all tiles of an utterance stay on one XCD (one L2 holds its operands), so a launch of
// many tiles lasts as long as its fullest XCD; with utterance b on XCD b % 8 that is left to
// the order of the batch (ragged batches of 16 and 32 utterances: the fullest XCD 32 % and
// 19 % above the average).  The prep kernel therefore ranks the utterances by the cells of
// their windows (rank 0 = most) and the products deal them out by rank: rank r goes to XCD
// r % 8 in even rounds of eight and to 7 - r % 8 in odd ones, so that every XCD takes its
// larger utterances first (the same batches: 10 % and 1 % above the average; both products of
// the larger one 223 -> 210 us).  The utterance of rank r is kept, as an int, in
// row_x[r][S] -- the row sums of px_grad have no row S, nobody reads that entry as a number
// -- so a workgroup finds its utterance with one scalar load.  Batches of more than 64 and
// calls without a window rank by index.
template <typename R>
__device__ __forceinline__ int *rank_slot(R *row_x, int r, int S) {
  return reinterpret_cast<int *>(row_x + (long)r * (S + 1) + S);
}
// one wave: ranks the batch and leaves the utterance of every rank in its slot
template <typename R>
__device__ __forceinline__ void rank_utterances(R *row_x, const int64_t *window, int B, int S, int T,
                                                int lane) {
  if (!window || B > kWave) {
    for (int i = lane; i < B; i += kWave) *rank_slot(row_x, i, S) = i;
    return;
  }
  unsigned key = 0;  // lanes without an utterance rank behind every utterance
  if (lane < B) {
    const Limits w = limits_of(window, lane, S, T);
    const long cells = (long)max(w.s_end - w.s_begin + 1, 0) * max(w.t_end - w.t_begin, 0);
    // (distinct keys: equal sizes rank by index)
    key = ((unsigned)min(cells, 1L << 24) << 6 | (unsigned)(kWave - 1 - lane)) + 1u;
  }
  int rank = 0;
  for (int j = 0; j < B; ++j) rank += (unsigned)__builtin_amdgcn_readlane((int)key, j) > key ? 1 : 0;
  if (lane < B) *rank_slot(row_x, rank, S) = lane;
}
// With fewer than 32 utterances a unit of placement is a PART of an utterance: its tiles
// of every 2^part_shift-th stretch of the vocabulary (such tiles share D but nothing of lm or
// am), enough parts for eight units per XCD while a part keeps four tiles along the
// vocabulary.  A batch of two then reaches all eight XCDs instead of two (B = 2, S = 100,
// T = 400, C = 5000: both products 117 -> 36 us), and a batch of sixteen is dealt out in 64
// units (fullest XCD 2 % above the average instead of 10 %: 212 -> 201 us).
inline int part_shift_for(int B, int c_tiles) {
  if (B >= 32) return 0;
  int shift = 0;
  while ((B << shift) < 64 && (8 << shift) <= c_tiles) ++shift;
  return shift;
}
// n / d for n < 2^32, the reciprocal made on the host (the round-up method of Granlund and
// Montgomery): a multiplication and three more scalar instructions instead of the compiler's thirty.
struct Divisor {
  unsigned d, reciprocal, shift1, shift2;
  explicit Divisor(unsigned d_) : d(d_) {
    unsigned l = 0;
    while (l < 32 && (1ull << l) < d) ++l;
    reciprocal = (unsigned)((((1ull << l) - d) << 32) / d + 1);
    shift1 = l < 1 ? l : 1, shift2 = l < 1 ? 0 : l - 1;
  }
  __device__ __forceinline__ unsigned divide(unsigned n) const {
    const unsigned t = __umulhi(reciprocal, n);
    return (t + ((n - t) >> shift1)) >> shift2;
  }
};
// One product's share of the grid: its tiles of c_per stretches of the vocabulary, rows of tiles
// outermost, for the units of one XCD one after the other.
struct Placement {
  Divisor c_per, unit_tiles;
  int c_tiles, part_shift;
  unsigned blocks;
  Placement(int c_tiles_, int row_tiles, int B, int part_shift_)
      : c_per((c_tiles_ + (1 << part_shift_) - 1) >> part_shift_),
        unit_tiles(row_tiles > 0 ? c_per.d * row_tiles : 1), c_tiles(c_tiles_), part_shift(part_shift_) {
    const long units = (long)B << part_shift;
    blocks = row_tiles > 0
                 ? (unsigned)(dgemm::kXcds * ((units + dgemm::kXcds - 1) / dgemm::kXcds) * unit_tiles.d)
                 : 0;
  }
};
// (utterance, row of tiles, tile along the vocabulary) of workgroup `id`
__device__ __forceinline__ bool place_block(unsigned id, const Placement &at, int B,
                                            const float *row_x, int S, int &b, int &row_idx,
                                            int &c_idx) {
  using dgemm::kXcds;
  const unsigned xcd = id % kXcds, slot = id / kXcds, round = at.unit_tiles.divide(slot);
  const unsigned within = slot - round * at.unit_tiles.d;
  const int unit = round * kXcds + ((round & 1) ? kXcds - 1 - xcd : xcd);
  const int rank = unit >> at.part_shift, part = unit & ((1 << at.part_shift) - 1);
  row_idx = at.c_per.divide(within);
  c_idx = part * at.c_per.d + (within - row_idx * at.c_per.d);
  if (rank >= B || c_idx >= at.c_tiles) return false;
  b = *reinterpret_cast<const int *>(row_x + (long)rank * (S + 1) + S);
  return true;
}

template <typename R>
__device__ __forceinline__ R wave_max(R v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const R o = __shfl_xor(v, off, 64);
    v = o > v ? o : v;
  }
  return v;
}
template <typename R>
__device__ __forceinline__ R wave_sum(R v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// One wave per row of lm (first n_lm rows) or am (the rest): max over C.
template <typename R>
__global__ void __launch_bounds__(256)
    row_max_kernel(const R *__restrict__ lm, const R *__restrict__ am, R *__restrict__ lm_max,
                   R *__restrict__ am_max, long n_lm, long n_am, int C) {
  const long row = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= n_lm + n_am) return;
  const R *src = row < n_lm ? lm + row * C : am + (row - n_lm) * C;
  R m = Num<R>::neg_inf();
  for (int c = lane; c < C; c += kWave) {
    const R v = src[c];
    m = (v > m || v != v) ? v : m;  // NaN propagates, like torch.max
  }
  {
    // reduce, keeping NaN if any lane saw one
    R r = m;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const R o = __shfl_xor(r, off, 64);
      r = (o > r || o != o) ? o : r;
    }
    m = r;
  }
  if (lane == 0) {
    if (row < n_lm)
      lm_max[row] = m;
    else
      am_max[row - n_lm] = m;
  }
}

template <typename R>
__device__ __forceinline__ R tiny_of();
template <>
__device__ __forceinline__ float tiny_of<float>() {
  return 1.17549435e-38f;
}
template <>
__device__ __forceinline__ double tiny_of<double>() {
  return 2.2250738585072014e-308;
}
template <typename R>
__device__ __forceinline__ R accurate_log(R x);
template <>
__device__ __forceinline__ float accurate_log<float>(float x) {
  return logf(x);
}
template <>
__device__ __forceinline__ double accurate_log<double>(double x) {
  return log(x);
}

// grid = (ceil(T/64), ceil((S+1)/64), B)
template <typename R>
__global__ void __launch_bounds__(kGemmThreads)
    simple_fwd_kernel(const R *__restrict__ lm, const R *__restrict__ am,
                      const int64_t *__restrict__ symbols, const int64_t *__restrict__ boundary,
                      const R *__restrict__ lm_max, const R *__restrict__ am_max,
                      R *__restrict__ px, R *__restrict__ py, R *__restrict__ norm_raw,
                      Delay<R> delay, int S, int T, int C, int term, int rnnt_type) {
  __shared__ R lds[4 * TileK<R>::value * kPitch];
  const int b = blockIdx.z;
  const int s_tile = blockIdx.y * kTileM, t_tile = blockIdx.x * kTileN;
  const int S1 = S + 1;
  const int T1 = rnnt_type == kRegular ? T + 1 : T;
  const R *lmb = lm + (long)b * S1 * C;
  const R *amb = am + (long)b * T * C;
  const R *lmx = lm_max + (long)b * S1;
  const R *amx = am_max + (long)b * T;

  WaveAcc<R> acc;
  tile_matmul<R, LoaderKFast<R, true>, LoaderKFast<R, true>>(acc, lds, lmb, C, lmx, s_tile, S1,
                                                             amb, C, amx, t_tile, T, C);

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t t_mask = (rnnt_type == kRegular && boundary) ? boundary[4 * b + 3] : -1;
  const int64_t *symb = symbols + (long)b * S;
  R *pxb = px + (long)b * S * T1;
  R *pyb = py + (long)b * S1 * T;
  R *nrb = norm_raw ? norm_raw + (long)b * S1 * T : nullptr;
  acc.for_each((wave >> 1) * 32, (wave & 1) * 32, lane, [&](int m, int n, R sum) {
    const int s = s_tile + m, t = t_tile + n;
    if (s >= S1 || t >= T) return;
    const R raw = accurate_log<R>(sum + tiny_of<R>());
    if (nrb) nrb[(long)s * T + t] = raw;
    const R norm = raw + lmx[s] + amx[t];
    pyb[(long)s * T + t] = (amb[(long)t * C + term] + lmb[(long)s * C + term]) - norm;
    if (s < S) {
      const int64_t sym = symb[s];
      R v;
      if (sym < 0 || sym >= C)
        v = std::numeric_limits<R>::quiet_NaN();  // out-of-vocabulary symbol
      else
        v = (amb[(long)t * C + sym] + lmb[(long)s * C + sym]) - norm;
      if (t == t_mask) v = Num<R>::neg_inf();
      pxb[(long)s * T1 + t] = delay.at(v, boundary, b, t, T);
    }
  });
  // the extra column of the regular lattice: nothing can be emitted after the last frame
  if (rnnt_type == kRegular && blockIdx.x == 0) {
    for (int m = threadIdx.x; m < kTileM; m += kGemmThreads)
      if (s_tile + m < S) pxb[(long)(s_tile + m) * T1 + T] = Num<R>::neg_inf();
  }
}

// constrained lattice: px[b,s,t] += py[b,s+1,t]   (rnnt_loss.py:224-225), then the delay penalty
template <typename R>
__global__ void __launch_bounds__(256)
    add_next_row_kernel(R *__restrict__ px, const R *__restrict__ py,
                        const int64_t *__restrict__ boundary, Delay<R> delay, long total, int S,
                        int T) {
  const long idx = (long)blockIdx.x * 256 + threadIdx.x;
  if (idx >= total) return;
  const long b = idx / ((long)S * T);
  const long rem = idx - b * (long)S * T;
  const int s = (int)(rem / T), t = (int)(rem - (long)s * T);
  px[idx] = delay.at(px[idx] + py[(b * (S + 1) + s + 1) * T + t], boundary, (int)b, t, T);
}

// ---- backward ------------------------------------------------------------------------
// `n` consecutive values of an array, one wave's row (its address is wave-uniform)
template <typename R>
struct Row {
  R *base;
  int n;
  __device__ __forceinline__ Row(R *base_, int n_) : base(base_), n(n_) {}
  __device__ __forceinline__ R get(bool there, int t) const { return there && t < n ? base[t] : (R)0; }
  __device__ __forceinline__ void put(bool there, int t, R v) const {
    if (there && t < n) base[t] = v;
  }
};
template <>
struct Row<float> {
  __amdgpu_buffer_rsrc_t rs;
  __device__ __forceinline__ Row(float *base, int n) : rs(buffer_of(base, 4 * n)) {}
  __device__ __forceinline__ float get(bool there, int t) const { return get_float(rs, there, 4 * t); }
  __device__ __forceinline__ void put(bool there, int t, float v) const {
    put_float(rs, there, 4 * t, v);
  }
};

constexpr int kProdK = 32;  // k per chunk of the float32 gradient products: two k-steps
// 256-thread workgroups.  The first ceil(B*(S+1)/4) of them give each wave one
// lattice row (b, s): D[b,s,:] and the two row sums.  With `score_grad` the wave first scales
// its row of the occupation gradients in place (scale_by_batch_kernel's work, for lattices whose
// rows do not read each other's: one pass over them less).  `joint`: what they count for in D
// (1, less in the smoothed loss).  Loads are issued in batches of
// four before anything is stored, so a row costs one memory round trip, not one per 64 frames.
// Bound by memory; cells outside the windows, a third of a ragged batch, are neither read nor written
// (B 64, S 120, T 600: 20.6 -> 15.7 us).
// In double the next workgroups take 64 frames of one utterance each and form the column
// sums, the four waves splitting the lattice rows (the float product forms those it needs).  The
// last workgroup ranks the utterances for the gradient products (rank_utterances).
template <typename R>
__global__ void __launch_bounds__(256)
    simple_bwd_prep_kernel(R *__restrict__ gpx, R *__restrict__ gpy,
                           const R *__restrict__ norm_raw, const int64_t *__restrict__ boundary,
                           const int64_t *__restrict__ window, const R *__restrict__ score_grad,
                           int stride, R scale, R joint, R *__restrict__ dmat, R *__restrict__ row_x,
                           R *__restrict__ row_y, R *__restrict__ col_y, int B, int S, int T,
                           int ldd, int rnnt_type) {
  __shared__ R partial[4][kWave];
  const int S1 = S + 1;
  const int T1 = rnnt_type == kRegular ? T + 1 : T;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long n_rows = (long)B * S1;
  const long row_blocks = (n_rows + 3) / 4;
  const bool constrained = rnnt_type == kConstrained;
  if (blockIdx.x < row_blocks) {
    const long row = (long)blockIdx.x * 4 + wave;
    if (row >= n_rows) return;
    const int b = (int)(row / S1), s = (int)(row % S1);
    const int t_mask = (rnnt_type == kRegular && boundary) ? (int)boundary[4 * b + 3] : -1;
    // outside the window nothing counts (the normalizers there may be undefined): D = 0
    const Limits lim = limits_of(window, b, S, T);
    const bool row_in = s >= lim.s_begin && s <= lim.s_end;
    // (a float row is read and written through a buffer resource over it: no branch around a
    // load, which would end in a wait for all of them; rows that do not exist are empty)
    const Row<R> gx_row(gpx + ((long)b * S + min(s, S - 1)) * T1, s < S ? T1 : 0);
    const Row<R> gx_prev(gpx + ((long)b * S + max(s - 1, 0)) * T1, constrained && s >= 1 ? T1 : 0);
    const Row<R> gy_row(gpy + row * T, T), nr_row(const_cast<R *>(norm_raw) + row * T, T);
    R *d_row = dmat + row * ldd;
    const bool scaled = score_grad != nullptr;
    const R g = scaled ? scale * score_grad[(long)b * stride] : (R)1;
    // What is scaled: all of the row, or, where the zeros outside the window stay zeros, what lies
    // inside (the lattice's last column with it).  What of D the products look at: their sums over
    // rows and frames stop at the first multiple of a chunk past the window, and D is 0 up to there.
    const bool whole = !window || !(g - g == 0);
    const int scaled_lo = whole ? 0 : lim.t_begin;
    const int scaled_hi = !scaled ? 0 : whole ? T1 : row_in ? min(lim.t_end + 1, T1) : 0;
    const int d_hi = !window ? ldd
                     : s < (lim.s_end + kProdK) / kProdK * kProdK
                         ? min(ldd, (lim.t_end + kProdK - 1) / kProdK * kProdK)
                         : 0;
    R sx = 0, sy = 0;
    for (int t0 = 0; t0 < max(scaled_hi, d_hi); t0 += 4 * kWave) {
      R gx[4], gy[4], above[4], nr[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int t = t0 + u * kWave + lane;
        const bool ok = t < T && row_in && t >= lim.t_begin && t < lim.t_end;
        const bool there = ok || (t >= scaled_lo && t < scaled_hi);
        gx[u] = gx_row.get(there, t);
        gy[u] = gy_row.get(there, t);
        above[u] = constrained ? gx_prev.get(ok && t != t_mask, t) : (R)0;
        nr[u] = nr_row.get(ok, t);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int t = t0 + u * kWave + lane;
        const bool ok = t < T && row_in && t >= lim.t_begin && t < lim.t_end;
        gy[u] += above[u];
        gx[u] *= g;
        gy[u] *= g;
        if (scaled) {
          gx_row.put(t >= scaled_lo && t < scaled_hi, t, gx[u]);
          gy_row.put(t >= scaled_lo && t < scaled_hi, t, gy[u]);
        }
        gx[u] = ok && t != t_mask ? gx[u] : (R)0;
        gy[u] = ok ? gy[u] : (R)0;
        if (t < d_hi) d_row[t] = -(gx[u] * joint + gy[u] * joint) * fast_exp<R>(-nr[u]);
        sx += gx[u];
        sy += gy[u];
      }
    }
    sx = wave_sum(sx);
    sy = wave_sum(sy);
    if (lane == 0) {
      if (s < S) row_x[row] = sx;  // (entry S of a row belongs to rank_utterances)
      row_y[row] = sy;
    }
  } else if (blockIdx.x == gridDim.x - 1) {
    if (wave == 0) rank_utterances(row_x, window, B, S, T, lane);
  } else {
    const int tiles = (T + kWave - 1) / kWave;
    const long cb = blockIdx.x - row_blocks;
    const int b = (int)(cb / tiles), t = (int)(cb % tiles) * kWave + lane;
    const int t_mask = (rnnt_type == kRegular && boundary) ? (int)boundary[4 * b + 3] : -1;
    const Limits lim = limits_of(window, b, S, T);
    const bool ok = t < T && t >= lim.t_begin && t < lim.t_end;
    R acc = 0;
    for (int s0 = wave; s0 < S1; s0 += 16) {
      R v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int s = s0 + 4 * u;
        v[u] = (ok && s < S1) ? gpy[((long)b * S1 + s) * T + t] : (R)0;
        if (constrained && ok && s >= 1 && s < S1 && t != t_mask)
          v[u] += gpx[((long)b * S + s - 1) * T1 + t];
      }
      acc += (v[0] + v[1]) + (v[2] + v[3]);
    }
    partial[wave][lane] = acc;
    __syncthreads();
    if (wave == 0 && t < T)
      col_y[(long)b * T + t] = (partial[0][lane] + partial[1][lane]) + (partial[2][lane] + partial[3][lane]);
  }
}

// px_grad[b,:,:] *= g_b, py_grad[b,:,:] *= g_b in place, with
// g_b = scale * score_grad[b * stride].  blockIdx.y is the utterance; a workgroup
// takes 1024 consecutive elements of its px_grad part or of its py_grad part.
template <typename R>
__global__ void __launch_bounds__(256)
    scale_by_batch_kernel(R *__restrict__ gpx, R *__restrict__ gpy,
                          const R *__restrict__ score_grad, int stride, R scale, int per_x,
                          int per_y, int x_blocks) {
  const int b = blockIdx.y;
  const R g = scale * score_grad[(long)b * stride];
  const bool is_x = (int)blockIdx.x < x_blocks;
  R *base = is_x ? gpx + (long)b * per_x : gpy + (long)b * per_y;
  const int n = is_x ? per_x : per_y;
  const int first = (is_x ? blockIdx.x : blockIdx.x - x_blocks) * 1024 + threadIdx.x;
  R v[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) v[u] = (first + 256 * u < n) ? base[first + 256 * u] : (R)0;
#pragma unroll
  for (int u = 0; u < 4; ++u)
    if (first + 256 * u < n) base[first + 256 * u] = v[u] * g;
}

// loss = -scores, -mean(scores) or -sum(scores); one wave
template <typename R>
__global__ void __launch_bounds__(kWave)
    loss_reduce_kernel(const R *__restrict__ scores, R *__restrict__ loss, int B, int reduction) {
  reduce_scores(scores, loss, B, reduction, (int)threadIdx.x);
}

// lm gradient: grid = (ceil(C/64), ceil((S+1)/64), B); K runs over frames.
template <typename R>
__global__ void __launch_bounds__(kGemmThreads)
    simple_bwd_lm_kernel(const R *__restrict__ lm, const R *__restrict__ am,
                         const int64_t *__restrict__ symbols, const R *__restrict__ lm_max,
                         const R *__restrict__ am_max, const R *__restrict__ dmat,
                         const R *__restrict__ row_x, const R *__restrict__ row_y,
                         R *__restrict__ lm_grad, int S, int T, int C, int ldd, int term) {
  __shared__ R lds[4 * TileK<R>::value * kPitch];
  const int b = blockIdx.z;
  const int s_tile = blockIdx.y * kTileM, c_tile = blockIdx.x * kTileN;
  const int S1 = S + 1;
  const R *lmb = lm + (long)b * S1 * C;
  const R *amb = am + (long)b * T * C;
  const R *lmx = lm_max + (long)b * S1;
  const R *amx = am_max + (long)b * T;
  const R *db = dmat + (long)b * S1 * ldd;

  WaveAcc<R> acc;
  tile_matmul<R, LoaderKFast<R, false>, LoaderRowFast<R, true>>(acc, lds, db, ldd, nullptr, s_tile,
                                                                S1, amb, C, amx, c_tile, C, T);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  acc.for_each((wave >> 1) * 32, (wave & 1) * 32, lane, [&](int m, int n, R sum) {
    const int s = s_tile + m, c = c_tile + n;
    if (s >= S1 || c >= C) return;
    R g = fast_exp<R>(lmb[(long)s * C + c] - lmx[s]) * sum;
    if (s < S && symbols[(long)b * S + s] == c) g += row_x[(long)b * S1 + s];
    if (c == term) g += row_y[(long)b * S1 + s];
    lm_grad[((long)b * S1 + s) * C + c] = g;
  });
}

// am gradient: grid = (ceil(C/64), ceil(T/64), B); K runs over lattice rows.
template <typename R>
__global__ void __launch_bounds__(kGemmThreads)
    simple_bwd_am_kernel(const R *__restrict__ lm, const R *__restrict__ am,
                         const R *__restrict__ lm_max, const R *__restrict__ am_max,
                         const R *__restrict__ dmat, const R *__restrict__ col_y,
                         R *__restrict__ am_grad, int S, int T, int C, int ldd, int term) {
  __shared__ R lds[4 * TileK<R>::value * kPitch];
  const int b = blockIdx.z;
  const int t_tile = blockIdx.y * kTileM, c_tile = blockIdx.x * kTileN;
  const int S1 = S + 1;
  const R *lmb = lm + (long)b * S1 * C;
  const R *amb = am + (long)b * T * C;
  const R *lmx = lm_max + (long)b * S1;
  const R *amx = am_max + (long)b * T;
  const R *db = dmat + (long)b * S1 * ldd;

  WaveAcc<R> acc;
  tile_matmul<R, LoaderRowFast<R, false>, LoaderRowFast<R, true>>(acc, lds, db, ldd, nullptr, t_tile,
                                                                  T, lmb, C, lmx, c_tile, C, S1);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  acc.for_each((wave >> 1) * 32, (wave & 1) * 32, lane, [&](int m, int n, R sum) {
    const int t = t_tile + m, c = c_tile + n;
    if (t >= T || c >= C) return;
    R g = fast_exp<R>(amb[(long)t * C + c] - amx[t]) * sum;
    if (c == term) g += col_y[(long)b * T + t];
    am_grad[((long)b * T + t) * C + c] = g;
  });
}

// am_grad[b,t,sym[b,s]] += gx[b,s,t]: one thread per (b,t), rows visited in
// order, so repeated symbols accumulate deterministically.
template <typename R>
__global__ void __launch_bounds__(256)
    simple_bwd_symbols_kernel(const R *__restrict__ gpx, const int64_t *__restrict__ symbols,
                              const int64_t *__restrict__ boundary, R *__restrict__ am_grad,
                              int B, int S, int T, int C, int rnnt_type) {
  const long idx = (long)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (long)B * T) return;
  const int b = (int)(idx / T), t = (int)(idx % T);
  const int T1 = rnnt_type == kRegular ? T + 1 : T;
  if (rnnt_type == kRegular && boundary && boundary[4 * b + 3] == t) return;
  R *row = am_grad + idx * C;
  for (int s = 0; s < S; ++s) {
    const int64_t sym = symbols[(long)b * S + s];
    if (sym >= 0 && sym < C) row[sym] += gpx[((long)b * S + s) * T1 + t];
  }
}

// ---- float32 gradient products on the bfloat16 matrix cores ----------------------------------
//   lm.grad[s,c] = exp(lm[s,c] - max[s]) * sum_t D[s,t] exp(am[t,c] - max[t]) + one-hots
//   am.grad[t,c] = exp(am[t,c] - max[t]) * sum_s D[s,t] exp(lm[s,c] - max[s]) + one-hots
// A workgroup of four waves takes kM rows (lattice rows of lm.grad, frames of am.grad) x 64
// vocabulary entries, a wave 32 rows x 64 or 32 of them as 32 x 32 accumulators.  k (frames, lattice
// rows) runs in chunks of 32.  D belongs to one wave's rows: it goes from memory straight
// into the lanes that multiply it and is split into bfloat16 parts (split_pair) there.  The
// operand along the vocabulary is shared: a thread fetches eight consecutive k of one entry, loads
// that are contiguous over the lanes, takes exp, splits, and has its 16-byte piece of the operand
// without any transposition; the pieces lie in LDS as [octet of k][part][entry], where consecutive
// lanes write and read consecutive pieces.  Two such images alternate: a chunk is staged while the
// one before it is multiplied, one barrier per chunk.
// What bounds it: instructions issued.  Of 250 000 cycles per SIMD (counters, B 16, S 120, T 400,
// C 5000, the matrix cores busy for 71 000) almost every group of four issues one.  Taking 12
// million of 21 million scalar instructions out (offsets made once instead of per load, reciprocals
// instead of divisions, a list that ends with its last hit) took 116 to 108 us, while the same kernel
// without any loads of D takes 104, with fewer and wider tiles (128 entries: 110), with its L2
// requests down by 15 % (eight waves, 128 entries: 130) or with its reads of HBM down by a third
// (the tiles of both products that read the same entries side by side: 119) gains nothing.
// Measured (both products; B 32, S 80, T 250, C 500 / B 64, S 120, T 600, C 500 / B 16, S 120, T 400,
// C 5000): 23.5 / 83 / 124 us when both operands went through one LDS image, 20 / 72.5 / 108 now.
constexpr int kProdThreads = 256;
constexpr int kProdC = 64;      // vocabulary entries of a tile
constexpr int kProdPerCu = 4;   // workgroups that share a compute unit
constexpr long kMinWideTiles = 256;
constexpr int kPartBytes = 16 * kProdC;            // one part of an octet of k
constexpr int kImageBytes = 4 * 3 * kPartBytes;    // a chunk of the operand along the vocabulary
template <int kM>
struct ProdShape {
  static constexpr int kWavesM = kM / 32, kWavesC = 4 / kWavesM;
  static constexpr int kWaveC = kProdC / kWavesC, kTiles = kWaveC / 32;  // 32-column tiles of a wave
  static constexpr int kMColumns = kM / 64;  // frames per thread of a sum over lattice rows
};
typedef int intx4 __attribute__((ext_vector_type(4)));
// k-octet `octet` (0 .. 3) of entry `c` in a chunk's LDS image
__device__ __forceinline__ int octet_at(int c, int octet) { return octet * 3 * kPartBytes + c * 16; }
__device__ __forceinline__ void split_octet(const float (&e)[8], uintx4 &hi, uintx4 &mid, uintx4 &lo) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    unsigned h, m, l;
    split_pair(e[2 * q], e[2 * q + 1], h, m, l);
    hi[q] = h, mid[q] = m, lo[q] = l;
  }
}
__device__ __forceinline__ void write_octet(char *to, const float (&e)[8]) {
  uintx4 hi, mid, lo;
  split_octet(e, hi, mid, lo);
  *reinterpret_cast<uintx4 *>(to) = hi;
  *reinterpret_cast<uintx4 *>(to + kPartBytes) = mid;
  *reinterpret_cast<uintx4 *>(to + 2 * kPartBytes) = lo;
}
__device__ __forceinline__ Split8 read_octet(const char *at) {
  Split8 o;
  o.hi = *reinterpret_cast<const bf16x8 *>(at);
  o.mid = *reinterpret_cast<const bf16x8 *>(at + kPartBytes);
  o.lo = *reinterpret_cast<const bf16x8 *>(at + 2 * kPartBytes);
  return o;
}
// (the gradients that a product writes are FRNNT_F32, FRNNT_F16 or FRNNT_BF16, or kStreamed:
// float32 with the non-temporal hint)
constexpr int kStreamed = 16;
__device__ __forceinline__ int out_bytes(int type) {
  return type == FRNNT_F32 || type == kStreamed ? 4 : 2;
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t out_buffer(void *base, long first, int count,
                                                             int type) {
  const int size = out_bytes(type);
  return __builtin_amdgcn_make_buffer_rsrc(static_cast<char *>(base) + first * size, 0, count * size,
                                           0x00020000);
}
// f(store) with store(resource, there, element, uniform element, value) for the type
template <typename F>
__device__ __forceinline__ void with_store(int type, F f) {
  if (type == FRNNT_F32)
    f([](__amdgpu_buffer_rsrc_t rs, bool there, int at, int uniform, float x) {
      put_float(rs, there, 4 * at, x, 4 * uniform);
    });
  else if (type == kStreamed)
    f([](__amdgpu_buffer_rsrc_t rs, bool there, int at, int uniform, float x) {
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_int(x), rs, there ? 4 * at : kNowhere,
                                            4 * uniform, 2);
    });
  else
    f([type](__amdgpu_buffer_rsrc_t rs, bool there, int at, int uniform, float x) {
      const uint16_t half = HalfIO::store(x), bf16 = (uint16_t)pack_bf16(x, 0.f);
      __builtin_amdgcn_raw_buffer_store_b16((short)(type == FRNNT_F16 ? half : bf16), rs,
                                            there ? 2 * at : kNowhere, 2 * uniform, 0);
    });
}
// acc[n] += D (rows of this wave's 32) times exp(x - max) (its 32-column tiles) over k < k_lim.
// kFrames: the rows are frames and k the lattice rows (am.grad), else the other way round.  `x` holds
// the rows of the operand along the vocabulary, one per k; `live`: this wave's rows count.  `early()` is
// called once the first chunk is staged, `late()` before the end, to request what follows.
template <int kM, bool kFrames, typename Early, typename Late>
__device__ __forceinline__ void accumulate_products(
    char *lds, __amdgpu_buffer_rsrc_t d_rs, int row, int ldd, __amdgpu_buffer_rsrc_t x_rs,
    const float *x_max, int c_tile, int C, int k_lim, bool live, int wave, int lane,
    dgemm::floatx16 (&acc)[ProdShape<kM>::kTiles], Early early, Late late) {
  using Shape = ProdShape<kM>;
  const int half = lane >> 5, r32 = lane & 31;
  const int c_wave = Shape::kWaveC * (wave / Shape::kWavesM);
  // D: a lane's operand is eight consecutive k of its row, straight from memory.  It is 0 wherever a
  // row or a frame does not count, and up to the end of its rows of ldd; nothing is read past them.
  float d[2][8];
  const int d_off = kFrames ? (8 * half * ldd + row) * 4 : (row * ldd + 8 * half) * 4;
  auto fetch_d = [&](int g, int k0) {
    if constexpr (kFrames) {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        d[g][i] = get_float(d_rs, true, d_off + k0 * ldd * 4, (16 * g + i) * ldd * 4);
    } else {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int k = 16 * g + 4 * j;
        const intx4 raw = __builtin_amdgcn_raw_buffer_load_b128(
            d_rs, 8 * half + k < ldd - k0 ? d_off + 4 * (k0 + k) : kNowhere, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) d[g][4 * j + i] = __int_as_float(raw[i]);
      }
    }
  };
  // the operand along the vocabulary: eight consecutive k of one entry per thread.  The
  // resource ends with row k_lim - 1: what follows reads as 0 with a shift of 0, a factor of 1.
  float x[8], shift;  // (lane i: the shift of k i)
  const int x_off = (8 * wave * C + c_tile + lane) * 4;
  auto fetch_x = [&](int k0) {
    const int k = k0 + 8 * wave + (lane & 7);
    const float mx = x_max[min(k, k_lim - 1)];
    shift = k < k_lim ? -mx * kLog2e : 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = get_float(x_rs, true, x_off + k0 * C * 4, i * C * 4);
  };
  auto stage_x = [&](char *image) {
    float e[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) e[i] = exp_shifted(x[i], read_lane(shift, i));
    write_octet(image + octet_at(lane, wave), e);
  };
  auto multiply = [&](int g, const char *image) {
    uintx4 hi, mid, lo;
    split_octet(d[g], hi, mid, lo);
    Split8 d_op;
    __builtin_memcpy(&d_op.hi, &hi, 16);
    __builtin_memcpy(&d_op.mid, &mid, 16);
    __builtin_memcpy(&d_op.lo, &lo, 16);
#pragma unroll
    for (int n = 0; n < Shape::kTiles; ++n)
      acc[n] = multiply_add(
          d_op, read_octet(image + octet_at(c_wave + 32 * n + r32, 2 * g + half)), acc[n]);
  };
  if (k_lim <= 0) {
    early();
    late();
    lds_barrier();
    return;
  }
  fetch_x(0);
  fetch_d(0, 0);
  fetch_d(1, 0);
  early();
  stage_x(lds);
  fetch_x(kProdK);
  lds_barrier();
  int image = 0, k0 = 0;
  for (; k0 + kProdK < k_lim; k0 += kProdK) {
    const char *from = lds + image;
    image ^= kImageBytes;
    stage_x(lds + image);
    fetch_x(k0 + 2 * kProdK);
    if (live) {
      multiply(0, from);
      fetch_d(0, k0 + kProdK);
      multiply(1, from);
      fetch_d(1, k0 + kProdK);
    }
    lds_barrier();
  }
  if (live) {
    multiply(0, lds + image);
    multiply(1, lds + image);
  }
  late();
}

template <int kM, bool kSmooth>
__device__ __forceinline__ void simple_bwd_lm_body(
    int b, int row_idx, int c_idx, const float *__restrict__ lm, const float *__restrict__ am,
    const int64_t *__restrict__ symbols, const float *__restrict__ lm_max,
    const float *__restrict__ am_max, const float *__restrict__ dmat,
    const float *__restrict__ row_x, const float *__restrict__ row_y,
    void *__restrict__ lm_grad, const int64_t *__restrict__ window, int S, int T, int C, int ldd,
    int term, int out_type, const SmoothTerms &smooth) {
  using Shape = ProdShape<kM>;
  using namespace dgemm;
  extern __shared__ __align__(16) char prod_lds[];
  __shared__ float row_mx[kM], row_rx[kM], row_ry[kM];
  __shared__ float row_w[kSmooth ? kM : 1], row_inv[kSmooth ? kM : 1];  // (times exp(lm - max): lm-only terms)
  __shared__ int row_sym[kM];
  const int S1 = S + 1;
  const Limits lim = limits_of(window, b, S, T);
  const int s_tile = row_idx * kM, c_tile = c_idx * kProdC;
  const float *lmb = lm + (long)b * S1 * C;
  const float *amb = am + (long)b * T * C;
  const float *amx = am_max + (long)b * T;
  const float *db = dmat + (long)b * S1 * ldd;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5, r32 = lane & 31;
  // With a window, D vanishes at frames >= t_end and on rows > s_end: the sum over frames
  // stops at t_end (the row maxima of later frames may not even be defined) and rows past s_end
  // get exact zeros.
  const int t_lim = __builtin_amdgcn_readfirstlane(lim.t_end);
  const int s_lim = __builtin_amdgcn_readfirstlane(min(S1, lim.s_end + 1));
  // The loads go through buffer resources that cover D[b] and am[b]: one instruction each, no
  // branch; rows past the last one read as 0 or as other rows of D and only feed rows that are never
  // written.  Vocabulary columns at and past C belong to the next row: they only feed output
  // columns that are never written.
  const __amdgpu_buffer_rsrc_t d_rs = buffer_of(db, S1 * ldd * 4);
  const __amdgpu_buffer_rsrc_t am_rs = buffer_of(amb, t_lim * C * 4);
  const int m_wave = 32 * (wave % Shape::kWavesM);
  floatx16 acc[Shape::kTiles];
#pragma unroll
  for (int n = 0; n < Shape::kTiles; ++n)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[n][v] = 0.f;
  const __amdgpu_buffer_rsrc_t lm_rs = buffer_of(lmb, S1 * C * 4);
  const __amdgpu_buffer_rsrc_t out_rs = out_buffer(lm_grad, (long)b * S1 * C, S1 * C, out_type);
  const int m0 = m_wave + 4 * half, c0 = c_tile + Shape::kWaveC * (wave / Shape::kWavesM) + r32;
  auto row_of = [&](int v) { return m0 + 8 * (v / 4) + v % 4; };
  const int first = (s_tile + m0) * C + c0;  // (element)
  auto below = [&](int v) { return (8 * (v / 4) + v % 4) * C; };  // (uniform)
  float in[Shape::kTiles][16];
  accumulate_products<kM, false>(
      prod_lds, d_rs, s_tile + m_wave + r32, ldd, am_rs, amx, c_tile, C, t_lim, s_tile + m_wave < s_lim,
      wave, lane, acc,
      [&] {
        if (tid < kM) {
          const int s = s_tile + tid, at = 4 * s;
          const long first_row = (long)b * S1;
          float mx = get_float(buffer_of((kSmooth ? smooth.lm_max : lm_max) + first_row, S1 * 4),
                               s < (kSmooth ? S1 : s_lim), at);
          const float rx = get_float(buffer_of(row_x + first_row, S1 * 4), s < S, at);
          const float ry = get_float(buffer_of(row_y + first_row, S1 * 4), s < S1, at);
          if (kSmooth) {
            const float sum = get_float(buffer_of(smooth.lm_sum + first_row, S1 * 4), s < S1, at);
            const float dot = smooth.am_scale != 0.f
                                  ? get_float(buffer_of(smooth.lm_dot + first_row, S1 * 4), s < S1, at)
                                  : 0.f;
            if (smooth.am_scale == 0.f) mx += *smooth.unigram;
            const float inv = 1.f / sum;
            row_w[tid] = (-dot * smooth.per_row - smooth.lm_scale * (rx + ry)) * inv;
            row_inv[tid] = smooth.per_row * inv;
          }
          const float times = kSmooth ? smooth.joint + smooth.lm_scale : 1.f;
          row_sym[tid] = get_symbol(symbols_of(symbols + (long)b * S, S), s < S, s, C);
          row_mx[tid] = mx, row_rx[tid] = rx * times, row_ry[tid] = ry * times;
        }
      },
      [&] {
#pragma unroll
        for (int n = 0; n < Shape::kTiles; ++n)
#pragma unroll
          for (int v = 0; v < 16; ++v)
            in[n][v] = get_float(lm_rs, c0 + 32 * n < C, 4 * first + 128 * n, 4 * below(v));
      });

  // ---- results: a lane holds column r32 of rows 8 (v / 4) + 4 half + v % 4 of its tiles (row_of)
  auto zero_past_end = [&] {
    if (s_tile + m_wave + 32 > s_lim) {  // (uniform)
#pragma unroll
      for (int n = 0; n < Shape::kTiles; ++n)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          acc[n][v] = s_tile + row_of(v) < s_lim ? acc[n][v] : 0.f;
    }
  };
  if (kSmooth) {
    zero_past_end();  // (the lm-only model's rows all count)
#pragma unroll
    for (int n = 0; n < Shape::kTiles; ++n)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[n][v] += row_w[row_of(v)];
    if (smooth.am_scale != 0.f) {  // (uniform)
#pragma unroll
      for (int n = 0; n < Shape::kTiles; ++n) {
        const float gu = get_float(buffer_of(smooth.g_unigram, C * 4), c0 + 32 * n < C, 4 * (c0 + 32 * n));
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[n][v] += gu * row_inv[row_of(v)];
      }
    }
  }
#pragma unroll
  for (int n = 0; n < Shape::kTiles; ++n)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[n][v] *= __expf(in[n][v] - row_mx[row_of(v)]);
  const bool symbols_here = __any((unsigned)(row_sym[m_wave + r32] - c_tile) < (unsigned)kProdC);
  if (symbols_here || (unsigned)(term - c_tile) < (unsigned)kProdC) {  // (uniform)
#pragma unroll
    for (int n = 0; n < Shape::kTiles; ++n)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        // (selects: branches around elements of a vector register make the compiler move all of it)
        const int m = row_of(v), c = c0 + 32 * n;
        const float rx = c == row_sym[m] ? row_rx[m] : 0.f, ry = c == term ? row_ry[m] : 0.f;
        acc[n][v] = (acc[n][v] + rx) + ry;
      }
  }
  if (!kSmooth) zero_past_end();
  with_store(out_type, [&](auto store) {
#pragma unroll
    for (int n = 0; n < Shape::kTiles; ++n)
#pragma unroll
      for (int v = 0; v < 16; ++v)
        store(out_rs, c0 + 32 * n < C, first + 32 * n, below(v), acc[n][v]);
  });
}

// The per-symbol term of am.grad,  sum_s [c = sym[b,s]] gx[b,s,t],  is a second product, gx^T times
// a one-hot matrix made in registers from the symbols, on the float32 matrix instruction: it is
// exact (products by 0 or 1) and has a fixed summation order.  The lattice rows whose symbol lies
// in the workgroup's vocabulary range are listed in order, sixteen at a time, and multiplied two
// rows at a time onto the finished dense results; the first sixteen are requested before the dense
// products and wait in registers.
constexpr int kListed = 16;
template <int kM, bool kSmooth>
__device__ __forceinline__ void simple_bwd_am_body(
    int b, int row_idx, int c_idx, const float *__restrict__ lm, const float *__restrict__ am,
    const int64_t *__restrict__ symbols, const int64_t *__restrict__ boundary,
    const float *__restrict__ lm_max, const float *__restrict__ am_max,
    const float *__restrict__ dmat, const float *__restrict__ gpx,
    const float *__restrict__ gpy, const float *__restrict__ row_x,
    void *__restrict__ am_grad, const int64_t *__restrict__ window, int S, int T, int C, int ldd,
    int term, int rnnt_type, int out_type, const SmoothTerms &smooth) {
  using Shape = ProdShape<kM>;
  using namespace dgemm;
  extern __shared__ __align__(16) char prod_lds[];
  __shared__ float frame_mx[kM], frame_y[kM], frame_w[kSmooth ? kM : 1];
  const int S1 = S + 1;
  const int T1 = rnnt_type == kRegular ? T + 1 : T;
  const Limits lim = limits_of(window, b, S, T);
  const int t_tile = row_idx * kM, c_tile = c_idx * kProdC;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5, r32 = lane & 31;
  const float *lmb = lm + (long)b * S1 * C;
  const float *amb = am + (long)b * T * C;
  const float *lmx = lm_max + (long)b * S1;
  const float *db = dmat + (long)b * S1 * ldd;
  const float *gxb = gpx + (long)b * S * T1;
  const __amdgpu_buffer_rsrc_t sym_rs = symbols_of(symbols + (long)b * S, S);
  const int t_mask = (rnnt_type == kRegular && boundary) ? (int)boundary[4 * b + 3] : -1;
  // With a window, D vanishes on rows > s_end and at frames >= t_end, where the frames'
  // maxima may not even be defined: such frames get exact zeros, the sum over the lattice
  // rows stops at s_end.
  const int t_lim = __builtin_amdgcn_readfirstlane(lim.t_end);
  const int k_lim = __builtin_amdgcn_readfirstlane(min(S1, lim.s_end + 1));
  const bool live = t_tile < t_lim;
  const __amdgpu_buffer_rsrc_t am_rs = buffer_of(amb, T * C * 4);
  const __amdgpu_buffer_rsrc_t out_rs = out_buffer(am_grad, (long)b * T * C, T * C, out_type);
  const int m_wave = 32 * (wave % Shape::kWavesM);
  const int m0 = m_wave + 4 * half, c_lo = c_tile + Shape::kWaveC * (wave / Shape::kWavesM),
            c0 = c_lo + r32;
  auto row_of = [&](int v) { return m0 + 8 * (v / 4) + v % 4; };
  const int first = (t_tile + m0) * C + c0;  // (element)
  auto below = [&](int v) { return (8 * (v / 4) + v % 4) * C; };  // (uniform)
  floatx16 acc[Shape::kTiles];
#pragma unroll
  for (int n = 0; n < Shape::kTiles; ++n)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[n][v] = 0.f;
  float in[Shape::kTiles][16];
  const __amdgpu_buffer_rsrc_t gx_rs = buffer_of(gxb, S * T1 * 4);
  // ---- the listed rows, from 128 symbols at a time: two masks of those in this tile
  const int s_count = live ? min(k_lim, S) : 0;
  int sym[2];
  unsigned long long hits[2];
  int column[kListed];        // (uniform) entry of the tile, -1 for none
  float value[kListed / 2];   // of rows 2 i + half at this lane's frame
  auto find_hits = [&](int s0) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int s = s0 + 64 * u + lane;
      sym[u] = get_symbol(sym_rs, s < s_count, s, C) - c_tile;
    }
#pragma unroll
    for (int u = 0; u < 2; ++u)
      hits[u] = __ballot(s0 + 64 * u + lane < s_count && (unsigned)sym[u] < (unsigned)kProdC);
  };
  auto fetch_listed = [&](int s0) {
    const int t = t_tile + m_wave + r32;
    const bool there = t < T && t != t_mask;
#pragma unroll
    for (int i = 0; i < kListed / 2; ++i) column[2 * i] = -1;
#pragma unroll
    for (int i = 0; i < kListed / 2; ++i) {
      if (!(hits[0] | hits[1])) break;  // (uniform)
      int row[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const bool low = hits[0] != 0, any = (hits[0] | hits[1]) != 0;
        unsigned long long &mask = low ? hits[0] : hits[1];
        const int at = any ? __builtin_ctzll(mask) : 0;
        row[u] = any ? s0 + at + (low ? 0 : kWave) : -1;
        column[2 * i + u] = any ? __builtin_amdgcn_readlane(low ? sym[0] : sym[1], at) : -1;
        mask &= mask - 1;
      }
      const int mine = half ? row[1] : row[0];
      value[i] = get_float(gx_rs, there && mine >= 0, (mine * T1 + t) * 4);
    }
  };
  if (live)
    accumulate_products<kM, true>(
        prod_lds, buffer_of(db, S1 * ldd * 4), t_tile + m_wave + r32, ldd, buffer_of(lmb, k_lim * C * 4),
        lmx, c_tile, C, k_lim, t_tile + m_wave < t_lim, wave, lane, acc,
        [&] {
          if (tid < kM) {
            const int t = t_tile + tid;
            const float mx = get_float(buffer_of(am_max + (long)b * T, T * 4), t < t_lim, 4 * t);
            frame_mx[tid] = kSmooth && smooth.am_scale == 0.f ? mx + *smooth.unigram : mx;
            if (kSmooth && smooth.am_scale != 0.f) {
              const float g = get_float(buffer_of(smooth.am_g + (long)b * T, T * 4), t < t_lim, 4 * t);
              const float z = get_float(buffer_of(smooth.am_z + (long)b * T, T * 4), t < t_lim, 4 * t);
              frame_w[tid] = t < t_lim ? -smooth.am_scale * g / z : 0.f;
            }
          }
          find_hits(0);
          fetch_listed(0);
        },
        [&] {
#pragma unroll
          for (int n = 0; n < Shape::kTiles; ++n)
#pragma unroll
            for (int v = 0; v < 16; ++v)
              in[n][v] = get_float(am_rs, c0 + 32 * n < C, 4 * first + 128 * n, 4 * below(v));
        });

  // ---- results: a lane holds column r32 of rows 8 (v / 4) + 4 half + v % 4 of its tiles (row_of)
  if (live) {
    // The termination symbol's term, sum_s gy[s,t], in the workgroups that hold its column: every
    // wave sums a quarter of the lattice rows.
    const __amdgpu_buffer_rsrc_t gx_rs = buffer_of(gxb, S * T1 * 4);
    if ((unsigned)(term - c_tile) < (unsigned)kProdC) {  // (uniform)
      const __amdgpu_buffer_rsrc_t gy_rs = buffer_of(gpy + (long)b * S1 * T, S1 * T * 4);
      lds_barrier();  // the operands have been read
      float *part = reinterpret_cast<float *>(prod_lds);
      float sum[Shape::kMColumns] = {};
      constexpr int kRowsAhead = 8;
      auto add_rows = [&](__amdgpu_buffer_rsrc_t rs, int rows, int pitch) {
        for (int s0 = wave; s0 < rows; s0 += 4 * kRowsAhead) {
          float y[kRowsAhead][Shape::kMColumns];
#pragma unroll
          for (int u = 0; u < kRowsAhead; ++u)
#pragma unroll
            for (int w = 0; w < Shape::kMColumns; ++w) {
              const int s = s0 + 4 * u, t = t_tile + lane + 64 * w;
              y[u][w] = get_float(rs, s < rows && t >= lim.t_begin && t < t_lim, 4 * t, s * pitch * 4);
            }
#pragma unroll
          for (int u = 0; u < kRowsAhead; ++u)
#pragma unroll
            for (int w = 0; w < Shape::kMColumns; ++w) sum[w] += y[u][w];
        }
      };
      add_rows(gy_rs, k_lim, T);
      // (constrained: py[s + 1] also went into px[s])
      if (rnnt_type == kConstrained) add_rows(gx_rs, min(k_lim, S), T1);
#pragma unroll
      for (int w = 0; w < Shape::kMColumns; ++w) part[wave * kM + lane + 64 * w] = sum[w];
      lds_barrier();
      if (tid < kM)
        frame_y[tid] = ((part[tid] + part[kM + tid]) + (part[2 * kM + tid] + part[3 * kM + tid])) *
                       (kSmooth ? smooth.symbol_scale : 1.f);
      lds_barrier();
    }
    float unigram[Shape::kTiles];
    if (kSmooth && smooth.am_scale != 0.f)
#pragma unroll
      for (int n = 0; n < Shape::kTiles; ++n)
        unigram[n] = get_float(buffer_of(smooth.unigram, C * 4), c0 + 32 * n < C, 4 * (c0 + 32 * n));
#pragma unroll
    for (int n = 0; n < Shape::kTiles; ++n) {
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int m = row_of(v);
        if (kSmooth && smooth.am_scale != 0.f) acc[n][v] += frame_w[m] * unigram[n];
        acc[n][v] *= __expf(in[n][v] - frame_mx[m]);
        if (c0 + 32 * n == term) acc[n][v] += frame_y[m];
      }
    }
    auto add_listed = [&] {
#pragma unroll
      for (int i = 0; i < kListed / 2; ++i) {
        if (column[2 * i] < 0) break;  // (uniform)
        const int mine = half ? column[2 * i + 1] : column[2 * i];
#pragma unroll
        for (int n = 0; n < Shape::kTiles; ++n) {
          const int at = Shape::kWaveC * (wave / Shape::kWavesM) + 32 * n;
          if ((unsigned)(column[2 * i] - at) >= 32u && (unsigned)(column[2 * i + 1] - at) >= 32u) continue;
          const float one = mine == at + r32 ? (kSmooth ? smooth.symbol_scale : 1.f) : 0.f;
          acc[n] = __builtin_amdgcn_mfma_f32_32x32x2f32(value[i], one, acc[n], 0, 0, 0);
        }
      }
    };
    add_listed();
    for (int s0 = 0; s0 < s_count; s0 += 2 * kWave) {
      if (s0 > 0) find_hits(s0);
      while (hits[0] | hits[1]) {  // (uniform)
        fetch_listed(s0);
        add_listed();
      }
    }
  }
  if (t_tile + m_wave + 32 > t_lim) {  // (uniform)
#pragma unroll
    for (int n = 0; n < Shape::kTiles; ++n)
#pragma unroll
      for (int v = 0; v < 16; ++v)
        acc[n][v] = t_tile + row_of(v) < t_lim ? acc[n][v] : 0.f;
  }
  with_store(out_type, [&](auto store) {
#pragma unroll
    for (int n = 0; n < Shape::kTiles; ++n)
#pragma unroll
      for (int v = 0; v < 16; ++v)
        store(out_rs, c0 + 32 * n < C, first + 32 * n, below(v), acc[n][v]);
  });
}

// launchers: float goes to the product kernels above, double to the LDS-tiled ones
void launch_fwd_gemm(const float *lm, const float *am, const int64_t *symbols,
                     const int64_t *boundary, float *lm_max, float *am_max, float *px,
                     float *py, float *norm_raw, const int64_t *window, double delay_penalty, int B, int S, int T, int C, int term, int rnnt_type,
                     const SmoothMix *mix, float *workspace, hipStream_t stream) {
  launch_normalizer_f32(lm, am, symbols, boundary, lm_max, am_max, px, py, norm_raw, window,
                        delay_penalty, B, S, T, C, term, rnnt_type, mix, workspace, stream);
}
void launch_fwd_gemm(const double *lm, const double *am, const int64_t *symbols,
                     const int64_t *boundary, const double *lm_max, const double *am_max,
                     double *px, double *py, double *norm_raw, const int64_t *, double delay_penalty, int B, int S, int T, int C, int term, int rnnt_type,
                     const SmoothMix *, float *, hipStream_t stream) {
  // (the double kernels compute the whole lattice whether or not a window is given)
  const int t_tiles = T > 0 ? (T + kTileN - 1) / kTileN : 1;
  const dim3 grid(t_tiles, (S + 1 + kTileM - 1) / kTileM, B);
  hipLaunchKernelGGL(simple_fwd_kernel<double>, grid, dim3(kGemmThreads), 0, stream, lm, am,
                     symbols, boundary, lm_max, am_max, px, py, norm_raw,
                     Delay<double>{delay_penalty}, S, T, C, term, rnnt_type);
}
// Both gradient products in one launch: the first lm_blocks workgroups take tiles of
// lm.grad, the rest tiles of am.grad.  The two only read what the prep kernel left, so
// their workgroups share the chip.  lm_blocks is a multiple of 8, so a workgroup's XCD is the same
// in both numberings.  (One after the other they take as long at the large sizes and 5 to 10 us
// longer where either leaves the chip partly idle.)
template <int kMl, int kMa, bool kSmooth>
__global__ void __launch_bounds__(kProdThreads, kProdPerCu)
    simple_bwd_am_lm_kernel(const float *__restrict__ lm, const float *__restrict__ am,
                            const int64_t *__restrict__ symbols,
                            const int64_t *__restrict__ boundary,
                            const float *__restrict__ lm_max, const float *__restrict__ am_max,
                            const float *__restrict__ dmat, const float *__restrict__ gpx,
                            const float *__restrict__ gpy, const float *__restrict__ row_x,
                            const float *__restrict__ row_y, void *__restrict__ lm_grad,
                            void *__restrict__ am_grad, const int64_t *__restrict__ window, int B,
                            int S, int T, int C, int ldd, int term, int rnnt_type,
                            Placement lm_at, Placement am_at, int out_type, SmoothTerms smooth) {
  int b, row_idx, c_idx;
  if (blockIdx.x < lm_at.blocks) {
    if (!place_block(blockIdx.x, lm_at, B, row_x, S, b, row_idx, c_idx)) return;
    simple_bwd_lm_body<kMl, kSmooth>(b, row_idx, c_idx, lm, am, symbols, lm_max, am_max, dmat,
                                         row_x, row_y, lm_grad, window, S, T, C, ldd, term,
                                         out_type, smooth);
  } else {
    if (!place_block(blockIdx.x - lm_at.blocks, am_at, B, row_x, S, b, row_idx, c_idx)) return;
    simple_bwd_am_body<kMa, kSmooth>(b, row_idx, c_idx, lm, am, symbols, boundary, lm_max, am_max,
                                         dmat, gpx, gpy, row_x, am_grad, window, S, T, C, ldd, term,
                                         rnnt_type, out_type, smooth);
  }
}
template <int kMl, int kMa, bool kSmooth>
void launch_bwd_t(const float *lm, const float *am, const int64_t *symbols,
                  const int64_t *boundary, const float *lm_max, const float *am_max,
                  const float *dmat, const float *gpx, const float *gpy, const float *row_x,
                  const float *row_y, void *lm_grad, void *am_grad, const int64_t *window, int B,
                  int S, int T, int C, int ldd, int term, int rnnt_type, int out_type,
                  const SmoothTerms &smooth, hipStream_t stream) {
  const int c_tiles = (C + kProdC - 1) / kProdC, shift = part_shift_for(B, c_tiles);
  const Placement lm_at(c_tiles, lm_grad ? (S + kMl) / kMl : 0, B, shift);
  const Placement am_at(c_tiles, am_grad && T > 0 ? (T + kMa - 1) / kMa : 0, B, shift);
  if (lm_at.blocks + am_at.blocks == 0) return;
  hipLaunchKernelGGL((simple_bwd_am_lm_kernel<kMl, kMa, kSmooth>), dim3(lm_at.blocks + am_at.blocks),
                     dim3(kProdThreads), 2 * kImageBytes, stream, lm, am, symbols, boundary, lm_max, am_max,
                     dmat, gpx, gpy, row_x, row_y, lm_grad, am_grad, window, B, S, T, C, ldd,
                     term, rnnt_type, lm_at, am_at, out_type, smooth);
}
// Rows of a workgroup's tile, each product's by its own.  128 rows read and convert the operand
// along the vocabulary half as often as 64 (both products at B 64, S 120, T 600, C 500: 74 against 90
// us; B 16, S 120, T 400, C 5000: 108 against 132), which is what counts once the chip is full; they
// lose where the padding of the last tile outweighs that (lm.grad's up to 64 rows: 20 against 17 us at
// B 21, S 47, T 333, C 503) or where fewer of them than fill the chip remain.
bool wide_tile(long columns_of_tiles, int rows) {
  const long wide = (rows + 127) / 128, narrow = (rows + 63) / 64;
  return narrow > 1 && 14 * wide <= 8 * narrow && columns_of_tiles * wide >= kMinWideTiles;
}
template <bool kSmooth>
void launch_bwd_f32(const float *lm, const float *am, const int64_t *symbols,
                    const int64_t *boundary, const float *lm_max, const float *am_max,
                    const float *dmat, const float *gpx, const float *gpy, const float *row_x,
                    const float *row_y, void *lm_grad, void *am_grad, const int64_t *window, int B,
                    int S, int T, int C, int ldd, int term, int rnnt_type, int out_type,
                    const SmoothTerms &smooth, hipStream_t stream) {
  // Where lm, am and their gradients together outgrow the last-level cache (256 MB) the gradients
  // are streamed past it, which leaves it to lm and am: these are read by both products.  Whole pass
  // of the loss, with the hint against without: C 5000, S 120, T 400: B 14, 278 MB: 291 / 299 us;
  // B 24, 476 MB: 452 / 476; B 64, S 120, T 600, C 1000, 352 MB: 424 / 444; C 500, B 128, 352 MB:
  // 545 / 547; B 8, S 200, T 1000, C 5000, 366 MB: 558 / 589.  Below, either way: B 10, C 5000,
  // 198 MB: 267 / 263; B 32, S 60, T 300, C 2500, 220 MB: 188 / 188; B 45, C 1000, 247 MB: 320 / 327.
  if (out_type == FRNNT_F32 && 8L * B * (S + 1 + T) * C > (256L << 20)) out_type = kStreamed;
  const long columns = (long)B * ((C + kProdC - 1) / kProdC);
  const bool wide_l = wide_tile(columns, S + 1), wide_a = wide_tile(columns, T);
  auto launch = wide_l ? wide_a ? launch_bwd_t<128, 128, kSmooth> : launch_bwd_t<128, 64, kSmooth>
                       : wide_a ? launch_bwd_t<64, 128, kSmooth> : launch_bwd_t<64, 64, kSmooth>;
  launch(lm, am, symbols, boundary, lm_max, am_max, dmat, gpx, gpy, row_x, row_y, lm_grad, am_grad,
         window, B, S, T, C, ldd, term, rnnt_type, out_type, smooth, stream);
}
void launch_bwd(const float *lm, const float *am, const int64_t *symbols, const int64_t *boundary,
                const float *lm_max, const float *am_max, const float *dmat, const float *gpx,
                const float *gpy, const float *row_x, const float *row_y, const float *, void *lm_grad,
                void *am_grad, const int64_t *window, int B, int S, int T, int C, int ldd, int term,
                int rnnt_type, int out_type, const SmoothTerms *smooth, hipStream_t stream) {
  if (smooth)
    launch_bwd_f32<true>(lm, am, symbols, boundary, lm_max, am_max, dmat, gpx, gpy, row_x, row_y,
                         lm_grad, am_grad, window, B, S, T, C, ldd, term, rnnt_type, out_type,
                         *smooth, stream);
  else
    launch_bwd_f32<false>(lm, am, symbols, boundary, lm_max, am_max, dmat, gpx, gpy, row_x, row_y,
                          lm_grad, am_grad, window, B, S, T, C, ldd, term, rnnt_type, out_type, {},
                          stream);
}
void launch_bwd(const double *lm, const double *am, const int64_t *symbols,
                const int64_t *boundary, const double *lm_max, const double *am_max,
                const double *dmat, const double *gpx, const double *, const double *row_x,
                const double *row_y, const double *col_y, void *lm_grad_, void *am_grad_,
                const int64_t *, int B, int S, int T, int C, int ldd, int term, int rnnt_type, int,
                const SmoothTerms *, hipStream_t stream) {
  double *lm_grad = static_cast<double *>(lm_grad_), *am_grad = static_cast<double *>(am_grad_);
  const unsigned c_tiles = (C + kTileN - 1) / kTileN;
  if (lm_grad)
    hipLaunchKernelGGL(simple_bwd_lm_kernel<double>, dim3(c_tiles, (S + 1 + kTileM - 1) / kTileM, B),
                       dim3(kGemmThreads), 0, stream, lm, am, symbols, lm_max, am_max, dmat, row_x,
                       row_y, lm_grad, S, T, C, ldd, term);
  if (!am_grad || T <= 0) return;
  hipLaunchKernelGGL(simple_bwd_am_kernel<double>, dim3(c_tiles, (T + kTileM - 1) / kTileM, B),
                     dim3(kGemmThreads), 0, stream, lm, am, lm_max, am_max, dmat, col_y, am_grad, S,
                     T, C, ldd, term);
  if (S > 0) {  // the double path keeps the separate per-symbol scatter
    const long n = (long)B * T;
    hipLaunchKernelGGL(simple_bwd_symbols_kernel<double>, dim3((unsigned)((n + 255) / 256)),
                       dim3(256), 0, stream, gpx, symbols, boundary, am_grad, B, S, T, C,
                       rnnt_type);
  }
}

template <typename R>
void launch_scale(R *px_grad, R *py_grad, const R *score_grad, int score_grad_stride,
                  double score_grad_scale, int B, int S, int T, int modified, hipStream_t stream) {
  const int per_x = S * (modified ? T : T + 1), per_y = (S + 1) * T;
  const int x_blocks = (per_x + 1023) / 1024, y_blocks = (per_y + 1023) / 1024;
  if (x_blocks + y_blocks > 0)
    hipLaunchKernelGGL(scale_by_batch_kernel<R>, dim3(x_blocks + y_blocks, B), dim3(256), 0, stream,
                       px_grad, py_grad, score_grad, score_grad_stride, (R)score_grad_scale, per_x,
                       per_y, x_blocks);
}

template <typename R>
int fwd_impl(const R *lm, const R *am, const int64_t *symbols, const int64_t *boundary, R *px,
             R *py, R *lm_max, R *am_max, R *norm_raw, double delay_penalty, int B,
             int S, int T, int C, int term, int rnnt_type, int window_only, void *stream_,
             const SmoothMix *mix = nullptr, float *workspace = nullptr) {
  if (B < 0 || S < 0 || T < 0 || C < 1) return fail(FRNNT_EINVAL, "simple_logprobs_fwd: bad size");
  if (rnnt_type < 0 || rnnt_type > 2)
    return fail(FRNNT_EINVAL, "simple_logprobs_fwd: rnnt_type must be 0, 1 or 2");
  if (term < 0 || term >= C)
    return fail(FRNNT_EINVAL, "simple_logprobs_fwd: termination symbol outside [0, C)");
  if (B == 0) return FRNNT_OK;
  if (!lm || !am || (!symbols && S > 0) || !px || !py || !lm_max || !am_max)
    return fail(FRNNT_EINVAL, "simple_logprobs_fwd: null pointer");
  // (the float32 kernel addresses an utterance's lm / am rows by 32-bit byte offsets)
  if (std::is_same<R, float>::value &&
      ((long)(S + 1) * C * 4 >= (1L << 31) || (long)T * C * 4 >= (1L << 31)))
    return fail(FRNNT_ELIMIT, "simple_logprobs_fwd: one utterance's lm or am exceeds 2 GiB");
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  const long n_lm = (long)B * (S + 1), n_am = (long)B * T;
  const long rows = n_lm + n_am;
  // (the fp32 GEMM kernel finds the row maxima itself)
  if (!std::is_same<R, float>::value)
    hipLaunchKernelGGL(row_max_kernel<R>, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, stream,
                       lm, am, lm_max, am_max, n_lm, n_am, C);
  // (the grid always has at least one column of tiles, so that the -inf column of
  // an empty-frame regular lattice is still written)
  const bool constrained = rnnt_type == kConstrained;
  launch_fwd_gemm(lm, am, symbols, boundary, lm_max, am_max, px, py, norm_raw,
                  window_only ? boundary : nullptr, constrained ? 0.0 : delay_penalty, B,
                  S, T, C, term, rnnt_type, mix, workspace, stream);
  if (constrained && S > 0 && T > 0) {
    const long total = (long)B * S * T;
    hipLaunchKernelGGL(add_next_row_kernel<R>, dim3((unsigned)((total + 255) / 256)), dim3(256), 0,
                       stream, px, py, boundary, Delay<R>{(R)delay_penalty}, total, S, T);
  }
  return check_launch("simple_logprobs_fwd");
}

template <typename R>
int bwd_impl(const R *lm, const R *am, const int64_t *symbols, const int64_t *boundary,
             const R *lm_max, const R *am_max, const R *norm_raw, const R *score_grad,
             int score_grad_stride, double score_grad_scale, R *px_grad, R *py_grad, R *dmat,
             R *row_x, R *row_y, R *col_y, void *lm_grad, void *am_grad, int B, int S, int T, int C,
             int term, int rnnt_type, int window_only, int out_type, void *stream_,
             const SmoothTerms *smooth = nullptr, const std::function<void()> *between = nullptr) {
  constexpr bool is_float = std::is_same<R, float>::value;
  if (B < 0 || S < 0 || T < 0 || C < 1) return fail(FRNNT_EINVAL, "simple_logprobs_bwd: bad size");
  if (rnnt_type < 0 || rnnt_type > 2 || term < 0 || term >= C)
    return fail(FRNNT_EINVAL, "simple_logprobs_bwd: bad rnnt_type or termination symbol");
  if (B == 0) return FRNNT_OK;
  if (!lm || !am || (!symbols && S > 0) || !lm_max || !am_max || !norm_raw || !px_grad ||
      !py_grad || !dmat || !row_x || !row_y || (!is_float && !col_y))
    return fail(FRNNT_EINVAL, "simple_logprobs_bwd: null pointer");
  // (the float32 kernels address an utterance's lm / am / D rows by 32-bit byte offsets)
  if (std::is_same<R, float>::value &&
      ((long)(S + 1) * C * 4 >= (1L << 31) || (long)T * C * 4 >= (1L << 31) ||
       (long)(S + 1) * (T + 3) * 4 >= (1L << 31)))
    return fail(FRNNT_ELIMIT, "simple_logprobs_bwd: one utterance's lm, am or lattice exceeds 2 GiB");
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  if (score_grad && score_grad_stride != 0 && score_grad_stride != 1)
    return fail(FRNNT_EINVAL, "simple_logprobs_bwd: score_grad_stride must be 0 or 1");
  // The occupation gradients are scaled as they are read, except where other workgroups than
  // the one that scales a row read it: the row above's in the constrained lattice, the
  // columns in double.  (B 64, S 120, T 600: 20 us instead of 30 in two launches.)
  const bool fused = is_float && rnnt_type != kConstrained;
  if (score_grad && !fused) {
    launch_scale(px_grad, py_grad, score_grad, score_grad_stride, score_grad_scale, B, S, T,
                 rnnt_type != kRegular, stream);
    score_grad = nullptr;
  }
  const int ldd = (T + 3) & ~3;  // leading dimension of dmat: 16-byte rows
  // (the double kernels ignore the window: they take the whole lattice as it is)
  const int64_t *window = (window_only && is_float) ? boundary : nullptr;
  const long prep_blocks = ((long)B * (S + 1) + 3) / 4 + 1 +
                           (is_float ? 0 : (long)B * ((T + kWave - 1) / kWave));
  hipLaunchKernelGGL(simple_bwd_prep_kernel<R>, dim3((unsigned)prep_blocks), dim3(256), 0, stream,
                     px_grad, py_grad, norm_raw, boundary, window, score_grad, score_grad_stride,
                     (R)score_grad_scale, smooth ? (R)smooth->joint : (R)1, dmat, row_x, row_y, col_y, B,
                     S, T, ldd, rnnt_type);
  if (between) (*between)();
  launch_bwd(lm, am, symbols, boundary, lm_max, am_max, dmat, px_grad, py_grad, row_x, row_y, col_y,
             lm_grad, am_grad, window, B, S, T, C, ldd, term, rnnt_type, out_type, smooth, stream);
  return check_launch("simple_logprobs_bwd");
}

// px_grad[b] and py_grad[b] times score_grad_scale * score_grad[b * stride], in place: the
// scaling step of the recursion's autograd backward (mutual_information.py:173-181).
template <typename R>
int scale_grads_impl(R *px_grad, R *py_grad, const R *score_grad, int score_grad_stride,
                     double score_grad_scale, int B, int S, int T, int modified, void *stream) {
  if (B < 0 || S < 0 || T < 0) return fail(FRNNT_EINVAL, "mi_scale_grads: negative size");
  if (score_grad_stride != 0 && score_grad_stride != 1)
    return fail(FRNNT_EINVAL, "mi_scale_grads: score_grad_stride must be 0 or 1");
  if (B == 0) return FRNNT_OK;
  if (!px_grad || !py_grad || !score_grad)
    return fail(FRNNT_EINVAL, "mi_scale_grads: null pointer");
  launch_scale(px_grad, py_grad, score_grad, score_grad_stride, score_grad_scale, B, S, T, modified,
               static_cast<hipStream_t>(stream));
  return check_launch("mi_scale_grads");
}

template <typename R>
int reduce_impl(const R *scores, R *loss, int B, int reduction, void *stream) {
  if (B < 0 || reduction < 0 || reduction > 2)
    return fail(FRNNT_EINVAL, "loss_reduce: bad size or reduction");
  if (!loss || (B > 0 && !scores)) return fail(FRNNT_EINVAL, "loss_reduce: null pointer");
  if (B == 0 && reduction == 0) return FRNNT_OK;
  hipLaunchKernelGGL(loss_reduce_kernel<R>, dim3(1), dim3(kWave), 0,
                     static_cast<hipStream_t>(stream), scores, loss, B, reduction);
  return check_launch("loss_reduce");
}

// 2-byte inputs as float32: a thread takes four groups of four elements, a workgroup's groups side by
// side, in 8-byte loads where the input is aligned to them and 16-byte stores (the output always
// is).  Bound by memory.
constexpr int kWidenBlock = 4 * 4 * 256;  // elements
template <typename IO>
__global__ void __launch_bounds__(256)
    widen_kernel(const uint16_t *__restrict__ lm, const uint16_t *__restrict__ am,
                 float *__restrict__ lm_wide, float *__restrict__ am_wide, long n_lm, long n_am,
                 unsigned lm_blocks) {
  const bool is_lm = blockIdx.x < lm_blocks;
  const uint16_t *from = is_lm ? lm : am;
  float *to = is_lm ? lm_wide : am_wide;
  const long n = is_lm ? n_lm : n_am;
  const long first = (long)(is_lm ? blockIdx.x : blockIdx.x - lm_blocks) * kWidenBlock;
  const long at = first + 4 * threadIdx.x;
  if ((reinterpret_cast<uintptr_t>(from) & 7) == 0 && first + kWidenBlock <= n) {
    uintx2 raw[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) raw[u] = *reinterpret_cast<const uintx2 *>(from + at + 1024 * u);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      dgemm::floatx4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = IO::load((uint16_t)(raw[u][i / 2] >> (16 * (i % 2))));
      *reinterpret_cast<dgemm::floatx4 *>(to + at + 1024 * u) = v;
    }
  } else {
    for (int u = 0; u < 4; ++u)
      for (int i = 0; i < 4; ++i)
        if (at + 1024 * u + i < n) to[at + 1024 * u + i] = IO::load(from[at + 1024 * u + i]);
  }
}

// ---- scratch that the library owns: for callers that cannot allocate --------------------
// One array per GPU, part of the code object, held until the process ends.  In host code
// the array's name is only a handle: its device address is looked up once per device
// (with that device current) and kept; kernels and everything else get that address.
constexpr size_t kOwnScratchFloats = (size_t)4 << 20;  // 16 MiB
static __device__ __align__(256) float own_scratch[kOwnScratchFloats];
constexpr int kMaxDevices = 64;

float *own_scratch_address() {
  static std::mutex guard;
  static float *address[kMaxDevices] = {nullptr};
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lock(guard);
  if (!address[device]) {
    void *found = nullptr;
    if (hipGetSymbolAddress(&found, HIP_SYMBOL(own_scratch)) != hipSuccess) {
      (void)hipGetLastError();
      return nullptr;
    }
    address[device] = static_cast<float *>(found);
  }
  return address[device];
}

}  // namespace

int simple_logprobs_fwd(const float *lm, const float *am, const int64_t *symbols,
                        const int64_t *boundary, float *px, float *py, float *lm_max,
                        float *am_max, float *norm_raw, double delay_penalty, int B, int S, int T, int C, int term, int rnnt_type, int window_only,
                        void *stream, const SmoothMix *mix, float *workspace) {
  return fwd_impl<float>(lm, am, symbols, boundary, px, py, lm_max, am_max, norm_raw,
                         delay_penalty, B, S, T, C, term, rnnt_type, window_only, stream, mix, workspace);
}
int simple_logprobs_fwd(const double *lm, const double *am, const int64_t *symbols,
                        const int64_t *boundary, double *px, double *py, double *lm_max,
                        double *am_max, double *norm_raw, double delay_penalty, int B, int S, int T, int C, int term, int rnnt_type, int window_only,
                        void *stream) {
  return fwd_impl<double>(lm, am, symbols, boundary, px, py, lm_max, am_max, norm_raw,
                          delay_penalty, B, S, T, C, term, rnnt_type, window_only, stream);
}
int simple_logprobs_bwd_smoothed(const float *lm, const float *am, const int64_t *symbols,
                                 const int64_t *boundary, const float *lm_max, const float *am_max,
                                 const float *norm_raw, const float *score_grad,
                                 int score_grad_stride, double score_grad_scale, float *px_grad,
                                 float *py_grad, float *dmat, float *row_x, float *row_y,
                                 const SmoothTerms &smooth, const std::function<void()> &between,
                                 float *lm_grad, float *am_grad, int B, int S, int T, int C, int term,
                                 int rnnt_type, void *stream) {
  return bwd_impl<float>(lm, am, symbols, boundary, lm_max, am_max, norm_raw, score_grad,
                         score_grad_stride, score_grad_scale, px_grad, py_grad, dmat, row_x, row_y,
                         nullptr, lm_grad, am_grad, B, S, T, C, term, rnnt_type, boundary != nullptr,
                         FRNNT_F32, stream, &smooth, &between);
}
void widen_inputs(int dtype, const void *lm, const void *am, float *lm_wide, float *am_wide,
                  long n_lm, long n_am, hipStream_t stream) {
  const unsigned lm_blocks = (unsigned)((n_lm + kWidenBlock - 1) / kWidenBlock);
  const unsigned am_blocks = (unsigned)((n_am + kWidenBlock - 1) / kWidenBlock);
  if (lm_blocks + am_blocks == 0) return;
  hipLaunchKernelGGL((dtype == FRNNT_F16 ? widen_kernel<HalfIO> : widen_kernel<Bf16IO>),
                     dim3(lm_blocks + am_blocks), dim3(256), 0, stream,
                     static_cast<const uint16_t *>(lm), static_cast<const uint16_t *>(am), lm_wide,
                     am_wide, n_lm, n_am, lm_blocks);
}

}  // namespace frnnt

extern "C" {

int frnnt_additive_loss_bwd(int dtype, const void *lm, const void *am, const int64_t *symbols,
                            const int64_t *boundary, const void *lm_max, const void *am_max,
                            const void *norm_raw, const void *score_grad, int score_grad_stride,
                            double score_grad_scale, void *px_grad, void *py_grad, void *dmat,
                            void *row_x, void *row_y, void *col_y, void *lm_grad, void *am_grad,
                            int B, int S, int T, int C, int termination_symbol, int rnnt_type,
                            void *stream) {
  if (dtype < FRNNT_F32 || dtype > FRNNT_BF16)
    return frnnt::fail(FRNNT_EINVAL, "additive_loss_bwd: unknown dtype");
  auto call = [&](auto r) {
    using R = decltype(r);
    auto in = [](const void *p) { return static_cast<const R *>(p); };
    auto out = [](void *p) { return static_cast<R *>(p); };
    return frnnt::bwd_impl<R>(in(lm), in(am), symbols, boundary, in(lm_max), in(am_max),
                              in(norm_raw), in(score_grad), score_grad_stride, score_grad_scale,
                              out(px_grad), out(py_grad), out(dmat), out(row_x), out(row_y),
                              out(col_y), lm_grad, am_grad, B, S, T, C, termination_symbol,
                              rnnt_type, boundary != nullptr, dtype, stream);
  };
  return dtype == FRNNT_F64 ? call(double()) : call(float());
}

int frnnt_simple_logprobs_bwd_noalloc_f32(const float *lm, const float *am, const int64_t *symbols,
                                          const int64_t *boundary, const float *lm_max,
                                          const float *am_max, const float *norm_raw,
                                          const float *score_grad, int score_grad_stride,
                                          double score_grad_scale, float *px_grad,
                                          float *py_grad, float *lm_grad, float *am_grad, int B,
                                          int S, int T, int C, int termination_symbol,
                                          int rnnt_type, int window_only, void *stream) {
  using frnnt::fail;
  if (B < 0 || S < 0 || T < 0) return fail(FRNNT_EINVAL, "simple_logprobs_bwd_noalloc: bad size");
  // dmat | row_x | row_y | col_y, each starting 16-byte aligned
  const size_t ldd = ((size_t)T + 3) & ~(size_t)3;
  const size_t n_rows = ((size_t)B * (S + 1) + 3) & ~(size_t)3;
  const size_t n_cols = ((size_t)B * T + 3) & ~(size_t)3;
  const size_t n_dmat = (size_t)B * (S + 1) * ldd;
  const size_t need = n_dmat + 2 * n_rows + n_cols;
  if (need > frnnt::kOwnScratchFloats)
    return fail(FRNNT_ELIMIT,
                "simple_logprobs_bwd_noalloc: B=%d S=%d T=%d needs %zu bytes of scratch, the "
                "library's own buffer holds %zu; use frnnt_simple_logprobs_bwd_f32 with a "
                "caller-provided workspace",
                B, S, T, need * sizeof(float), frnnt::kOwnScratchFloats * sizeof(float));
  // the array is the current device's copy: the buffers must live on that device
  if (px_grad) {
    hipPointerAttribute_t where;
    int current = -1;
    if (hipPointerGetAttributes(&where, px_grad) != hipSuccess) {
      (void)hipGetLastError();
      return fail(FRNNT_EINVAL, "simple_logprobs_bwd_noalloc: px_grad is not a device pointer");
    }
    if (hipGetDevice(&current) != hipSuccess || where.device != current)
      return fail(FRNNT_EINVAL,
                  "simple_logprobs_bwd_noalloc: the buffers live on device %d but device %d is "
                  "current; make the buffers' device current before the call",
                  where.device, current);
  }
  float *base = frnnt::own_scratch_address();
  if (!base) return fail(FRNNT_ELAUNCH, "simple_logprobs_bwd_noalloc: hipGetSymbolAddress failed");
  float *dmat = base, *row_x = dmat + n_dmat, *row_y = row_x + n_rows, *col_y = row_y + n_rows;
  return frnnt::bwd_impl<float>(lm, am, symbols, boundary, lm_max, am_max, norm_raw, score_grad,
                                score_grad_stride, score_grad_scale, px_grad, py_grad, dmat, row_x,
                                row_y, col_y, lm_grad, am_grad, B, S, T, C, termination_symbol,
                                rnnt_type, window_only, FRNNT_F32, stream);
}

int64_t frnnt_loss_scratch(int B, int S, int T, int C, int has_boundary) {
  if (B < 1 || S < 0 || T < 0 || C < 1) return 0;
  const long lattice = (long)B * (S + 1) * (T + 1);
  const long work = frnnt::normalizer_workspace(B, S, T, C, has_boundary != 0);
  return lattice > work ? lattice : work;
}

int frnnt_simple_logprobs_fwd_f32(const float *lm, const float *am, const int64_t *symbols,
                                  const int64_t *boundary, float *px, float *py, float *lm_max,
                                  float *am_max, float *norm_raw, int B, int S, int T, int C,
                                  int termination_symbol, int rnnt_type, int window_only,
                                  void *stream) {
  return frnnt::fwd_impl<float>(lm, am, symbols, boundary, px, py, lm_max, am_max, norm_raw,
                                0.0, B, S, T, C, termination_symbol, rnnt_type,
                                window_only, stream);
}
int frnnt_simple_logprobs_fwd_f64(const double *lm, const double *am, const int64_t *symbols,
                                  const int64_t *boundary, double *px, double *py, double *lm_max,
                                  double *am_max, double *norm_raw, int B, int S, int T, int C,
                                  int termination_symbol, int rnnt_type, int window_only,
                                  void *stream) {
  return frnnt::fwd_impl<double>(lm, am, symbols, boundary, px, py, lm_max, am_max, norm_raw,
                                 0.0, B, S, T, C, termination_symbol, rnnt_type,
                                 window_only, stream);
}
int frnnt_simple_logprobs_bwd_f32(const float *lm, const float *am, const int64_t *symbols,
                                  const int64_t *boundary, const float *lm_max,
                                  const float *am_max, const float *norm_raw,
                                  const float *score_grad, int score_grad_stride,
                                  double score_grad_scale, float *px_grad, float *py_grad,
                                  float *dmat, float *row_x, float *row_y, float *col_y,
                                  float *lm_grad, float *am_grad, int B, int S, int T, int C,
                                  int termination_symbol, int rnnt_type, int window_only,
                                  void *stream) {
  return frnnt::bwd_impl<float>(lm, am, symbols, boundary, lm_max, am_max, norm_raw, score_grad,
                                score_grad_stride, score_grad_scale, px_grad, py_grad, dmat, row_x,
                                row_y, col_y, lm_grad, am_grad, B, S, T, C, termination_symbol,
                                rnnt_type, window_only, FRNNT_F32, stream);
}
int frnnt_simple_logprobs_bwd_f64(const double *lm, const double *am, const int64_t *symbols,
                                  const int64_t *boundary, const double *lm_max,
                                  const double *am_max, const double *norm_raw,
                                  const double *score_grad, int score_grad_stride,
                                  double score_grad_scale, double *px_grad, double *py_grad,
                                  double *dmat, double *row_x, double *row_y, double *col_y,
                                  double *lm_grad, double *am_grad, int B, int S, int T, int C,
                                  int termination_symbol, int rnnt_type, int window_only,
                                  void *stream) {
  return frnnt::bwd_impl<double>(lm, am, symbols, boundary, lm_max, am_max, norm_raw, score_grad,
                                 score_grad_stride, score_grad_scale, px_grad, py_grad, dmat,
                                 row_x, row_y, col_y, lm_grad, am_grad, B, S, T, C,
                                 termination_symbol, rnnt_type, window_only, FRNNT_F32, stream);
}

int frnnt_mi_scale_grads_f32(float *px_grad, float *py_grad, const float *score_grad,
                             int score_grad_stride, double score_grad_scale, int B, int S, int T,
                             int modified, void *stream) {
  return frnnt::scale_grads_impl<float>(px_grad, py_grad, score_grad, score_grad_stride,
                                        score_grad_scale, B, S, T, modified, stream);
}
int frnnt_mi_scale_grads_f64(double *px_grad, double *py_grad, const double *score_grad,
                             int score_grad_stride, double score_grad_scale, int B, int S, int T,
                             int modified, void *stream) {
  return frnnt::scale_grads_impl<double>(px_grad, py_grad, score_grad, score_grad_stride,
                                         score_grad_scale, B, S, T, modified, stream);
}
int frnnt_loss_reduce_f32(const float *scores, float *loss, int B, int reduction, void *stream) {
  return frnnt::reduce_impl<float>(scores, loss, B, reduction, stream);
}
int frnnt_loss_reduce_f64(const double *scores, double *loss, int B, int reduction, void *stream) {
  return frnnt::reduce_impl<double>(scores, loss, B, reduction, stream);
}

}  // extern "C"

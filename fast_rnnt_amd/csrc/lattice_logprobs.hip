// px / py from joiner logits: the unpruned loss (logits [B][T][S+1][C],
// fast_rnnt/python/fast_rnnt/rnnt_loss.py:343-449) and the pruned loss
// (logits [B][T][R][C] plus ranges [B][T][R], rnnt_loss.py:856-1024) share one
// set of kernels; the unpruned case is R = S+1 with every range starting at 0.
//
// Forward, HBM-streaming: the logits are read once, a wave (or a part of one, for short rows)
// per logits row (b, t, j), which forms norm = logsumexp and the two picked log-probs
//   x = logits[b,t,j,sym(b, ranges[b,t,j])] - norm   (sym(b, S) = termination symbol)
//   y = logits[b,t,j,term] - norm.
// Without the constrained step every cell of px / py comes from one row, which writes it: row j of
// frame t lands at lattice row (j + ranges[b,t,0]) mod (S+1).  The cells around the rows' --
// everything else is -inf, and the -inf columns of the regular lattice -- are written by
// workgroups of their own in the same launch.  The constrained "px += py[:, 1:]" step needs two rows
// in one cell: there (and in float64) the picks go to xr / yr and a second, small kernel lays
// them out.  (The backward: lattice_gradient.hip.)
#include "lattice_rows.hip.h"

namespace frnnt {
namespace {

// Where a row's results go: norm always; the picks to px / py at once (direct) or to xr / yr.
template <typename R>
struct Picks {
  R *norm, *xr, *yr, *px, *py;
  Delay<R> delay;
  bool direct;
  int *arrived;  // (may be NULL) to be 0, and *loss NaN, when the recursion starts (LossOf)
  R *loss;
  __device__ __forceinline__ void start() const {
    if (arrived && (blockIdx.x | blockIdx.y | blockIdx.z | threadIdx.x) == 0) {
      *arrived = 0;
      *loss = std::numeric_limits<R>::quiet_NaN();
    }
  }
  // the cell (s, t_end) of the regular lattice, and its last column: no symbol is emitted there
  // (rnnt_loss.py:45-63)
  __device__ __forceinline__ void close(const Lattice &L, int b, int s, int t) const {
    if (s < L.S) px[((long)b * L.S + s) * (L.T + 1) + t] = Num<R>::neg_inf();
  }
  __device__ __forceinline__ void write(const Lattice &L, const Row &row, R lse, R x, R y) const {
    norm[row.index] = lse;
    if (!direct) {
      xr[row.index] = x;
      yr[row.index] = y;
      return;
    }
    py[((long)row.b * (L.S + 1) + row.s) * L.T + row.t] = y;
    if (row.s == L.S) return;
    const bool regular = L.rnnt_type == kRegular;
    const int T1 = regular ? L.T + 1 : L.T;
    const long t_end = regular && L.boundary ? (long)L.boundary[4 * row.b + 3] : L.T;
    R *cell = px + ((long)row.b * L.S + row.s) * T1 + row.t;
    *cell = row.t == t_end ? Num<R>::neg_inf() : delay.at(x, L.boundary, row.b, row.t, L.T);
    if (regular && (row.t + 1 == t_end || row.t + 1 == L.T)) cell[1] = Num<R>::neg_inf();
  }
  // A window without frames has no live row, but the recursion looks at its column t_end.
  __device__ __forceinline__ void skip(const Lattice &L, const Row &row) const {
    if (!direct || L.rnnt_type != kRegular || !L.window || row.t >= L.T) return;
    const int64_t *w = L.window + 4 * row.b;
    if (w[1] != w[3]) return;
    if (row.t == w[3] || row.t + 1 == w[3]) close(L, row.b, row.s, (int)w[3]);
  }
};

// any element type, any row length: lanes stride over the row (float64, and vocabularies beyond 32-bit
// offsets)
template <typename P, typename R = typename AccumOf<P>::type>
__global__ void __launch_bounds__(256)
    row_norm_plain_kernel(const typename P::Elem *__restrict__ logits, Lattice L, Picks<R> out) {
  const int b = block_batch();
  const unsigned r = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (b >= L.B) return;
  const Row row = locate(L, b, r);
  if (!row.live) {
    if (lane == 0) out.skip(L, row);
    return;
  }
  const typename P::Elem *x = logits + row.index * L.C;
  R m = Num<R>::neg_inf();
  for (int c = lane; c < L.C; c += kWave) {
    const R v = P::load(x[c]);
    m = (v > m || v != v) ? v : m;
  }
  m = group_max(m, 64);
  const R shift = (m - m == 0) ? m : (R)0;  // torch.logsumexp: infinite max -> shift by 0
  R sum = 0;
  for (int c = lane; c < L.C; c += kWave) sum += exp_acc<R>(P::load(x[c]) - shift);
  sum = group_sum(sum, 64);
  const R lse = log_acc<R>(sum) + shift;
  if (lane == 0) {
    const int sym = row_symbol(L, row);
    out.write(L, row, lse, sym >= 0 ? P::load(x[sym]) - lse : std::numeric_limits<R>::quiet_NaN(),
              P::load(x[L.term]) - lse);
  }
}

// entry c of a row whose pieces one wave holds (c is wave-uniform and inside the row)
template <typename P, int kVecs>
__device__ __forceinline__ float row_entry(const intx4 (&raw)[kVecs], int off, int c) {
  const int piece = (c + off) / P::kPer, e = (c + off) % P::kPer;
  const int vec = piece / kWave, owner = piece % kWave;
  constexpr int kPerWord = P::kPer / 4;
  int cand = raw[0][0];
#pragma unroll
  for (int i = 0; i < kVecs; ++i)
#pragma unroll
    for (int w = 0; w < 4; ++w) cand = (i == vec && w == e / kPerWord) ? raw[i][w] : cand;
  const int word = __builtin_amdgcn_readlane(cand, owner);
  return P::at(intx4{word, word, word, word}, e % kPerWord);
}

// The cells of px / py that no row of the logits is placed at: tiles of 64 columns x 32 lattice rows
// like assemble_kernel's, lanes along t, the first `blocks` of an utterance's workgroups.  They write
// nothing that a row writes, but for the -inf of closed columns, so that neither waits for the
// other.  (With a launch of its own after the rows', which laid out what they had left in xr / yr,
// B 32, S 80, T 250, C 500, five rows a frame, took 20.2 + 5.7 us, now 24.0; B 8, S 200, T 1200, C 400,
// eight rows: 38.4 + 13.2, now 42.3.)
constexpr int kAssembleRows = 32;
struct Surround {
  unsigned blocks;
  int t_tiles;
  __device__ __forceinline__ void fill(const Lattice &L, int b, unsigned block, float *px,
                                       float *py) const {
    const bool regular = L.rnnt_type == kRegular;
    const int T1 = regular ? L.T + 1 : L.T, S1 = L.S + 1;
    const int t = (int)(block % t_tiles) * 64 + (threadIdx.x & 63);
    const int s0 = (int)(block / t_tiles) * kAssembleRows + (threadIdx.x >> 6);
    if (L.window) {
      const int64_t *w = L.window + 4 * b;
      if ((t & ~63) > w[3] || (t | 63) < w[1] || (s0 & ~3) > w[2] || (s0 & ~3) + kAssembleRows <= w[0])
        return;
    }
    const int r0 = placed_at(L.ranges[((long)b * L.T + min(t, L.T - 1)) * L.Rr], 0, L.S);
    const bool closed = regular && L.boundary && L.boundary[4 * b + 3] == t;
    float *px_b = px + (long)b * L.S * T1, *py_b = py + (long)b * S1 * L.T;
#pragma unroll
    for (int k = 0; k < kAssembleRows / 4; ++k) {
      const int s = s0 + 4 * k, rel = s - r0 < 0 ? s - r0 + S1 : s - r0;
      const bool placed = rel < L.Rr && t < L.T;
      if (s < L.S && t < T1 && (!placed || closed)) px_b[(long)s * T1 + t] = Num<float>::neg_inf();
      if (s < S1 && t < L.T && !placed) py_b[(long)s * L.T + t] = Num<float>::neg_inf();
    }
  }
};

// What of a row's pieces (the vectors from piece p0 on) is a neighbour's becomes -inf (whole pieces of a whole
// wave need no test; kAligned: no piece is shared); the largest entry of a lane's pieces, without the NaNs, which
// come back through the sum.
template <typename P, int kLanes, int kVecs, bool kAligned = false>
__device__ __forceinline__ float largest_of_lane(intx4 (&raw)[kVecs], const RowPieces<P, kLanes> &q, int p0,
                                                 int lane, int C) {
#pragma unroll
  for (int i = 0; i < kVecs; ++i) {
    const int first_piece = p0 + kLanes * i;
    if (kLanes == kWave && first_piece + kLanes <= q.whole && (first_piece > 0 || q.off == 0)) continue;
    if (kAligned) {
      intx4 none = {};
#pragma unroll
      for (int e = 0; e < P::kPer; ++e) P::drop(none, e);
      raw[i] = first_piece + lane < q.pieces ? raw[i] : none;
      continue;
    }
#pragma unroll
    for (int e = 0; e < P::kPer; ++e)
      if ((unsigned)((first_piece + lane) * P::kPer + e - q.off) >= (unsigned)C) P::drop(raw[i], e);
  }
  float here = -__builtin_huge_valf();
#pragma unroll
  for (int i = 0; i < kVecs; ++i)
#pragma unroll
    for (int e = 0; e < P::kPer; e += 2)
      here = max3_raw(P::at(raw[i], e), P::at(raw[i], e + 1), here);
  // (the pieces stay packed: unpacked twice rather than kept as floats)
#pragma unroll
  for (int i = 0; i < kVecs; ++i)
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      int word = raw[i][w];
      asm("" : "+v"(word));
      raw[i][w] = word;
    }
  return here;
}

template <typename P, int kLanes, int kVecs, bool kLoop, bool kStream>
__global__ void __launch_bounds__(256)
    row_norm_kernel(const typename P::Elem *__restrict__ logits, Lattice L, Picks<float> out,
                    Surround around) {
  constexpr int kAux = kStream ? 2 : 0;
  constexpr int kRows = kWave / kLanes;
  out.start();
  // (from the last row to the first: the caller has left what it wrote last in the cache)
  const int b = L.B - 1 - block_batch();
  if (b < 0) return;
  if (blockIdx.x < around.blocks) return around.fill(L, b, blockIdx.x, out.px, out.py);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // in a scalar register
  const int lane = threadIdx.x & (kLanes - 1);
  const unsigned r0 = ((gridDim.x - 1 - blockIdx.x) * 4 + wave) * kRows;
  const unsigned r = kRows == 1 ? r0 : r0 + (threadIdx.x & 63) / kLanes;
  const Row row = locate(L, b, r);
  if (!row.live && lane == 0) out.skip(L, row);
  if (kRows == 1 ? !row.live : !__any(row.live)) return;
  const long first = (long)b * L.T * L.Rr + r0;
  const uintptr_t base = wave_base<P, kLanes>(logits, first, L.C);
  const __amdgpu_buffer_rsrc_t rs = resource(base, wave_bytes<P, kLanes>(L.C));
  const RowPieces<P, kLanes> q =
      pieces_of<P, kLanes>(base, reinterpret_cast<uintptr_t>(logits + row.index * L.C), L.C);
  const float ninf = -__builtin_huge_valf();
  float m = ninf, sum = 0, shift = 0;
  intx4 raw[kVecs];
  for (int p0 = 0; p0 < (kLoop ? q.pieces : 1); p0 += kLanes * kVecs) {
#pragma unroll
    for (int i = 0; i < kVecs; ++i) {
      const int p = p0 + lane + kLanes * i;
      const bool wanted = (kRows == 1 || row.live) && p < q.pieces;
      raw[i] = __builtin_amdgcn_raw_buffer_load_b128(rs, wanted ? q.at + 16 * p : kOutOfRange, 0, kAux);
    }
    const float here = over_group(largest_of_lane<P, kLanes>(raw, q, p0, lane, L.C), kLanes,
                                  [](float a, float b) { return max3_raw(a, b, b); });
    if (kLoop) {
      // (a NaN is ignored by the maximum and comes back through the sum)
      const float to = here > m ? here : m;
      const float next = (to - to == 0) ? to : 0.f;
      if (p0 > 0) sum *= __expf((m - m == 0 ? m : (m < 0 ? next : 0.f)) - next);
      m = to;
      shift = next;
    } else {
      m = here;
      shift = (m - m == 0) ? m : 0.f;  // torch.logsumexp: infinite max -> shift by 0
    }
#pragma unroll
    for (int i = 0; i < kVecs; ++i)
#pragma unroll
      for (int e = 0; e < P::kPer; ++e) sum += __expf(P::at(raw[i], e) - shift);
  }
  const int sym = row.live ? row_symbol(L, row) : -1;
  float at_sym = 0, at_term = 0;
  if (kRows > 1 || kLoop) {
    const typename P::Elem *x = logits + row.index * L.C;
    if (row.live && lane == 0) {
      at_term = P::load(x[L.term]);
      if (sym >= 0) at_sym = P::load(x[sym]);
    }
  } else {
    at_term = row_entry<P, kVecs>(raw, q.off, L.term);
    if (sym >= 0) at_sym = row_entry<P, kVecs>(raw, q.off, sym);
  }
  sum = group_sum(sum, kLanes);
  const float lse = logf(sum) + shift;
  if (row.live && lane == 0)
    out.write(L, row, lse, sym >= 0 ? at_sym - lse : std::numeric_limits<float>::quiet_NaN(),
              at_term - lse);
}

// ---- several short rows per wave ------------------------------------------------------------------
// Four rows are reduced together: where the halves and quarters of a wave would be joined for each of them, two
// rows' change places, and a quarter of the wave ends with each row.  The order in which a row's lanes are joined
// is over_group's.
template <int kLanes, typename F>
__device__ __forceinline__ float over_four_rows(const float (&v)[kLanes / 16], F f) {
  auto halves = [&](float a, float b) {
    const auto pair = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return f(__uint_as_float(pair[0]), __uint_as_float(pair[1]));
  };
  auto quarters = [&](float a, float b) {
    const auto pair = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return f(__uint_as_float(pair[0]), __uint_as_float(pair[1]));
  };
  if constexpr (kLanes == 64) return over_group(quarters(halves(v[0], v[1]), halves(v[2], v[3])), 16, f);
  if constexpr (kLanes == 32) return over_group(quarters(v[0], v[1]), 16, f);
  if constexpr (kLanes == 16) return over_group(v[0], 16, f);
}
// For short rows: a lane group takes kIter rows, in steps of four a wave.  A row's chain of dependent loads -- its
// range, its symbol, that entry -- is walked for all rows of a wave at once, a lane per row, beside the pieces,
// which are all requested first, and that lane writes its row's results.
// Bound by the latency of the loads of the waves that fit, and by issue: a wave per row is 604 bytes in flight at
// float16, C 302, five rows a frame, B 34, T 1028, S 148: 83 -> 49 us (1.7 TB/s of what counts); bfloat16, B 128,
// T 200, C 80: 18.4 -> 13.0; float32, B 100, T 500, C 500: 126 -> 86 (4.7 TB/s); B 32, T 500, C 256: 38 -> 23.7;
// B 32, T 250, C 500: 23.6 -> 22.2, C 700: 24.0 -> 22.2; B 8, T 200, C 500: 7.2 -> 6.6.  Where rows are longer, a row is enough
// in flight for a wave (float32, C 1000: 26.7 -> 29.9; bfloat16: 25.9 -> 26.7), and few rows do not
// fill the chip (B 4, T 100, C 500: 4.3 -> 4.8; bfloat16, B 8, T 100: 5.1 -> 5.7).
template <typename P, int kLanes, int kVecs, int kIter, bool kStream, bool kAligned>
__global__ void __launch_bounds__(256)
    row_norm_rows_kernel(const typename P::Elem *__restrict__ logits, Lattice L, Picks<float> out,
                         Surround around) {
  constexpr int kAux = kStream ? 2 : 0;
  constexpr int kRows = kWave / kLanes, kN = kRows * kIter, kSteps = 4 / kRows;
  static_assert(kN % 4 == 0 && kN <= kWave, "a lane per row");
  out.start();
  const int b = L.B - 1 - block_batch();
  if (b < 0) return;
  if (blockIdx.x < around.blocks) return around.fill(L, b, blockIdx.x, out.px, out.py);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // in a scalar register
  const int at = threadIdx.x & 63, lane = at & (kLanes - 1);
  const unsigned r0 = ((gridDim.x - 1 - blockIdx.x) * 4 + wave) * kN;
  if (r0 >= (unsigned)(L.T * L.Rr)) return;
  // this lane's row: of the fours, number at % 16
  const bool mine = at % 16 < kN / 4;
  Row row = placed_in_frame(L, b, r0 + (mine ? 4 * (at % 16) + row_of_quarter(at / 16) : 0));
  // (a row whose range begins outside the window is read all the same)
  const unsigned long long there = __ballot(mine && row.live);
  if (there == 0 && !__any(mine && row.t < L.T)) return;
  const long first = (long)b * L.T * L.Rr + r0;
  const uintptr_t base = wave_base<P, kLanes>(logits, first, L.C);
  const __amdgpu_buffer_rsrc_t rs =
      resource(base, ((long)kN * L.C * (long)sizeof(typename P::Elem) + 31) & ~15L);
  intx4 raw[kIter][kVecs];
  RowPieces<P, kLanes> q[kIter];
#pragma unroll
  for (int n = 0; n < kIter; ++n) {
    const int group = kRows == 4 ? row_of_quarter(at / 16) : kRows == 2 ? at / 32 : 0;
    const int nth = kRows * n + group;
    q[n] = pieces_of<P, kLanes>(base, reinterpret_cast<uintptr_t>(logits + (first + nth) * L.C), L.C);
    if (kAligned) q[n].off = 0, q[n].whole = q[n].pieces = L.C / P::kPer;
    const bool wanted = there >> (16 * row_of_quarter(nth % 4) + nth / 4) & 1;
#pragma unroll
    for (int i = 0; i < kVecs; ++i) {
      const int p = lane + kLanes * i;
      raw[n][i] = __builtin_amdgcn_raw_buffer_load_b128(
          rs, (int)wanted & (int)(p < q[n].pieces) ? q[n].at + 16 * p : kOutOfRange, 0, kAux);
    }
  }
  place(L, row);
  const bool live = mine && row.live;
  if (mine && !row.live) out.skip(L, row);
  const int sym = live ? row_symbol(L, row) : -1;
  float at_sym = 0, at_term = 0;
  if (live) {
    const typename P::Elem *x = logits + row.index * L.C;
    at_term = P::load(x[L.term]);
    if (sym >= 0) at_sym = P::load(x[sym]);
  }
  float my_sum = 0, my_shift = 0;
#pragma unroll
  for (int n0 = 0; n0 < kIter; n0 += kSteps) {
    float v[kSteps];
#pragma unroll
    for (int n = 0; n < kSteps; ++n)
      v[n] = largest_of_lane<P, kLanes, kVecs, kAligned>(raw[n0 + n], q[n0 + n], 0, lane, L.C);
    const float m = over_four_rows<kLanes>(v, [](float a, float b) { return max3_raw(a, b, b); });
    const float shift = (m - m == 0) ? m : 0.f;  // torch.logsumexp: infinite max -> shift by 0
    float shifts[kSteps];
    to_rows<kLanes>(shift, shifts);
#pragma unroll
    for (int n = 0; n < kSteps; ++n) {
      v[n] = 0;
#pragma unroll
      for (int i = 0; i < kVecs; ++i)
#pragma unroll
        for (int e = 0; e < P::kPer; ++e) v[n] += __expf(P::at(raw[n0 + n][i], e) - shifts[n]);
    }
    const float sum = over_four_rows<kLanes>(v, [](float a, float b) { return a + b; });
    const bool here = at % 16 == n0 / kSteps;
    my_sum = here ? sum : my_sum;
    my_shift = here ? shift : my_shift;
  }
  const float lse = logf(my_sum) + my_shift;
  if (live)
    out.write(L, row, lse, sym >= 0 ? at_sym - lse : std::numeric_limits<float>::quiet_NaN(), at_term - lse);
}

// (rows in 16-byte pieces; else the plain kernel takes them)
template <typename P>
bool rows_in_pieces(int C) {
  return !std::is_same<P, DoublePiece>::value && (long)C * (long)sizeof(typename P::Elem) < (1L << 26);
}
template <typename P, typename R>
void launch_row_norm(const typename P::Elem *logits, const Lattice &L, const Picks<R> &out,
                     bool read_again, hipStream_t stream) {
  const long rows = (long)L.T * L.Rr;
  if constexpr (!std::is_same<P, DoublePiece>::value) {
    if (rows_in_pieces<P>(L.C)) {
      Surround around{0, 1};
      if (L.ranges && out.direct) {
        around.t_tiles = (L.T + (L.rnnt_type == kRegular ? 1 : 0) + 63) / 64;
        around.blocks = (unsigned)around.t_tiles * ((L.S + kAssembleRows) / kAssembleRows);
      }
      const bool big = rows * L.B * L.C * (long)sizeof(typename P::Elem) >
                       (read_again ? 2 * kCacheBytes : kCacheBytes);
      with_row_split<P>(logits, L.C, [&](auto lanes, auto vecs, auto loop) {
        if constexpr (vecs <= (P::kPer == 4 ? 3 : 1) && !loop) {
          constexpr int kIter = lanes == 64 && vecs == 1 && P::kPer == 4 ? 8 : 4;
          constexpr int kRowsOfBlock = kIter * 256 / lanes;
          if (several_rows(rows * L.B, kRowsOfBlock)) {
            auto launch = [&](auto stream_hint, auto aligned) {
              hipLaunchKernelGGL((row_norm_rows_kernel<P, lanes, vecs, kIter, stream_hint, aligned>),
                                 batch_grid(around.blocks + (rows + kRowsOfBlock - 1) / kRowsOfBlock, L.B),
                                 dim3(256), 0, stream, logits, L, out, around);
            };
            constexpr std::integral_constant<bool, lanes == 64> hint;
            if (big)
              rows_aligned<P>(logits, L.C) ? launch(hint, std::true_type{}) : launch(hint, std::false_type{});
            else
              rows_aligned<P>(logits, L.C) ? launch(std::false_type{}, std::true_type{})
                                           : launch(std::false_type{}, std::false_type{});
            return;
          }
        }
        const dim3 grid = batch_grid(around.blocks + (rows + 256 / lanes - 1) / (256 / lanes), L.B);
        if (big && lanes == 64)
          hipLaunchKernelGGL((row_norm_kernel<P, lanes, vecs, loop, lanes == 64>), grid, dim3(256),
                             0, stream, logits, L, out, around);
        else
          hipLaunchKernelGGL((row_norm_kernel<P, lanes, vecs, loop, false>), grid, dim3(256), 0,
                             stream, logits, L, out, around);
      });
      return;
    }
  }
  hipLaunchKernelGGL((row_norm_plain_kernel<P>), batch_grid((rows + 3) / 4, L.B), dim3(256), 0,
                     stream, logits, L, out);
}

// px / py of a tile of 64 columns x 32 lattice rows: lanes along t (coalesced stores), a frame's
// first range entry read once per lane, four waves with eight rows each.  Tiles that the
// recursion cannot reach are left alone when the caller allows it.
template <typename R>
__global__ void __launch_bounds__(256)
    assemble_kernel(const R *__restrict__ xr, const R *__restrict__ yr, Lattice L,
                    Delay<R> delay, R *__restrict__ px, R *__restrict__ py, int t_tiles) {
  const int b = block_batch();
  if (b >= L.B) return;
  const bool regular = L.rnnt_type == kRegular;
  const int T1 = regular ? L.T + 1 : L.T, S1 = L.S + 1;
  const int t = (blockIdx.x % t_tiles) * 64 + (threadIdx.x & 63);
  const int s0 = (blockIdx.x / t_tiles) * kAssembleRows + (threadIdx.x >> 6);
  if (L.window) {
    const int64_t *w = L.window + 4 * b;
    if ((t & ~63) > w[3] || (t | 63) < w[1] || (s0 & ~3) > w[2] ||
        (s0 & ~3) + kAssembleRows <= w[0])
      return;
  }
  const R ninf = Num<R>::neg_inf();
  // (loads without a branch around them, so that all of them are in flight at once: what is not
  // there is looked for in the frame's first row and replaced afterwards)
  const long frame = ((long)b * L.T + min(t, L.T - 1)) * L.Rr;
  const int r0 = L.ranges ? placed_at(L.ranges[frame], 0, L.S) : 0;
  const bool closed = regular && L.boundary && L.boundary[4 * b + 3] == t;
  const bool constrained = L.rnnt_type == kConstrained;
  auto slot = [&](int s) {
    int rel = s - r0;
    if (rel < 0) rel += S1;
    return rel < L.Rr && t < L.T ? rel : -1;
  };
  R x[kAssembleRows / 4], y[kAssembleRows / 4], up[kAssembleRows / 4];
#pragma unroll
  for (int k = 0; k < kAssembleRows / 4; ++k) {
    const int at = max(slot(s0 + 4 * k), 0);
    x[k] = xr[frame + at];
    y[k] = yr[frame + at];
    up[k] = 0;
    if (constrained) up[k] = yr[frame + max(slot(s0 + 4 * k + 1), 0)];
  }
  R *px_b = px + (long)b * L.S * T1, *py_b = py + (long)b * S1 * L.T;
#pragma unroll
  for (int k = 0; k < kAssembleRows / 4; ++k) {
    const int s = s0 + 4 * k;
    const bool here = slot(s) >= 0;
    R v = here && !closed ? x[k] : ninf;
    if (constrained) v += slot(s + 1) >= 0 ? up[k] : ninf;
    v = delay.at(v, L.boundary, b, t, L.T);
    if (s < L.S && t < T1) px_b[(long)s * T1 + t] = v;
    if (s < S1 && t < L.T) py_b[(long)s * L.T + t] = here ? y[k] : ninf;
  }
}

template <typename R>
__global__ void __launch_bounds__(256) fill_neg_inf_kernel(R *__restrict__ x, long n) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i < n) x[i] = Num<R>::neg_inf();
}
template <typename R>
void launch_fill_neg_inf(R *x, long n, hipStream_t stream) {
  if (n > 0)
    hipLaunchKernelGGL(fill_neg_inf_kernel<R>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                       stream, x, n);
}

template <typename P, typename R>
int fwd_impl(const void *logits_, const int64_t *symbols, const int64_t *ranges,
             const int64_t *boundary, R *px, R *py, R *norm, R *xr, R *yr, int B, int S, int T,
             int Rr, int C, int term, int rnnt_type, int window_only, double delay_penalty,
             bool read_again, int *arrived, R *loss, void *stream_) {
  if (B < 0 || S < 0 || T < 0 || Rr < 1 || C < 1)
    return fail(FRNNT_EINVAL, "lattice_logprobs_fwd: bad size");
  if (Rr > S + 1) return fail(FRNNT_EINVAL, "lattice_logprobs_fwd: more range rows than S + 1");
  if (!ranges && Rr != S + 1)
    return fail(FRNNT_EINVAL, "lattice_logprobs_fwd: without ranges the logits need S + 1 rows");
  if (rnnt_type < 0 || rnnt_type > 2 || term < 0 || term >= C)
    return fail(FRNNT_EINVAL, "lattice_logprobs_fwd: bad rnnt_type or termination symbol");
  if (B == 0) return FRNNT_OK;
  if (!logits_ || (!symbols && S > 0) || !px || !py || !norm || !xr || !yr)
    return fail(FRNNT_EINVAL, "lattice_logprobs_fwd: null pointer");
  if ((long)T * Rr >= (1L << 31))
    return fail(FRNNT_ELIMIT, "lattice_logprobs_fwd: an utterance has 2^31 logits rows or more");
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  const Lattice L{symbols, ranges, boundary, window_only ? boundary : nullptr, B, S, T, Rr, C,
                  term, rnnt_type};
  const Delay<R> delay{(R)delay_penalty};
  const bool direct = rnnt_type != kConstrained && (!ranges || rows_in_pieces<P>(C));
  if (T > 0)
    launch_row_norm<P, R>(static_cast<const typename P::Elem *>(logits_), L,
                          Picks<R>{norm, xr, yr, px, py, delay, direct, arrived, loss}, read_again, stream);
  const int T1 = rnnt_type == kRegular ? T + 1 : T;
  if (T == 0 && T1 > 0) {
    // no frames: nothing but the closed column
    launch_fill_neg_inf(px, (long)B * S, stream);
  } else if (!direct && T1 > 0) {
    const int t_tiles = (T1 + 63) / 64, s_tiles = (S + 1 + kAssembleRows - 1) / kAssembleRows;
    hipLaunchKernelGGL(assemble_kernel<R>, batch_grid((long)t_tiles * s_tiles, B), dim3(256), 0,
                       stream, xr, yr, L, delay, px, py, t_tiles);
  }
  return check_launch("lattice_logprobs_fwd");
}

// A whole loss on logits up to its scores' gradient: px / py, then what every loss shares.
template <typename P, typename R>
int loss_fwd_impl(const void *logits, const int64_t *symbols, const int64_t *ranges,
                  const int64_t *boundary, R *px, R *py, R *norm, R *xr, R *yr, R *p, R *scores,
                  R *px_grad, R *py_grad, R *loss, int B, int S, int T, int Rr, int C, int term,
                  int rnnt_type, double delay_penalty, int reduction, int checks, int32_t *status,
                  void *stream) {
  // the recursion's forward can form the loss if it finds a counter cleared; the rows' picks leave xr to it
  // where they go to px and py themselves
  const bool counted = std::is_same<R, float>::value && rnnt_type != kConstrained && T > 0 && loss &&
                       rows_in_pieces<P>(C);
  int *arrived = counted ? reinterpret_cast<int *>(xr) : nullptr;
  const int rc = fwd_impl<P, R>(logits, symbols, ranges, boundary, px, py, norm, xr, yr, B, S, T,
                                Rr, C, term, rnnt_type, boundary != nullptr, delay_penalty,
                                px_grad != nullptr, arrived, loss, stream);
  if (rc != FRNNT_OK) return rc;
  return mi_loss(px, py, boundary, p, scores, px_grad, py_grad, loss, B, S, T, rnnt_type != kRegular,
                 reduction, checks, status, arrived, stream);
}

}  // namespace
}  // namespace frnnt

extern "C" {

#define FRNNT_LATTICE_ENTRY(sfx, io, P, R)                                                       \
  int frnnt_lattice_logprobs_fwd_##sfx(                                                          \
      const io *logits, const int64_t *symbols, const int64_t *ranges, const int64_t *boundary,   \
      R *px, R *py, R *norm, R *xr, R *yr, int B, int S, int T, int Rr, int C,                    \
      int termination_symbol, int rnnt_type, int window_only, void *stream) {                    \
    return frnnt::fwd_impl<frnnt::P, R>(logits, symbols, ranges, boundary, px, py, norm, xr, yr,  \
                                        B, S, T, Rr, C, termination_symbol, rnnt_type,            \
                                        window_only, 0.0, true, nullptr, nullptr, stream);                         \
  }                                                                                              \
  int frnnt_lattice_loss_fwd_##sfx(                                                              \
      const io *logits, const int64_t *symbols, const int64_t *ranges, const int64_t *boundary,   \
      R *px, R *py, R *norm, R *xr, R *yr, R *p, R *scores, R *px_grad, R *py_grad, R *loss,      \
      int B, int S, int T, int Rr, int C, int termination_symbol, int rnnt_type,                 \
      double delay_penalty, int reduction, int checks, int32_t *status, void *stream) {          \
    return frnnt::loss_fwd_impl<frnnt::P, R>(                                                    \
        logits, symbols, ranges, boundary, px, py, norm, xr, yr, p, scores, px_grad,             \
        py_grad, loss, B, S, T, Rr, C, termination_symbol, rnnt_type, delay_penalty, reduction,  \
        checks, status, stream);                                                                 \
  }
FRNNT_LATTICE_ENTRY(f32, float, FloatPiece, float)
FRNNT_LATTICE_ENTRY(f64, double, DoublePiece, double)
FRNNT_LATTICE_ENTRY(f16, void, HalfPiece, float)
FRNNT_LATTICE_ENTRY(bf16, void, Bf16Piece, float)
#undef FRNNT_LATTICE_ENTRY

}  // extern "C"

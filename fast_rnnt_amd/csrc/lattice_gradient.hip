// The gradient of the losses on joiner logits (the forward: lattice_logprobs.hip), HBM-streaming: a
// wave or a part of one per logits row,
//   dlogits[c] = -softmax[c] * (gx + gy) + [c = sym] gx + [c = term] gy
// with gx / gy the px / py gradients of the lattice cell the row was placed at, times the
// gradient of the utterance's score when that has not been applied to them yet.
#include "lattice_rows.hip.h"

namespace frnnt {
namespace {

// What the gradient of a row needs besides the row: the px / py gradients of its cell, its
// symbol and its normalizer.
template <typename R>
struct RowScalars {
  R gx, gy, lse;
  int sym;
};
template <typename R>
struct Grads {
  const R *norm, *gpx, *gpy;
  const R *score_grad;  // NULL: gpx / gpy are scaled already
  int score_stride;
  R score_scale;
  __device__ __forceinline__ RowScalars<R> of(const Lattice &L, const Row &row) const {
    const bool regular = L.rnnt_type == kRegular;
    const int T1 = regular ? L.T + 1 : L.T;
    const bool masked = regular && L.boundary && L.boundary[4 * row.b + 3] == row.t;
    const R f = score_grad ? score_scale * score_grad[(long)row.b * score_stride] : (R)1;
    auto gx_at = [&](int s) -> R {
      if (s < 0 || s >= L.S || masked) return (R)0;
      return f * gpx[((long)row.b * L.S + s) * T1 + row.t];
    };
    RowScalars<R> k;
    k.gx = gx_at(row.s);
    k.gy = f * gpy[((long)row.b * (L.S + 1) + row.s) * L.T + row.t];
    if (L.rnnt_type == kConstrained) k.gy += gx_at(row.s - 1);
    k.sym = row_symbol(L, row);
    k.lse = norm[row.index];
    return k;
  }
};

// any element type, any row length: lanes stride over the row (float64, vocabularies beyond 32-bit
// offsets, and gradients whose 16-byte pieces do not lie where the logits' do)
template <typename P, typename R = typename AccumOf<P>::type>
__global__ void __launch_bounds__(256)
    row_grad_plain_kernel(const typename P::Elem *__restrict__ logits, Lattice L, Grads<R> in,
                          typename P::Elem *__restrict__ glogits) {
  const int b = block_batch();
  const unsigned r = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (b >= L.B) return;
  const Row row = locate(L, b, r);
  if (row.t >= L.T) return;
  typename P::Elem *g = glogits + row.index * L.C;
  if (!row.live) {
    for (int c = lane; c < L.C; c += kWave) g[c] = 0;
    return;
  }
  const RowScalars<R> k = in.of(L, row);
  const R w = -(k.gx + k.gy);
  const typename P::Elem *x = logits + row.index * L.C;
  for (int c = lane; c < L.C; c += kWave) {
    R v = exp_acc<R>(P::load(x[c]) - k.lse) * w;
    if (c == k.sym) v += k.gx;
    if (c == L.term) v += k.gy;
    g[c] = P::store(v);
  }
}

// The gradient leaves as 16-byte stores; the pieces that a row shares with its neighbours leave
// as single elements.  A row outside the window (when the caller says the gradients
// vanish there) is not read: exact zeros are stored.
// kAligned: every row begins and ends on 16 bytes.  No piece is shared then, and a row's code is one
// straight line from its loads to its stores, with the symbol's and the blank's terms selected in
// every piece: a branch around them, or around the shared pieces, holds the loads that follow it back
// (float32, B 8, S 60, T 200, C 1000: 122 -> 115 us; B 16, T 400, C 3000, five rows a frame:
// 130 -> 117; bfloat16, C 5000: 113 -> 100; it takes the compiler's "max-ilp" order as well, see the
// Makefile: with the default one 121, 130 and 115).
template <typename P, int kLanes, int kVecs, bool kLoop, bool kStream, bool kAligned>
__global__ void __launch_bounds__(256)
    row_grad_kernel(const typename P::Elem *__restrict__ logits, Lattice L, Grads<float> in,
                    typename P::Elem *__restrict__ glogits) {
  constexpr int kAux = kStream ? 2 : 0;
  constexpr int kRows = kWave / kLanes;
  const int b = block_batch();
  if (b >= L.B) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // in a scalar register
  const int lane = threadIdx.x & (kLanes - 1);
  const unsigned r0 = (blockIdx.x * 4 + wave) * kRows;
  const unsigned r = kRows == 1 ? r0 : r0 + (threadIdx.x & 63) / kLanes;
  const Row row = locate(L, b, r);
  const bool inside = row.t < L.T;
  if (kRows == 1 ? !inside : !__any(inside)) return;
  const long first = (long)b * L.T * L.Rr + r0;
  const uintptr_t base = wave_base<P, kLanes>(logits, first, L.C);
  const uintptr_t gbase = wave_base<P, kLanes>(glogits, first, L.C);
  const long bytes = wave_bytes<P, kLanes>(L.C);
  const __amdgpu_buffer_rsrc_t in_rs = resource(base, bytes), out_rs = resource(gbase, bytes);
  RowPieces<P, kLanes> q =
      pieces_of<P, kLanes>(base, reinterpret_cast<uintptr_t>(logits + row.index * L.C), L.C);
  if (kAligned) q.off = 0, q.whole = q.pieces = L.C / P::kPer;  // (as constants of the code)
  RowScalars<float> k{0.f, 0.f, 0.f, -1};
  intx4 raw[kVecs];
  for (int p0 = 0; p0 < (kLoop ? q.pieces : 1); p0 += kLanes * kVecs) {
#pragma unroll
    for (int i = 0; i < kVecs; ++i) {
      const int p = p0 + lane + kLanes * i;
      const bool wanted = row.live && p < q.pieces;
      raw[i] = __builtin_amdgcn_raw_buffer_load_b128(in_rs, wanted ? q.at + 16 * p : kOutOfRange,
                                                     0, kAux);
    }
    if (row.live && p0 == 0) k = in.of(L, row);
    const float w = -(k.gx + k.gy);
    const int sym_vec = row.live && k.sym >= 0 ? (k.sym + q.off) / P::kPer / kLanes : -1;
    const int term_vec = row.live ? (L.term + q.off) / P::kPer / kLanes : -1;
#pragma unroll
    for (int i = 0; i < kVecs; ++i) {
      const int first_piece = p0 + kLanes * i, p = first_piece + lane;
      const int c = p * P::kPer - q.off;
      float v[P::kPer];
#pragma unroll
      for (int e = 0; e < P::kPer; ++e) v[e] = __expf(P::at(raw[i], e) - k.lse) * w;
      const int vec = p0 / kLanes + i;
      if (kAligned || kRows > 1 || vec == sym_vec || vec == term_vec) {
#pragma unroll
        for (int e = 0; e < P::kPer; ++e) {
          if (c + e == k.sym) v[e] += k.gx;
          if (c + e == L.term) v[e] += k.gy;
        }
      }
      if (!row.live) {
#pragma unroll
        for (int e = 0; e < P::kPer; ++e) v[e] = 0.f;
      }
      const intx4 o = P::pack(v);
      const bool whole = inside && p < q.whole && (p > 0 || q.off == 0);
      __builtin_amdgcn_raw_buffer_store_b128(o, out_rs, whole ? q.at + 16 * p : kOutOfRange, 0,
                                             kAux);
      // pieces shared with a neighbouring row, if this vector holds any
      const bool ragged = (first_piece == 0 && q.off != 0) ||
                          (q.pieces > q.whole && (unsigned)(q.whole - first_piece) < kLanes);
      if (!kAligned && (kRows > 1 || ragged)) {
#pragma unroll
        for (int e = 0; e < P::kPer; ++e) {
          const bool own = inside && !whole && (unsigned)(c + e) < (unsigned)L.C;
          const int to = own ? q.at + 16 * p + e * (int)sizeof(typename P::Elem) : kOutOfRange;
          if (sizeof(typename P::Elem) == 4)
            __builtin_amdgcn_raw_buffer_store_b32(o[e & 3], out_rs, to, 0, kAux);
          else
            __builtin_amdgcn_raw_buffer_store_b16(
                (short)((unsigned)o[e >> 1] >> (16 * (e & 1))), out_rs, to, 0, kAux);
        }
      }
    }
  }
}

// For short rows, kIter of them per lane group, in steps of four a wave: what a row's gradient needs besides the row,
// a chain of dependent loads, is fetched for all rows of a wave at once, a lane per row, beside the pieces, which are
// all requested first.
// Bound by the latency of the loads of the waves that fit: float16, C 302, five rows a frame, B 34, T 1028: 81 -> 61
// us; float32, B 32, T 500, C 256: 32.4 -> 26.0 (5.5 TB/s); B 64, T 300, C 128: 23.2 -> 18.3; bfloat16, B 128, T 200,
// C 80: 18.4 -> 14.1; B 32, T 250, C 500: 22.8 -> 21.7.  Rows of two pieces a lane have enough in flight without
// (float32, C 500: 143.8 -> 152.3 at B 100, T 500; bfloat16, C 1000: 26.2 -> 31.7), and few rows do not fill the chip
// (bfloat16, B 8, T 100, C 500: 5.6 -> 7.0; float32, B 16, T 150, C 60: 4.9 -> 5.2).
template <int kLanes, int kAt>
__device__ __forceinline__ void of_rows(float x, float (&v)[kLanes / 16]) {
  // (in lane kAt of the quarters)
  if constexpr (kLanes == 64)
    to_rows<64>(x, v, kAt);
  else
    to_rows<kLanes>(__int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x150 + kAt, 0xf, 0xf, true)), v);
}
template <typename P, int kLanes, int kVecs, int kIter, bool kStream, bool kAligned>
__global__ void __launch_bounds__(256)
    row_grad_rows_kernel(const typename P::Elem *__restrict__ logits, Lattice L, Grads<float> in,
                         typename P::Elem *__restrict__ glogits) {
  constexpr int kAux = kStream ? 2 : 0;
  constexpr int kRows = kWave / kLanes, kN = kRows * kIter, kSteps = 4 / kRows;
  static_assert(kN % 4 == 0 && kN <= 8, "of_rows");
  const int b = block_batch();
  if (b >= L.B) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // in a scalar register
  const int at = threadIdx.x & 63, lane = at & (kLanes - 1);
  const unsigned r0 = (blockIdx.x * 4 + wave) * kN, rows = (unsigned)(L.T * L.Rr);
  if (r0 >= rows) return;
  // this lane's row: of the fours, number at % 16
  const bool mine = at % 16 < kN / 4;
  Row row = placed_in_frame(L, b, r0 + (mine ? 4 * (at % 16) + row_of_quarter(at / 16) : 0));
  // (a row whose range begins outside the window is read all the same)
  const unsigned long long there = __ballot(mine && row.live);
  const long first = (long)b * L.T * L.Rr + r0;
  const uintptr_t base = wave_base<P, kLanes>(logits, first, L.C);
  const uintptr_t gbase = wave_base<P, kLanes>(glogits, first, L.C);
  const long bytes = ((long)kN * L.C * (long)sizeof(typename P::Elem) + 31) & ~15L;
  const __amdgpu_buffer_rsrc_t in_rs = resource(base, bytes), out_rs = resource(gbase, bytes);
  intx4 raw[kIter][kVecs];
  RowPieces<P, kLanes> q[kIter];
  auto number = [&](int n) {
    return kRows * n + (kRows == 4 ? row_of_quarter(at / 16) : kRows == 2 ? at / 32 : 0);
  };
  auto bit_of = [&](unsigned long long mask, int nth) {
    return (int)(mask >> (16 * row_of_quarter(nth % 4) + nth / 4) & 1);
  };
#pragma unroll
  for (int n = 0; n < kIter; ++n) {
    const int nth = number(n);
    q[n] = pieces_of<P, kLanes>(base, reinterpret_cast<uintptr_t>(logits + (first + nth) * L.C), L.C);
    if (kAligned) q[n].off = 0, q[n].whole = q[n].pieces = L.C / P::kPer;
    const int wanted = bit_of(there, nth);
#pragma unroll
    for (int i = 0; i < kVecs; ++i) {
      const int p = lane + kLanes * i;
      raw[n][i] = __builtin_amdgcn_raw_buffer_load_b128(
          in_rs, wanted & (int)(p < q[n].pieces) ? q[n].at + 16 * p : kOutOfRange, 0, kAux);
    }
  }
  place(L, row);
  RowScalars<float> mine_k{0.f, 0.f, 0.f, -1};
  float my_w = 0.f;  // (exact zeros for a row that does not count: its pieces are 0 as well)
  if (mine && row.live) {
    mine_k = in.of(L, row);
    my_w = -(mine_k.gx + mine_k.gy);
  }
  const unsigned long long live = __ballot(mine && row.live);
  auto four = [&](auto which) {
    constexpr int kAt = which;
    float gx[kSteps], gy[kSteps], lse[kSteps], w[kSteps], sym[kSteps];
    of_rows<kLanes, kAt>(mine_k.gx, gx);
    of_rows<kLanes, kAt>(mine_k.gy, gy);
    of_rows<kLanes, kAt>(mine_k.lse, lse);
    of_rows<kLanes, kAt>(my_w, w);
    of_rows<kLanes, kAt>(__int_as_float(mine_k.sym), sym);
#pragma unroll
    for (int m = 0; m < kSteps; ++m) {
      const int n = kAt * kSteps + m, nth = number(n);
      const bool inside = r0 + nth < rows;
      const bool counts = bit_of(live, nth) != 0;
#pragma unroll
      for (int i = 0; i < kVecs; ++i) {
        const int first_piece = kLanes * i, p = first_piece + lane, c = p * P::kPer - q[n].off;
        const intx4 x = counts ? raw[n][i] : intx4{0, 0, 0, 0};
        float v[P::kPer];
#pragma unroll
        for (int e = 0; e < P::kPer; ++e) {
          v[e] = __expf(P::at(x, e) - lse[m]) * w[m];
          if (c + e == __float_as_int(sym[m])) v[e] += gx[m];
          if (c + e == L.term) v[e] += gy[m];
        }
        const intx4 o = P::pack(v);
        const bool whole = inside && p < q[n].whole && (p > 0 || q[n].off == 0);
        __builtin_amdgcn_raw_buffer_store_b128(o, out_rs, whole ? q[n].at + 16 * p : kOutOfRange, 0, kAux);
        // pieces shared with a neighbouring row, if this vector holds any
        const bool ragged = (first_piece == 0 && q[n].off != 0) ||
                            (q[n].pieces > q[n].whole && (unsigned)(q[n].whole - first_piece) < kLanes);
        if (!kAligned && (kRows > 1 || ragged)) {
#pragma unroll
          for (int e = 0; e < P::kPer; ++e) {
            const bool own = inside && !whole && (unsigned)(c + e) < (unsigned)L.C;
            const int to = own ? q[n].at + 16 * p + e * (int)sizeof(typename P::Elem) : kOutOfRange;
            if (sizeof(typename P::Elem) == 4)
              __builtin_amdgcn_raw_buffer_store_b32(o[e & 3], out_rs, to, 0, kAux);
            else
              __builtin_amdgcn_raw_buffer_store_b16((short)((unsigned)o[e >> 1] >> (16 * (e & 1))), out_rs, to, 0,
                                                    kAux);
          }
        }
      }
    }
  };
  four(std::integral_constant<int, 0>{});
  if constexpr (kN > 4) four(std::integral_constant<int, 1>{});
}

template <typename P, typename R>
void launch_row_grad(const typename P::Elem *logits, const Lattice &L, const Grads<R> &in,
                     typename P::Elem *glogits, hipStream_t stream) {
  const long rows = (long)L.T * L.Rr;
  if constexpr (!std::is_same<P, DoublePiece>::value) {
    if ((long)L.C * (long)sizeof(typename P::Elem) < (1L << 26) &&
        ((reinterpret_cast<uintptr_t>(logits) ^ reinterpret_cast<uintptr_t>(glogits)) & 15) == 0) {
      const bool big = rows * L.B * L.C * (long)sizeof(typename P::Elem) > kStreamBytes;
      with_row_split<P>(logits, L.C, [&](auto lanes, auto vecs, auto loop) {
        if constexpr (vecs == 1 && !loop) {
          constexpr int kIter = lanes == 16 ? 2 : 4, kRowsOfBlock = kIter * 256 / lanes;
          if (several_rows(rows * L.B, kRowsOfBlock)) {
            auto launch = [&](auto stream_hint, auto aligned) {
              hipLaunchKernelGGL((row_grad_rows_kernel<P, lanes, vecs, kIter, stream_hint, aligned>),
                                 batch_grid((rows + kRowsOfBlock - 1) / kRowsOfBlock, L.B), dim3(256), 0, stream,
                                 logits, L, in, glogits);
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
        const dim3 grid = batch_grid((rows + 256 / lanes - 1) / (256 / lanes), L.B);
        auto launch = [&](auto stream_hint, auto aligned) {
          hipLaunchKernelGGL((row_grad_kernel<P, lanes, vecs, loop, stream_hint, aligned>), grid,
                             dim3(256), 0, stream, logits, L, in, glogits);
        };
        constexpr std::integral_constant<bool, lanes == 64> hint;
        if (big)
          rows_aligned<P>(logits, L.C) ? launch(hint, std::true_type{}) : launch(hint, std::false_type{});
        else
          rows_aligned<P>(logits, L.C) ? launch(std::false_type{}, std::true_type{})
                                       : launch(std::false_type{}, std::false_type{});
      });
      return;
    }
  }
  hipLaunchKernelGGL((row_grad_plain_kernel<P>), batch_grid((rows + 3) / 4, L.B), dim3(256), 0,
                     stream, logits, L, in, glogits);
}

template <typename P, typename R>
int bwd_impl(const void *logits_, const int64_t *symbols, const int64_t *ranges,
             const int64_t *boundary, const R *norm, const R *px_grad, const R *py_grad,
             void *logits_grad, const R *score_grad, int score_grad_stride,
             double score_grad_scale, int B, int S, int T, int Rr, int C, int term, int rnnt_type,
             int window_only, void *stream_) {
  if (B < 0 || S < 0 || T < 0 || Rr < 1 || C < 1 || Rr > S + 1 || (!ranges && Rr != S + 1))
    return fail(FRNNT_EINVAL, "lattice_logprobs_bwd: bad size");
  if (rnnt_type < 0 || rnnt_type > 2 || term < 0 || term >= C)
    return fail(FRNNT_EINVAL, "lattice_logprobs_bwd: bad rnnt_type or termination symbol");
  if (score_grad_stride != 0 && score_grad_stride != 1)
    return fail(FRNNT_EINVAL, "lattice_logprobs_bwd: score_grad_stride must be 0 or 1");
  if (B == 0 || T == 0) return FRNNT_OK;
  if (!logits_ || (!symbols && S > 0) || !norm || !px_grad || !py_grad || !logits_grad)
    return fail(FRNNT_EINVAL, "lattice_logprobs_bwd: null pointer");
  if ((long)T * Rr >= (1L << 31))
    return fail(FRNNT_ELIMIT, "lattice_logprobs_bwd: an utterance has 2^31 logits rows or more");
  const Lattice L{symbols, ranges, boundary, window_only ? boundary : nullptr, B, S, T, Rr, C,
                  term, rnnt_type};
  launch_row_grad<P, R>(
      static_cast<const typename P::Elem *>(logits_), L,
      Grads<R>{norm, px_grad, py_grad, score_grad, score_grad_stride, (R)score_grad_scale},
      static_cast<typename P::Elem *>(logits_grad), static_cast<hipStream_t>(stream_));
  return check_launch("lattice_logprobs_bwd");
}

}  // namespace
}  // namespace frnnt

extern "C" {

#define FRNNT_LATTICE_ENTRY(sfx, io, P, R)                                                       \
  int frnnt_lattice_logprobs_bwd_##sfx(                                                          \
      const io *logits, const int64_t *symbols, const int64_t *ranges, const int64_t *boundary,   \
      const R *norm, const R *px_grad, const R *py_grad, io *logits_grad, int B, int S, int T,    \
      int Rr, int C, int termination_symbol, int rnnt_type, int window_only, void *stream) {     \
    return frnnt::bwd_impl<frnnt::P, R>(logits, symbols, ranges, boundary, norm, px_grad,         \
                                        py_grad, logits_grad, nullptr, 0, 1.0, B, S, T, Rr, C,    \
                                        termination_symbol, rnnt_type, window_only, stream);     \
  }                                                                                              \
  int frnnt_lattice_loss_bwd_##sfx(                                                              \
      const io *logits, const int64_t *symbols, const int64_t *ranges, const int64_t *boundary,   \
      const R *norm, const R *score_grad, int score_grad_stride, double score_grad_scale,        \
      const R *px_grad, const R *py_grad, io *logits_grad, int B, int S, int T, int Rr, int C,    \
      int termination_symbol, int rnnt_type, void *stream) {                                     \
    return frnnt::bwd_impl<frnnt::P, R>(logits, symbols, ranges, boundary, norm, px_grad,         \
                                        py_grad, logits_grad, score_grad, score_grad_stride,     \
                                        score_grad_scale, B, S, T, Rr, C, termination_symbol,    \
                                        rnnt_type, boundary != nullptr, stream);                 \
  }
FRNNT_LATTICE_ENTRY(f32, float, FloatPiece, float)
FRNNT_LATTICE_ENTRY(f64, double, DoublePiece, double)
FRNNT_LATTICE_ENTRY(f16, void, HalfPiece, float)
FRNNT_LATTICE_ENTRY(bf16, void, Bf16Piece, float)
#undef FRNNT_LATTICE_ENTRY

}  // extern "C"

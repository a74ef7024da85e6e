// What the forward (lattice_logprobs.hip) and the backward (lattice_gradient.hip) of the losses on
// joiner logits share: element types, which lattice cell a logits row belongs to, and how a row is
// held in registers.
#pragma once
#include "common.hip.h"

namespace frnnt {
namespace {

enum { kRegular = 0, kModified = 1, kConstrained = 2 };

typedef int intx4 __attribute__((ext_vector_type(4)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
constexpr int kOutOfRange = (int)0x80000000;  // an offset outside every buffer resource

// ---- element types of the logits: what a 16-byte piece of a row holds ---------------------
// float16 / bfloat16 logits are read as they are -- half the bytes of the dominant stream --
// and everything after the load is float32 (the reference's recursion has no half form,
// mutual_information_cuda.cu:37-38); only logits.grad goes back out in the 2-byte type.
struct FloatPiece {
  typedef float Elem;
  static constexpr int kPer = 4;
  static __device__ __forceinline__ float load(Elem x) { return x; }
  static __device__ __forceinline__ Elem store(float x) { return x; }
  static __device__ __forceinline__ float at(intx4 raw, int e) { return __int_as_float(raw[e]); }
  static __device__ __forceinline__ void drop(intx4 &raw, int e) { raw[e] = (int)0xff800000; }
  static __device__ __forceinline__ intx4 pack(const float (&v)[kPer]) {
    return intx4{__float_as_int(v[0]), __float_as_int(v[1]), __float_as_int(v[2]),
                 __float_as_int(v[3])};
  }
};
template <typename IO, typename Hw, unsigned kMinusInf>
struct NarrowPiece {
  typedef uint16_t Elem;
  static constexpr int kPer = 8;
  static __device__ __forceinline__ float load(Elem x) { return IO::load(x); }
  static __device__ __forceinline__ Elem store(float x) { return IO::store(x); }
  static __device__ __forceinline__ float at(intx4 raw, int e) {
    const unsigned w = (unsigned)raw[e >> 1];
    return IO::load((uint16_t)((e & 1) ? w >> 16 : w & 0xffffu));
  }
  static __device__ __forceinline__ void drop(intx4 &raw, int e) {
    const unsigned w = (unsigned)raw[e >> 1];
    raw[e >> 1] = (int)((e & 1) ? (w & 0xffffu) | kMinusInf << 16 : (w & 0xffff0000u) | kMinusInf);
  }
  // (two values per conversion instruction, rounded to nearest even)
  static __device__ __forceinline__ intx4 pack(const float (&v)[kPer]) {
    typedef Hw hwx2 __attribute__((ext_vector_type(2)));
    intx4 o;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const hwx2 h = __builtin_convertvector((floatx2{v[2 * q], v[2 * q + 1]}), hwx2);
      int w;
      __builtin_memcpy(&w, &h, 4);
      o[q] = w;
    }
    return o;
  }
};
typedef NarrowPiece<HalfIO, _Float16, 0xfc00u> HalfPiece;
typedef NarrowPiece<Bf16IO, __bf16, 0xff80u> Bf16Piece;
struct DoublePiece {  // (only its element type is used: doubles take the plain kernels)
  typedef double Elem;
  static __device__ __forceinline__ double load(Elem x) { return x; }
  static __device__ __forceinline__ Elem store(double x) { return x; }
};
template <typename P>
struct AccumOf {
  typedef float type;
};
template <>
struct AccumOf<DoublePiece> {
  typedef double type;
};

// Sums and maxima over the kLanes lanes of a group, in every one of them.  In float32 through the vector unit's own
// lane exchanges, one instruction a step (a shuffle goes through the LDS unit and waits for it): the other half of
// the wave, the other row of 16 lanes, then rotations within the row, whose partners are those of an exchange with
// lane ^ 8, 4, 2, 1, since what has been combined already repeats.
template <int kControl>
__device__ __forceinline__ float rotated_in_row(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), kControl, 0xf, 0xf, true));
}
template <typename F>
__device__ __forceinline__ float over_group(float v, int lanes, F f) {
  auto joined = [&](auto pair) { return f(__uint_as_float(pair[0]), __uint_as_float(pair[1])); };
  if (lanes > 32)
    v = joined(__builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false));
  if (lanes > 16)
    v = joined(__builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false));
  v = f(v, rotated_in_row<0x128>(v));
  v = f(v, rotated_in_row<0x124>(v));
  v = f(v, rotated_in_row<0x122>(v));
  return f(v, rotated_in_row<0x121>(v));
}
// (NaN if any is)
__device__ __forceinline__ float group_max(float v, int lanes) {
  return over_group(v, lanes, [](float a, float b) { return b > a || b != b ? b : a; });
}
__device__ __forceinline__ float group_sum(float v, int lanes) {
  return over_group(v, lanes, [](float a, float b) { return a + b; });
}
__device__ __forceinline__ double group_max(double v, int lanes) {
  for (int off = lanes / 2; off > 0; off >>= 1) {
    const double o = __shfl_xor(v, off, 64);
    v = (o > v || o != o) ? o : v;
  }
  return v;
}
__device__ __forceinline__ double group_sum(double v, int lanes) {
  for (int off = lanes / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

template <typename R>
__device__ __forceinline__ R exp_acc(R x);
template <>
__device__ __forceinline__ float exp_acc<float>(float x) {
  return __expf(x);
}
template <>
__device__ __forceinline__ double exp_acc<double>(double x) {
  return exp(x);
}
template <typename R>
__device__ __forceinline__ R log_acc(R x);
template <>
__device__ __forceinline__ float log_acc<float>(float x) {
  return logf(x);
}
template <>
__device__ __forceinline__ double log_acc<double>(double x) {
  return log(x);
}

// What every kernel here knows of a call.
struct Lattice {
  const int64_t *symbols, *ranges, *boundary;
  const int64_t *window;  // == boundary when the caller goes on to the recursion with it
  int B, S, T, Rr, C, term, rnnt_type;
};

// Logits row r (= t * Rr + j) of utterance b.
struct Row {
  int b, t, j;
  int s;      // lattice row it is placed at
  long index; // b * T * Rr + r
  bool live;  // false: past the end, or outside the window
};

// Lattice row of row j of a frame whose ranges begin at r0: (r0 + j) mod (S + 1) -- the roll
// of rnnt_loss.py:968-984, whatever the frame's other range entries hold (the reference
// accepts ranges that are not consecutive and rolls by the first entry alone).
__device__ __forceinline__ int placed_at(int64_t r0, int j, int S) {
  int64_t s = r0 + j;
  if ((uint64_t)s > (uint64_t)S) {
    s %= S + 1;
    s = s < 0 ? s + S + 1 : s;
  }
  return (int)s;
}

// Which row, and whether it counts.  A row (b, t) x lattice row s outside utterance b's boundary
// window [s_begin, s_end] x [t_begin, t_end) is never looked at by the recursion, which hands
// it a gradient of exact zeros: callers that go on to it with the same boundary (the loss
// functions) let the kernels skip such rows -- about a third of a ragged batch.
//
// In two steps: what is known without the ranges -- `live` as far as the frame and, where there are none, the
// lattice row decide -- and the rest.
__device__ __forceinline__ Row placed_in_frame(const Lattice &L, int b, unsigned r) {
  Row o;
  o.b = b;
  o.t = (int)(r / (unsigned)L.Rr);
  o.j = (int)(r - (unsigned)o.t * (unsigned)L.Rr);
  o.s = o.j;
  o.index = (long)b * L.T * L.Rr + r;
  o.live = o.t < L.T;
  if (o.live && L.window) {
    const int64_t *w = L.window + 4 * b;
    o.live = o.t >= w[1] && o.t < w[3] && (L.ranges || (o.s >= w[0] && o.s <= w[2]));
  }
  return o;
}
__device__ __forceinline__ void place(const Lattice &L, Row &o) {
  if (!L.ranges || o.t >= L.T) return;
  o.s = placed_at(L.ranges[o.index - o.j], o.j, L.S);
  if (o.live && L.window) {
    const int64_t *w = L.window + 4 * o.b;
    o.live = o.s >= w[0] && o.s <= w[2];
  }
}
__device__ __forceinline__ Row locate(const Lattice &L, int b, unsigned r) {
  Row o = placed_in_frame(L, b, r);
  place(L, o);
  return o;
}

// Symbol scored by a row: symbols[b][s] for s < S, the termination symbol for s == S; -1 if
// the range entry is out of [0, S].
__device__ __forceinline__ int row_symbol(const Lattice &L, const Row &row) {
  const int64_t s = L.ranges ? L.ranges[row.index] : row.j;
  if (s < 0 || s > L.S) return -1;
  const int64_t sym = s == L.S ? (int64_t)L.term : L.symbols[(long)row.b * L.S + s];
  return sym >= 0 && sym < L.C ? (int)sym : -1;
}

__device__ __forceinline__ int block_batch() { return blockIdx.z * 65535 + blockIdx.y; }
inline dim3 batch_grid(long blocks, int B) {
  return dim3((unsigned)blocks, (unsigned)(B < 65535 ? B : 65535), (unsigned)((B + 65534) / 65535));
}

// ---- rows held in registers as 16-byte pieces ----------------------------------------------
// kLanes lanes own a row, kVecs pieces each: all of a wave for rows of more than 32 pieces, half
// or a quarter of it for shorter ones (with a whole wave per row of 64 floats three quarters of
// the lanes idle and a launch is bound by the waves it starts, not by bytes).  Pieces lie on
// 16-byte boundaries of the ADDRESS, so any row length and any alignment takes the same path:
// a row of odd length begins `off` elements into its first piece, and the elements of the first
// and the last piece that belong to its neighbours are masked.  Every load of a row is in flight
// before the first is used, through a raw buffer resource over the wave's rows: a piece that is
// not wanted gets an offset outside it, reads as 0 and moves no data -- no branch stands between
// the loads.  kLoop: rows of more pieces than registers, in chunks of kLanes * kVecs.
// kStream: see kCacheBytes and kStreamBytes.
template <typename P, int kLanes>
struct RowPieces {
  int off;      // elements of the first piece that lie before the row
  int whole;    // pieces [off > 0, whole) lie wholly inside the row
  int pieces;   // pieces that hold any of it
  int at;       // byte offset of the first piece in the resource
};
template <typename P, int kLanes>
__device__ __forceinline__ RowPieces<P, kLanes> pieces_of(uintptr_t base, uintptr_t row, int C) {
  RowPieces<P, kLanes> o;
  o.off = (int)(row & 15) / (int)sizeof(typename P::Elem);
  o.whole = (o.off + C) / P::kPer;
  o.pieces = (o.off + C + P::kPer - 1) / P::kPer;
  o.at = (int)((row & ~(uintptr_t)15) - base);
  return o;
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t resource(uintptr_t base, long bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void *>(base), 0, (int)bytes,
                                           0x00020000);
}
// the rows of a wave, as a resource that begins at its first row's first piece
template <typename P, int kLanes>
__device__ __forceinline__ uintptr_t wave_base(const typename P::Elem *logits, long first, int C) {
  return reinterpret_cast<uintptr_t>(logits + first * C) & ~(uintptr_t)15;
}
template <typename P, int kLanes>
__device__ __forceinline__ long wave_bytes(int C) {
  return ((long)(kWave / kLanes) * C * (long)sizeof(typename P::Elem) + 31) & ~15L;
}

// ---- the last-level cache (256 MB) ---------------------------------------------------------------
// A joiner writes the logits from the first row to the last and leaves the last ones in the cache; its
// backward reads the gradient from the first row on.  So the forward pass goes from the last row to the
// first, and finds what the joiner has left, and the backward from the first to the last, and finds what
// the forward has left.  (With a forward from the first row on, which pushes out what it has yet to come
// to, and a backward from the last, behind a linear layer that writes the logits: B 8, S 60, T 200, C 1000,
// 372 MiB: 71 + 97 us, now 58 + 103; bfloat16, B 16, T 400, five rows a frame, C 5000, 305 MiB: 69 + 92,
// now 54 + 99; float32, B 20, T 500, C 1500, 286 MiB: 50 + 79, now 45 + 84.  On logits that lie in memory
// untouched the two are worth the same to 2 %: 53 + 95 and 52 + 98 at 372 MiB.)
//
// Logits of more than two caches that the backward will read, or of more than one that it will not, are
// read with the non-temporal hint: too little of them would still be there when it is wanted, and read
// past the cache they leave it to what the joiner wrote last.  Without the hint and with it, behind that
// layer: forward and backward, pruned bfloat16, 763 MiB: 411 and 362 us, 534 MiB: 281 and 254, 458 MiB:
// 233 and 219; the whole lattice, 605 MiB: 286 and 272, 512 MiB: 224 and 228, 465 MiB: 202 and 210, 372
// MiB: 162 and 169; a forward alone, 372 MiB: 60 and 53, 305 MiB: 51 and 49, 298 MiB: 43 and 42, 248 MiB:
// 38 and 38, 208 MiB: 38.6 and 39.5, 183 MiB: 32 and 36.
constexpr long kCacheBytes = 256L << 20;
// The gradient is read and written with that hint from this many bytes of logits on, which leaves the
// cache to what the joiner's backward reads beside it.  Forward, backward, and the linear layer and its
// gradients around them, without the hint and with it: bfloat16, 104 MiB: 465 and 462 us; 122 MiB: 488 and
// 479; 153 MiB: 616 and 607; 183 MiB: 614 and 599; float32, 107 to 210 MiB: 0.1 to 0.3 % less with it at
// six sizes, 0.3 % more at a seventh; float16, 122 MiB: 857 and 865.  The gradient pass itself is 13 %
// slower to 3 % faster with it below 200 MiB and faster above (372 MiB: 113 and 103).  Below the line
// the hint costs (80 MiB: 851 and 855).
constexpr long kStreamBytes = 96L << 20;

// Whether every row begins and ends on 16 bytes.
template <typename P>
bool rows_aligned(const void *logits, int C) {
  return C % P::kPer == 0 && reinterpret_cast<uintptr_t>(logits) % 16 == 0;
}

// Several short rows of a wave, in fours: quarter `seg` of the wave (16 lanes) has the results or the parameters of
// row row_of_quarter(seg) of the four, `to_rows` brings them to the lanes that hold a row's pieces: of a whole wave
// each (v[0 .. 3]), of a half (rows 0 and 1, then 2 and 3), or its own quarter.
__device__ __forceinline__ constexpr int row_of_quarter(int seg) { return (seg & 1) * 2 + seg / 2; }
template <int kLanes>
__device__ __forceinline__ void to_rows(float of_quarters, float (&v)[kLanes / 16], int at = 0) {
  if constexpr (kLanes == 64) {
#pragma unroll
    for (int n = 0; n < 4; ++n)
      v[n] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(of_quarters), 16 * row_of_quarter(n) + at));
  } else if constexpr (kLanes == 32) {
    const unsigned w = __float_as_uint(of_quarters);
    const auto pair = __builtin_amdgcn_permlane16_swap(w, w, false, false);
    v[0] = __uint_as_float(pair[0]), v[1] = __uint_as_float(pair[1]);
  } else {
    v[0] = of_quarters;
  }
}

// Whether a launch with several rows per lane group has enough workgroups (of rows_of_block rows) to be worth it:
// each is a longer chain, which shows where they do not all but fill the chip (figures at the kernels).
inline bool several_rows(long rows, int rows_of_block) { return rows >= 384L * rows_of_block; }

// Calls f(lanes, vecs, loop) with the split of a row's pieces as compile-time constants: the
// fewest pieces per lane that hold the row, so that little is computed on padding; chunks of
// eight pieces where 80 registers of pieces do not hold it.  Two rows per lane group were
// measured slower (3 - 10 % on 390 MB and on 80 MB of float32 logits).
template <typename P, typename F>
void with_row_split(const void *logits, int C, F f) {
  const long pieces = (C + (rows_aligned<P>(logits, C) ? 0 : P::kPer - 1) + P::kPer - 1) / P::kPer;
  using std::integral_constant;
#define FRNNT_SPLIT(LANES, VECS, LOOP) \
  f(integral_constant<int, LANES>{}, integral_constant<int, VECS>{}, integral_constant<bool, LOOP>{})
  if (pieces <= 16) return FRNNT_SPLIT(16, 1, false);
  if (pieces <= 32) return FRNNT_SPLIT(32, 1, false);
  if (pieces <= 64) return FRNNT_SPLIT(64, 1, false);
  if (pieces <= 128) return FRNNT_SPLIT(64, 2, false);
  if (pieces <= 192) return FRNNT_SPLIT(64, 3, false);
  if (pieces <= 256) return FRNNT_SPLIT(64, 4, false);
  if (pieces <= 384) return FRNNT_SPLIT(64, 6, false);
  if (pieces <= 512) return FRNNT_SPLIT(64, 8, false);
  if (pieces <= 640) return FRNNT_SPLIT(64, 10, false);
  if constexpr (P::kPer == 4) {
    if (pieces <= 896) return FRNNT_SPLIT(64, 14, false);
    if (pieces <= 1280) return FRNNT_SPLIT(64, 20, false);
  }
  FRNNT_SPLIT(64, 8, true);
#undef FRNNT_SPLIT
}

}  // namespace
}  // namespace frnnt

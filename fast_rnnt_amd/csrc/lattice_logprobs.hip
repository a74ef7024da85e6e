// px / py from joiner logits: the unpruned loss (logits [B][T][S+1][C],
// fast_rnnt/python/fast_rnnt/rnnt_loss.py:343-449) and the pruned loss
// (logits [B][T][R][C] plus ranges [B][T][R], rnnt_loss.py:856-1024) share one
// set of kernels; the unpruned case is R = S+1 with every range starting at 0.
//
// Forward, HBM-streaming: the logits are read once, a wave (or a part of one, for short rows)
// per logits row (b, t, j), which forms norm = logsumexp and the two picked log-probs
//   x = logits[b,t,j,sym(b, ranges[b,t,j])] - norm   (sym(b, S) = termination symbol)
//   y = logits[b,t,j,term] - norm.
// Without ranges (and without the constrained step) every cell of px / py comes from one row,
// which writes it.  Otherwise the picks go to xr / yr and a second, small kernel lays them
// out: row j of frame t lands at lattice row (j + ranges[b,t,0]) mod (S+1), everything
// else is -inf, plus the -inf columns of the regular lattice and the constrained
// "px += py[:, 1:]" step.
//
// Backward, HBM-streaming: the same split,
//   dlogits[c] = -softmax[c] * (gx + gy) + [c = sym] gx + [c = term] gy
// with gx / gy the px / py gradients of the lattice cell the row was placed at, times the
// gradient of the utterance's score when that has not been applied to them yet.
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

template <typename R>
__device__ __forceinline__ R group_max(R v, int lanes) {
  for (int off = lanes / 2; off > 0; off >>= 1) {
    const R o = __shfl_xor(v, off, 64);
    v = (o > v || o != o) ? o : v;
  }
  return v;
}
template <typename R>
__device__ __forceinline__ R group_sum(R v, int lanes) {
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
__device__ __forceinline__ Row locate(const Lattice &L, int b, unsigned r) {
  Row o;
  o.b = b;
  o.t = (int)(r / (unsigned)L.Rr);
  o.j = (int)(r - (unsigned)o.t * (unsigned)L.Rr);
  o.s = o.j;
  o.index = (long)b * L.T * L.Rr + r;
  o.live = o.t < L.T;
  if (o.live) {
    if (L.ranges) o.s = placed_at(L.ranges[o.index - o.j], o.j, L.S);
    if (L.window) {
      const int64_t *w = L.window + 4 * b;
      o.live = o.t >= w[1] && o.t < w[3] && o.s >= w[0] && o.s <= w[2];
    }
  }
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

// Where a row's results go: norm always; the picks to px / py at once (direct) or to xr / yr.
template <typename R>
struct Picks {
  R *norm, *xr, *yr, *px, *py;
  Delay<R> delay;
  bool direct;
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

__device__ __forceinline__ int block_batch() { return blockIdx.z * 65535 + blockIdx.y; }
inline dim3 batch_grid(long blocks, int B) {
  return dim3((unsigned)blocks, (unsigned)(B < 65535 ? B : 65535), (unsigned)((B + 65534) / 65535));
}

// ---- any element type, any row length: lanes stride over the row ---------------------------
// (float64, vocabularies beyond 32-bit offsets, and gradients whose 16-byte pieces do not lie
// where the logits' do)
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
// kStream: logits that the last-level cache cannot hold until the backward pass are read
// with the non-temporal hint.
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

template <typename P, int kLanes, int kVecs, bool kLoop, bool kStream>
__global__ void __launch_bounds__(256)
    row_norm_kernel(const typename P::Elem *__restrict__ logits, Lattice L, Picks<float> out) {
  constexpr int kAux = kStream ? 2 : 0;
  constexpr int kRows = kWave / kLanes;
  const int b = block_batch();
  if (b >= L.B) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // in a scalar register
  const int lane = threadIdx.x & (kLanes - 1);
  const unsigned r0 = (blockIdx.x * 4 + wave) * kRows;
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
      raw[i] = __builtin_amdgcn_raw_buffer_load_b128(rs, wanted ? q.at + 16 * p : kOutOfRange, 0,
                                                     kAux);
    }
    // entries that are not the row's become -inf (whole pieces of a whole wave need no test)
#pragma unroll
    for (int i = 0; i < kVecs; ++i) {
      const int first_piece = p0 + kLanes * i;
      if (kRows == 1 && first_piece + kLanes <= q.whole && (first_piece > 0 || q.off == 0)) continue;
#pragma unroll
      for (int e = 0; e < P::kPer; ++e)
        if ((unsigned)((first_piece + lane) * P::kPer + e - q.off) >= (unsigned)L.C)
          P::drop(raw[i], e);
    }
    float here = ninf;
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
    here = group_max(here, kLanes);
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

// The gradient leaves as 16-byte stores; the pieces that a row shares with its neighbours leave
// as single elements.  A row outside the window (when the caller says the gradients
// vanish there) is not read: exact zeros are stored.
template <typename P, int kLanes, int kVecs, bool kLoop, bool kStream>
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
  const RowPieces<P, kLanes> q =
      pieces_of<P, kLanes>(base, reinterpret_cast<uintptr_t>(logits + row.index * L.C), L.C);
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
      if (kRows == 1 ? (vec == sym_vec || vec == term_vec) : true) {
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
      if (kRows > 1 || ragged) {
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

// Logits beyond this many bytes do not stay in the last-level cache between the forward
// and the backward pass: they are streamed (non-temporal hint), which leaves the cache to
// what is used again.  Below it the hint costs (a 80 MB gradient pass: 23.8 -> 26.6 us).
constexpr long kStreamBytes = 192L << 20;

// Calls f(lanes, vecs, loop) with the split of a row's pieces as compile-time constants: the
// fewest pieces per lane that hold the row, so that little is computed on padding; chunks of
// eight pieces where 80 registers of pieces do not hold it.  Two rows per lane group were
// measured slower (3 - 10 % on 390 MB and on 80 MB of float32 logits).
template <typename P, typename F>
void with_row_split(const void *logits, int C, F f) {
  const long item = sizeof(typename P::Elem);
  const bool aligned = (C * item) % 16 == 0 && reinterpret_cast<uintptr_t>(logits) % 16 == 0;
  const long pieces = (C + (aligned ? 0 : P::kPer - 1) + P::kPer - 1) / P::kPer;
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

template <typename P, typename R>
void launch_row_norm(const typename P::Elem *logits, const Lattice &L, const Picks<R> &out,
                     hipStream_t stream) {
  const long rows = (long)L.T * L.Rr;
  if constexpr (!std::is_same<P, DoublePiece>::value) {
    if ((long)L.C * (long)sizeof(typename P::Elem) < (1L << 26)) {
      const bool big = rows * L.B * L.C * (long)sizeof(typename P::Elem) > kStreamBytes;
      with_row_split<P>(logits, L.C, [&](auto lanes, auto vecs, auto loop) {
        const dim3 grid = batch_grid((rows + 256 / lanes - 1) / (256 / lanes), L.B);
        if (big && lanes == 64)
          hipLaunchKernelGGL((row_norm_kernel<P, lanes, vecs, loop, lanes == 64>), grid, dim3(256),
                             0, stream, logits, L, out);
        else
          hipLaunchKernelGGL((row_norm_kernel<P, lanes, vecs, loop, false>), grid, dim3(256), 0,
                             stream, logits, L, out);
      });
      return;
    }
  }
  hipLaunchKernelGGL((row_norm_plain_kernel<P>), batch_grid((rows + 3) / 4, L.B), dim3(256), 0,
                     stream, logits, L, out);
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
        const dim3 grid = batch_grid((rows + 256 / lanes - 1) / (256 / lanes), L.B);
        if (big && lanes == 64)
          hipLaunchKernelGGL((row_grad_kernel<P, lanes, vecs, loop, lanes == 64>), grid, dim3(256),
                             0, stream, logits, L, in, glogits);
        else
          hipLaunchKernelGGL((row_grad_kernel<P, lanes, vecs, loop, false>), grid, dim3(256), 0,
                             stream, logits, L, in, glogits);
      });
      return;
    }
  }
  hipLaunchKernelGGL((row_grad_plain_kernel<P>), batch_grid((rows + 3) / 4, L.B), dim3(256), 0,
                     stream, logits, L, in, glogits);
}

// px / py of a tile of 64 columns x 32 lattice rows: lanes along t (coalesced stores), a frame's
// first range entry read once per lane, four waves with eight rows each.  Tiles that the
// recursion cannot reach are left alone when the caller allows it.
constexpr int kAssembleRows = 32;
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
             void *stream_) {
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
  const bool direct = !ranges && rnnt_type != kConstrained;
  if (T > 0)
    launch_row_norm<P, R>(static_cast<const typename P::Elem *>(logits_), L,
                          Picks<R>{norm, xr, yr, px, py, delay, direct}, stream);
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

// A whole loss on logits up to its scores' gradient: px / py, then what every loss shares.
template <typename P, typename R, typename Tail>
int loss_fwd_impl(Tail tail, const void *logits, const int64_t *symbols, const int64_t *ranges,
                  const int64_t *boundary, R *px, R *py, R *norm, R *xr, R *yr, R *p, R *scores,
                  R *px_grad, R *py_grad, R *loss, int B, int S, int T, int Rr, int C, int term,
                  int rnnt_type, double delay_penalty, int reduction, int checks, int32_t *status,
                  void *stream) {
  const int rc = fwd_impl<P, R>(logits, symbols, ranges, boundary, px, py, norm, xr, yr, B, S, T,
                                Rr, C, term, rnnt_type, boundary != nullptr, delay_penalty, stream);
  if (rc != FRNNT_OK) return rc;
  return tail(px, py, boundary, p, scores, px_grad, py_grad, loss, B, S, T, rnnt_type != kRegular,
              reduction, checks, status, stream);
}

}  // namespace
}  // namespace frnnt

extern "C" {

#define FRNNT_LATTICE_ENTRY(sfx, io, P, R, tail)                                                 \
  int frnnt_lattice_logprobs_fwd_##sfx(                                                          \
      const io *logits, const int64_t *symbols, const int64_t *ranges, const int64_t *boundary,   \
      R *px, R *py, R *norm, R *xr, R *yr, int B, int S, int T, int Rr, int C,                    \
      int termination_symbol, int rnnt_type, int window_only, void *stream) {                    \
    return frnnt::fwd_impl<frnnt::P, R>(logits, symbols, ranges, boundary, px, py, norm, xr, yr,  \
                                        B, S, T, Rr, C, termination_symbol, rnnt_type,            \
                                        window_only, 0.0, stream);                               \
  }                                                                                              \
  int frnnt_lattice_logprobs_bwd_##sfx(                                                          \
      const io *logits, const int64_t *symbols, const int64_t *ranges, const int64_t *boundary,   \
      const R *norm, const R *px_grad, const R *py_grad, io *logits_grad, int B, int S, int T,    \
      int Rr, int C, int termination_symbol, int rnnt_type, int window_only, void *stream) {     \
    return frnnt::bwd_impl<frnnt::P, R>(logits, symbols, ranges, boundary, norm, px_grad,         \
                                        py_grad, logits_grad, nullptr, 0, 1.0, B, S, T, Rr, C,    \
                                        termination_symbol, rnnt_type, window_only, stream);     \
  }                                                                                              \
  int frnnt_lattice_loss_fwd_##sfx(                                                              \
      const io *logits, const int64_t *symbols, const int64_t *ranges, const int64_t *boundary,   \
      R *px, R *py, R *norm, R *xr, R *yr, R *p, R *scores, R *px_grad, R *py_grad, R *loss,      \
      int B, int S, int T, int Rr, int C, int termination_symbol, int rnnt_type,                 \
      double delay_penalty, int reduction, int checks, int32_t *status, void *stream) {          \
    return frnnt::loss_fwd_impl<frnnt::P, R>(                                                    \
        tail, logits, symbols, ranges, boundary, px, py, norm, xr, yr, p, scores, px_grad,       \
        py_grad, loss, B, S, T, Rr, C, termination_symbol, rnnt_type, delay_penalty, reduction,  \
        checks, status, stream);                                                                 \
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
FRNNT_LATTICE_ENTRY(f32, float, FloatPiece, float, frnnt_mi_loss_fwd_f32)
FRNNT_LATTICE_ENTRY(f64, double, DoublePiece, double, frnnt_mi_loss_fwd_f64)
FRNNT_LATTICE_ENTRY(f16, void, HalfPiece, float, frnnt_mi_loss_fwd_f32)
FRNNT_LATTICE_ENTRY(bf16, void, Bf16Piece, float, frnnt_mi_loss_fwd_f32)
#undef FRNNT_LATTICE_ENTRY

}  // extern "C"

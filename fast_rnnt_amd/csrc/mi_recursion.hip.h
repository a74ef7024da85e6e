// Lattice ("mutual information") recursion, forward and backward, for gfx950.
//
// Mapping.  One workgroup per utterance, one lane per lattice row.  A *sweep
// wave* owns 64 consecutive rows and walks the lattice along anti-diagonals: at
// local step e lane L works on column e - L, so the neighbour in the previous
// row is what lane L-1 produced one step earlier (regular lattice) or two steps
// earlier (modified lattice) and arrives through a DPP wave shift, and the
// neighbour in the same row is the lane's own previous result.
//
// A single wave issues about one instruction every 4.5 cycles (a dependent one every 8, a
// scalar test with its branch costs 18 cycles, 35 when taken) and nothing overlaps
// within it, so a sweep wave's time is its instruction count: everything that is not
// the dependent chain is kept off it, and tiles that need no tests run without them,
// each kind of tile in a loop of its own.  *Staging waves* of the same workgroup fetch
// px/py (forward) or p/px (backward) with coalesced, range-checked row loads, turn
// them into diagonal ("sheared") 64-row x 32-step tiles in LDS and -- for the
// backward sweep -- also evaluate the exp() of the gradient split (the forward kernel's do,
// where nobody wants p: kShares); the sweep wave
// pulls a tile into registers with 16-byte LDS reads and leaves the tile's results
// in the same LDS buffer with 16-byte writes.  The staging waves carry the results
// to memory as coalesced row segments through range-checked buffer stores (a cell
// outside the window gets an offset that the hardware drops instead of a branch)
// once they have refilled the buffer.  There are two or three buffers per sweep wave;
// sweep and staging waves meet only through monotone LDS counters (bounded
// spinning; one counter per buffer, which all staging waves of a sweep wave count up),
// never at a barrier, and the sweep wave looks at a counter one chunk (one tile) before
// it needs it.
//
// Rows beyond 64 go to further sweep waves; wave w+1 consumes the last row of
// wave w through an LDS seam row guarded by a progress counter and simply runs a
// few steps behind.  Lattices taller than the workgroup's sweep waves are
// processed band after band with the same seam mechanism; while there are compute
// units to spare, the bands of a long lattice go to workgroups of their own ("apart",
// below).  Forward, the seam is the staging waves' business alone: what the row above
// feeds into a band's first row is added to that row's x.  Backward there is no such
// operand, and the sweep wave takes the seam's values itself.
//
// The arithmetic follows the CPU reference operation for operation
// (fast_rnnt/csrc/mutual_information_cpu.cu:89-121 forward, :179-252 backward,
// log-add from fast_rnnt/csrc/mutual_information.h:36-65); only exp/log come
// from the GPU's own units.
#pragma once
#include "common.hip.h"

namespace frnnt {

// Polls before a wait gives up; set by frnnt_set_spin_limit(), which lets a test force the give-up
// path from the host (mi_recursion.hip).
extern int mi_spin_limit;

namespace {

constexpr int kMaxSweep = 4;           // sweep waves per workgroup
constexpr int kChunk = 8;              // steps between two writes of results / seam hand-over
constexpr int kTileSteps = 32;         // steps per staged tile
constexpr int kTilePitch = kTileSteps + 4;  // rows start 16-byte aligned and spread over the banks
constexpr int kTileElems = kWave * kTilePitch;
constexpr int kSeamPad = kChunk;        // slack on either side of a seam row, so that a whole
                                       // chunk of seam values is written without bounds tests
// The slack on the left is a little longer: the last lane's chunk that starts at step e0
// (a multiple of kChunk) goes to seam columns e0 - 63 ..., and with 11 elements of slack
// their address is a multiple of 16 bytes, so that a chunk is two 16-byte LDS writes.
constexpr int kSeamPadLeft = kSeamPad + 3;
static_assert((kSeamPadLeft - (kWave - 1)) % 4 == 0, "seam chunks are not 16-byte aligned");
constexpr int kSeamSlack = kSeamPadLeft + kSeamPad;
constexpr int kFwdStagers = 3;         // staging waves per sweep wave
constexpr int kBwdStagers = 3;
// With at most two sweep waves a workgroup has room for more staging waves per sweep wave.
// The backward kernel's evaluate d1 / d2 and are what its sweep waves wait for (B 32, S 80, T 250,
// when a launch took 17 us: 17.2 us with 6, 16.9 with 7: 16 waves, the most a workgroup holds); the
// forward kernel's only copy (then 18.45 us with 2, 18.05 with 3, 17.9 with 4).
constexpr int kFwdStagersFew = 4;
constexpr int kBwdStagersFew = 7;
// How many tiles ahead of the one it stages a forward staging wave requests inputs (see the loop below).
// (Doubles have no registers for a second set.  Backward the second set costs more than it gives: the
// code there has no scalar registers left, B 64, S 120, T 600: 37 -> 41 us.)
template <typename R>
constexpr int kFetchAhead = sizeof(R) == 4 ? 2 : 1;
// The kernels that pass shares (kShares) deal a sweep wave's tiles out to two groups of its staging waves in
// turn.  A wave's time per tile is mostly latency -- the look at the counter, the way through LDS, its own
// count -- and hardly shrinks with its rows: 2 000 - 2 600 cycles with five rows a lane (backward) and 2 800
// with eight (forward), where a sweep wave needs 1 200 and 2 400 for a tile.  All waves on every tile,
// forward: B 64, S 120, T 600 39.5 us instead of 34.6; backward, B 12, S 220, T 1500: 69 instead of 50.
// With as much time for a tile, inputs requested one tile ahead of a wave's next are enough; two sets of
// registers cost more in code to fetch at the start (1 000 - 2 400 cycles) than they give.
template <int kStagers, bool kShares>
constexpr int kStagerGroups = kShares && kStagers % 2 == 0 ? 2 : 1;

// Staging waves per sweep wave there, with two sweep waves, and waves of a backward workgroup that do what
// is on nobody's way: the zeros around the window and the loss.  (By the staging waves, between two tiles, they
// held up the sweep for 2 600 - 12 700 cycles.)
constexpr int kSharesStagers = 6;
// The same with one sweep wave, where there is room for more: a wave has fewer rows, and so less code to
// fetch at the start.  6 -> 8, forward and backward, B 8, S 60, T 200: 13.3 + 9.8 -> 12.8 + 9.0 us; B 46, S 47,
// T 204: 12.0 + 10.6 -> 11.8 + 9.5; B 15, S 33, T 153: 11.3 + 8.6 -> 10.6 + 7.6 (10: 12.6 + 8.8, 12.2 + 9.3,
// 10.8 + 7.8); in the backward kernel with bands apart, where a wave also hands on the seam, B 12, S 220,
// T 1500: 50.4 with 6, 49.2 with 8, 46.3 with 10.
constexpr int kSharesStagersOne = 8;
constexpr int kSharesStagersApart = 10;
template <int kSweepCap, bool kShares>
constexpr int kHelpers = kShares && kSweepCap <= 2 ? 2 : 0;
constexpr int kSpinLimit = 1 << 22;   // polls before a wait gives up (seconds, not microseconds)
struct Window {
  int s0, t0, ns, nt;  // origin and extent (ns = s_end - s_begin, ...)
  bool ok;
};
// `checks` bits and `status[0]` codes of the forward kernel (FRNNT_CHECK_* / FRNNT_STATUS_*
// of the public header)
constexpr int kCheckSymbols = 1, kCheckFrames = 2;
constexpr int kStatusWindow = 1, kStatusNoSymbols = 2, kStatusFewFrames = 3;

__device__ __forceinline__ Window load_window(const int64_t *boundary, int b, int S, int T) {
  Window w{0, 0, S, T, true};
  if (boundary) {
    const int64_t a = boundary[4 * b + 0], c = boundary[4 * b + 1];
    const int64_t d = boundary[4 * b + 2], e = boundary[4 * b + 3];
    w.ok = (0 <= a) && (a <= d) && (d <= S) && (0 <= c) && (c <= e) && (e <= T);
    w.s0 = (int)a;
    w.t0 = (int)c;
    w.ns = (int)(d - a);
    w.nt = (int)(e - c);
  }
  return w;
}

// Blocks until the counter reaches `target`; gives up (returns false) after a
// bounded number of polls so that no wave can spin forever.
// A wave that gives up must not leave quietly: the callers mark the utterance's outputs
// (see give_up below), so that a wait that never ends shows as NaN, not as a wrong number.
__device__ __forceinline__ bool wait_for(const int *counter, int target, int limit) {
  int spins = 0;
  while (__hip_atomic_load(counter, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) < target) {
    __builtin_amdgcn_s_sleep(1);
    if (++spins > limit) return false;
  }
  return true;
}
// Non-blocking look at a counter: the value is used a chunk or a tile later, when it
// has long arrived.  LDS serves the reads of one wave in order, so data read after
// the counter is at least as recent as the counter; the empty asm keeps the compiler
// from moving such reads ahead of it.
__device__ __forceinline__ int peek(const int *counter) {
  const int v = __hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  asm volatile("" ::: "memory");
  return v;
}
// Waits until this wave's LDS reads have arrived.  On the rare path that re-reads the seam
// it keeps the common path's wait at "the read issued a chunk ago", which the LDS writes
// issued since then do not hold up (after a join the compiler takes the stricter wait).
__device__ __forceinline__ void lds_reads_done() {
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0) only
}
__device__ __forceinline__ void count_in(int *counter) {
  __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void publish(int *counter, int value) {
  __hip_atomic_store(counter, value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// The same for a counter that only tells of LDS writes by this very wave: LDS carries
// out one wave's instructions in the order they were issued, so the counter's write
// lands after the data without the wave waiting for its writes to finish (a release
// makes it wait, ~190 cycles every time).  The empty asm keeps the compiler from
// moving the data's writes below the counter's.
__device__ __forceinline__ void publish_lds_writes(int *counter, int value) {
  asm volatile("" ::: "memory");
  __hip_atomic_store(counter, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  asm volatile("" ::: "memory");
}

// log(exp(a) + exp(c)) on the serial chain: same operation order as log_add(),
// written so that the only fix-up is the NaN that (-inf) - (-inf) produces.
__device__ __forceinline__ float chain_log_add(float a, float c) {
  const float d = a - c;
  const float hi = fmaxf(a, c);  // neither operand is ever NaN
  // -|d| * log2(e) is <= 0 or NaN ((-inf) - (-inf)).  The median with 0 and 1 is the exponential's
  // output clamp, no instruction of its own: it leaves [0, 1] alone and maps the NaN to 0, and the
  // result is then hi -- exactly the "return the larger operand" rule of the reference, without
  // a branch.  (A minimum before the exponential did it with one dependent instruction more:
  // B 64, S 120, T 600: 37.6 -> 37.0 us; B 12, S 220, T 1500: 69.8 -> 68.4.)
  const float t = -fabsf(d) * 1.44269504088896341f;
  const float e = __builtin_amdgcn_fmed3f(__builtin_amdgcn_exp2f(t), 0.0f, 1.0f);
  return __builtin_fmaf(__builtin_amdgcn_logf(1.0f + e), 0.693147180559945309f, hi);
}
__device__ __forceinline__ double chain_log_add(double a, double c) { return log_add(a, c); }

// Results go to memory through raw buffer stores: the resource covers one
// utterance's array, a lane passes a byte offset, and an offset of kDropped lies
// outside every resource, so the hardware's range check discards the store.  That
// turns "this lane has nothing to write here" into one select on the offset, with
// no branch and no change of the execution mask.
constexpr int kDropped = (int)0x80000000;
typedef int intx2 __attribute__((ext_vector_type(2)));
typedef int intx4 __attribute__((ext_vector_type(4)));

template <typename R>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(R *base, size_t elems) {
  // raw buffer (stride 0), 32-bit elements as far as the descriptor is concerned
  return __builtin_amdgcn_make_buffer_rsrc(base, 0, (int)(elems * sizeof(R)), 0x00020000);
}
__device__ __forceinline__ void put1(__amdgpu_buffer_rsrc_t rs, int off, float v) {
  __builtin_amdgcn_raw_buffer_store_b32(__float_as_int(v), rs, off, 0, 0);
}
__device__ __forceinline__ void put1(__amdgpu_buffer_rsrc_t rs, int off, double v) {
  const long long bits = __double_as_longlong(v);
  __builtin_amdgcn_raw_buffer_store_b64(intx2{(int)bits, (int)(bits >> 32)}, rs, off, 0, 0);
}
// Range-checked load: an offset outside the resource (negative ones included, they are
// huge when read as unsigned) reads as 0 and touches no memory.
__device__ __forceinline__ float get1(__amdgpu_buffer_rsrc_t rs, int off, float) {
  return __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, off, 0, 0));
}
__device__ __forceinline__ double get1(__amdgpu_buffer_rsrc_t rs, int off, double) {
  const intx2 v = __builtin_amdgcn_raw_buffer_load_b64(rs, off, 0, 0);
  return __longlong_as_double(((long long)v[1] << 32) | (unsigned int)v[0]);
}
// four consecutive elements (the address only needs element alignment)
__device__ __forceinline__ void put4(__amdgpu_buffer_rsrc_t rs, int off, float a, float b, float c,
                                     float d) {
  __builtin_amdgcn_raw_buffer_store_b128(
      intx4{__float_as_int(a), __float_as_int(b), __float_as_int(c), __float_as_int(d)}, rs, off,
      0, 0);
}
__device__ __forceinline__ void put4(__amdgpu_buffer_rsrc_t rs, int off, double a, double b,
                                     double c, double d) {
  const long long ab = __double_as_longlong(a), bb = __double_as_longlong(b);
  const long long cb = __double_as_longlong(c), db = __double_as_longlong(d);
  __builtin_amdgcn_raw_buffer_store_b128(
      intx4{(int)ab, (int)(ab >> 32), (int)bb, (int)(bb >> 32)}, rs, off, 0, 0);
  __builtin_amdgcn_raw_buffer_store_b128(
      intx4{(int)cb, (int)(cb >> 32), (int)db, (int)(db >> 32)}, rs, off == kDropped ? off : off + 16,
      0, 0);
}
// One lane's kTileSteps staged values, 16 bytes per LDS read.
template <typename R>
__device__ __forceinline__ void pull_row(R (&dst)[kTileSteps], const R *src) {
  constexpr int kPer = 16 / (int)sizeof(R);
  typedef R Piece __attribute__((ext_vector_type(kPer)));
  const Piece *s = reinterpret_cast<const Piece *>(src);
#pragma unroll
  for (int i = 0; i < kTileSteps / kPer; ++i) {
    const Piece v = s[i];
#pragma unroll
    for (int e = 0; e < kPer; ++e) dst[i * kPer + e] = v[e];
  }
}

// kChunk values, 16 bytes per LDS read.
template <typename R>
__device__ __forceinline__ void pull_chunk(R (&dst)[kChunk], const R *src) {
  constexpr int kPer = 16 / (int)sizeof(R);
  typedef R Piece __attribute__((ext_vector_type(kPer)));
  const Piece *s = reinterpret_cast<const Piece *>(src);
#pragma unroll
  for (int i = 0; i < kChunk / kPer; ++i) {
    const Piece v = s[i];
#pragma unroll
    for (int e = 0; e < kPer; ++e) dst[i * kPer + e] = v[e];
  }
}

// kChunk values of one lane into its tile row, 16 bytes per LDS write.
template <typename R>
__device__ __forceinline__ void push_chunk(R *dst, const R (&src)[kChunk]) {
  constexpr int kPer = 16 / (int)sizeof(R);
  typedef R Piece __attribute__((ext_vector_type(kPer)));
  Piece *d = reinterpret_cast<Piece *>(dst);
#pragma unroll
  for (int i = 0; i < kChunk / kPer; ++i) {
    Piece v;
#pragma unroll
    for (int e = 0; e < kPer; ++e) v[e] = src[i * kPer + e];
    d[i] = v;
  }
}

// The first (kHalf = 0) or second half of a chunk into its place in the tile row.  An LDS
// write takes its data out of the registers over some 30 cycles after it has been issued,
// and an instruction that overwrites one of them waits for that; so a sweep wave writes
// the first half of a chunk as soon as it is complete, in the middle of the chunk, and
// the second half at its end: each half then has four steps' time before the next chunk
// comes to its registers.
template <int kHalf, typename R>
__device__ __forceinline__ void push_half(R *dst, const R (&src)[kChunk]) {
  constexpr int kPer = 16 / (int)sizeof(R);
  typedef R Piece __attribute__((ext_vector_type(kPer)));
  Piece *d = reinterpret_cast<Piece *>(dst);
#pragma unroll
  for (int i = kHalf * (kChunk / 2 / kPer); i < (kHalf + 1) * (kChunk / 2 / kPer); ++i) {
    Piece v;
#pragma unroll
    for (int e = 0; e < kPer; ++e) v[e] = src[i * kPer + e];
    d[i] = v;
  }
}

// Two values to neighbouring elements, in one LDS write (the address is a multiple of two elements).
template <typename R>
__device__ __forceinline__ void push_two(R *dst, R a, R b) {
  typedef R Pair __attribute__((ext_vector_type(2)));
  *reinterpret_cast<Pair *>(dst) = Pair{a, b};
}
static_assert(kTilePitch >= kTileSteps + 2 && kTilePitch % 2 == 0, "no room in front of a tile's rows");

// Keeps the registers of a half chunk that has just been written to LDS from being given
// to the next results at once (see push_half): called four steps later, it makes them
// count as still in use until then.  Emits no instruction.
template <typename R>
__device__ __forceinline__ void still_in_use(const R (&v)[kChunk], int first) {
  if constexpr (sizeof(R) == 4) {
    asm volatile("" ::"v"(v[first]), "v"(v[first + 1]), "v"(v[first + 2]), "v"(v[first + 3]));
  }
}

struct Counters {
  int failed;                             // set by a wave whose bounded wait ran out
  int ready[kMaxSweep];                   // seam columns published by sweep wave w
  int written[kMaxSweep];                 // tiles whose results sweep wave w has left in LDS
  // (forward, kShares) per sweep wave and tile buffer, as in `loaded`: how many times a staging wave has taken a
  // tile's results out of it
  int taken[16];
  // per sweep wave w and tile buffer k (index w * buffers + k): how many times a staging
  // wave has finished staging a tile into that buffer, all of the waves that stage it and all
  // tiles together -- the buffer's n-th tile is complete at n * those.  One counter for
  // all staging waves: a sweep wave pays for every test it makes.
  int loaded[16];
};

// Geometry of what sweep wave `w` does in band `band`; identical on the sweep
// wave and on its staging waves.
struct Band {
  int row0, nrows, nsteps, ntiles;
};
__device__ __forceinline__ Band band_of(int band, int w, int nsweep, int NS, int NT) {
  Band g;
  g.row0 = (band * nsweep + w) * kWave;
  g.nrows = min(kWave, NS + 1 - g.row0);
  g.nsteps = NT + g.nrows;
  g.ntiles = (g.nsteps + kTileSteps - 1) / kTileSteps;
  return g;
}

// The tiles [lo, hi) of a sweep wave's band that are plain: all 32 steps exist
// ((m + 1) * 32 <= nsteps), the step that holds the wave's result (fin_step, if any) is not
// among them and, for a wave with a seam above it, every seam column that the tile and the
// first chunk after it look at exists (0 <= 32 m - shift, 32 (m + 1) + 7 - shift <= NT).
struct PlainTiles {
  int lo, hi;
};
__device__ __forceinline__ PlainTiles plain_tiles(const Band &g, int fin_step, bool up, int shift, int NT) {
  PlainTiles t;
  t.lo = (up && shift > 0) ? 1 : 0;
  t.hi = g.nsteps / kTileSteps;
  if (fin_step >= 0) t.hi = min(t.hi, fin_step / kTileSteps);
  if (up) t.hi = min(t.hi, max(NT - (kChunk - 1) + shift, 0) / kTileSteps);
  t.lo = min(t.lo, g.ntiles);
  t.hi = max(min(t.hi, g.ntiles), t.lo);
  return t;
}

// ---- a workgroup per band of 64 rows ("apart") ---------------------------------------------
// A compute unit that runs several sweep waves and their staging waves gives each of them less:
// measured per step of the sweep, 33 ns (forward) and 27 ns (backward) with one sweep wave, 40
// and 46 with two, 72 and 93 with four.  While there are compute units to spare, every band of 64
// rows of an utterance therefore gets a workgroup of its own.  What a band's last row feeds into
// the next band is a row of the output (p forward, px_grad backward): the staging wave that
// holds it puts it into LDS as soon as a tile is done, a courier wave stores it, and one of the next
// band's workgroup polls it, value by value: the row has been filled with a mark beforehand
// (mark_seams_kernel), a signalling NaN, which no arithmetic instruction ever returns.  The
// values are stored and loaded with agent scope, past the XCDs' own L2.  The workgroups of a
// launch need not all be resident: an utterance's bands run on one XCD, producers have the lower
// block numbers, and an XCD starts its workgroups in their order, so that a producer is running or
// done before its consumer starts.
constexpr int kSeamMark = 0x7fa5a5a5;
// What a courier wave of a band does: takes the seam's `total` values from memory -- value c at
// from + c * stride -- to the seam row in LDS as they arrive, and counts them in.  A wave of its
// own: a staging wave's waits are for everything it has requested and stored, in order.
// `again`: marks what it has taken, for the next launch that finds its seam there.
__device__ __forceinline__ bool bring_seam(float *from, int stride, int total, float *seam,
                                           int *ready, int lane, int limit, bool again) {
  for (int done = 0, spins = 0; done < total;) {
    int bits = kSeamMark;
    if (done + lane < total)
      bits = __hip_atomic_load(reinterpret_cast<int *>(from + (long)(done + lane) * stride),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned long long missing = __ballot(bits == kSeamMark);
    const int n = missing ? __builtin_ctzll(missing) : kWave;
    if (n == 0) {
      if (++spins > limit) return false;
      __builtin_amdgcn_s_sleep(1);
      continue;
    }
    if (lane < n) seam[done + lane] = __int_as_float(bits);
    if (again && lane < n)
      __hip_atomic_store(reinterpret_cast<int *>(from + (long)(done + lane) * stride), kSeamMark,
                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    done += n;
    spins = 0;
    if (lane == 0) publish_lds_writes(ready, done);
  }
  return true;
}
// What the other courier wave does: carries the seam that the band leaves in LDS to memory.
__device__ __forceinline__ bool send_seam(float *to, int stride, int total, const float *seam,
                                          const int *ready, int lane, int limit) {
  for (int done = 0; done < total;) {
    if (!wait_for(ready, done + 1, limit)) return false;
    const int n = min(min(__builtin_amdgcn_readfirstlane(peek(ready)), total) - done, kWave);
    if (lane < n)
      __hip_atomic_store(reinterpret_cast<int *>(to + (long)(done + lane) * stride),
                         __float_as_int(seam[done + lane]), __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    done += n;
  }
  return true;
}
__device__ __forceinline__ bool bring_seam(double *, int, int, double *, int *, int, int, bool) {
  return false;
}
__device__ __forceinline__ bool send_seam(double *, int, int, const double *, const int *, int, int) {
  return false;
}

// The word of the share d1 of a cell that passes nothing on, in LDS: the largest finite number, which all
// that is not finite (mutual_information_cpu.cu:203-206: such a cell has no shares) or negative (no cell
// of the window's) becomes.  And the bit of Counters::loaded for a buffer that has held such a cell.
constexpr unsigned kNoShares = 0x7f7fffff;
constexpr int kNoSharesHere = 1 << 30;
// Where p of lattice row s, the last of a band, passes to the next band if p itself is not stored: T + 1
// elements from row s of py_grad on, which nothing else uses before the backward kernel writes all of
// it.  (The element past the row's end is the first of the row after it, which exists and is no band's
// last.)
template <typename R>
__device__ __forceinline__ R *mail_row(R *py_grad, int b, int s, int S, int T) {
  return py_grad + ((size_t)b * (S + 1) + s) * T;
}

// Or, with a post, where the seam behind band `band` passes in either direction: a row of its own, T + 1 elements for
// each band but the last.  Marked once, by the forward's call; who has read a value leaves a mark again.
template <typename R>
__device__ __forceinline__ R *post_row(R *post, int b, int band, int S, int T) {
  return post + ((size_t)b * (S / kWave) + band) * (T + 1);
}

// A word that any of an utterance's workgroups may make NaN (a wait of theirs ran out) and that the
// last one gives its value: the value replaces what the word held before the launch and nothing
// else, the NaN replaces anything.  Whichever comes first, the NaN stays.
__device__ __forceinline__ void store_nan(float *word) {
  __hip_atomic_store(reinterpret_cast<int *>(word),
                     __float_as_int(std::numeric_limits<float>::quiet_NaN()), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void store_once(float *word, int before, float value) {
  __hip_atomic_compare_exchange_strong(reinterpret_cast<int *>(word), &before,
                                       __float_as_int(value), __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
}

// The marks of an utterance's seam rows: in p or, with `mail`, in the rows that stand for p's (mail_row or, if it is
// a post, post_row; both may be NULL) where rows s0 + 63, s0 + 127, ... of the window feed the next one, in px_grad
// (which may be NULL) where the reversed rows do; and, with p or mail, the utterance's score (see store_once).
// A block per utterance and seam.
__global__ void __launch_bounds__(256)
    mark_seams_kernel(const int64_t *__restrict__ boundary, float *__restrict__ p, float *__restrict__ mail,
                      float *__restrict__ ans, float *__restrict__ px_grad, int S, int T,
                      int modified, int posted) {
  const int b = blockIdx.x, last = (int)blockIdx.y * kWave + kWave - 1;  // (row, or reversed row)
  if ((p || mail) && blockIdx.y == 0 && threadIdx.x == 0) ans[b] = __int_as_float(kSeamMark);
  const Window win = load_window(boundary, b, S, T);
  if (!win.ok || last + 1 > win.ns) return;
  const float mark = __int_as_float(kSeamMark);
  if (p || mail) {
    int *row = reinterpret_cast<int *>(
        posted ? post_row(mail, b, blockIdx.y, S, T)
               : (mail ? mail_row(mail, b, win.s0 + last, S, T) : p + ((size_t)b * (S + 1) + win.s0 + last) * (T + 1)) +
                     win.t0);
    for (int j = threadIdx.x; j <= win.nt; j += 256) row[j] = __float_as_int(mark);
  }
  if (px_grad) {
    const int T1 = modified ? T : T + 1;
    int *row = reinterpret_cast<int *>(px_grad + ((size_t)b * S + win.s0 + win.ns - last - 1) * T1 + win.t0);
    for (int j = threadIdx.x; j <= win.nt - modified; j += 256) row[j] = __float_as_int(mark);
  }
}

// =============================== forward =====================================
// Staged per step and row: x = px feeding the cell from the row below,
// y = py feeding it from the left; -inf where that edge does not exist, and
// y = 0 at the origin cell so that the chain produces p = 0 there.
// A sweep wave only runs the chain: it takes a tile's x / y from an LDS buffer and
// leaves the tile's p in the place of y (16 bytes per LDS write); the staging waves
// carry p to memory, each for the rows it stages, before they refill the buffer.
// kSweepCap: most sweep waves the launch may use; it only sets the register budget.
// kApart: a workgroup per band; `pitch` workgroups per band, one per utterance (of B).
// kShares: what a cell hands down of its gradient, d1 = exp(term1 - p), is stored in the place of p (see
// the backward kernel); the seams of workgroups apart then go through `mail` (see mail_row; posted: post_row).
// rows (may be NULL): takes a copy of the boundary.
template <typename R, bool kModified, int kSweepCap, int kStagers, int kBuffers, bool kApart, bool kShares>
__global__ void __launch_bounds__(((1 + kStagers) * kSweepCap + (kApart ? 2 : 0)) * kWave)
    mi_forward_kernel(const R *__restrict__ px, const R *__restrict__ py,
                      const int64_t *__restrict__ boundary, R *__restrict__ p,
                      R *__restrict__ ans, int S, int T, int spin_limit, int checks,
                      int *__restrict__ status, int B, int pitch, R *mail, int posted, int64_t *rows,
                      R *loss, int reduction, int *arrived) {
  // (lattices of one band -- a cap of one sweep wave -- have no seams)
  constexpr bool kSeams = kApart || kSweepCap > 1;
  extern __shared__ __align__(16) unsigned char dyn_lds[];
  __shared__ Counters cnt;

  const int b = kApart ? blockIdx.x % pitch : blockIdx.x, part = kApart ? blockIdx.x / pitch : 0;
  if (kApart && b >= B) return;
  const int nsweep = blockDim.x / (kWave * (1 + kStagers));
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);  // in a scalar register
  const int lane = threadIdx.x % kWave;
  const int T1 = kModified ? T : T + 1;
  const int TP = T + 1;
  const int shift = kModified ? 1 : 0;
  const R ninf = Num<R>::neg_inf();

  const Window win = load_window(boundary, b, S, T);
  // What the loss functions assert of a boundary row before they call the recursion
  // (rnnt_loss.py:25-42), for callers that do not want to wait for a host copy of the rows:
  // a row that fails is treated like one whose window is out of range, and `status` -- memory
  // the host can read, e.g. pinned host memory -- names the failed test and the row.
  int bad = win.ok ? 0 : kStatusWindow;
  if (checks != 0 && boundary != nullptr && win.ok) {
    if ((checks & kCheckSymbols) && win.s0 + win.ns < 1) bad = kStatusNoSymbols;
    else if ((checks & kCheckFrames) && win.t0 + win.nt < win.s0 + win.ns) bad = kStatusFewFrames;
  }
  if (kShares && rows && boundary && part == 0 && threadIdx.x < 4)
    rows[4 * b + threadIdx.x] = boundary[4 * b + threadIdx.x];
  // What the lane that holds the utterance's score does with it (not apart: `loss` is NULL there), and, in the
  // workgroup that comes last, the rest of its wave: the loss, for which no launch of its own is then needed (a
  // validation pass of two small kernels, B 5, S 19, T 77, C 131, float16, 14.7 -> 12.6 us).
  // `arrived` counts the workgroups; it was 0, and the loss NaN, before the launch.  The scores are stored
  // and read past the XCDs' own L2.
  auto store_score = [&](R v) {
    __hip_atomic_store(&ans[b], v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0) only: the score has arrived
    asm volatile("" ::: "memory");
  };
  auto count_for_loss = [&](R v, int holder) {
    if (!loss) return;
    if (reduction == 0) {
      if (lane == holder) loss[b] = -v;
      return;
    }
    int before = 0;
    if (lane == holder)
      before = __hip_atomic_fetch_add(arrived, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (__builtin_amdgcn_readlane(before, holder) == (int)gridDim.x - 1) {
      asm volatile("" ::: "memory");
      reduce_scores([&](int i) { return __hip_atomic_load(&ans[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); },
                    loss, (int)gridDim.x, reduction, lane);
    }
  };
  if (bad != 0) {
    if (wave == 0 && part == 0) {
      const R nan = std::numeric_limits<R>::quiet_NaN();
      if (lane == 0) {
        store_score(nan);
        if (status) {
          status[1] = b;
          status[0] = bad;
        }
      }
      count_for_loss(nan, 0);
    }
    return;
  }
  if (threadIdx.x < (int)(sizeof(Counters) / sizeof(int)))
    reinterpret_cast<int *>(&cnt)[threadIdx.x] = 0;
  __syncthreads();

  const int NS = win.ns, NT = win.nt, cols = NT + 1;
  const int band_rows = kWave * nsweep;
  const int last_row = kApart ? part * kWave : NS;  // (of those that may begin a band here)
  if (kApart && part * kWave > NS) return;
  const R *pxb = px + (size_t)b * S * T1;
  const R *pyb = py + (size_t)b * (S + 1) * T;
  R *pb = p + (size_t)b * (S + 1) * TP;
  R *seam = reinterpret_cast<R *>(dyn_lds);
  const int seam_pitch = (TP + 3) & ~3;  // keeps the tiles 16-byte aligned
  // (apart: the seam that comes in, and the one that goes out)
  R *tiles = seam + (size_t)(kApart ? 2 : nsweep) * seam_pitch;  // per sweep wave: kBuffers x tiles, then as many y tiles
  // A wave whose bounded wait ran out: the utterance's score becomes NaN (also for the
  // wave that would store it later), so the failure cannot pass for a result.
  auto give_up = [&]() {
    if (lane == 0) {
      publish(&cnt.failed, 1);
      if constexpr (kApart) {
        store_nan(&ans[b]);
      } else {
        const R nan = std::numeric_limits<R>::quiet_NaN();
        store_score(nan);
        if (loss) loss[reduction == 0 ? b : 0] = nan;
      }
    }
  };

  // (apart) where p of the window's row i passes from one workgroup to the next
  auto seam_row = [&](int i) -> R * {
    if (kShares && posted) return post_row(mail, b, i / kWave, S, T);
    return (kShares ? mail_row(mail, b, win.s0 + i, S, T) : pb + (size_t)(win.s0 + i) * TP) + win.t0;
  };
  if (kApart && wave >= 1 + kStagers) {
    // ------------------------------- courier waves -------------------------------
    if (wave == 1 + kStagers) {
      const int next = (part + 1) * kWave;
      if (next <= NS && !send_seam(seam_row(next - 1), 1, cols, seam + seam_pitch, &cnt.ready[1], lane,
                                   spin_limit))
        give_up();
      return;
    }
    if (part > 0 &&
        !bring_seam(seam_row(part * kWave - 1), 1, cols, seam, &cnt.ready[0], lane, spin_limit, kShares && posted))
      give_up();
    return;
  }
  if (wave >= nsweep) {
    // ------------------------------ staging wave -------------------------------
    constexpr int kGroups = kStagerGroups<kStagers, kShares>, kPer = kStagers / kGroups;
    const int w = (wave - nsweep) / kStagers, l = (wave - nsweep) % kPer;
    const int group = (wave - nsweep) % kStagers / kPer;  // which of the tiles m = group, group + kGroups, ...
    const int prev = (w + nsweep - 1) % nsweep;
    const R *up_seam = seam + (size_t)prev * seam_pitch;
    R *my_seam = seam + (size_t)(kApart ? 1 : w) * seam_pitch;
    R *base = tiles + (size_t)w * 2 * kBuffers * kTileElems;
    const int half = lane >> 5, q = lane & 31;
    // rows of a tile this wave stages: r(u) = 2*l + half + 2*kPer*u
    constexpr int kRows = (kWave + 2 * kPer - 1) / (2 * kPer);
    constexpr int kAhead = kShares ? 1 : kFetchAhead<R>;
    struct Staged {
      R x[kRows], y[kRows];
    };
    // Global fetches (into registers) are issued kAhead tiles before they are staged, so that their
    // latency overlaps the sweep.  The loads are range-checked and otherwise unconditional: what a lane
    // reads for cells outside the window is either replaced at staging time (row 0, column 0: the -inf
    // that closes the lattice) or never reaches a cell of the window (columns before a row's start or
    // beyond its end only feed cells at least as far out).
    const __amdgpu_buffer_rsrc_t px_rsrc = buffer_of(const_cast<R *>(pxb), (size_t)S * T1);
    const __amdgpu_buffer_rsrc_t py_rsrc = buffer_of(const_cast<R *>(pyb), (size_t)(S + 1) * T);
    // (what is stored: the rows of the window, so that a row beyond them is outside the resource)
    const __amdgpu_buffer_rsrc_t p_rsrc = buffer_of(pb + (size_t)win.s0 * TP, (size_t)(NS + 1) * TP);
    constexpr int kStep = 2 * kPer;
    constexpr int kSize = (int)sizeof(R);
    const int r_first = 2 * l + half;
    auto fetch = [&](Staged &in, const Band &g, int m) {
      const int s_first = win.s0 + g.row0 + r_first;
      const int j_first = m * kTileSteps + q - r_first;
      const int x0 = m < g.ntiles ? ((s_first - 1) * T1 + win.t0 + j_first - shift) * kSize : kDropped;
      const int y0 = m < g.ntiles ? (s_first * T + win.t0 + j_first - 1) * kSize : kDropped;
#pragma unroll
      for (int u = 0; u < kRows; ++u) {
        // kStep rows further up: as many rows down in memory, as many columns left
        in.x[u] = get1(px_rsrc, x0 + u * (kStep * (T1 - 1) * kSize), R());
        in.y[u] = get1(py_rsrc, y0 + u * (kStep * (T - 1) * kSize), R());
      }
    };
    // p of tile pm of the band that starts at row0, left by the sweep wave in buffer `buf`:
    // element (row r, step q) is the cell (row0 + r, 32 pm + q - r) of the window.  Taking
    // it out of the buffer and storing it are two steps: the stores of a tile go out after
    // the buffer has been refilled and handed back to the sweep wave, not before.
    // (kShares: and what the cell below had and the edge between the two, for the share of the cell's
    // gradient that goes down.  That cell's p is one step back (modified: two) in the row below; the
    // last steps of the tile before lie in front of each row, where the sweep wave has left them.)
    struct Drained {
      R v[kRows], below[kShares ? kRows : 1], x[kShares ? kRows : 1];
      int row0, pm;
    };
    constexpr int kNowhere = -(1 << 20);  // (a tile with no cell in the window)
    // As many stores as a tile's, all dropped: outside the resources that the loads come from, which
    // keeps the compiler from moving them before the loads.
    auto store_nothing = [&]() {
#pragma unroll
      for (int u = 0; u < kRows; ++u) put1(u & 1 ? py_rsrc : px_rsrc, kDropped + u * kSize, (R)0);
    };
    auto take = [&](Drained &d, int row0, int pm, int buf) {
      const R *xs = base + buf * kTileElems + r_first * kTilePitch + q;
      const R *ps = xs + kBuffers * kTileElems;
      d.row0 = row0;
      d.pm = pm;
#pragma unroll
      for (int u = 0; u < kRows; ++u) {
        if (r_first + kStep * u >= kWave) continue;
        d.v[u] = ps[u * kStep * kTilePitch];
        if constexpr (kShares) {
          d.below[u] = ps[(u * kStep - 1) * kTilePitch - 1 - shift];  // (row 0: not a cell's, replaced below)
          d.x[u] = xs[u * kStep * kTilePitch];
        }
      }
    };
    // The tile's last row, for the sweep wave below (one staging wave holds it): to the seam row, as
    // soon as the tile is done.
    constexpr int kLastL = (kWave / 2 - 1) % kPer, kLastU = (kWave / 2 - 1) / kPer;
    auto hand_on = [&](const Drained &d) -> bool {
      if (!kSeams || l != kLastL || d.row0 + kWave > NS) return true;  // (wave-uniform)
      const int col = d.pm * kTileSteps + q - (kWave - 1);
      if (half == 1 && (unsigned)col <= (unsigned)NT) my_seam[col] = d.v[kLastU];
      const int done = max(0, min(d.pm * kTileSteps + kTileSteps - (kWave - 1), cols));
      const int before = kApart ? 0 : (d.row0 / kWave - w) / nsweep * cols;
      int *ready = &cnt.ready[kApart ? 1 : w];
      // The tile before may be the other group's, which counts its columns in first.  (A tile without
      // columns counts nothing: that could come after, and would take back, what a later tile has counted.)
      if (kGroups > 1) {
        const int already = max(0, min(d.pm * kTileSteps - (kWave - 1), cols));
        if (done == already) return true;
        if (!wait_for(ready, before + already, spin_limit)) return false;
      }
      if (lane == 0) publish_lds_writes(ready, before + done);
      return true;
    };
    auto store = [&](const Drained &d) {
      const int i0 = d.row0 + r_first;
      const int j0 = d.pm * kTileSteps + q - r_first;
      const int o0 = (i0 * TP + win.t0 + j0) * kSize;
      R out[kRows];
#pragma unroll
      for (int u = 0; u < kRows; ++u) {
        out[u] = d.v[u];
        if constexpr (kShares) {
          // mutual_information_cpu.cu:196-212.  A band's first row has what comes from below in its x.
          const R below = u == 0 && r_first == 0 ? (R)0 : d.below[u];
          R total = d.v[u];
          if (total - total != 0) total = 0;
          out[u] = Num<R>::exp_(below + d.x[u] - total);
        }
      }
      if constexpr (kShares) {
        // column 0 hands everything down (:219-226), in the modified lattice nothing
        if (d.pm * kTileSteps < kWave)
#pragma unroll
          for (int u = 0; u < kRows; ++u)
            if (j0 == kStep * u) out[u] = kModified ? (R)0 : (R)1;
      }
#pragma unroll
      for (int u = 0; u < kRows; ++u) {
        const bool ok = (unsigned)(j0 - kStep * u) <= (unsigned)NT && r_first + kStep * u < kWave;
        put1(p_rsrc, ok ? o0 + u * (kStep * (TP - 1) * kSize) : kDropped, out[u]);
      }
    };
    // The tile that a buffer held before tile m of the band that starts at row0.  Bands that
    // another one follows have whole_tiles tiles, two at least, so that it lies two bands back at most.
    const int whole_tiles = (NT + kWave + kTileSteps - 1) / kTileSteps;
    auto take_buffer = [&](Drained &d, int row0, int m, int buf) {
      int pm = m - kBuffers;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        row0 = pm < 0 ? row0 - band_rows : row0;
        pm = pm < 0 ? pm + whole_tiles : pm;
      }
      take(d, row0, pm, buf);
    };
    int tile_base = 0;
    int end_row0 = 0, end_tiles = 0;
    for (int band = part; band * band_rows <= last_row; ++band) {
      const Band g = band_of(band, w, nsweep, NS, NT);
      if (g.row0 > NS) break;
      // A wave's memory accesses are counted off in their order, so that a wait for a load is also one
      // for every access issued before it, and for those issued after it that the compiler cannot count
      // on.  With one tile requested at a time, behind the stores of the tile before, a tile's staging
      // took the latency of both, longer than the sweep needs for a tile.  Here two tiles' inputs are on
      // their way, in two sets of registers, and on every path exactly one tile's loads and one tile's
      // stores follow each other -- dropped ones where there is nothing to fetch or to store, and a wait
      // that ran out ends the loop only after both halves -- so that the wait for a tile's inputs leaves
      // the later loads and stores on their way.  (B 64, S 120, T 600: 37.4 -> 32.2 us, 29.4 with no
      // stores at all; B 12, S 220, T 1500: 68.0 -> 65.7; B 32, S 80, T 250: 17.0 -> 16.2.)
      Staged ahead[kAhead];
      Drained out = {};
      out.pm = kNowhere;
#pragma unroll
      for (int k = 0; k < kAhead; ++k) {
        fetch(ahead[k], g, group + k * kGroups);
        store_nothing();
      }
      auto stage = [&](const Staged &cur, int m) __attribute__((always_inline)) -> bool {
        const int gt = tile_base + m, buf = gt % kBuffers;
        if (gt >= kBuffers) {
          // the buffer still holds p of tile gt - kBuffers
          if (!wait_for(&cnt.written[w], gt - kBuffers + 1, spin_limit)) {
            give_up();
            return false;
          }
          take_buffer(out, g.row0, m, buf);
          // (kShares: the row below a staging wave's is another one's, who must not refill it before)
          if (kShares && lane == 0) count_in(&cnt.taken[w * kBuffers + buf]);
          if (!hand_on(out) ||
              (kShares && !wait_for(&cnt.taken[w * kBuffers + buf], kPer * (gt / kBuffers), spin_limit))) {
            give_up();
            return false;
          }
        }
        // The row above the band belongs to another sweep wave: what it feeds into the band's first
        // row is added to that row's x here (the sweep would add it with the same rounding), so
        // that a sweep wave runs the same steps whether it has a wave above it or not.
        R seam_value = 0;
        if (kSeams && l == 0 && g.row0 > 0) {  // (wave-uniform)
          const int col = m * kTileSteps + q - shift;
          const bool there = half == 0 && col >= 0 && col <= NT;
          const int need = min((m + 1) * kTileSteps - shift, cols);
          const int before = kApart ? 0 : (w > 0 ? band : band - 1) * cols;
          if (need > 0 && !wait_for(&cnt.ready[prev], before + need, spin_limit)) {
            give_up();
            return false;
          }
          seam_value = ninf;
          if (there) seam_value = up_seam[col];
        }
        // (the wait for this tile's inputs, on every path through what follows)
#pragma unroll
        for (int u = 0; u < kRows; ++u) asm volatile("" ::"v"(cur.x[u]), "v"(cur.y[u]));
        R *xdst = base + buf * kTileElems + r_first * kTilePitch + q;
        R *ydst = xdst + kBuffers * kTileElems;
        // only the first tiles hold a column 0 (local step = row), and only the first
        // band holds row 0
        const bool starts = m * kTileSteps <= kWave - 1 + shift;
#pragma unroll
        for (int u = 0; u < kRows; ++u) {
          const int r = r_first + kStep * u;
          if (r >= kWave) continue;
          R x = cur.x[u], y = cur.y[u];
          const int i = g.row0 + r;
          if (starts) {
            const int j = m * kTileSteps + q - r;
            if (j <= 0) y = (j == 0 && i == 0) ? (R)0 : ninf;
            if (j < shift) x = ninf;
          }
          if (u == 0 && i == 0) x = ninf;
          if (kSeams && u == 0 && r == 0) x += seam_value;
          xdst[u * kStep * kTilePitch] = x;
          ydst[u * kStep * kTilePitch] = y;
        }
        // every lane's LDS writes precede the release by lane 0 of the same wave
        if (lane == 0) count_in(&cnt.loaded[w * kBuffers + buf]);
        return true;
      };
      bool failed = false;
      for (int m = group; m < g.ntiles; m += kAhead * kGroups) {
#pragma unroll
        for (int k = 0; k < kAhead; ++k) {
          if (m + k * kGroups < g.ntiles && !failed)
            failed = !stage(ahead[k], m + k * kGroups);
          else
            out.pm = kNowhere;
          fetch(ahead[k], g, m + (k + kAhead) * kGroups);
          asm volatile("" ::: "memory");
          store(out);
        }
        if (failed) return;
      }
      tile_base += g.ntiles;
      end_row0 = g.row0;
      end_tiles = g.ntiles;
    }
    // the tiles still in the buffers
    const int first_left = max(tile_base - kBuffers, 0);
    for (int gt = first_left; gt < tile_base; ++gt) {
      if (gt % kGroups != group) continue;
      Drained out;
      if (!wait_for(&cnt.written[w], gt + 1, spin_limit)) {
        give_up();
        return;
      }
      take_buffer(out, end_row0, gt - tile_base + end_tiles + kBuffers, gt % kBuffers);
      if (!hand_on(out)) {
        give_up();
        return;
      }
      store(out);
    }
    return;
  }

  // -------------------------------- sweep wave ---------------------------------
  const int w = wave;
  R *base = tiles + (size_t)w * 2 * kBuffers * kTileElems;
  int tile_base = 0, buf = 0, rounds = 0;  // tile number modulo kBuffers, and divided by it
  for (int band = part; band * band_rows <= last_row; ++band) {
    const Band g = band_of(band, w, nsweep, NS, NT);
    if (g.row0 > NS) break;
    const int i = g.row0 + lane;
    // the answer is the cell (NS, NT): lane NS - row0 at step NT + NS - row0
    const int fin_lane = NS - g.row0;
    const int fin_step = (fin_lane < kWave) ? NT + fin_lane : -1;

    R own = (i == 0) ? (R)0 : ninf, own2 = ninf;
    R fin = ninf;
    // the counter is read one tile ahead of its use, so that the LDS round trip is off the
    // chain; a stale value only costs a re-read
    int seen_loaded = 0;
    // One tile, specialised at compile time on kPlain: a tile whose 32 steps all exist and do
    // not hold the answer's step.  A single wave pays for every instruction it issues, scalar
    // tests and branches included, so plain tiles run without the tests; and either kind of tile
    // has a loop of its own (below): with both in one loop body the compiler's code for the steps
    // themselves took twice as long.
    auto one_tile = [&](int m, auto plain_c) __attribute__((always_inline)) -> bool {
      constexpr bool kPlain = decltype(plain_c)::value;
      const int gt = tile_base + m;
      constexpr int kPer = kStagers / kStagerGroups<kStagers, kShares>;
      if (__builtin_amdgcn_readfirstlane(seen_loaded) < kPer * (rounds + 1) &&
          !wait_for(&cnt.loaded[w * kBuffers + buf], kPer * (rounds + 1), spin_limit)) {
        give_up();
        return false;
      }
      // this lane's 32 steps of inputs go to registers in one burst
      R xq[kTileSteps], yq[kTileSteps];
      const R *x_row = base + buf * kTileElems + lane * kTilePitch;
      R *y_row = base + (kBuffers + buf) * kTileElems + lane * kTilePitch;  // y in, p out
      pull_row(xq, x_row);
      pull_row(yq, y_row);
      // the two steps before the tile's, in the two unused elements in front of the lane's row
      if constexpr (kShares) push_two(y_row - 2, own2, own);
      buf = buf + 1 == kBuffers ? 0 : buf + 1;
      rounds += buf == 0;

      R last[kChunk];  // the chunk before
#pragma unroll
      for (int k = 0; k < kChunk; ++k) last[k] = 0;
      // one chunk of kChunk steps
      auto chunk = [&](int c4, int e0) __attribute__((always_inline)) {
        if (c4 == kTileSteps / kChunk - 1) seen_loaded = peek(&cnt.loaded[w * kBuffers + buf]);
        R vals[kChunk];
#pragma unroll
        for (int k = 0; k < kChunk; ++k) {
          const int kk = c4 * kChunk + k;
          // lane 0 receives a 0: its x is -inf in lattice row 0, and holds what comes from the
          // row above elsewhere
          const R up = from_lane_below_zero(kModified ? own2 : own);
          const R v = chain_log_add(up + xq[kk], own + yq[kk]);
          vals[k] = v;
          own2 = own;
          own = v;
          if (k == kChunk / 2 - 1) {
            // the chunk's p takes the place of its y in the tile: first half
            push_half<0>(y_row + c4 * kChunk, vals);
            still_in_use(last, kChunk / 2);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
        still_in_use(vals, 0);
        if (!kPlain) {
          const int kf = fin_step - e0;  // wave-uniform
          if ((unsigned)kf < (unsigned)kChunk) {
#pragma unroll
            for (int k = 0; k < kChunk; ++k)
              if (k == kf) fin = vals[k];
          }
        }
        push_half<1>(y_row + c4 * kChunk, vals);
#pragma unroll
        for (int k = kChunk / 2; k < kChunk; ++k) last[k] = vals[k];
      };
#pragma unroll
      for (int c4 = 0; c4 < kTileSteps / kChunk; ++c4) {
        const int e0 = m * kTileSteps + c4 * kChunk;
        if (kPlain || e0 < g.nsteps) chunk(c4, e0);
      }
      if (lane == 0) publish_lds_writes(&cnt.written[w], gt + 1);
      return true;
    };
    // the band's tiles: the plain ones, then the rest
    const int plain = plain_tiles(g, fin_step, false, shift, NT).hi;
    for (int m = 0; m < plain; ++m)
      if (!one_tile(m, std::true_type{})) return;
    for (int m = plain; m < g.ntiles; ++m)
      if (!one_tile(m, std::false_type{})) return;
    if (kApart && lane == fin_lane) {
      // (one that gave up here or in another band's workgroup has stored, or will store, its NaN)
      if constexpr (kApart) store_once(&ans[b], kSeamMark, fin);
    } else if (fin_lane >= 0 && fin_lane < kWave) {  // (wave-uniform)
      R score = peek(&cnt.failed) ? std::numeric_limits<R>::quiet_NaN() : fin;
      if (lane == fin_lane) {
        store_score(score);
        // A staging wave may give up between that look and the store, and its NaN must not be
        // covered by the score: once the store has left, look again.  A wave that gives up
        // after this second look stores its NaN after it, and so after the score.
        if (__hip_atomic_load(&cnt.failed, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP)) {
          score = std::numeric_limits<R>::quiet_NaN();
          store_score(score);
        }
      }
      count_for_loss(score, fin_lane);
    }
    tile_base += g.ntiles;
  }
}

// =============================== backward ====================================
// Rows and columns are counted from the end of the window (r = NS - i,
// c = NT - j); lane L of a sweep wave owns reversed row r and works on reversed
// column e - L at local step e.  A cell's gradient is what the row above hands
// down plus what its right neighbour hands left; it is then split into a d1
// share for the cell below and a d2 share for the cell to the left.  The staging
// waves evaluate d1 / d2 (mutual_information_cpu.cu:196-212 and the two edge
// loops :219-235).  A single wave issues one instruction every 4-5 cycles, and a sweep
// wave that also computes addresses and stores its results spends ~140 cycles per
// step where the dependent chain (shift, add, multiply) needs ~25; so the sweep wave
// only leaves the px / py gradients of a tile in the LDS buffer it has just read that
// tile's d1 / d2 from (a lane's 32 steps, 16 bytes per write), and the staging waves
// carry them to memory, each for the rows it stages, before they refill the buffer.
// kApart, pitch: as in the forward kernel.
// kShares: the forward kernel has left d1 in `p`, borders and all.  The staging waves then only copy it to
// LDS, a third of the loads and no exp; the sweep wave takes d2 = 1 - d1 itself, off the chain, and leaves
// the cells' gradients, one value per cell in LDS instead of two; and the staging waves split those as they
// carry them to memory.  Same operations, same bits.  The forward kernel's staging waves, of which the
// sweep needs less, do the exp.  Both kernels and the marks, from p and px -> with shares, full windows: B 12, S 220,
// T 1500 139 -> 120 us; B 64, S 120, T 600 64.6 -> 58.4; B 32, S 80, T 250 33.6 -> 32.4 (17.1 + 16.5 -> 18.4 + 14.0);
// B 8, S 60, T 200 23.7 -> 21.7.
template <typename R, bool kModified, int kSweepCap, int kStagers, int kBuffers, bool kApart, bool kShares>
__global__ void __launch_bounds__(((1 + kStagers) * kSweepCap + (kApart ? 2 : 0) +
                                   kHelpers<kSweepCap, kShares>) * kWave)
    mi_backward_kernel(const R *__restrict__ px, const int64_t *__restrict__ boundary,
                       const R *__restrict__ p, R *ans_grad, R *__restrict__ px_grad,
                       R *__restrict__ py_grad, int S, int T, int seed_stride, int overwrite_ans_grad,
                       const R *__restrict__ scores, R *__restrict__ loss, int B, int reduction,
                       int spin_limit, int pitch, R *post) {
  extern __shared__ __align__(16) unsigned char dyn_lds[];
  __shared__ Counters cnt;

  const int b = kApart ? blockIdx.x % pitch : blockIdx.x, part = kApart ? blockIdx.x / pitch : 0;
  if (kApart && b >= B) return;
  constexpr int kHelp = kHelpers<kSweepCap, kShares>;
  const int nsweep = (blockDim.x / kWave - (kApart ? 2 : 0) - kHelp) / (1 + kStagers);
  const int nwaves = blockDim.x / kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);  // in a scalar register
  const int lane = threadIdx.x % kWave;
  const int T1 = kModified ? T : T + 1;
  const int TP = T + 1;
  const int shift = kModified ? 1 : 0;

  const Window win = load_window(boundary, b, S, T);
  R *gxb = px_grad + (size_t)b * S * T1;
  R *gyb = py_grad + (size_t)b * (S + 1) * T;
  const __amdgpu_buffer_rsrc_t gx_rsrc = buffer_of(gxb, (size_t)S * T1);
  const __amdgpu_buffer_rsrc_t gy_rsrc = buffer_of(gyb, (size_t)(S + 1) * T);

  const R seed = ans_grad ? ans_grad[(size_t)b * seed_stride] : (R)1;
  // What a cell without a gradient holds.  mi_backward takes a seed as it is: 0.  The pair that passes shares stands for
  // gradients of ones that are scaled afterwards, all of them: 0 times the seed, NaN if that is not finite.
  const R nothing = kShares ? seed - seed : (R)0;
  // That everywhere the sweep does not write, by wave `part` of `parts`, off the critical path (a
  // barrier after these stores would have to wait until they have all reached memory).  An array's
  // window leaves a run before it, one after it and, all of one length, those between its rows: four rows'
  // to an instruction, 16 lanes each (row by row, with a run's ends tested for each, two waves took
  // longer than the sweep: 24 000 cycles at S 80, T 250, a third of it outside).
  auto zero_run = [&](__amdgpu_buffer_rsrc_t rs, int begin, int end, int first, int lanes) {
    // elements [begin, end), by lanes `first` .. of `lanes` that step through it together; overlapping the
    // last four, so that all stores are whole
    const R z = nothing;
    if (end - begin < 4) {
      put1(rs, first < end - begin ? (begin + first) * (int)sizeof(R) : kDropped, z);
      return;
    }
    for (int t = begin + 4 * first; t - 4 * first < end; t += 4 * lanes)
      put4(rs, t < end ? min(t, end - 4) * (int)sizeof(R) : kDropped, z, z, z, z);
  };
  // rows [r_lo, r_hi) and columns [lo, hi) of the array's rows x width are the sweep's
  auto zero_around = [&](__amdgpu_buffer_rsrc_t rs, int rows, int width, int r_lo, int r_hi, int lo, int hi,
                         int part, int parts) {
    if (r_hi <= r_lo) {
      zero_run(rs, 0, rows * width, part * kWave + lane, parts * kWave);
      return;
    }
    zero_run(rs, 0, r_lo * width + lo, part * kWave + lane, parts * kWave);
    zero_run(rs, (r_hi - 1) * width + hi, rows * width, part * kWave + lane, parts * kWave);
    const int gap = width - hi + lo, q = lane & 15;
    if (gap <= 0) return;
    for (int r = r_lo + 4 * part; r < r_hi - 1; r += 4 * parts) {
      const int row = r + (lane >> 4), begin = row * width + hi;
      const bool there = row < r_hi - 1;
      if (gap < 4) {
        put1(rs, there && q < gap ? (begin + q) * (int)sizeof(R) : kDropped, nothing);
      } else {
        for (int t = 4 * q; t - 4 * q < gap; t += 64)
          put4(rs, there && t < gap ? (begin + min(t, gap - 4)) * (int)sizeof(R) : kDropped, nothing,
               nothing, nothing, nothing);
      }
    }
  };
  auto zero_outside = [&](int part, int parts) {
    if (!boundary) return;
    const int s_hi = win.ok ? win.s0 + win.ns : 0, s_lo = win.ok ? win.s0 : 0;
    const int t_hi = win.t0 + win.nt;
    zero_around(gx_rsrc, S, T1, s_lo, s_hi, win.t0, t_hi - shift + 1, part, parts);
    zero_around(gy_rsrc, S + 1, T, s_lo, win.ok ? s_hi + 1 : 0, win.t0, t_hi, part, parts);
  };
  if (kApart && part > 0 && (!win.ok || part * kWave > win.ns)) return;
  if (!win.ok) {
    zero_outside(wave, nwaves);
    if (loss && b == 0 && wave == 0) reduce_scores(scores, loss, B, reduction, lane);
    return;
  }
  if (threadIdx.x < (int)(sizeof(Counters) / sizeof(int)))
    reinterpret_cast<int *>(&cnt)[threadIdx.x] = 0;
  __syncthreads();

  const int NS = win.ns, NT = win.nt, cols = NT + 1;
  const int band_rows = kWave * nsweep;
  const int last_row = kApart ? part * kWave : NS;  // (of those that may begin a band here)
  const R *pxb = px + (size_t)b * S * T1;
  const R *pb = p + (size_t)b * (S + 1) * TP;
  R *seam = reinterpret_cast<R *>(dyn_lds);
  const int seam_pitch = (TP + kSeamSlack + 3) & ~3;  // keeps the tiles 16-byte aligned
  // (apart: the seam that comes in, and the one that goes out)
  R *tiles = seam + (size_t)(kApart ? 2 : nsweep) * seam_pitch;  // per sweep wave: kBuffers d1 tiles, then as many d2 tiles
  // (apart) per buffer: what the row above the band hands to the tile's steps
  R *handed_down = tiles + (size_t)nsweep * 2 * kBuffers * kTileElems;
  // A wave whose bounded wait ran out leaves NaN where the window starts -- in px_grad,
  // in py_grad and, when it is written back, in ans_grad -- so that the utterance's
  // gradients cannot pass for a result; every staging wave repeats that when it is done
  // and finds the mark, so no later store of a good value covers it up.  (apart: and where the
  // band's first row starts, because another workgroup, which does not see the mark, may store
  // the window's start later; nobody else stores the band's rows.)
  auto poison = [&]() {
    if (lane != 0) return;
    const R nan = std::numeric_limits<R>::quiet_NaN();
    if (NS > 0 && NT >= shift) put1(gx_rsrc, (win.s0 * T1 + win.t0) * (int)sizeof(R), nan);
    if (NT > 0) put1(gy_rsrc, (win.s0 * T + win.t0) * (int)sizeof(R), nan);
    if constexpr (kApart) {
      const int i = NS - part * kWave;  // the band's first row
      if (i > 0 && NT >= shift)
        put1(gx_rsrc, ((win.s0 + i - 1) * T1 + win.t0) * (int)sizeof(R), nan);
      if (NT > 0) put1(gy_rsrc, ((win.s0 + i) * T + win.t0) * (int)sizeof(R), nan);
      if (overwrite_ans_grad && ans_grad) store_nan(&ans_grad[b]);
    } else {
      if (overwrite_ans_grad && ans_grad) ans_grad[b] = nan;
    }
  };
  auto give_up = [&]() {
    if (lane == 0) publish(&cnt.failed, 1);
    poison();
  };

  if (kHelp > 0 && wave >= nwaves - kHelp) {
    // -------------------------------- helpers ------------------------------------
    const int parts = kApart ? (NS + kWave) / kWave : 1;  // (the bands' workgroups)
    zero_outside(part * kHelp + nwaves - 1 - wave, parts * kHelp);
    if (loss && b == 0 && part == 0 && wave == nwaves - 1) reduce_scores(scores, loss, B, reduction, lane);
    return;
  }
  if (kApart && wave >= 1 + kStagers) {
    // ------------------------------- courier waves -------------------------------
    // where the gradients that band `of` hands down pass: through its last row of px_grad, from the end, or the post
    const bool posted = kShares && post != nullptr;
    const int stride = posted ? 1 : -1;
    auto seam_row = [&](int of) -> R * {
      if (posted) return post_row(post, b, of, S, T);
      return gxb + (size_t)(win.s0 + NS - (of + 1) * kWave) * T1 + win.t0 + NT - shift;
    };
    if (wave == 1 + kStagers) {
      if ((part + 1) * kWave <= NS && !send_seam(seam_row(part), stride, cols - shift, seam + seam_pitch,
                                                 &cnt.ready[1], lane, spin_limit))
        give_up();
      return;
    }
    if (part > 0 && !bring_seam(seam_row(part - 1), stride, cols - shift, seam, &cnt.ready[0], lane, spin_limit,
                                posted))
      give_up();
    return;
  }
  if (wave >= nsweep) {
    // ------------------------------ staging wave -------------------------------
    constexpr int kGroups = kStagerGroups<kStagers, kShares>, kPer = kStagers / kGroups;
    const int w = (wave - nsweep) / kStagers, l = (wave - nsweep) % kPer;
    const int group = (wave - nsweep) % kStagers / kPer;  // as in the forward kernel
    R *base = tiles + (size_t)w * 2 * kBuffers * kTileElems;
    const int half = lane >> 5, q = lane & 31;
    // rows of a tile this wave stages: r(u) = 2*l + half + 2*kPer*u
    constexpr int kRows = (kWave + 2 * kPer - 1) / (2 * kPer);
    struct Staged {
      R here[kRows], below[kRows], x[kRows];  // (kShares: here = d1, and nothing else)
    };
    // Global fetches of tile m+1 are issued (into registers) as soon as tile m is staged,
    // before this wave waits for the next LDS buffer, so their latency overlaps the
    // sweep.  The loads are range-checked and otherwise unconditional; staging replaces
    // what was read for cells outside the window.
    const __amdgpu_buffer_rsrc_t p_rsrc = buffer_of(const_cast<R *>(pb), (size_t)(S + 1) * TP);
    const __amdgpu_buffer_rsrc_t px_rsrc = buffer_of(const_cast<R *>(pxb), (size_t)S * T1);
    constexpr int kStep = 2 * kPer;
    constexpr int kSize = (int)sizeof(R);
    const int r_first = 2 * l + half;
    auto fetch = [&](Staged &in, const Band &g, int m) {
      // element offsets of row u = 0; each further u is kStep rows up the reversed
      // lattice, i.e. that many rows down in memory and as many columns right
      const int s_first = win.s0 + NS - (g.row0 + r_first);
      const int j_first = NT - (m * kTileSteps + q - r_first);
      const int below0 = ((s_first - 1) * TP + win.t0 + j_first - shift) * kSize;
      const int x0 = ((s_first - 1) * T1 + win.t0 + j_first - shift) * kSize;
      const int here0 = (s_first * TP + win.t0 + j_first) * kSize;
#pragma unroll
      for (int u = 0; u < kRows; ++u) {
        in.below[u] = get1(p_rsrc, below0 - u * (kStep * (TP - 1) * kSize), R());
        in.x[u] = get1(px_rsrc, x0 - u * (kStep * (T1 - 1) * kSize), R());
        in.here[u] = get1(p_rsrc, here0 - u * (kStep * (TP - 1) * kSize), R());
      }
    };
    // Gradients of tile m of band g, left by the sweep wave in buffer `buf`: element
    // (row r, step q) is the cell in reversed column c = 32 m + q - r, i.e. column
    // j = NT - c of lattice row i = NS - (row0 + r); gx goes to px_grad[s-1][t0 + j - shift],
    // gy to py_grad[s][t0 + j - 1], where those exist (mutual_information_cpu.cu:213-216).
    // The straight-line form below (every row group handled alike, borders by select) is
    // faster than variants that skip the rows past the window's top or branch to a
    // mask-free copy for tiles inside the window: those were 1 to 5 us slower per launch.
    // Taking a tile's gradients out of the buffer and storing them are two steps: a wave's
    // wait for a load also waits for every store it has issued before, so the stores go
    // out after the buffer has been refilled and handed back to the sweep wave.
    struct Drained {
      R vx[kRows], vy[kRows];
      int row0, pm;
    };
    auto take = [&](Drained &d, int pg_row0, int pm, int buf) {
      const R *gxs = base + buf * kTileElems + r_first * kTilePitch + q;
      const R *gys = gxs + kBuffers * kTileElems;
      d.row0 = pg_row0;
      d.pm = pm;
#pragma unroll
      for (int u = 0; u < kRows; ++u) {
        if (r_first + kStep * u >= kWave) continue;
        d.vx[u] = gxs[u * kStep * kTilePitch];
        d.vy[u] = gys[u * kStep * kTilePitch];
      }
    };
    // (kShares) what a tile holds are d1 and the cells' gradients, 0 where d1 is kNoShares; the + 0 makes a
    // -0 of that 0
    auto split = [&](Drained &d) {
      if constexpr (kShares)
#pragma unroll
        for (int u = 0; u < kRows; ++u) {
          const R d1 = d.vx[u], cell = d.vy[u];
          d.vx[u] = d1 * cell;
          d.vy[u] = __builtin_fmaf((R)1 - d1, cell, (R)0);
        }
    };
    // (apart) The gradients that the tile's last row hands down go to the outgoing seam as soon as
    // the tile is done: the workgroup of the next band waits for them.
    constexpr int kLastL = (kWave / 2 - 1) % kPer, kLastU = (kWave / 2 - 1) / kPer;
    auto hand_on = [&](const Drained &d) -> bool {
      if (!kApart || l != kLastL || d.row0 + kWave > NS) return true;  // (wave-uniform)
      const int col = d.pm * kTileSteps + q - (kWave - 1);
      if (half == 1 && (unsigned)col <= (unsigned)NT) seam[seam_pitch + col] = kShares ? d.vx[kLastU] * d.vy[kLastU] : d.vx[kLastU];
      const int done = max(0, min(d.pm * kTileSteps + kTileSteps - (kWave - 1), cols));
      if (kGroups > 1) {  // as in the forward kernel
        const int already = max(0, min(d.pm * kTileSteps - (kWave - 1), cols));
        if (done == already) return true;
        if (!wait_for(&cnt.ready[1], already, spin_limit)) return false;
      }
      if (lane == 0) publish_lds_writes(&cnt.ready[1], done);
      return true;
    };
    auto store = [&](const Drained &d) {
      constexpr int kMinX = kModified ? 1 : 0;
      const int i0 = NS - d.row0 - r_first;                   // lattice row of u = 0
      const int j0 = NT - (d.pm * kTileSteps + q - r_first);  // and its column
      const int x0 = ((win.s0 + i0 - 1) * T1 + win.t0 - shift + j0) * kSize;
      const int y0 = ((win.s0 + i0) * T + win.t0 - 1 + j0) * kSize;
#pragma unroll
      for (int u = 0; u < kRows; ++u) {
        if (r_first + kStep * u >= kWave) continue;
        // one row group further: kStep rows up in memory and as many columns right
        const int xo = x0 - u * (kStep * (T1 - 1) * kSize), yo = y0 - u * (kStep * (T - 1) * kSize);
        const int i = i0 - kStep * u, j = j0 + kStep * u;
        const bool okx = i > 0 && (unsigned)(j - kMinX) < (unsigned)(NT + 1 - kMinX);
        const bool oky = i >= 0 && (unsigned)(j - 1) < (unsigned)NT;
        put1(gx_rsrc, okx ? xo : kDropped, d.vx[u]);
        put1(gy_rsrc, oky ? yo : kDropped, d.vy[u]);
      }
    };
    // which tile each buffer holds: its band's first row and its number in the band
    int held_row0[kBuffers], held_m[kBuffers];
#pragma unroll
    for (int k = 0; k < kBuffers; ++k) held_row0[k] = held_m[k] = 0;
    auto take_buffer = [&](Drained &d, int buf) {
      int row0 = held_row0[0], pm = held_m[0];
#pragma unroll
      for (int k = 1; k < kBuffers; ++k) {
        row0 = buf == k ? held_row0[k] : row0;
        pm = buf == k ? held_m[k] : pm;
      }
      take(d, row0, pm, buf);
    };
    int tile_base = 0, buf = 0;  // buf = tile number modulo kBuffers
    bool zeroed = false;
    if constexpr (kShares) {
      // As in the forward kernel: several tiles' d1 are on their way, each in a set of registers, and one
      // tile's loads and one tile's stores follow each other on every path.
      auto request = [&](Staged &in, const Band &g, int m) {
        const int s_first = win.s0 + NS - (g.row0 + r_first);
        const int j_first = NT - (m * kTileSteps + q - r_first);
        const int at = m < g.ntiles ? (s_first * TP + win.t0 + j_first) * kSize : kDropped;
#pragma unroll
        for (int u = 0; u < kRows; ++u) in.here[u] = get1(p_rsrc, at - u * (kStep * (TP - 1) * kSize), R());
      };
      constexpr int kAhead = kGroups > 1 ? 1 : kFetchAhead<R>;
      constexpr int kNowhere = -(1 << 20);  // (a tile with no cell in the window)
      // the tile that a buffer held before tile m of the band that starts at row0
      const int whole_tiles = (NT + kWave + kTileSteps - 1) / kTileSteps;
      auto take_before = [&](Drained &d, int row0, int m, int buf) {
        int pm = m - kBuffers;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          row0 = pm < 0 ? row0 - band_rows : row0;
          pm = pm < 0 ? pm + whole_tiles : pm;
        }
        take(d, row0, pm, buf);
      };
      int end_row0 = 0, end_tiles = 0;
      for (int band = part; band * band_rows <= last_row; ++band) {
        const Band g = band_of(band, w, nsweep, NS, NT);
        if (g.row0 > NS) break;
        Staged ahead[kAhead];
        Drained out = {};
        out.pm = kNowhere;
#pragma unroll
        for (int k = 0; k < kAhead; ++k) {
          request(ahead[k], g, group + k * kGroups);
#pragma unroll
          for (int u = 0; u < 2 * kRows; ++u) put1(p_rsrc, kDropped + u * kSize, (R)0);
        }
        auto stage = [&](const Staged &cur, int m) __attribute__((always_inline)) -> bool {
          const int gt = tile_base + m, buf = gt % kBuffers;
          if (gt >= kBuffers) {
            // the buffer still holds the gradients of tile gt - kBuffers
            if (!wait_for(&cnt.written[w], gt - kBuffers + 1, spin_limit)) return false;
            take_before(out, g.row0, m, buf);
            if (!hand_on(out)) return false;
          }
          if (kApart && l == 0 && g.row0 > 0) {  // (wave-uniform) the row above is another workgroup's
            const int col = m * kTileSteps + q - shift;
            const int need = min((m + 1) * kTileSteps - shift, cols - shift);
            if (need > 0 && !wait_for(&cnt.ready[0], need, spin_limit)) return false;
            R v = 0;
            if (half == 0 && col >= 0 && col < cols - shift) v = seam[col];
            if (half == 0) handed_down[buf * kTileSteps + q] = v;
          }
          // (the wait for this tile's inputs, on every path through what follows)
#pragma unroll
          for (int u = 0; u < kRows; ++u) asm volatile("" ::"v"(cur.here[u]));
          R *dst = base + buf * kTileElems + r_first * kTilePitch + q;
          // (cells outside the window: any finite value)
          unsigned most = 0;
#pragma unroll
          for (int u = 0; u < kRows; ++u) {
            if (r_first + kStep * u >= kWave) continue;
            const unsigned d1 = min(__float_as_uint(cur.here[u]), kNoShares);
            most = max(most, d1);
            dst[u * kStep * kTilePitch] = __uint_as_float(d1);
          }
          // cells of the window that pass nothing on, if there are any: the sweep then looks at each cell
          if (__ballot(most == kNoShares)) {
            bool there = false;
#pragma unroll
            for (int u = 0; u < kRows; ++u) {
              const int r = r_first + kStep * u;
              there = there || (r < kWave && g.row0 + r <= NS && __float_as_uint(cur.here[u]) >= kNoShares &&
                                (unsigned)(m * kTileSteps + q - r) <= (unsigned)NT);
            }
            if (__ballot(there) && lane == 0)
              __hip_atomic_fetch_or(&cnt.loaded[w * kBuffers + buf], kNoSharesHere, __ATOMIC_RELAXED,
                                    __HIP_MEMORY_SCOPE_WORKGROUP);
          }
          // every lane's LDS writes precede the release by lane 0 of the same wave
          if (lane == 0) count_in(&cnt.loaded[w * kBuffers + buf]);
          return true;
        };
        bool failed = false;
        for (int m = group; m < g.ntiles; m += kAhead * kGroups) {
#pragma unroll
          for (int k = 0; k < kAhead; ++k) {
            if (m + k * kGroups < g.ntiles && !failed)
              failed = !stage(ahead[k], m + k * kGroups);
            else
              out.pm = kNowhere;
            request(ahead[k], g, m + (k + kAhead) * kGroups);
            asm volatile("" ::: "memory");
            split(out);
            store(out);
          }
          if (failed) {
            give_up();
            return;
          }
          if (kHelp == 0 && !zeroed && m + kAhead * kGroups >= kBuffers) {
            // the sweep wave is that many tiles behind now: time for the zeros around the window
            if (part == 0) zero_outside(wave - nsweep, nsweep * kStagers);
            zeroed = true;
          }
        }
        tile_base += g.ntiles;
        end_row0 = g.row0;
        end_tiles = g.ntiles;
      }
      // the tiles still in the buffers
      for (int gt = max(tile_base - kBuffers, 0); gt < tile_base; ++gt) {
        if (gt % kGroups != group) continue;
        Drained out;
        if (!wait_for(&cnt.written[w], gt + 1, spin_limit)) {
          give_up();
          return;
        }
        take_before(out, end_row0, gt - tile_base + end_tiles + kBuffers, gt % kBuffers);
        if (!hand_on(out)) {
          give_up();
          return;
        }
        split(out);
        store(out);
      }
      if (kHelp == 0) {
        if (!zeroed && part == 0) zero_outside(wave - nsweep, nsweep * kStagers);
        if (loss && b == 0 && part == 0 && wave == nsweep) reduce_scores(scores, loss, B, reduction, lane);
      }
      if (peek(&cnt.failed)) poison();
      return;
    }
    for (int band = part; band * band_rows <= last_row && !kShares; ++band) {
      const Band g = band_of(band, w, nsweep, NS, NT);
      if (g.row0 > NS) break;
      Staged cur;
      fetch(cur, g, 0);
      for (int m = 0; m < g.ntiles; ++m) {
        const int gt = tile_base + m;
        Drained out;
        const bool refill = gt >= kBuffers;
        if (refill) {
          // the buffer still holds the gradients of tile gt - kBuffers
          if (!wait_for(&cnt.written[w], gt - kBuffers + 1, spin_limit)) {
            give_up();
            return;
          }
          take_buffer(out, buf);
          hand_on(out);
        }
#pragma unroll
        for (int k = 0; k < kBuffers; ++k) {
          held_row0[k] = buf == k ? g.row0 : held_row0[k];
          held_m[k] = buf == k ? m : held_m[k];
        }
        if (kApart && l == 0 && g.row0 > 0) {  // (wave-uniform) the row above is another workgroup's
          const int col = m * kTileSteps + q - shift;
          const int need = min((m + 1) * kTileSteps - shift, cols - shift);
          if (need > 0 && !wait_for(&cnt.ready[0], need, spin_limit)) {
            give_up();
            return;
          }
          R v = 0;
          if (half == 0 && col >= 0 && col < cols - shift) v = seam[col];
          if (half == 0) handed_down[buf * kTileSteps + q] = v;
        }
        R *d1dst = base + buf * kTileElems + r_first * kTilePitch + q;
        R *d2dst = d1dst + kBuffers * kTileElems;
        // Only two borders of the window need care here.  Column 0 hands everything down
        // (mutual_information_cpu.cu:219-226; nothing at all in the modified lattice) and
        // the top row hands everything left (:228-235).  Everywhere else outside the
        // window the sweep needs no zeros: cells a row passes before its first column keep
        // a gradient of exactly 0 (nothing has reached them, and d1 / d2 are finite), and
        // what is computed past column 0 or above the top row only feeds cells further
        // out, none of which is stored or handed to another wave.
        const int at_col0 = NT - m * kTileSteps;  // q - r of the cells in column 0
        const int top_r = NS - g.row0;            // the top row, if it lies in this band
#pragma unroll
        for (int u = 0; u < kRows; ++u) {
          const int r = r_first + kStep * u;
          if (r >= kWave) continue;
          // mutual_information_cpu.cu:196-212
          const R term1 = cur.below[u] + cur.x[u];
          R total = cur.here[u];
          if (total - total != 0) total = 0;
          R d1 = Num<R>::exp_(term1 - total);
          R d2 = (R)1 - d1;
          if (d1 - d1 != 0) d1 = d2 = 0;
          if (q - r == at_col0) d1 = kModified ? (R)0 : (R)1;
          if (r == top_r) d2 = 1;
          d1dst[u * kStep * kTilePitch] = d1;
          d2dst[u * kStep * kTilePitch] = d2;
        }
        // every lane's LDS writes precede the release by lane 0 of the same wave
        if (lane == 0) count_in(&cnt.loaded[w * kBuffers + buf]);
        if (refill) store(out);
        // the next tile's inputs, fetched while this wave waits for its buffer
        if (m + 1 < g.ntiles) fetch(cur, g, m + 1);
        buf = buf + 1 == kBuffers ? 0 : buf + 1;
        if (gt == kBuffers - 1) {
          // the sweep wave is that many tiles behind now: time for the zeros around the window
          if (part == 0) zero_outside(wave - nsweep, nsweep * kStagers);
          zeroed = true;
        }
      }
      tile_base += g.ntiles;
    }
    // the tiles still in the buffers
    const int first_left = max(tile_base - kBuffers, 0);
    buf = first_left % kBuffers;
    for (int gt = first_left; gt < tile_base; ++gt) {
      if (!wait_for(&cnt.written[w], gt + 1, spin_limit)) {
        give_up();
        return;
      }
      Drained out;
      take_buffer(out, buf);
      hand_on(out);
      store(out);
      buf = buf + 1 == kBuffers ? 0 : buf + 1;
    }
    if (!zeroed && part == 0) zero_outside(wave - nsweep, nsweep * kStagers);
    if (peek(&cnt.failed)) poison();
    // the loss, if asked for: the scores are the forward kernel's, complete before this
    // kernel started, and this wave has nothing left to do
    if (loss && b == 0 && part == 0 && wave == nsweep) reduce_scores(scores, loss, B, reduction, lane);
    return;
  }

  // -------------------------------- sweep wave ---------------------------------
  const int w = wave;
  const int prev = (w + nsweep - 1) % nsweep;
  R *my_seam = seam + (size_t)w * seam_pitch + kSeamPadLeft;
  const R *up_seam = seam + (size_t)prev * seam_pitch + kSeamPadLeft;
  R *base = tiles + (size_t)w * 2 * kBuffers * kTileElems;
  int tile_base = 0, buf = 0, rounds = 0;  // tile number modulo kBuffers, and divided by it
  for (int band = part; band * band_rows <= last_row; ++band) {
    const Band g = band_of(band, w, nsweep, NS, NT);
    if (g.row0 > NS) break;
    const int r = g.row0 + lane;
    const bool has_up = g.row0 > 0;
    const int up_base = (w > 0 ? band : band - 1) * cols;
    const int my_base = band * cols;
    // the gradient of the origin cell: lane NS - row0 at step NT + NS - row0
    const int fin_lane = NS - g.row0;
    const int fin_step = (fin_lane < kWave) ? NT + fin_lane : -1;

    // the seed enters as "handed left" into the first cell of the reversed sweep
    // (shares: a seed that is not finite makes cells that it does not reach NaN as well)
    R to_below = nothing, to_below2 = nothing, to_left = (r == 0) ? seed : nothing;
    R g_origin = 0;
    const R *seam_at = up_seam + (lane - shift);  // seam_at[e]: what lane 0 needs at step e + lane
    // rows below this wave's: someone reads the seam
    const bool has_down = !kApart && g.row0 + kWave <= NS;
    int seen_ready = 0;
    R seen_seam = 0;
    int seen_loaded = 0;
    // waits until the tile is staged; kShares: and notes whether any so far held a cell that passes nothing
    // on, which only the tiles that are not plain look for
    bool some_keep = false;
    auto staged = [&]() __attribute__((always_inline)) -> bool {
      constexpr int kMask = kShares ? kNoSharesHere - 1 : -1;
      constexpr int kPer = kStagers / kStagerGroups<kStagers, kShares>;
      int *loaded = &cnt.loaded[w * kBuffers + buf];
      int seen = __builtin_amdgcn_readfirstlane(seen_loaded);
      for (int spins = 0; (seen & kMask) < kPer * (rounds + 1);) {
        seen = __builtin_amdgcn_readfirstlane(
            __hip_atomic_load(loaded, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP));
        if ((seen & kMask) >= kPer * (rounds + 1)) break;
        __builtin_amdgcn_s_sleep(1);
        if (++spins > spin_limit) {
          give_up();
          return false;
        }
      }
      some_keep = kShares && (seen & kNoSharesHere) != 0;
      seen_loaded = seen;  // (asked again where a loop of plain tiles ends before its time)
      return true;
    };
    // one tile, specialised at compile time on whether the wave takes from a seam (kUp) and feeds
    // one (kDown), and on kPlain, with a loop for each kind, for the forward kernel's reasons
    auto one_tile = [&](int m, auto up_c, auto down_c, auto plain_c) __attribute__((always_inline)) -> bool {
      constexpr bool kUp = decltype(up_c)::value;
      constexpr bool kDown = decltype(down_c)::value;
      constexpr bool kPlain = decltype(plain_c)::value;
      const int gt = tile_base + m;
      R d1q[kTileSteps], d2q[kShares ? 1 : kTileSteps];
      const R *handed_at = handed_down + buf * kTileSteps;
      R arrived[kChunk];  // (apart) what lane 0 receives in the chunk's steps
      if constexpr (kApart && kUp) pull_chunk(arrived, handed_at);
      R *gx_row = base + buf * kTileElems + lane * kTilePitch;               // d1 in, gx out
      R *gy_row = base + (kBuffers + buf) * kTileElems + lane * kTilePitch;  // d2 in, gy out
      // (kShares: d1 in and left there; cells out)
      buf = buf + 1 == kBuffers ? 0 : buf + 1;
      rounds += buf == 0;
      pull_row(d1q, gx_row);
      if constexpr (!kShares) pull_row(d2q, gy_row);

      bool failed = false;
      auto chunk = [&](int c4, int e0) __attribute__((always_inline)) {
        R handed = 0, next[kChunk];
        if constexpr (kApart && kUp) {
          if (c4 + 1 < kTileSteps / kChunk) {
            pull_chunk(next, handed_at + (c4 + 1) * kChunk);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
        if (kUp && !kApart) {
          const int need = kPlain ? e0 + kChunk - shift : min(e0 + kChunk - shift, cols);
          handed = seen_seam;
          if ((kPlain || need > 0) && __builtin_amdgcn_readfirstlane(seen_ready) < up_base + need) {
            // (a wait that has run out is not tried again: the tile is finished on whatever the
            // seam holds, and the wave gives up afterwards)
            if (!failed && !wait_for(&cnt.ready[prev], up_base + need, spin_limit)) failed = true;
            const int col = e0 + lane - shift;
            handed = (lane < kChunk && col >= 0 && col <= NT) ? up_seam[col] : (R)0;
            lds_reads_done();
          }
          // next chunk's counter, then its seam values (LDS serves a wave in order)
          seen_ready = peek(&cnt.ready[prev]);
          if (kPlain) {
            seen_seam = seam_at[e0 + kChunk];  // every column exists; lanes 8 .. 63 do not matter
          } else {
            const int col = e0 + kChunk + lane - shift;
            seen_seam = 0;
            if (lane < kChunk && col >= 0 && col <= NT) seen_seam = up_seam[col];
          }
          // (the reads above are for the next chunk: they are issued here, before the steps)
          __builtin_amdgcn_sched_barrier(0);
        }
        if (c4 == kTileSteps / kChunk - 1) seen_loaded = peek(&cnt.loaded[w * kBuffers + buf]);
        R down[kChunk], left[kChunk], cell[kChunk];
#pragma unroll
        for (int k = 0; k < kChunk; ++k) {
          const int kk = c4 * kChunk + k;
          R from_above;
          if (kUp && kApart) {
            from_above = from_lane_below_or(kModified ? to_below2 : to_below, arrived[k]);
          } else if (kUp) {
            from_above = from_lane_below_or(kModified ? to_below2 : to_below, handed);
            handed = from_lane_above(handed);
          } else {
            from_above = from_lane_below_zero(kModified ? to_below2 : to_below);
          }
          // cells outside the window carry d1 = d2 = 0, so nothing leaks in or out
          cell[k] = from_above + to_left;
          if constexpr (kShares && !kPlain) cell[k] = d1q[kk] == __uint_as_float(kNoShares) ? (R)0 : cell[k];
          down[k] = d1q[kk] * cell[k];
          left[k] = (kShares ? (R)1 - d1q[kk] : d2q[kShares ? 0 : kk]) * cell[k];
          to_below2 = to_below;
          to_below = down[k];
          to_left = left[k];
          if (k == kChunk / 2 - 1) {
            // the chunk's gradients take the place of its d1 / d2 in the tile: first half
            if constexpr (!kShares) push_half<0>(gx_row + c4 * kChunk, down);
            push_half<0>(gy_row + c4 * kChunk, kShares ? cell : left);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
        if (!kPlain) {
          const int kf = fin_step - e0;  // wave-uniform
          if ((unsigned)kf < (unsigned)kChunk) {
#pragma unroll
            for (int k = 0; k < kChunk; ++k)
              if (k == kf) g_origin = cell[k];
          }
        }
        // seam: the last lane's reversed columns e0 - 63 ... (the pads take what falls
        // outside)
        if (kDown && e0 + kChunk > kWave - 1) {
          if (lane == kWave - 1) {
            push_chunk(my_seam + (e0 - (kWave - 1)), down);
            const int done = max(0, min(e0 + kChunk - (kWave - 1), cols));
            publish_lds_writes(&cnt.ready[w], my_base + done);
          }
        }
        if constexpr (!kShares) push_half<1>(gx_row + c4 * kChunk, down);
        push_half<1>(gy_row + c4 * kChunk, kShares ? cell : left);
        if constexpr (kApart && kUp) {
          if (c4 + 1 < kTileSteps / kChunk)
#pragma unroll
            for (int k = 0; k < kChunk; ++k) arrived[k] = next[k];
        }
      };
#pragma unroll
      for (int c4 = 0; c4 < kTileSteps / kChunk; ++c4) {
        const int e0 = m * kTileSteps + c4 * kChunk;
        // the window's edges need no care here: d1 = d2 = 0 outside it
        if (kPlain || e0 < g.nsteps) chunk(c4, e0);
      }
      if (failed) {
        give_up();
        return false;
      }
      if (lane == 0) publish_lds_writes(&cnt.written[w], gt + 1);
      return true;
    };
    auto sweep_tiles = [&](auto up_c, auto down_c) __attribute__((always_inline)) -> bool {
      const PlainTiles plain = plain_tiles(g, fin_step, !kApart && decltype(up_c)::value, shift, NT);
      int m = 0;
      for (; m < plain.lo; ++m)
        if (!staged() || !one_tile(m, up_c, down_c, std::false_type{})) return false;
      for (; m < plain.hi; ++m) {
        if (!staged()) return false;
        if (kShares && some_keep) break;
        if (!one_tile(m, up_c, down_c, std::true_type{})) return false;
      }
      for (; m < g.ntiles; ++m)
        if (!staged() || !one_tile(m, up_c, down_c, std::false_type{})) return false;
      return true;
    };
    bool done;
    if constexpr (!kApart && kSweepCap == 1)  // (lattices of one band)
      done = sweep_tiles(std::false_type{}, std::false_type{});
    else if (has_up)
      done = has_down ? sweep_tiles(std::true_type{}, std::true_type{})
                      : sweep_tiles(std::true_type{}, std::false_type{});
    else
      done = has_down ? sweep_tiles(std::false_type{}, std::true_type{})
                      : sweep_tiles(std::false_type{}, std::false_type{});
    if (!done) return;
    if (lane == fin_lane && overwrite_ans_grad && ans_grad) {
      if constexpr (kApart) {
        // (a NaN found as the seed is the caller's or another workgroup's: it stays either way)
        if (seed == seed) store_once(&ans_grad[b], __float_as_int(seed), g_origin);
      } else {
        ans_grad[b] = peek(&cnt.failed) ? std::numeric_limits<R>::quiet_NaN() : g_origin;
      }
    }
    tile_base += g.ntiles;
  }
}

constexpr size_t kLdsBudget = 156 * 1024;

// Dynamic LDS of a launch: per sweep wave a seam row and 2 x buffers tiles.
size_t lds_bytes(int nsweep, int T, int buffers, size_t elem) {
  return (size_t)nsweep *
         ((size_t)((T + 1 + kSeamSlack + 3) & ~3) + (size_t)buffers * 2 * kTileElems) * elem;
}

// Sweep waves per workgroup: one per 64 rows, as many as LDS allows.
int pick_sweep_waves(int S, int T, size_t elem) {
  int n = (S + 1 + kWave - 1) / kWave;
  n = n < 1 ? 1 : (n > kMaxSweep ? kMaxSweep : n);
  while (n > 1 && lds_bytes(n, T, 2, elem) > kLdsBudget) --n;
  return n;
}

// Dynamic LDS of a workgroup that has a band to itself: one sweep wave's share, a second seam row and
// (backward) what the row above hands to each buffer's steps.
constexpr int kApartBuffers = 3;
size_t apart_lds_bytes(int T) {
  return lds_bytes(1, T, kApartBuffers, sizeof(float)) +
         (size_t)(((T + 1 + kSeamSlack + 3) & ~3) + kApartBuffers * kTileSteps) * sizeof(float);
}

// Whether every band of 64 rows gets a workgroup of its own.  It costs a fixed time -- the marks, and
// the way of a seam from one workgroup to the next -- and saves some of each of the sweep's steps;
// both measured (microseconds, nanoseconds), for 2, 3 and 4 bands.
// (B 12, S 220, T 1500: 134 + 164 -> 72 + 80 us; B 3, S 250, T 1335: 120 + 149 -> 67 + 74;
// B 10, S 137, T 817: 51 + 60 -> 43 + 48.)
// Both seam rows must fit into LDS (T up to 12 988; the other launch goes to 30 700).  Two workgroups of the
// forward kernel share a compute unit while their LDS allows it (T up to 3 004; the backward's ten waves have too
// many registers for that).  Otherwise a band that finds no unit
// of its own starts when an earlier one is done: two bands, which one workgroup sweeps almost as fast
// as two, then stay together (B 136, S 100, T 6000: 595 + 599 apart, 407 + 555 together; B 136, S 70,
// T 5000: 443 + 438, 281 + 318); three and four are still better off apart (B 128, S 250, T 5000:
// 674 + 831 apart, 763 + 1125 together; B 96, S 180, T 6000: 656 + 696, 681 + 862).
//
// The kernels that pass shares have faster steps apart (kSharesStagersApart).  Three bands then pay for any length
// while each has a compute unit: forward and backward with the marks, together and apart, B 8, S 130, T 140: 41.5 and
// 37.9 us; S 160, T 300: 58.5 and 48.2; T 600: 85 and 64; B 64, S 190, T 200: 56.5 and 49.0.  (With more
// of them than units the rule is that of the other kernels: B 100, S 130, T 600: 88 and 92; B 168, S 160, T 300: 67 and 74.  Two bands
// gain from where they did: B 24, S 80, T 600: 55.7 and 56.3; T 900: 72.5 and 71.1.)  Their workgroups, of eleven waves
// with 88 registers and fifteen with 65, have a unit each whatever their LDS (a unit's registers hold 20 and 28 such
// waves), so that two bands stay together as soon as there are more of them than units: together and
// apart, both kernels and the marks, ragged batches of up to S 100, T 1500: B 128 159 and 138, B 160 178 and 203, B 256
// 274 and 288; S 100, T 3000, B 160: 378 and 423; S 70, T 3000, B 200: 310 and 382.  Three and four gain apart with two
// to a unit's place as well (S 130, T 1500, B 100: 211 and 147; S 190, T 3000, B 168: 764 and 656; S 250, T 1500, B 128:
// 466 and 335).
template <typename R, bool kShares>
bool bands_apart(int B, int S, int T, bool backward) {
  const int bands = (S + kWave) / kWave;
  if (sizeof(R) != 4 || bands < 2 || bands > kMaxSweep || T < 1) return false;
  size_t per_cu = kLdsBudget / apart_lds_bytes(T);
  if (per_cu == 0) return false;
  if (kShares) per_cu = 1;
  const long workgroups = (long)((B + 7) / 8 * 8) * bands;
  if (workgroups > (bands == 2 && per_cu == 1 ? 256 : 512)) return false;
  if (kShares && bands == 3 && workgroups <= 256) return true;
  constexpr double kCost[2][3] = {{6, 7, 10}, {11, 16, 20}}, kSaved[2][3] = {{6.7, 7, 39}, {13, 28, 60}};
  return 1e-3 * kSaved[backward][bands - 2] * (S + T) > kCost[backward][bands - 2];
}
inline void mark_seams(const int64_t *boundary, float *p, float *mail, float *ans, float *px_grad, int B,
                       int S, int T, int modified, bool posted, hipStream_t stream) {
  hipLaunchKernelGGL(mark_seams_kernel, dim3(B, (S + kWave) / kWave - 1), dim3(256), 0, stream,
                     boundary, p, mail, ans, px_grad, S, T, modified, (int)posted);
}
// What a caller's buffer holds behind the shares: the post, if there is a seam to pass, and a copy of the boundary.
inline int64_t shares_floats(int B, int S, int T) { return (int64_t)B * (S + 1) * (T + 1); }
inline int64_t post_floats(int B, int S, int T) {
  const bool seams = bands_apart<float, true>(B, S, T, false) || bands_apart<float, true>(B, S, T, true);
  return seams ? (int64_t)B * (S / kWave) * (T + 1) : 0;
}
inline int64_t rows_at(int B, int S, int T) { return (shares_floats(B, S, T) + post_floats(B, S, T) + 1) / 2 * 2; }

// `px_grad`: if given, its seams are marked as well (for a backward_impl that follows and is told so).
// kShares (float only): p is filled for a backward_impl with kShares; py_grad is its py_grad or, posted, the post of both.
// `loss`: if it can, the kernel forms the loss (see count_for_loss) and sets loss->formed.
template <typename R, bool kShares = false>
int forward_impl(const R *px, const R *py, const int64_t *boundary, R *p, R *ans, int B, int S,
                 int T, int modified, void *stream, int checks = 0, int *status = nullptr,
                 R *px_grad = nullptr, R *py_grad = nullptr, LossOf<R> *loss = nullptr, bool posted = false,
                 int64_t *rows = nullptr) {
  static_assert(!kShares || sizeof(R) == 4, "shares are float's");
  R *loss_out = loss && loss->out && (loss->reduction == 0 || loss->arrived) ? loss->out : nullptr;
  const int reduction = loss ? loss->reduction : 0;
  int *arrived = loss ? loss->arrived : nullptr;
  if (B < 0 || S < 0 || T < 0) return fail(FRNNT_EINVAL, "mi_forward: negative size");
  if (B == 0) return FRNNT_OK;
  if (!px || !py || !p || !ans) return fail(FRNNT_EINVAL, "mi_forward: null pointer");
  if ((size_t)(S + 1) * (T + 1) * sizeof(R) >= ((size_t)1 << 30))
    return fail(FRNNT_ELIMIT, "mi_forward: one utterance's lattice exceeds 1 GiB");
  const int n = pick_sweep_waves(S, T, sizeof(R));
  if (lds_bytes(n, T, 2, sizeof(R)) > kLdsBudget)
    return fail(FRNNT_ELIMIT, "mi_forward: T=%d needs %zu bytes of LDS", T, lds_bytes(n, T, 2, sizeof(R)));
  // With at most two sweep waves there is room, for floats, for a third tile buffer, which
  // gives a staging wave two tiles' time instead of one to empty and refill a buffer.
  constexpr int kFewBuffers = sizeof(R) == 4 ? 3 : 2;
  static_assert(kMaxSweep * 2 <= 16 && 2 * kFewBuffers <= 16, "Counters::loaded is too short");
  const bool few = n <= 2 && lds_bytes(n, T, kFewBuffers, sizeof(R)) <= kLdsBudget;
  // (doubles keep two staging waves per sweep wave: with more waves in the workgroup a sweep
  // wave's two tile rows of doubles no longer fit its share of the registers)
  constexpr int kMany = sizeof(R) == 4 ? kFwdStagers : 2;
  constexpr int kFew = kShares ? kSharesStagers : sizeof(R) == 4 ? kFwdStagersFew : 2;
  constexpr int kOne = kShares ? kSharesStagersOne : kFew;  // with one sweep wave
  if constexpr (sizeof(R) == 4) {
    const bool apart = bands_apart<R, kShares>(B, S, T, false);
    const bool later = (px_grad || posted) && bands_apart<R, kShares>(B, S, T, true);
    if (apart || later)
      mark_seams(boundary, apart && !kShares ? p : nullptr, (apart && kShares) || posted ? py_grad : nullptr, ans,
                 later ? px_grad : nullptr, B, S, T, modified, posted, static_cast<hipStream_t>(stream));
    if (apart) {
      const int pitch = (B + 7) / 8 * 8;  // (an utterance's bands on one XCD)
      const size_t lds = apart_lds_bytes(T);
      auto kernel = modified ? mi_forward_kernel<R, true, 1, kOne, kApartBuffers, true, kShares>
                             : mi_forward_kernel<R, false, 1, kOne, kApartBuffers, true, kShares>;
      if (!allow_lds(reinterpret_cast<const void *>(kernel), lds))
        return check_launch("mi_forward: hipFuncSetAttribute");
      hipLaunchKernelGGL(kernel, dim3(pitch * ((S + kWave) / kWave)), dim3((3 + kOne) * kWave), lds,
                         static_cast<hipStream_t>(stream), px, py, boundary, p, ans, S, T,
                         mi_spin_limit, checks, status, B, pitch, py_grad, (int)posted, rows, nullptr, 0,
                         nullptr);
      return check_launch("mi_forward");
    }
  }
  const bool one_band = few && S + 1 <= kWave;
  const int stagers = one_band ? kOne : few ? kFew : kMany;
  const size_t lds = lds_bytes(n, T, few ? kFewBuffers : 2, sizeof(R));
  auto kernel = one_band ? (modified ? mi_forward_kernel<R, true, 1, kOne, kFewBuffers, false, kShares>
                                     : mi_forward_kernel<R, false, 1, kOne, kFewBuffers, false, kShares>)
              : few      ? (modified ? mi_forward_kernel<R, true, 2, kFew, kFewBuffers, false, kShares>
                                     : mi_forward_kernel<R, false, 2, kFew, kFewBuffers, false, kShares>)
                         : (modified ? mi_forward_kernel<R, true, kMaxSweep, kMany, 2, false, kShares>
                                     : mi_forward_kernel<R, false, kMaxSweep, kMany, 2, false, kShares>);
  if (!allow_lds(reinterpret_cast<const void *>(kernel), lds))
    return check_launch("mi_forward: hipFuncSetAttribute");
  hipLaunchKernelGGL(kernel, dim3(B), dim3(n * (1 + stagers) * kWave), lds,
                     static_cast<hipStream_t>(stream), px, py, boundary, p, ans, S, T, mi_spin_limit,
                     checks, status, B, B, py_grad, (int)posted, rows, loss_out, reduction, arrived);
  if (loss) loss->formed = loss_out != nullptr;
  return check_launch("mi_forward");
}

// kShares: p is what a forward_impl with kShares has left; px is not read.  post: that of such a forward_impl.
template <typename R, bool kShares = false>
int backward_impl(const R *px, const R *py, const int64_t *boundary, const R *p, R *ans_grad,
                  R *px_grad, R *py_grad, int B, int S, int T, int modified,
                  int overwrite_ans_grad, void *stream, const R *scores = nullptr,
                  R *loss = nullptr, int reduction = 0, bool marked = false, int seed_stride = 1,
                  R *post = nullptr) {
  (void)py;  // the d2 = 1 - d1 split needs only p and px
  if (loss && (!scores || reduction < 0 || reduction > 2))
    return fail(FRNNT_EINVAL, "mi_backward: loss without scores, or bad reduction");
  if (B < 0 || S < 0 || T < 0) return fail(FRNNT_EINVAL, "mi_backward: negative size");
  if (B == 0) return FRNNT_OK;
  if ((!px && !kShares) || !p || !px_grad || !py_grad)
    return fail(FRNNT_EINVAL, "mi_backward: null pointer");
  if ((size_t)(S + 1) * (T + 1) * sizeof(R) >= ((size_t)1 << 30))
    return fail(FRNNT_ELIMIT, "mi_backward: one utterance's lattice exceeds 1 GiB");
  const int n = pick_sweep_waves(S, T, sizeof(R));
  if (lds_bytes(n, T, 2, sizeof(R)) > kLdsBudget)
    return fail(FRNNT_ELIMIT, "mi_backward: T=%d needs %zu bytes of LDS", T, lds_bytes(n, T, 2, sizeof(R)));
  // With at most two sweep waves there is room for more staging waves per sweep wave and,
  // for floats, for a third tile buffer, which gives a staging wave two tiles' time instead
  // of one to empty and refill a buffer.  (A workgroup of 16 waves leaves each 128
  // registers, too few for a sweep wave's two tile rows of doubles.)
  constexpr bool kFloat = sizeof(R) == 4;
  constexpr int kFew = kShares ? kSharesStagers : kFloat ? kBwdStagersFew : kBwdStagers;
  constexpr int kOne = kShares ? kSharesStagersOne : kFew;  // with one sweep wave
  constexpr int kAlone = kShares ? kSharesStagersApart : kFew;  // bands apart
  constexpr int kFewBuffers = kFloat ? 3 : 2;
  static_assert(kMaxSweep * 2 <= 16 && 2 * kFewBuffers <= 16, "Counters::loaded is too short");
  const bool few = n <= 2 && lds_bytes(n, T, kFewBuffers, sizeof(R)) <= kLdsBudget;
  if constexpr (kFloat) {
    if (bands_apart<R, kShares>(B, S, T, true)) {
      if (!marked && !post)
        mark_seams(boundary, nullptr, nullptr, nullptr, px_grad, B, S, T, modified, false,
                   static_cast<hipStream_t>(stream));
      const int pitch = (B + 7) / 8 * 8;
      const size_t lds = apart_lds_bytes(T);
      auto kernel = modified ? mi_backward_kernel<R, true, 1, kAlone, kApartBuffers, true, kShares>
                             : mi_backward_kernel<R, false, 1, kAlone, kApartBuffers, true, kShares>;
      if (!allow_lds(reinterpret_cast<const void *>(kernel), lds))
        return check_launch("mi_backward: hipFuncSetAttribute");
      hipLaunchKernelGGL(kernel, dim3(pitch * ((S + kWave) / kWave)),
                         dim3((3 + kAlone + kHelpers<1, kShares>) * kWave), lds,
                         static_cast<hipStream_t>(stream), px, boundary, p, ans_grad, px_grad,
                         py_grad, S, T, seed_stride, overwrite_ans_grad, scores, loss, B, reduction,
                         mi_spin_limit, pitch, post);
      return check_launch("mi_backward");
    }
  }
  const bool one_band = kShares && few && S + 1 <= kWave;
  const int stagers = one_band ? kOne : few ? kFew : kBwdStagers;
  const size_t lds = lds_bytes(n, T, few ? kFewBuffers : 2, sizeof(R));
  constexpr int kOneCap = kShares ? 1 : 2;  // (without shares: the kernel for two)
  auto kernel = one_band ? (modified ? mi_backward_kernel<R, true, kOneCap, kOne, kFewBuffers, false, kShares>
                                     : mi_backward_kernel<R, false, kOneCap, kOne, kFewBuffers, false, kShares>)
              : few ? (modified ? mi_backward_kernel<R, true, 2, kFew, kFewBuffers, false, kShares>
                                : mi_backward_kernel<R, false, 2, kFew, kFewBuffers, false, kShares>)
                    : (modified ? mi_backward_kernel<R, true, kMaxSweep, kBwdStagers, 2, false, kShares>
                                : mi_backward_kernel<R, false, kMaxSweep, kBwdStagers, 2, false, kShares>);
  if (!allow_lds(reinterpret_cast<const void *>(kernel), lds))
    return check_launch("mi_backward: hipFuncSetAttribute");
  const int helpers = few ? kHelpers<2, kShares> : kHelpers<kMaxSweep, kShares>;
  hipLaunchKernelGGL(kernel, dim3(B), dim3((n * (1 + stagers) + helpers) * kWave), lds,
                     static_cast<hipStream_t>(stream), px, boundary, p, ans_grad, px_grad,
                     py_grad, S, T, seed_stride, overwrite_ans_grad, scores, loss, B, reduction,
                     mi_spin_limit, B, post);
  return check_launch("mi_backward");
}

}  // namespace
}  // namespace frnnt

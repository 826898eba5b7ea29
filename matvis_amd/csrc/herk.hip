// (d) V = conj(Z) Z^T as a Hermitian rank-k update on MFMA tiles.
//
// Rows are cut into panels (64 rows; 32 in complex128) and only the panel
// pairs (i, j) with i <= j of the upper triangle are computed, in groups of
// four pairs a workgroup (one pair a wave); the accumulator is defined on
// r <= c.
//
// K (the source axis, times nax) is cut into slices.  A work item is one
// (group, slice); its waves write their partial pairs to the workspace, and a
// reduce kernel sums the slices in FP64 in a fixed order, so results are
// deterministic.  The number of active slices is chosen on the device from
// the device-side column count (sources above the horizon are only known
// there): enough slices that no FP32 accumulation chain exceeds `cmax` K
// tiles, then the count among the next 64 that best fills the resident
// workgroup slots.  The grid is at most one workgroup per slot; workgroups
// loop over items, each XCD owning a contiguous run of slice-major items so
// that workgroups sharing an L2 read the same K range of Z.
//
// Complex arithmetic on real MFMA: with X_r = (re_0, im_0, re_1, im_1, ...)
// the row of Z read as reals, and Y_r = (im_0, -re_0, im_1, -re_1, ...),
//   Re V[r, c] = X_r . X_c        Im V[r, c] = X_r . Y_c
// so each output tile needs two real products over 2K reals: 8 flop per
// complex multiply-add, with no extra passes over Z.  (The split forms'
// terms order the reals of each 4 columns as re_0..re_3, im_0..im_3: the dot
// products are the same sums, and Y is a register reorder of X.)
#include <map>
#include <mutex>
#include <type_traits>
#include <utility>

#include "common.h"

namespace mv {
namespace {

constexpr int kXcd = 8;

__host__ __device__ inline int icdiv(int a, int b) { return (a + b - 1) / b; }

// Upper-triangle tile index -> (bi, bj) with bi <= bj, row-major over bi.
__device__ __forceinline__ void tile_coords(int t, int nb, int &bi, int &bj) {
  int i = 0;
  while (t >= nb - i) {
    t -= nb - i;
    ++i;
  }
  bi = i;
  bj = i + t;
}

// HERKs of one shape in one launch (the frequencies of a time): instance b's
// Z starts b z_stride elements (complex, or 32-bit words of a split term)
// after the first, its partials b ws_stride bytes, its accumulator
// b vacc_stride complex elements.  The slice count is that of one instance, so
// that each result has the same bits alone and in any batch.
struct HerkBatch {
  int n;
  int64_t z_stride, ws_stride, vacc_stride;
  const double *scales;  // device, one an instance, or null: the one scale
};

struct SliceCfg {
  int max_slices;  // partial slots per tile in the workspace
  int slots;       // workgroups resident at once (multiple of kXcd)
  int cmax;        // at most this many K tiles per slice
  int ovh;         // per-item cost beyond its K tiles, in K-tile units
  int reach;       // counts from the least one on that are considered
  int full;        // an instance that leaves slots idle keeps chains as
                   // short as the fullest of 64 counts has them
};

// Active slice count for `ktiles` K tiles over `ntiles` items a slice (panel
// groups): enough slices that no chain exceeds cmax K tiles; then, where the
// counts within reach (at most the capacity and ktiles) can fill the resident
// slots, the one of the first 64 with the least cost = rounds of slots x (K
// tiles per slice + per-item overhead), the smallest count on ties.  Where they
// cannot (small_slices), a power of two: an instance that leaves slots idle
// shares its launch with others (frequencies, HerkBatch), and counts that
// divide the slots leave no nearly empty last round.  The largest of at most
// sqrt(30 ktiles): a slice more costs its share of the reduce, about a thirtieth
// of the time of a K tile in a launch that leaves most slots idle (3.5 us,
// FP64), and shortens every chain by ktiles / ns^2 of them.
// The plain forms and fp16 terms, whose error is that of the chains, go on to
// the power of two whose chains are no longer than those of the fullest of 64
// counts, and reach for 128.  (Without: errors over |V|, 2 x 18k columns, 256
// rows of fp16 terms 64 slices 6.7e-8, 75 6.4e-8, 128 5.3e-8; 200 of complex64
// 64 slices 9.9e-8, 128 7.0e-8; 32 of 1.8k complex64 columns 32 slices 7.8e-8, 64
// 6.5e-8.  Times at 64 and 128 slices: m = 128, 20k columns, complex64 42 and 38
// us, FP64 65 and 54.)  Two bf16 terms are coarser than any chain, and of three
// each wave sums half the columns.
// Pure integer function of its arguments: the compute and reduce kernels and
// the host agree on it.
// Measured, HERK and reduce of a time: 16 frequencies of 128 antennas, 1,866
// K tiles, 72 -> 64 slices (1,152 -> 1,024 items for 512 slots, and one launch
// instead of two) 254 -> 214 us.
__host__ __device__ inline void slice_range(int ktiles, const SliceCfg &c,
                                            int &lo, int &hi) {
  lo = icdiv(ktiles, c.cmax);
  lo = lo < 1 ? 1 : (lo > c.max_slices ? c.max_slices : lo);
  hi = lo + c.reach - 1;
  if (hi > c.max_slices) hi = c.max_slices;
  if (hi > ktiles) hi = ktiles > lo ? ktiles : lo;
}
__host__ __device__ inline int64_t slice_cost(int ktiles, int ntiles, int ns,
                                              const SliceCfg &c) {
  const int per_x = c.slots / kXcd > 0 ? c.slots / kXcd : 1;
  const int rounds = icdiv(icdiv(ntiles * ns, kXcd), per_x);
  return (int64_t)rounds * (icdiv(ktiles, ns) + c.ovh);
}
// Whether even hi slices leave slots idle, and then the count.
__host__ __device__ inline bool small_slices(int ktiles, int ntiles, int lo,
                                             int hi, const SliceCfg &c,
                                             int &ns) {
  if ((int64_t)ntiles * hi > c.slots) return false;
  ns = 1;
  const int most = hi < lo + 63 ? hi : lo + 63;
  const int chain = c.full ? icdiv(ktiles, most) : ktiles;
  while (2 * ns <= hi && (4 * (int64_t)ns * ns <= 30 * (int64_t)ktiles ||
                          icdiv(ktiles, ns) > chain))
    ns *= 2;
  if (ns < lo) ns = lo;
  return true;
}
__host__ __device__ inline int active_slices(int ktiles, int ntiles,
                                             const SliceCfg &c) {
  if (ktiles <= 0) return 1;
  int lo, hi, ns;
  slice_range(ktiles, c, lo, hi);
  if (small_slices(ktiles, ntiles, lo, hi, c, ns)) return ns;
  if (hi > lo + 63) hi = lo + 63;
  int best = lo;
  int64_t best_cost = INT64_MAX;
  for (ns = lo; ns <= hi; ++ns) {
    const int64_t cost = slice_cost(ktiles, ntiles, ns, c);
    if (cost < best_cost) {
      best_cost = cost;
      best = ns;
    }
  }
  return best;
}
// The same value with one candidate per lane of a full wave (wave-uniform
// arguments): the least (cost, count) over the lanes.
__device__ inline int active_slices_wave(int ktiles, int ntiles,
                                         const SliceCfg &c) {
  if (ktiles <= 0) return 1;
  int lo, hi;
  slice_range(ktiles, c, lo, hi);
  int small;
  if (small_slices(ktiles, ntiles, lo, hi, c, small)) return small;
  const int lane = (int)(threadIdx.x & 63);
  const int ns = lo + lane;
  // cost < 2^48 (rounds and K tiles per slice are below 2^24); the lane in
  // the low bits breaks ties toward the smaller count
  uint64_t key = ns <= hi
                     ? ((uint64_t)slice_cost(ktiles, ntiles, ns, c) << 6) | lane
                     : UINT64_MAX;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const uint64_t o = __shfl_xor(key, off, 64);
    key = o < key ? o : key;
  }
  // every lane holds the least key: a scalar, so that what depends on it is
  return lo + __builtin_amdgcn_readfirstlane((int)(key & 63));
}

// Columns of each segment: the device count never exceeds the host bound the
// buffers were sized for.
__device__ __forceinline__ int64_t seg_columns(int64_t host,
                                               const int32_t *dev) {
  if (!dev) return host;
  const int64_t d = *dev;
  return d < 0 ? 0 : (d < host ? d : host);
}

// Item loop: workgroup b runs on XCD x = b % 8, which holds w_x =
// ceil((g - x) / 8) of the g workgroups.  Each XCD owns a contiguous item
// range proportional to w_x (empty when w_x = 0) and its workgroups sweep it.
template <class F>
__device__ __forceinline__ void for_items(int64_t items, F &&body) {
  const int g = gridDim.x, b = blockIdx.x;
  const int x = b % kXcd, j = b / kXcd;
  int before = 0;
  for (int y = 0; y < x; ++y) before += (g - y + kXcd - 1) / kXcd;
  const int workers = (g - x + kXcd - 1) / kXcd;
  const int64_t lo = items * before / g;
  const int64_t hi = items * (before + workers) / g;
  for (int64_t it = lo + j; it < hi; it += workers) body(it);
}

// Workgroup barrier ordering LDS accesses only.  __syncthreads() is a
// release/acquire fence for all address spaces and so also waits for every
// global load in flight; the K loops keep the next tiles' loads in flight
// across their barriers, and wait for them where the registers are used.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// 16 bytes from global memory per lane straight into LDS: lane l's bytes
// land at byte 16 l of the wave-uniform destination `lds`.
__device__ __forceinline__ void copy16_to_lds(const uint32_t *src,
                                              uint32_t *lds) {
  __builtin_amdgcn_global_load_lds(src, lds, 16, 0, 0);
}
// Wait until this wave's global loads, LDS copies included, have landed.
__device__ __forceinline__ void wait_global_loads() {
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0), other counters unchecked
}

// ------------------------------------------------------------ panel groups

// The upper triangle of the n x n grid of P-row panels is cut into groups of
// panel pairs (i, j), i <= j, that touch at most four panels: a workgroup
// stages the group's panels and its four waves compute the pairs, a pair a
// wave or, where there are fewer than four, parts of pairs.  A wave of a
// diagonal pair leaves out the blocks below the diagonal, and what a group
// takes is its longest wave (a whole pair 4 quadrants, a diagonal one 3):
//   Off the diagonal: blocks I < J of two panels, all four pairs; 4.
//   n even, diagonal: of whole fours of blocks the pairs (2I, 2I),
//     (2I, 2I + 1), (2I + 1, 2I + 1) in sequence, four a group (at most four
//     adjacent panels), 4; of the last one to three blocks each block by
//     itself, (2I, 2I + 1) as two halves, 3.
//   n odd, last panel L = n - 1: per block (2I, 2I), (2I, 2I + 1), (2I, L),
//     (2I + 1, L), 4; then the pairs (2I + 1, 2I + 1) and (L, L), four a
//     group, 3, or the last two as halves, 2, or the last one as quadrants, 1.
// Square tiles of 2 x 2 pairs leave a wave idle on every diagonal tile and
// two on every tile of a half-empty last column (11 panels: 21 tiles).
// Measured against whole pairs, four a group in sequence: m = 128 split, 2 x
// 15k columns, 47 -> 42 us; m = 32 complex64, 3.6k columns, 9.6 -> 7.0; 6
// frequencies of 61 antennas (m = 122) FP64 (three real products), a time 283 ->
// 258; 24 grouped instances of 64-350 antennas 458 -> 417; m = 700 1% less.
__host__ __device__ inline int panel_groups(int n) {
  const int h = n / 2;
  const int off = h * (h - 1) / 2;
  return off + (n & 1 ? h + icdiv(h + 1, 4) : icdiv(3 * h, 4));
}

// Row-major index of pair (i, j), i <= j, in the upper triangle of n panels.
__host__ __device__ inline int pair_index(int i, int j, int n) {
  return i * n - i * (i - 1) / 2 + (j - i);
}

// The part of a panel pair's blocks that a wave computes, in quadrants
// (half a panel's rows by half a panel's columns).
enum PairPart : int {
  kWhole,    // all four
  kDiagonal, // a diagonal pair's: all but the one below the diagonal, and in
             // the others no block below the diagonal
  kTop,      // the first panel's first half
  kBottom,   // the first panel's second half
  kQuad00, kQuad01, kQuad11,  // one quadrant
};

// What wave w of group g does: it stages panel `load` into slot w (none if
// negative) and computes `part` of the pair of panels (i, j), held in slots
// si and sj (none if i is negative).
// norm: the slot of a panel whose row norms (the split forms' exact diagonal)
// the group sums as its w-th, -1 if none.  Each panel's are summed once, by a
// group that stages it: the work would otherwise gather in the last groups.
// Blocks I, I + 1 off the diagonal take the odd panel of I; the even panels
// and the last odd one stay with the group of their diagonal pair.
struct WavePair {
  int load, i, j, si, sj, norm, part;
};
__host__ __device__ inline WavePair group_wave(int g, int n, int w) {
  const int h = n / 2;
  const int off = h * (h - 1) / 2;
  WavePair p;
  if (g < off) {
    int I = 0, t = g;
    while (t >= h - 1 - I) {
      t -= h - 1 - I;
      ++I;
    }
    const int J = I + 1 + t;
    p.si = w >> 1;
    p.sj = 2 + (w & 1);
    p.i = 2 * I + p.si;
    p.j = 2 * J + (w & 1);
    p.load = w < 2 ? 2 * I + w : 2 * J + w - 2;
    p.norm = w == 1 && J == I + 1 ? 1 : -1;
    p.part = kWhole;
    return p;
  }
  g -= off;
  if (!(n & 1)) {
    const int fours = 3 * (h / 4);  // groups of the whole fours of blocks
    if (g < fours) {
      // pair s of the sequence: block s / 3, entry s % 3
      const int s0 = 4 * g, s = s0 + w;
      const int first = 2 * (s0 / 3) + (s0 % 3 == 2);  // row panel of pair s0
      p.load = first + w < n ? first + w : -1;
      p.i = 2 * (s / 3) + (s % 3 == 2);
      p.j = 2 * (s / 3) + (s % 3 != 0);
      p.si = p.i - first;
      p.sj = p.j - first;
      p.norm = s % 3 == 0 || s == 3 * h - 1 ? p.si : -1;
      p.part = s % 3 == 1 ? kWhole : kDiagonal;
      return p;
    }
    const int I = h / 4 * 4 + g - fours;
    p.load = w < 2 ? 2 * I + w : -1;
    p.si = w == 1 ? 1 : 0;
    p.sj = w == 0 ? 0 : 1;
    p.i = 2 * I + p.si;
    p.j = 2 * I + p.sj;
    p.norm = w == 0 ? 0 : (w == 1 && I == h - 1 ? 1 : -1);
    p.part = w < 2 ? kDiagonal : (w == 2 ? kTop : kBottom);
    return p;
  }
  const int L = n - 1;
  if (g < h) {
    // slots: 0 = 2g, 1 = 2g + 1, 2 = L
    p.load = w < 2 ? 2 * g + w : (w == 2 ? L : -1);
    p.si = w == 3 ? 1 : 0;
    p.sj = w < 2 ? w : 2;
    p.i = 2 * g + p.si;
    p.j = w < 2 ? 2 * g + w : L;
    p.norm = w == 0 ? 0 : -1;
    p.part = w == 0 ? kDiagonal : kWhole;
    return p;
  }
  // pairs e0 .. e0 + count - 1 of (2e + 1, 2e + 1), the last one (L, L)
  const int e0 = 4 * (g - h);
  const int count = h + 1 - e0 < 4 ? h + 1 - e0 : 4;
  const int s = count > 2 ? w : (count == 2 ? w >> 1 : 0);  // the wave's pair
  p.load = w < count ? (e0 + w < h ? 2 * (e0 + w) + 1 : L) : -1;
  p.norm = w < count && e0 + w >= h - 1 ? w : -1;
  p.si = p.sj = s;
  p.i = e0 + s < h ? 2 * (e0 + s) + 1 : L;
  p.part = count > 2 ? kDiagonal
           : count == 2 ? (w & 1 ? kQuad11 : kTop)
                        : (w == 0 ? kQuad00 : (w == 1 ? kQuad01 : kQuad11));
  if (s >= count || (count == 1 && w == 3)) {
    p.i = -1;
    p.si = p.sj = 0;
    p.part = kQuad11;
  }
  p.j = p.i;
  return p;
}
template <int V> using Int = std::integral_constant<int, V>;

// First row and column quadrant of a part.
__host__ __device__ inline int part_row(int part) {
  return part == kBottom || part == kQuad11 ? 1 : 0;
}
__host__ __device__ inline int part_col(int part) {
  return part >= kQuad01 ? 1 : 0;
}

// ------------------------------------------------------------ plain forms

template <typename T> struct PlainMfma;
// Both take A[i][k] from lane i + 16 k and B[k][j] from lane j + 16 k; they
// differ in where D lands: register r of lane l holds D[row(l, r)][l % 16].
template <> struct PlainMfma<double> {
  typedef v4d acc;
  __device__ static acc op(double a, double b, acc c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static constexpr int kRowStep = 4;
  __device__ static int row(int g, int r) { return g + kRowStep * r; }
};
template <> struct PlainMfma<float> {
  typedef v4f acc;
  __device__ static acc op(float a, float b, acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static constexpr int kRowStep = 1;
  __device__ static int row(int g, int r) { return 4 * g + kRowStep * r; }
};

constexpr int kPT = 64;  // side the accumulator of the plain forms is padded to
constexpr int kPK = 16;  // complex columns of a K tile as slices count them
// Complex columns per LDS stage: 128 bytes a row.  FP64 stages of 8 columns
// make 32 KB a workgroup, so that three share a CU (160 KB, 168 registers)
// and the matrix cores have work while two wait for copies or operands: m =
// 700, 2 x 29.9k columns, 16 columns and two workgroups 1.49 ms, 8 and two 1.52,
// 8 and three 1.44 (these with three real products a complex one).
template <typename T> constexpr int kPStageK = sizeof(T) == 8 ? 8 : 16;

// Bytes of a panel row in LDS (one stage) and the 16-byte chunks it has.
template <typename T> constexpr int kPRowBytes =
    kPStageK<T> * 2 * (int)sizeof(T);

// Where column c of row r of a panel sits in LDS: rows are not padded; the
// row's eight 16-byte chunks are permuted by an XOR with (r / 2) % 8, so that
// the 16 rows of one column that an operand read touches fall in distinct
// banks: rows 2q and 2q + 1 are the two halves of the 64 banks.  Conflicts
// take 5% of the kernel's cycles in complex128 and 8% in complex64.
__device__ __forceinline__ int plain_swz(int r) { return (r >> 1) & 7; }
template <typename T> __device__ __forceinline__ int plain_pos(int r, int c) {
  const int b = c * 2 * (int)sizeof(T);  // byte within the row
  return r * kPRowBytes<T> + (((b >> 4) ^ plain_swz(r)) << 4) + (b & 15);
}

// One stage of a group's four panels; the two stages of a kernel are
// separate __shared__ objects (see the split forms' stages).
template <typename T, int P> struct alignas(16) PlainStage {
  char x[4][P * kPRowBytes<T>];
};

// One plain HERK instance as the kernels read it.
template <typename T> struct PlainProblem {
  const cplx<T> *z;
  int64_t ldz, seg_stride;
  cplx<T> *part;
  int m, n, ngroups, npairs;  // rows, panels, groups, panel pairs
  int wide;  // rows are 16-byte aligned and offsets fit 32-bit 16-byte units
};

// Whether the 16-byte copies apply: every row and segment starts on 16 bytes
// and a row's offset fits 32 bits of 16-byte units.
template <typename T>
__host__ __device__ inline int plain_wide(const PlainProblem<T> &Q, int nseg) {
  constexpr int per = 16 / (2 * (int)sizeof(T));  // columns in 16 bytes
  return (uintptr_t)Q.z % 16 == 0 && Q.ldz % per == 0 &&
         (nseg == 1 || Q.seg_stride % per == 0) &&
         (int64_t)Q.m * Q.ldz / per < ((int64_t)1 << 32);
}

// The P x P panel pairs of one (slice, group) item, each wave its own pair as
// (P / 16)^2 blocks of 16x16.
//
// Two real products over 2K reals, as the top of this file has them: one
// 16x16x4 MFMA each per 2 complex columns, lane group g = l / 16 supplying part
// g % 2 of column g / 2.  An imaginary part is thus a single chain whose terms
// a d and -b c of a column follow one another: its partial sums, and with them
// its rounding, stay as small as Im V is where the rows are nearly in phase
// (short baselines, the feeds of one antenna).  Three real products a complex
// one (Im as a difference of their sums) take a quarter fewer MFMAs, but round
// Im at the size of |V|: phases within 0.01 rad, 60k columns, errors of Im /
// |V| 2e-11 -> 8e-7 in complex64 and 5e-20 -> 1.4e-16 in complex128.  The
// real part's chain, whose terms do add up, is cut into two over alternate
// columns, and slices are short (form_cmax).  Chains are the same at either
// panel side, so that a problem's bits do not depend on a group's largest one.
//
// Measured with the reduce, m = 700, 59.7k columns, against square tiles with
// copies through registers, a mask on every element and half of each operand
// read thrown away: FP64 2.39 -> 2.01 ms, FP32 1.34 -> 1.04 ms, 74% and 72% of
// the peak (78.6 and 157 TFLOP/s); m = 64, 3.6k columns 26 -> 19 and 22 -> 16
// us.  (Three products 1.50 and 0.78 ms.)
// Errors against 64 bits (complex128: extended precision) over sqrt(V_ii
// V_jj), m = 160, 60k columns, one chain a real part and 64-78 slices -> two
// and 128 (slice_reach): Re, phases within 0.3 rad 6.6e-8 -> 1.9e-8 and 1.5e-16
// -> 7.2e-17, incoherent Z 2.1e-9 -> 1.1e-9 and 4.2e-18 -> 2.2e-18; Im 6.9e-10
// -> 5.3e-10 and 1.4e-18 -> 1.0e-18, incoherent 2.0e-9 -> 1.5e-9 and 4.1e-18 ->
// 3.0e-18.  A time of the 350-antenna sky in complex64 9.6e-7 -> 2.3e-7 of |V|.
// The diagonal is exactly real.
//
// Copies go straight from global memory into the other LDS stage
// (global_load_lds: 16 bytes a lane where rows are 16-byte aligned, else 4:
// complex64 rows of an odd length, m = 700, 59.7k columns 1.28 ms for 1.04),
// each wave one panel, while the current K tile is computed; the last K tile
// of a segment that is not whole goes through registers with a column mask.
// Rows past m are read as row m - 1: they reach output rows and columns past
// m only.
template <typename T, int P>
__device__ __forceinline__ void plain_item(const PlainProblem<T> &Q,
                                           int64_t seg_len, int slice,
                                           int group, int ns, int ktiles,
                                           int kps, PlainStage<T, P> &L0,
                                           PlainStage<T, P> &L1) {
  typedef typename PlainMfma<T>::acc acc_t;
  typedef T vec2 __attribute__((ext_vector_type(2)));
  constexpr int PK = kPStageK<T>;
  constexpr int RB = kPRowBytes<T>, CH = RB / 16;  // row bytes, chunks a row
  constexpr int NB = P / 16;                       // 16-row blocks a panel
  constexpr int NI = P * RB / 1024;                // 1 KB copies a panel
  // the wave's index in a scalar register: what it does is uniform over it
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int g = lane >> 4, rl = lane & 15;
  const WavePair wp = group_wave(group, Q.n, wave);
  const int kt0 = (int)((int64_t)slice * ktiles / ns);
  const int kt1 = (int)((int64_t)(slice + 1) * ktiles / ns);

  // this lane's part of copy u: row u 1024 / RB + lane / CH of the panel,
  // LDS chunk lane % CH, i.e. logical chunk (lane % CH) ^ swz(row)
  uint32_t off[NI];
  const int prow0 = wp.load * P;
  if (wp.load >= 0 && Q.wide) {
#pragma unroll
    for (int u = 0; u < NI; ++u) {
      const int r = u * (1024 / RB) + lane / CH;
      const int gr = prow0 + r < Q.m ? prow0 + r : Q.m - 1;
      const int c = (lane % CH) ^ plain_swz(r);
      off[u] = (uint32_t)((int64_t)gr * Q.ldz * (2 * (int)sizeof(T)) / 16) + c;
    }
  }
  int sg = kt0 / (kps > 0 ? kps : 1), kc = kt0 - sg * kps;
  auto copy = [&](PlainStage<T, P> &D) {
    const int64_t c0 = (int64_t)kc * PK;
    if (wp.load >= 0) {
      const cplx<T> *src = Q.z + sg * Q.seg_stride + c0;
      if (c0 + PK <= seg_len) {
        if (Q.wide) {
#pragma unroll
          for (int u = 0; u < NI; ++u)
            copy16_to_lds(
                (const uint32_t *)((const char *)src + ((uint64_t)off[u] << 4)),
                (uint32_t *)&D.x[wave][u * 1024]);
        } else {
#pragma unroll 1
          for (int u = 0; u < 4 * NI; ++u) {
            const int b = u * 256 + lane * 4, r = b / RB, x = b % RB;
            const int gr = prow0 + r < Q.m ? prow0 + r : Q.m - 1;
            const char *row = (const char *)(src + (int64_t)gr * Q.ldz);
            __builtin_amdgcn_global_load_lds(
                (const uint32_t *)(row + (((x >> 4) ^ plain_swz(r)) << 4) +
                                   (x & 15)),
                (uint32_t *)&D.x[wave][u * 256], 4, 0, 0);
          }
        }
      } else {
        const int valid = (int)(seg_len - c0);  // 1 .. PK - 1 columns
#pragma unroll 1
        for (int e = lane; e < P * PK; e += 64) {
          const int r = e / PK, c = e % PK;
          const int gr = prow0 + r < Q.m ? prow0 + r : Q.m - 1;
          const cplx<T> v = src[(int64_t)gr * Q.ldz + (c < valid ? c : 0)];
          *(vec2 *)&D.x[wave][plain_pos<T>(r, c)] =
              c < valid ? vec2{v.re, v.im} : vec2{(T)0, (T)0};
        }
      }
    }
    if (++kc == kps) {
      kc = 0;
      ++sg;
    }
  };

  // The K loop of a wave that computes NI rows and NJ columns of blocks from
  // (oi, oj), without those below the diagonal where DIAG.  A loop for each
  // part: the waves of a group run different ones, with the same barriers.
  // (Branches around the parts' MFMAs within one loop spill accumulators.)
  auto run = [&](auto ni_, auto nj_, auto diag_, int oi, int oj) {
    constexpr int NI = decltype(ni_)::value, NJ = decltype(nj_)::value;
    constexpr bool DIAG = decltype(diag_)::value;
    acc_t re[2][NI][NJ], im[NI][NJ];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) re[0][i][j] = re[1][i][j] = im[i][j] = acc_t{};

    auto compute = [&](const PlainStage<T, P> &D) {
      const char *A = D.x[wp.si] + oi * 16 * RB, *B = D.x[wp.sj] + oj * 16 * RB;
#pragma unroll
      for (int ks = 0; ks < PK / 2; ++ks) {
        const int pos = plain_pos<T>(rl, 2 * ks + (g >> 1));
        T a[NI], bre[NJ], bim[NJ];
#pragma unroll
        for (int i = 0; i < NI; ++i)
          a[i] = ((const T *)&A[i * 16 * RB + pos])[g & 1];
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          const vec2 b = *(const vec2 *)&B[j * 16 * RB + pos];
          bre[j] = g & 1 ? b[1] : b[0];
          bim[j] = g & 1 ? -b[0] : b[1];
        }
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
          for (int i = 0; i < NI; ++i) {
            if (DIAG && i > j) continue;
            acc_t &x = re[ks & 1][i][j], &y = im[i][j];
            x = PlainMfma<T>::op(a[i], bre[j], x);
            y = PlainMfma<T>::op(a[i], bim[j], y);
          }
        // operand reads stay in their step: hoisted over the unrolled steps
        // they would spill (the other waves of the SIMD cover their latency)
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    // one stage computed from C while the next is copied into N
    auto step = [&](PlainStage<T, P> &C, PlainStage<T, P> &N, int kt) {
      if (kt + 1 < kt1) copy(N);
      if (wp.i >= 0) compute(C);
      wait_global_loads();  // this wave's copies into N
      lds_barrier();
    };
    for (int kt = kt0; kt < kt1; kt += 2) {
      step(L0, L1, kt);
      if (kt + 1 < kt1) step(L1, L0, kt + 1);
    }
    // every wave is past the last barrier: LDS is free for the next item

    if (wp.i < 0) return;
    // 16x16 accumulator: lane l = 16 g + rl, register r -> row
    // PlainMfma<T>::row(g, r), column rl
    // (the base is opaque so that the store addresses are formed here)
    cplx<T> *out = Q.part + ((int64_t)slice * Q.npairs +
                             pair_index(wp.i, wp.j, Q.n)) * P * P;
    int obase =
        (PlainMfma<T>::row(g, 0) + oi * 16) * P + rl + oj * 16;
    asm volatile("" : "+v"(obase));
    out += obase;
    constexpr int rstep = PlainMfma<T>::kRowStep * P;
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        if (DIAG && i > j) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          out[i * 16 * P + r * rstep + j * 16] =
              cplx<T>{re[0][i][j][r] + re[1][i][j][r], im[i][j][r]};
      }
  };

  if (kt0 < kt1) copy(L0);
  wait_global_loads();
  lds_barrier();
  constexpr int HB = NB / 2;  // blocks a quadrant's side
  constexpr Int<NB> whole{};
  constexpr Int<HB> half{};
  const int oi = part_row(wp.part) * HB, oj = part_col(wp.part) * HB;
  if (wp.part == kWhole) run(whole, whole, Int<0>{}, 0, 0);
  else if (wp.part == kDiagonal) run(whole, whole, Int<1>{}, 0, 0);
  else if (wp.part <= kBottom) run(half, whole, Int<0>{}, oi, 0);
  else run(half, half, Int<0>{}, oi, oj);
}

// Workgroups a CU holds (kPStageK).
template <typename T> constexpr int kPlainWgs = sizeof(T) == 8 ? 3 : 2;

template <typename T, int P>
__global__ __launch_bounds__(256, kPlainWgs<T>) void herk_plain_kernel(
    const PlainProblem<T> Q0, int nseg, int64_t seg_len_host,
    const int32_t *__restrict__ seg_len_dev, SliceCfg cfg, HerkBatch hb) {
  __shared__ PlainStage<T, P> L0, L1;
  const int64_t seg_len = seg_columns(seg_len_host, seg_len_dev);
  const int ns = active_slices_wave((int)cdiv(seg_len, (int64_t)kPK) * nseg,
                                    Q0.ngroups, cfg);
  // stages per segment
  const int kps = (int)cdiv(seg_len, (int64_t)kPStageK<T>);
  const int64_t per = (int64_t)Q0.ngroups * ns;
  for_items(per * hb.n, [&](int64_t it) {
    const int64_t b = it / per, i = it - b * per;
    PlainProblem<T> Q = Q0;
    Q.z += b * hb.z_stride;
    Q.part = (cplx<T> *)((char *)Q.part + b * hb.ws_stride);
    plain_item<T, P>(Q, seg_len, (int)(i / Q.ngroups), (int)(i % Q.ngroups),
                     ns, kps * nseg, kps, L0, L1);
  });
}

// ------------------------------------------------------------ split forms

constexpr int kST = 128;  // tile side, complex rows
constexpr int kSK = 16;   // complex columns per LDS stage (one K tile)

template <bool F16> struct SplitMfma;
template <> struct SplitMfma<false> {
  __device__ static v16f op(u32x4 a, u32x4 b, v16f c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(
        __builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
  }
};
template <> struct SplitMfma<true> {
  __device__ static v16f op(u32x4 a, u32x4 b, v16f c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(
        __builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), c, 0, 0, 0);
  }
};

// The imaginary-part operand Y of a 16-byte chunk of 4 columns in the split
// terms' layout (the 4 real parts, then the 4 imaginary parts, 16 bits
// each): (re x 4 | im x 4) -> (im x 4 | -re x 4), a register reorder and two
// sign flips of packed pairs.
__device__ __forceinline__ u32x4 swap_negate4(u32x4 v) {
  return u32x4{v[2], v[3], v[0] ^ 0x80008000u, v[1] ^ 0x80008000u};
}



// The two 16-bit halves of a packed (re, im) word as floats.
template <bool F16> __device__ __forceinline__ float lo_half(uint32_t w) {
  if constexpr (F16)
    return (float)__builtin_bit_cast(_Float16, (uint16_t)(w & 0xffffu));
  else
    return __builtin_bit_cast(float, w << 16);
}
template <bool F16> __device__ __forceinline__ float hi_half(uint32_t w) {
  if constexpr (F16)
    return (float)__builtin_bit_cast(_Float16, (uint16_t)(w >> 16));
  else
    return __builtin_bit_cast(float, w & 0xffff0000u);
}

// sum over 4 columns of |t0 + t1 (+ t2)|^2, in FP64 (two bf16 terms add
// exactly in FP32; three round once at 2^-24): the sum of the squares of all
// 8 summed components, whichever column each 16-bit half of a word belongs to
template <int NT, bool F16>
__device__ __forceinline__ double row_norm2(const u32x4 *r) {
  double s = 0.0;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    float re = 0.0f, im = 0.0f;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const uint32_t w = r[t][q];
      re += lo_half<F16>(w);
      im += hi_half<F16>(w);
    }
    s += (double)re * re + (double)im * im;
  }
  return s;
}

// One HERK instance of a split form as the kernels read it.  `part` holds
// `nslices` x ntiles partial panel pairs of 64 x 64 complex<float>, `dpart`
// the FP64 row norms of the panels (nslices x nb x 64).
//
// Split terms are stored K-tile-major: K tile q (columns 16 q .. 16 q + 15
// of the concatenated segments, seg_stride a multiple of 16) is `ldz` rows
// of 16 words, row r at word (q ldz + r) 16.  The rows one copy
// instruction reads (16 consecutive rows of one K tile) are 1 KB of
// contiguous memory and a panel of a K tile is one run of 64 x 64 bytes, where a row-major layout puts every row's 64 bytes on its
// own page.
struct SplitProblem {
  const uint32_t *t[3];
  int64_t ldz, seg_stride, seg_len_host;
  const int32_t *seg_len_dev;
  cplx<float> *part;
  double *dpart;
  cplx<double> *vacc;
  int64_t ldv;
  double scale;
  // nb panels, ntiles = nb (nb + 1) / 2 partial pairs a slice
  int m, nseg, nb, ntiles, accumulate;
  int ngroups;  // work items a slice (panel groups, or pairs)
};

// Workgroups of the split kernels: four or eight waves on a panel group (a
// launch's problems, and grouped ones), or one wave on one panel pair (grouped
// three-term problems of tile 64, wave_pairs).  Three terms' stages fill the LDS with one workgroup a CU, which with
// four waves leaves each SIMD a single one whose every wait shows: eight waves
// then share the four pairs, each taking half the columns of a K tile, and
// add their sums up through LDS (m = 700, 2 x 9.8k columns: 230 -> 196 us; 2 x
// 59.7k: 1,267 -> 1,167 us; 12 chunks of a sky, 2 frequencies: 6.6 -> 5.9 ms).
constexpr int kSP = 64;  // rows of a panel
template <int NT> constexpr int kGroupWaves = NT == 3 ? 8 : 4;

// LDS position of word w (a multiple of 4) of row r in a K-tile panel of
// 16 words a row: the row's 16-byte chunk c is stored at chunk c ^ swz(r).
// Four rows span the 64 banks, so the rows that a 16-byte operand read serves
// together have to differ in r / 4 mod 4 where they share r mod 4.  The read
// serves lanes 0-3, 12-15, 20-23, 24-27 (r / 4 = 0, 3, 5, 6), then 4-7, 8-11,
// 16-19, 28-31, and so on, not 16 adjacent lanes: with a swizzle conflict-free
// for the latter, conflicts took 10% of the kernel's cycles; with this one
// SQ_LDS_BANK_CONFLICT counts none (m = 700, 59.7k sources: 642 -> 627 us).
__device__ __forceinline__ int swz(int r) { return (r >> 2) & 3; }
__device__ __forceinline__ int lds_word(int r, int w) {
  return r * kSK + (((w >> 2) ^ swz(r)) << 2);
}

// One K-tile stage: every term of the group's panels.  The two stages of a
// kernel are separate __shared__ objects, so that the compiler sees that
// loads in flight into one do not alias reads from the other.
template <int NT, int WAVES> struct alignas(16) SplitStage {
  uint32_t x[WAVES == 1 ? 2 : 4][NT][kSP * kSK];
};

// [x lanes 0-31 | y lanes 0-31] and [x lanes 32-63 | y lanes 32-63] of each
// register: the lane-half exchange of v_permlane32_swap.
__device__ __forceinline__ u32x4 halves_lo(u32x4 x, u32x4 y) {
  u32x4 r;
#pragma unroll
  for (int d = 0; d < 4; ++d)
    r[d] = __builtin_amdgcn_permlane32_swap(x[d], y[d], false, false)[0];
  return r;
}
__device__ __forceinline__ u32x4 halves_hi(u32x4 x, u32x4 y) {
  u32x4 r;
#pragma unroll
  for (int d = 0; d < 4; ++d)
    r[d] = __builtin_amdgcn_permlane32_swap(x[d], y[d], false, false)[1];
  return r;
}

// A wave computes its 64x64 panel pair as 2x2 blocks of 32x32x16 MFMA, whose
// K = 16 reals are 8 from lanes 0-31 and 8 from lanes 32-63.
//
// Term products are grouped so that small ones share an instruction with a
// large one: a lane half h in {0, 1} supplies its term (a_h for A, b_h for B)
// over the same 4 complex columns, so one MFMA adds t_a0 t_b0 + t_a1 t_b1
// before its single FP32 rounding into the accumulator.
//   (2 terms, 3 products): [hi|lo] x [lo|hi] per 4 columns, and hi*hi over 8
//     columns, whose operands are the lane-half exchange of two [hi|lo]
//     (A) and [lo|hi] (B) fragments already in registers
//   (2 terms, 4 products): [hi|lo] x [hi|lo] and [hi|lo] x [lo|hi]
//   (3 terms, 6 products): [h|m] x [h|m], [h|m] x [m|h], [h|l] x [l|h]
// Each costs the same number of MFMAs as issuing the products separately.
// The imaginary-part operand Y = (im, -re) of a B fragment is formed in
// registers.
//
// K tiles go through two LDS stages.  Each wave copies its panel of the next
// tile straight from global memory into the other stage
// (global_load_lds_dwordx4: 16 bytes a lane, lane l to byte 16 l of a 1 KB
// run of 16 rows), then computes the current tile; one barrier per K tile
// publishes the copy and frees the stage just read.  Rows past m are read as
// row m - 1: they only reach output rows and columns past m, which nothing
// reads.  All threads of a group that has panels' row norms to sum add
// |t0 + t1 (+ t2)|^2 of those panels' staged rows in FP64 (the exact
// diagonal), a quarter of a row each.
//
// Measured at m = 700, 2 x 59.7k columns, 2 terms, 3 products: on panel
// groups instead of square 128-row tiles (17 items a slice, not 21; 68 panel
// copies, not 72) and with the row norms spread over the groups, 20
// frequencies of the 350-antenna sky took 16.2 ms (17.6), three terms on a
// chunked sky 6.6 ms (7.3); norms left with their diagonal pairs 16.4 and
// 7.25 ms.  What bounds it now is power: 627 us, 1.17M cycles at 1.88 GHz,
// 63% of them MFMA-busy.  Without the copies 480 us (2.10 GHz), without the
// norms 590 (1.83), without either 456 (2.05), copies from L2 alone 610: a
// stall taken out (operand reads a step ahead, copies spread between the
// MFMAs, three stages) comes back as a lower clock.
template <int NT, int MAXORD, bool F16, int WAVES>
__device__ __forceinline__ void split_item(const SplitProblem &P, int slice,
                                           int group, int ns, int ktiles,
                                           int kps,
                                           SplitStage<NT, WAVES> &L0,
                                           SplitStage<NT, WAVES> &L1) {
  typedef SplitStage<NT, WAVES> Stage;
  constexpr int kHalves = WAVES == 8 ? 2 : 1;  // waves a pair
  constexpr int kRuns = kSP / 16 / kHalves;    // 16-row runs a wave copies
  // the wave's index in a scalar register: what it does is uniform over it
  const int windex =
      WAVES > 1 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6) : 0;
  const int wave = windex & 3, half = windex >> 2;
  const int lane = threadIdx.x & 63;
  const int lr = lane & 31, lh = lane >> 5;
  WavePair wp;
  int second = -1;  // one wave stages its pair's other panel too
  if constexpr (WAVES > 1) {
    wp = group_wave(group, P.nb, wave);
  } else {
    tile_coords(group, P.nb, wp.i, wp.j);
    wp.load = wp.i;
    wp.si = 0;
    wp.sj = wp.i == wp.j ? 0 : 1;
    wp.norm = wp.i == wp.j ? 0 : -1;
    wp.part = wp.i == wp.j ? kDiagonal : kWhole;
    if (wp.i != wp.j) second = wp.j;
  }
  const int kt0 = (int)((int64_t)slice * ktiles / ns);
  const int kt1 = (int)((int64_t)(slice + 1) * ktiles / ns);
  // copy lanes: run u covers rows 16 u .. 16 u + 15 of the wave's part of the
  // panel; lane l fills LDS chunk l % 4 of row 16 u + l / 4, i.e. logical
  // chunk (l % 4) ^ swz(row) of that row
  constexpr int kPanels = WAVES == 1 ? 2 : 1;  // panels a wave copies
  const int row0 = half * kRuns * 16;
  uint32_t coff[kPanels][kRuns];
#pragma unroll
  for (int q = 0; q < kPanels; ++q)
#pragma unroll
    for (int u = 0; u < kRuns; ++u) {
      const int r = row0 + u * 16 + (lane >> 2);
      const int row = (q ? second : wp.load) * kSP + r;
      const int c = (lane & 3) ^ swz(r);
      coff[q][u] = (uint32_t)((row < P.m ? row : P.m - 1) * kSK + 4 * c);
    }
  // the panels whose row norms this group sums (slots, -1: none); with eight
  // waves every other of them a half
  constexpr int kNorms = WAVES == 1 ? 1 : 4;
  int dslot[kNorms];
  double dsum[kNorms];
  bool any_diag = false;
#pragma unroll
  for (int w = 0; w < kNorms; ++w) {
    const WavePair q = WAVES > 1 ? group_wave(group, P.nb, w) : wp;
    dslot[w] = kHalves == 1 || (w & 1) == half ? q.norm : -1;
    any_diag = any_diag || dslot[w] >= 0;
    dsum[w] = 0.0;
  }
  double dsum1[4] = {0.0, 0.0, 0.0, 0.0};  // the one wave's
  const int nrow = (int)(threadIdx.x & 255) >> 2;  // the row it norms

  // position of the K tile to copy next: segment sg, tile kc within it;
  // whole K tiles: columns [seg_len, round_up(seg_len, 16)) of every
  // segment are zero by contract
  int sg = kt0 / (kps > 0 ? kps : 1), kc = kt0 - sg * kps;
  const int64_t seg_tiles = P.seg_stride / kSK;
  auto copy = [&](Stage &D) {
    const int64_t k0 = (sg * seg_tiles + kc) * P.ldz * kSK;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int u = 0; u < kRuns; ++u) {
        const int run = (row0 + u * 16) * kSK;
        if (WAVES == 1 || wp.load >= 0)
          copy16_to_lds(P.t[t] + k0 + coff[0][u], &D.x[wave][t][run]);
        if (WAVES == 1 && second >= 0)
          copy16_to_lds(P.t[t] + k0 + coff[kPanels - 1][u], &D.x[1][t][run]);
      }
    if (++kc == kps) {
      kc = 0;
      ++sg;
    }
  };
  // thread t: quarter t % 4 (4 columns) of row t / 4, and with one wave the
  // rows 16, 32, 48 further on
  auto diag_sums = [&](const Stage &D) {
#pragma unroll
    for (int w = 0; w < kNorms; ++w) {
      if (dslot[w] < 0) continue;
#pragma unroll
      for (int q = 0; q < (WAVES == 1 ? 4 : 1); ++q) {
        const int row = q * 16 + nrow;
        u32x4 r[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t)
          r[t] = *(const u32x4 *)&D.x[dslot[w]][t][lds_word(row, (lane & 3) * 4)];
        if constexpr (WAVES > 1) dsum[w] += row_norm2<NT, F16>(r);
        else dsum1[q] += row_norm2<NT, F16>(r);
      }
    }
  };
  auto store_norms = [&]() {
    // the four threads of a row are lanes 4 q .. 4 q + 3
    auto store = [&](int panel, int row, double s) {
      s += __shfl_xor(s, 1, 64);
      s += __shfl_xor(s, 2, 64);
      if ((lane & 3) == 0)
        P.dpart[((int64_t)slice * P.nb + panel) * kSP + row] = s;
    };
    if constexpr (WAVES > 1) {
#pragma unroll
      for (int w = 0; w < kNorms; ++w)
        if (dslot[w] >= 0)
          store(group_wave(group, P.nb, dslot[w]).load, nrow, dsum[w]);
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) store(wp.i, q * 16 + (lane >> 2), dsum1[q]);
    }
  };
  // The K loop of a wave that computes NI x NJ blocks from block (oi, oj),
  // without the one below the diagonal where DIAG.  A loop for each part: the
  // waves of a group run different ones, with the same barriers.  (Branches
  // around the parts' MFMAs within one loop spill accumulators.)
  auto run = [&](auto ni_, auto nj_, auto diag_, int oi, int oj) {
    constexpr int NI = decltype(ni_)::value, NJ = decltype(nj_)::value;
    constexpr bool DIAG = decltype(diag_)::value;
    v16f acc_re[NI][NJ], acc_im[NI][NJ];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        acc_re[i][j] = v16f{};
        acc_im[i][j] = v16f{};
      }

    // the MFMAs of one K tile from stage D
    auto compute = [&](const Stage &D) {
      const uint32_t(*Ax)[kSP * kSK] = D.x[wp.si];
      const uint32_t(*Bx)[kSP * kSK] = D.x[wp.sj];
      // lane half lh reads term t_lh at word offset w_lh of its row
      auto ld_a = [&](int t0, int t1, int w0, int w1, u32x4 (&a)[NI]) {
        const uint32_t *base = Ax[lh ? t1 : t0] + oi * 32 * kSK;
        const int w = lh ? w1 : w0;
#pragma unroll
        for (int i = 0; i < NI; ++i)
          a[i] = *(const u32x4 *)&base[lds_word(i * 32 + lr, w)];
      };
      auto ld_b = [&](int t0, int t1, int w0, int w1, u32x4 (&b)[NJ]) {
        const uint32_t *base = Bx[lh ? t1 : t0] + oj * 32 * kSK;
        const int w = lh ? w1 : w0;
#pragma unroll
        for (int j = 0; j < NJ; ++j)
          b[j] = *(const u32x4 *)&base[lds_word(j * 32 + lr, w)];
      };
      auto mma = [&](const u32x4 (&a)[NI], const u32x4 (&b)[NJ]) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          const u32x4 y = swap_negate4(b[j]);
#pragma unroll
          for (int i = 0; i < NI; ++i) {
            if (DIAG && i > j) continue;
            acc_re[i][j] = SplitMfma<F16>::op(a[i], b[j], acc_re[i][j]);
            acc_im[i][j] = SplitMfma<F16>::op(a[i], y, acc_im[i][j]);
          }
        }
      };
      u32x4 a[NI], b[NJ];
      if constexpr (NT == 2 && MAXORD == 1) {
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
          u32x4 a1[NI], b1[NJ];
          ld_a(0, 1, 8 * ks, 8 * ks, a);  // [hi|lo] of columns 8ks..8ks+3
          ld_b(1, 0, 8 * ks, 8 * ks, b);  // [lo|hi]
          mma(a, b);
          ld_a(0, 1, 8 * ks + 4, 8 * ks + 4, a1);
          ld_b(1, 0, 8 * ks + 4, 8 * ks + 4, b1);
          mma(a1, b1);
          // hi of columns 8ks..8ks+3 in lanes 0-31 and of 8ks+4..8ks+7 in
          // lanes 32-63, for A and B alike
#pragma unroll
          for (int i = 0; i < NI; ++i) a[i] = halves_lo(a[i], a1[i]);
#pragma unroll
          for (int j = 0; j < NJ; ++j) b[j] = halves_hi(b[j], b1[j]);
          mma(a, b);
        }
      } else if constexpr (NT == 2) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          ld_a(0, 1, 4 * q, 4 * q, a);
          ld_b(0, 1, 4 * q, 4 * q, b);
          mma(a, b);
          ld_b(1, 0, 4 * q, 4 * q, b);
          mma(a, b);
        }
      } else {
        // the wave's columns: all 16, or 8 half .. 8 half + 7
#pragma unroll
        for (int p = 0; p < 4 / kHalves; ++p) {
          const int w = 4 * (p + half * (4 / kHalves));
          ld_a(0, 1, w, w, a);
          ld_b(0, 1, w, w, b);
          mma(a, b);
          ld_b(1, 0, w, w, b);
          mma(a, b);
          ld_a(0, 2, w, w, a);
          ld_b(2, 0, w, w, b);
          mma(a, b);
        }
      }
    };
    // one K tile computed from stage C while the next is copied into N
    auto step = [&](Stage &C, Stage &N, int kt) {
      if (kt + 1 < kt1) copy(N);
      if (any_diag) diag_sums(C);
      if (WAVES == 1 || wp.i >= 0) {
        // issue priority to waves in their MFMA phase over waves copying or
        // waiting at the barrier
        __builtin_amdgcn_s_setprio(1);
        compute(C);
        __builtin_amdgcn_s_setprio(0);
      }
      wait_global_loads();  // this wave's copies into N
      lds_barrier();
    };

    for (int kt = kt0; kt < kt1; kt += 2) {
      step(L0, L1, kt);
      if (kt + 1 < kt1) step(L1, L0, kt + 1);
    }
    // every wave is past the last barrier: LDS is free for the next item
    if (any_diag) store_norms();

    if constexpr (kHalves == 2) {
      // the second halves' sums go to the first through LDS, real parts and
      // then imaginary parts: 16 KB a wave, two waves' in each stage's memory
      static_assert(sizeof(Stage) >= 2 * 64 * 64 * 4, "two waves' sums a stage");
      float *sums = (wave & 2 ? (float *)&L1 : (float *)&L0) +
                    (wave & 1) * 64 * 64 + lane;
      auto fold = [&](v16f(&acc)[NI][NJ]) {
        if (half == 1) {
#pragma unroll
          for (int e = 0; e < NI * NJ * 16; ++e)
            sums[e * 64] = acc[(e >> 4) / NJ][(e >> 4) % NJ][e & 15];
        }
        lds_barrier();
        if (half == 0) {
#pragma unroll
          for (int e = 0; e < NI * NJ * 16; ++e)
            acc[(e >> 4) / NJ][(e >> 4) % NJ][e & 15] += sums[e * 64];
        }
        lds_barrier();
      };
      fold(acc_re);
      fold(acc_im);
      if (half == 1) return;
    }
    if (WAVES > 1 && wp.i < 0) return;  // no pair, no partials
    // 32x32 accumulator layout: lane l, register r ->
    //   row 8*(r/4) + 4*(l/32) + r%4, col l%32.
    // The thread's base offset is opaque to the optimizer so that the store
    // addresses are formed here rather than kept live across the K loop.
    cplx<float> *out =
        P.part + ((int64_t)slice * P.ntiles + pair_index(wp.i, wp.j, P.nb)) *
                     kSP * kSP;
    int obase = (4 * lh + oi * 32) * kSP + lr + oj * 32;
    asm volatile("" : "+v"(obase));
    out += obase;
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        if (DIAG && i > j) continue;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int row = i * 32 + 8 * (r >> 2) + (r & 3);
          out[row * kSP + j * 32] =
              cplx<float>{acc_re[i][j][r], acc_im[i][j][r]};
        }
      }
  };

  if (kt0 < kt1) copy(L0);
  wait_global_loads();
  lds_barrier();
  const int oi = part_row(wp.part), oj = part_col(wp.part);
  if (wp.part == kWhole) run(Int<2>{}, Int<2>{}, Int<0>{}, 0, 0);
  else if (wp.part == kDiagonal) run(Int<2>{}, Int<2>{}, Int<1>{}, 0, 0);
  else if constexpr (WAVES > 1) {
    if (wp.part <= kBottom) run(Int<1>{}, Int<2>{}, Int<0>{}, oi, 0);
    else run(Int<1>{}, Int<1>{}, Int<0>{}, oi, oj);
  }
}

// One split HERK: K tiles and the slice count from the device column count,
// items (instance, slice, group) swept per XCD.
template <int NT, int MAXORD, bool F16>
__global__ __launch_bounds__(64 * kGroupWaves<NT>, 2) void herk_split_kernel(
    const SplitProblem P0, SliceCfg cfg, HerkBatch hb) {
  constexpr int W = kGroupWaves<NT>;
  __shared__ SplitStage<NT, W> L0, L1;
  SplitProblem P = P0;
  const int64_t seg_len = seg_columns(P.seg_len_host, P.seg_len_dev);
  const int kps = (int)cdiv(seg_len, (int64_t)kSK);  // K tiles per segment
  const int ktiles = kps * P.nseg;
  const int ns = active_slices_wave(ktiles, P.ngroups, cfg);
  const int64_t per = (int64_t)P.ngroups * ns;
  for_items(per * hb.n, [&](int64_t it) {
    const int64_t b = it / per, i = it - b * per;
#pragma unroll
    for (int t = 0; t < NT; ++t) P.t[t] = P0.t[t] + b * hb.z_stride;
    P.part = (cplx<float> *)((char *)P0.part + b * hb.ws_stride);
    P.dpart = (double *)((char *)P0.dpart + b * hb.ws_stride);
    split_item<NT, MAXORD, F16, W>(P, (int)(i / P.ngroups),
                                   (int)(i % P.ngroups), ns, ktiles, kps, L0,
                                   L1);
  });
}

// ------------------------------------------------------------ grouped

// Per-launch plan of a grouped HERK, written by herk_group_plan_kernel into
// the head of the workspace: slice counts, item and tile prefix offsets.
struct GroupPlan {
  int32_t *ns;        // [nprob]
  int64_t *item_off;  // [nprob + 1]
  int32_t *tile_off;  // [nprob + 1]
};

// Single block: every problem's internal descriptor (tile or, with `panels`,
// panel grid of side ts, partial
// areas carved from `parts` in problem order: cap x ntiles x ts^2 partial
// elements of part_bytes each, then, with row_norms, cap x ntiles x ts FP64
// row norms), its slice count (enough slices that no chain exceeds its kchain
// and cmax K tiles, chain0 where it names none, at most its capacity: a
// function of the problem alone) and the prefix offsets.
__global__ __launch_bounds__(256) void herk_group_plan_kernel(
    const mv_herk_problem *__restrict__ pub, int nprob, int ts, int panels,
    int kc, int cmax, int chain0, int part_bytes, int row_norms,
    SplitProblem *__restrict__ probs, char *__restrict__ parts,
    GroupPlan plan) {
  // Prefix sums of items, partial tiles and partial bytes over the problems,
  // 256 at a time: each thread forms its problem's in registers and the block
  // scans them in LDS (one thread walking the descriptors took 9 us for 24
  // problems).
  __shared__ int64_t items_s[256], bytes_s[256];
  __shared__ int32_t tiles_s[256];
  int64_t items0 = 0, bytes0 = 0;
  int32_t tiles0 = 0;
  const int t = threadIdx.x;
  for (int p0 = 0; p0 < nprob; p0 += 256) {
    const int p = p0 + t;
    SplitProblem P;
    int64_t items = 0, bytes = 0, own = 0;
    int32_t tiles = 0;
    if (p < nprob) {
      const mv_herk_problem &q = pub[p];
      for (int k = 0; k < 3; ++k) P.t[k] = (const uint32_t *)q.z[k];
      P.ldz = q.ldz;
      P.seg_stride = q.seg_stride;
      P.seg_len_host = q.seg_len;
      P.seg_len_dev = (const int32_t *)q.seg_len_dev;
      P.vacc = (cplx<double> *)q.vacc;
      P.ldv = q.ldv;
      P.scale = q.scale;
      P.m = q.m;
      P.nseg = q.nseg;
      P.accumulate = q.accumulate;
      P.nb = icdiv(q.m, ts);
      P.ntiles = P.nb * (P.nb + 1) / 2;
      P.ngroups = panels ? panel_groups(P.nb) : P.ntiles;
      const int64_t seg_len = seg_columns(q.seg_len, P.seg_len_dev);
      const int ktiles = (int)(cdiv(seg_len, (int64_t)kc) * q.nseg);
      const int chain = q.kchain > 0 ? (q.kchain < cmax ? q.kchain : cmax)
                                     : chain0;
      int ns = ktiles > 0 ? icdiv(ktiles, chain) : 1;
      ns = ns < 1 ? 1 : (ns > q.nslices ? q.nslices : ns);
      plan.ns[p] = ns;
      own = (int64_t)q.nslices * P.ntiles * ts * ts * part_bytes;
      bytes = own + (row_norms ? (int64_t)q.nslices * P.nb * ts * 8 : 0);
      items = (int64_t)P.ngroups * ns;
      tiles = P.ntiles;
    }
    items_s[t] = items;
    bytes_s[t] = bytes;
    tiles_s[t] = tiles;
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {
      const int64_t i = t >= off ? items_s[t - off] : 0;
      const int64_t b = t >= off ? bytes_s[t - off] : 0;
      const int32_t n = t >= off ? tiles_s[t - off] : 0;
      __syncthreads();
      items_s[t] += i;
      bytes_s[t] += b;
      tiles_s[t] += n;
      __syncthreads();
    }
    if (p < nprob) {
      char *at = parts + bytes0 + bytes_s[t] - bytes;
      P.part = (cplx<float> *)at;
      P.dpart = row_norms ? (double *)(at + own) : nullptr;
      probs[p] = P;
      plan.item_off[p] = items0 + items_s[t] - items;
      plan.tile_off[p] = tiles0 + tiles_s[t] - tiles;
    }
    items0 += items_s[255];
    bytes0 += bytes_s[255];
    tiles0 += tiles_s[255];
    __syncthreads();
  }
  if (t == 0) {
    plan.item_off[nprob] = items0;
    plan.tile_off[nprob] = tiles0;
  }
}

// index p with off[p] <= x < off[p + 1]
template <typename T>
__device__ __forceinline__ int find_segment(const T *off, int n, T x) {
  int lo = 0, hi = n;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (off[mid] <= x) lo = mid;
    else hi = mid;
  }
  return lo;
}

// All problems' items in one persistent launch, problem-major then
// slice-major, swept per XCD as in the single-problem kernel.
template <int NT, int MAXORD, bool F16, int WAVES>
__global__ __launch_bounds__(64 * WAVES, NT == 2 || WAVES == 8 ? 2 : 1) void
herk_split_grouped_kernel(
    const SplitProblem *__restrict__ probs, int nprob, GroupPlan plan) {
  __shared__ SplitStage<NT, WAVES> L0, L1;
  const int64_t items = plan.item_off[nprob];
  for_items(items, [&](int64_t it) {
    const int p = find_segment(plan.item_off, nprob, it);
    const SplitProblem P = probs[p];
    const int ns = plan.ns[p];
    const int64_t local = it - plan.item_off[p];
    const int64_t seg_len = seg_columns(P.seg_len_host, P.seg_len_dev);
    const int kps = (int)cdiv(seg_len, (int64_t)kSK);
    split_item<NT, MAXORD, F16, WAVES>(P, (int)(local / P.ngroups),
                                       (int)(local % P.ngroups), ns,
                                       kps * P.nseg, kps, L0, L1);
  });
}

// Grouped plain HERK: the items of all problems, as the grouped split
// kernel; each problem's Z is its term pointer 0.
template <typename T, int P>
__global__ __launch_bounds__(256, kPlainWgs<T>) void herk_plain_grouped_kernel(
    const SplitProblem *__restrict__ probs, int nprob, GroupPlan plan) {
  __shared__ PlainStage<T, P> L0, L1;
  const int64_t items = plan.item_off[nprob];
  for_items(items, [&](int64_t it) {
    const int p = find_segment(plan.item_off, nprob, it);
    const SplitProblem &S = probs[p];
    PlainProblem<T> Q;
    Q.z = (const cplx<T> *)S.t[0];
    Q.ldz = S.ldz;
    Q.seg_stride = S.seg_stride;
    const int64_t seg_len = seg_columns(S.seg_len_host, S.seg_len_dev);
    Q.part = (cplx<T> *)S.part;
    Q.m = S.m;
    Q.n = S.nb;
    Q.ngroups = S.ngroups;
    Q.npairs = S.ntiles;
    Q.wide = plain_wide(Q, S.nseg);
    const int ns = plan.ns[p];
    const int64_t local = it - plan.item_off[p];
    const int kps = (int)cdiv(seg_len, (int64_t)kPStageK<T>);
    plain_item<T, P>(Q, seg_len, (int)(local / Q.ngroups), (int)(local % Q.ngroups), ns,
                     kps * S.nseg, kps, L0, L1);
  });
}

// ------------------------------------------------------------ epilogues

// Elements of upper tile `tile`: the sum of their `ns` slice partials in
// FP64 (fixed order), scaled, stored or added into the accumulator.  With
// `dpart` (split forms) the diagonal elements of diagonal tiles take the row
// norms summed there instead of the MFMA sums.
//
// A wave takes 32 groups of kReduceEpt adjacent elements of one row; each
// group's sum over slices s = 8q + j is eight independent chains j, chains
// 0-3 in lanes 0-31 and chains 4-7 in lanes 32-63, so that each lane keeps
// four loads in flight and a launch has twice the workgroups of one lane per
// group.  The chains combine in a fixed order, ((c0 + c1) + (c2 + c3)) +
// ((c4 + c5) + (c6 + c7)); lane half h then stores element h of the group.
// (Four elements a lane halve the grid and measured slower.)
// Below the diagonal of a diagonal tile nothing is read (the compute kernels
// leave its blocks out): what is above it is stored there too, conjugated.
template <typename TP> constexpr int kReduceEpt = 2;

// The first element of the calling lane's group and its lane half.
template <typename TP>
__device__ __forceinline__ int64_t reduce_group(int &half) {
  const int lane = (int)(threadIdx.x & 63);
  half = lane >> 5;
  return kReduceEpt<TP> * ((int64_t)blockIdx.x * 128 +
                           (int64_t)(threadIdx.x >> 6) * 32 + (lane & 31));
}

template <typename TP, bool DTILE>
__device__ __forceinline__ void reduce_elems_t(
    const cplx<TP> *__restrict__ part, const double *__restrict__ dpart,
    int ntiles, int nb, int bi, int bj, int ts, int tile, int64_t e, int h,
    int ns, double scale, cplx<double> *__restrict__ vacc, int64_t ldv,
    int accumulate) {
  constexpr int E = kReduceEpt<TP>;
  static_assert(E == 2, "lane half h stores element h of its group");
  const int64_t tsz = (int64_t)ts * ts;
  const int64_t r = e / ts, c = e % ts;
  if (bi == bj && r > c + 1) return;  // both lane halves
  // what is accumulated onto is loaded before the sums, not waited for after
  cplx<double> *tile0 = vacc + (int64_t)bi * ts * ldv + (int64_t)bj * ts;
  cplx<double> *dst = tile0 + r * ldv + c + h;
  cplx<double> *mirror = tile0 + (c + h) * ldv + r;
  const bool above = bi != bj || r <= c + h, mirrored = bi == bj && r < c + h;
  cplx<double> old = {0.0, 0.0}, old_m = {0.0, 0.0};
  if (accumulate) {
    if (above) old = *dst;
    if (mirrored) old_m = *mirror;
  }
  const cplx<TP> *src = part + (int64_t)tile * tsz + e;
  const int64_t step = (int64_t)ntiles * tsz;
  // diagonal tiles (DTILE) also sum the row norms of the group's row, in the
  // same loop (every lane of the tile, so no lane runs extra rounds of
  // dependent loads after it)
  constexpr bool dtile = DTILE;
  const double *dp = dtile ? dpart + (int64_t)bi * ts + r : nullptr;
  const int64_t dstep = (int64_t)nb * ts;
  double re[E][4], im[E][4], dn[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    dn[j] = 0.0;
#pragma unroll
    for (int k = 0; k < E; ++k) re[k][j] = im[k][j] = 0.0;
  }
  // FP32 partials: all four chains' loads before the first sum, in source
  // order the compiler waits for each (16 frequencies of 128 antennas, 64
  // slices, 28.0 -> 18.6 us; m = 700, 59.7k sources 36.6 -> 28.3; 12 chunks of
  // 9.8k 24.7 -> 21.8; two rounds at once 24.4, 33.0 and 33.2).  FP64 partials
  // take twice the registers and lose waves with it (m = 700 12.4 -> 14.2).
  constexpr bool AHEAD = sizeof(TP) == 4;
  int s = 0;
  for (; s + 8 <= ns; s += 8) {
    cplx<TP> v[4][E];
    double d[4];
    auto load = [&](int j) {
      const int64_t sl = s + 4 * h + j;  // chain 4 h + j
      const cplx<TP> *q = src + sl * step;
#pragma unroll
      for (int k = 0; k < E; ++k) v[j][k] = q[k];
      if constexpr (dtile) d[j] = dp[sl * dstep];
    };
    if constexpr (AHEAD) {
#pragma unroll
      for (int j = 0; j < 4; ++j) load(j);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if constexpr (!AHEAD) load(j);
      if constexpr (dtile) dn[j] += d[j];
#pragma unroll
      for (int k = 0; k < E; ++k) {
        re[k][j] += (double)v[j][k].re;
        im[k][j] += (double)v[j][k].im;
      }
    }
  }
  if (h == 0) {
    // the last ns % 8 slices join chain 0
#pragma unroll(AHEAD ? 4 : 1)
    for (; s < ns; ++s) {
      const cplx<TP> *q = src + (int64_t)s * step;
#pragma unroll
      for (int k = 0; k < E; ++k) {
        re[k][0] += (double)q[k].re;
        im[k][0] += (double)q[k].im;
      }
      if constexpr (dtile) dn[0] += dp[(int64_t)s * dstep];
    }
  }
  // this half's four chains, then (chains 0-3) + (chains 4-7) in both
  // halves (the same sum: an IEEE add commutes)
  auto both = [&](const double (&x)[4]) {
    const double a = (x[0] + x[1]) + (x[2] + x[3]);
    const double b = __shfl_xor(a, 32, 64);
    return h == 0 ? a + b : b + a;
  };
  double sr[E], si[E];
#pragma unroll
  for (int k = 0; k < E; ++k) {
    sr[k] = both(re[k]);
    si[k] = both(im[k]);
  }
  double vr = h == 0 ? sr[0] : sr[1];
  double vi = h == 0 ? si[0] : si[1];
  if constexpr (dtile) {
    const double d = both(dn);
    if (r == c + h) {
      // the diagonal: the FP64 sum of |terms|^2 the compute kernel kept
      vr = d;
      vi = 0.0;
    }
  } else if (bi == bj && r == c + h) {
    vi -= vi;  // the diagonal is real: 0, or NaN where it is not finite
  }
  vr *= scale;
  vi *= scale;
  if (accumulate) {
    if (above) *dst = cplx<double>{old.re + vr, old.im + vi};
    if (mirrored) *mirror = cplx<double>{old_m.re + vr, old_m.im - vi};
  } else {
    if (above) *dst = cplx<double>{vr, vi};
    if (mirrored) *mirror = cplx<double>{vr, -vi};
  }
}

template <typename TP>
__device__ __forceinline__ void reduce_elems(
    const cplx<TP> *__restrict__ part, const double *__restrict__ dpart,
    int ntiles, int nb, int ts, int tile, int64_t e, int h, int ns,
    double scale, cplx<double> *__restrict__ vacc, int64_t ldv,
    int accumulate) {
  int bi, bj;
  tile_coords(tile, nb, bi, bj);
  if (dpart && bi == bj)  // uniform over the block: one tile a block
    reduce_elems_t<TP, true>(part, dpart, ntiles, nb, bi, bj, ts, tile, e, h,
                             ns, scale, vacc, ldv, accumulate);
  else
    reduce_elems_t<TP, false>(part, dpart, ntiles, nb, bi, bj, ts, tile, e, h,
                              ns, scale, vacc, ldv, accumulate);
}

// Blocks of 256 threads (128 element groups), per tile (looped past the
// grid's 65535).
template <typename TP>
dim3 reduce_grid(int ts, int64_t ntiles, int nbatch = 1) {
  return dim3((unsigned)cdiv((int64_t)ts * ts,
                             (int64_t)128 * kReduceEpt<TP>),
              (unsigned)(ntiles < 65535 ? ntiles : 65535), (unsigned)nbatch);
}

// grid reduce_grid<TP>(ts, ntiles, instances); the slice count is found once
// per block
template <typename TP>
__global__ __launch_bounds__(256) void herk_reduce_kernel(
    const cplx<TP> *__restrict__ part, const double *__restrict__ dpart,
    int ntiles, int ngroups, int nb, int ts, int64_t seg_len_host,
    const int32_t *__restrict__ seg_len_dev, int nseg, int kc, SliceCfg cfg,
    HerkBatch hb, double scale, cplx<double> *__restrict__ vacc, int64_t ldv,
    int accumulate) {
  __shared__ int ns_shared;
  if (threadIdx.x < 64) {
    const int64_t seg_len = seg_columns(seg_len_host, seg_len_dev);
    const int ktiles = (int)(cdiv(seg_len, (int64_t)kc) * nseg);
    const int ns = active_slices_wave(ktiles, ngroups, cfg);
    if (threadIdx.x == 0) ns_shared = ns;
  }
  __syncthreads();
  int h;
  const int64_t e = reduce_group<TP>(h);
  if (e >= (int64_t)ts * ts) return;
  const int64_t b = blockIdx.z;
  part = (const cplx<TP> *)((const char *)part + b * hb.ws_stride);
  if (dpart) dpart = (const double *)((const char *)dpart + b * hb.ws_stride);
  vacc += b * hb.vacc_stride;
  if (hb.scales) scale = hb.scales[b];
  for (int tile = blockIdx.y; tile < ntiles; tile += gridDim.y)
    reduce_elems(part, dpart, ntiles, nb, ts, tile, e, h, ns_shared, scale,
                 vacc, ldv, accumulate);
}

// Grouped reduce: blockIdx.y runs over the tiles of all problems (prefix
// offsets from the plan); lanes and element groups as above.
template <typename TP>
__global__ __launch_bounds__(256) void herk_group_reduce_kernel(
    const SplitProblem *__restrict__ probs, int nprob, int ts,
    GroupPlan plan) {
  int h;
  const int64_t e = reduce_group<TP>(h);
  if (e >= (int64_t)ts * ts) return;
  // the grid covers the tiles of the problems' largest shapes (a graph
  // replayed with smaller ones keeps it); tiles past this plan's total idle
  const int32_t total = plan.tile_off[nprob];
  for (int32_t t = blockIdx.y; t < total; t += gridDim.y) {
    const int p = find_segment(plan.tile_off, nprob, t);
    const SplitProblem &P = probs[p];
    reduce_elems((const cplx<TP> *)P.part, P.dpart, P.ntiles, P.nb, ts,
                 (int)(t - plan.tile_off[p]), e, h, plan.ns[p], P.scale,
                 P.vacc, P.ldv, P.accumulate);
  }
}

__global__ __launch_bounds__(256) void vacc_sum_kernel(
    const double *__restrict__ src, int nsrc_v, int64_t stride,
    double *__restrict__ dst, int64_t count) {
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= count) return;
  double s = 0.0;
  for (int i = 0; i < nsrc_v; ++i) s += src[(int64_t)i * stride + e];
  dst[e] = s;
}

// out[p, a, b] = V[i nf + b, j nf + a] from the r <= c half of the
// accumulator, V[r, c] = conj(V[c, r]) for the other half; grid.y instances.
template <typename TO>
__global__ __launch_bounds__(256) void expand_kernel(
    const cplx<double> *__restrict__ vacc, int64_t ldv, int nant, int nf,
    const int32_t *__restrict__ pairs, int64_t npairs,
    cplx<TO> *__restrict__ out, int64_t vacc_stride, int64_t out_stride) {
  vacc += blockIdx.y * vacc_stride;
  out += blockIdx.y * out_stride;
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int per = nf * nf;
  if (idx >= npairs * per) return;
  const int64_t p = idx / per;
  const int a = (int)((idx / nf) % nf), b = (int)(idx % nf);
  int i, j;
  if (pairs) {
    i = pairs[2 * p];
    j = pairs[2 * p + 1];
  } else {
    i = (int)(p / nant);
    j = (int)(p % nant);
  }
  if (i < 0 || i >= nant || j < 0 || j >= nant) {
    out[idx] = cplx<TO>{(TO)0, (TO)0};
    return;
  }
  const int64_t r = (int64_t)i * nf + b, c = (int64_t)j * nf + a;
  cplx<double> v;
  if (r <= c) {
    v = vacc[r * ldv + c];
  } else {
    v = vacc[c * ldv + r];
    v.im = -v.im;
  }
  out[idx] = cplx<TO>{(TO)v.re, (TO)v.im};
}

int split_maxord(int nterms, int nprod) {
  if (nterms == 2 && nprod == 3) return 1;
  if (nterms == 2 && nprod == 4) return 2;
  if (nterms == 3 && nprod == 6) return 2;
  return -1;
}

// Longest accumulation chain per slice, in K tiles of 16 columns, for m rows.
// The split forms' diagonal is summed exactly, and off the diagonal the FP32
// chain error stays near 1e-7 relative at 62 tiles and grows about as the
// square root of the length; 192 tiles keeps it well under 1e-6 while the
// partial tiles written per launch stay small.  The plain forms' real parts grow
// with the length in the same way, in FP64 too.  96 K tiles: 59.7k sources of 350
// antennas in complex64 with 128 3.7e-7 of |V|, with 96 2.3e-7, in the same 8.69
// ms for 4 frequencies; complex128, m = 160, 60k columns, 9.0e-17 of
// sqrt(V_ii V_jj) where one slice a slot gave 1.5e-16.  Problems of few rows
// write few partials: 64.
int form_cmax(int form, int m) {
  switch (form) {
    case MV_FORM_C128: return 96;
    case MV_FORM_C64: return m > 128 ? 96 : 64;
    default: return 192;
  }
}

// Longest K-slice, in K tiles, of a grouped split problem that asks for none:
// half the accuracy limit.  Measured at 192, 96 and 64 K tiles: 24 instances
// of 64-350 antennas 628, 408 and 391 us, two of 350 antennas 274, 229 and
// 189, 256 that fill the GPU by themselves 20.99, 21.22 and 21.98 ms (the
// partials of more slices).
constexpr int kGroupChain = 96;

// Resident workgroups of `kernel` on the current device (CUs x blocks per
// CU), rounded down to a multiple of the XCD count; cached per device.
template <class K> int kernel_slots(K kernel, int block) {
  static std::mutex mu;
  static std::map<std::pair<const void *, int>, int> cache;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return -1;
  const std::pair<const void *, int> key((const void *)kernel, dev);
  std::lock_guard<std::mutex> lock(mu);
  auto f = cache.find(key);
  if (f != cache.end()) return f->second;
  int cus = 0, per = 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount,
                            dev) != hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernel, block, 0) !=
          hipSuccess)
    return -1;
  int slots = cus * (per > 0 ? per : 1);
  slots = slots >= kXcd ? slots / kXcd * kXcd : kXcd;
  cache[key] = slots;
  return slots;
}

// ts: side of the partial tiles (plain: of the panels), nb of them a side,
// ntiles partial tiles and ngroups work items a slice
struct HerkPlan {
  int ts, nb, ntiles, ngroups, kc, threads;
  SliceCfg cfg;
  int grid;
};

// Panel side of the plain forms for row count m (of the largest problem in a
// grouped launch): 32 for complex128, whose 64-row panels' accumulators would
// not fit the registers.
int panel_side(int form, int m) {
  return form == MV_FORM_C64 && m > 128 ? 64 : 32;
}

// Slice counts beyond the least that an instance may take (slice_range): 128
// where five panels or fewer leave slots idle with them (4 groups of 512 slots).
int slice_reach(int form, int m) {
  const int panel = form == MV_FORM_SPLIT_F16 ? 64 : panel_side(form, m);
  return form != MV_FORM_SPLIT_BF16 && m <= 5 * panel ? 128 : 64;
}

}  // namespace
}  // namespace mv

using namespace mv;

extern "C" int mv_herk_tile(int form) {
  switch (form) {
    case MV_FORM_C128:
    case MV_FORM_C64: return kPT;
    case MV_FORM_SPLIT_BF16:
    case MV_FORM_SPLIT_F16: return kST;
    default: return 0;
  }
}

namespace {
// split forms: FP32 partial tiles, then FP64 row norms of diagonal tiles
size_t split_partial_bytes(int m, int nslices) {
  const int64_t nb = cdiv((int64_t)m, (int64_t)kST);
  return (size_t)nslices * (nb * (nb + 1) / 2) * kST * kST * 8;
}
}  // namespace

extern "C" size_t mv_herk_workspace_bytes(int form, int m, int nslices) {
  const int ts = mv_herk_tile(form);
  if (ts == 0 || m <= 0 || nslices <= 0) return 0;
  const int64_t nb = cdiv((int64_t)m, (int64_t)ts);
  const int64_t ntiles = nb * (nb + 1) / 2;
  if (ts == kST)
    return split_partial_bytes(m, nslices) + (size_t)nslices * ntiles * kST * 8;
  const size_t elem = form == MV_FORM_C128 ? 16 : 8;
  return (size_t)nslices * ntiles * ts * ts * elem;
}

extern "C" int mv_herk_max_slices(int form, int m, int64_t kmax) {
  const int ts = mv_herk_tile(form);
  if (ts == 0 || m <= 0 || kmax < 0) return 0;
  const int64_t ktiles = cdiv(kmax, (int64_t)16);
  if (ktiles == 0) return 1;
  const int64_t lo = cdiv(ktiles, (int64_t)form_cmax(form, m));
  const int64_t most = lo + slice_reach(form, m);
  const int64_t ns = most < ktiles ? most : ktiles;
  return (int)(ns < 1 ? 1 : ns);
}

namespace {
// The kernel instantiation for (form, nterms, maxord, panel side) as a
// type-erased pointer for occupancy queries.
const void *herk_kernel(int form, int nterms, int maxord, int panel) {
  switch (form) {
    case MV_FORM_C128: return (const void *)&herk_plain_kernel<double, 32>;
    case MV_FORM_C64:
      return panel == 64 ? (const void *)&herk_plain_kernel<float, 64>
                         : (const void *)&herk_plain_kernel<float, 32>;
    default: break;
  }
  const bool f16 = form == MV_FORM_SPLIT_F16;
  if (nterms == 2 && maxord == 1)
    return f16 ? (const void *)&herk_split_kernel<2, 1, true>
               : (const void *)&herk_split_kernel<2, 1, false>;
  if (nterms == 2)
    return f16 ? (const void *)&herk_split_kernel<2, 2, true>
               : (const void *)&herk_split_kernel<2, 2, false>;
  return f16 ? (const void *)&herk_split_kernel<3, 2, true>
             : (const void *)&herk_split_kernel<3, 2, false>;
}

// Whether a grouped split launch gives a wave a panel pair instead of a
// workgroup a panel group: three terms at tile 64.  Two terms take panel
// groups at either tile since a group's waves share single panels' pairs: 64
// instances of m = 64, 5k-40k columns (one feed), 341 us a pair a wave, 304 in
// groups; 400 of them 2,325 and 1,833; 64 of m = 128, 928 and 638; 8 of m =
// 64, 136 and 83.  Three terms, in groups of eight waves: m = 64, 64 instances
// 481 and 528, 400 instances 2,965 and 3,146 (m = 128: 1,450 and 1,148).
bool wave_pairs(int nterms, int tile) { return nterms == 3 && tile == 64; }

// The grouped split kernel for (form, nterms, maxord, wave_pairs).
const void *grouped_kernel(bool f16, int nterms, int maxord, bool pairs) {
  constexpr int W2 = kGroupWaves<2>, W3 = kGroupWaves<3>;
  if (nterms == 2 && maxord == 1)
    return f16 ? (const void *)&herk_split_grouped_kernel<2, 1, true, W2>
               : (const void *)&herk_split_grouped_kernel<2, 1, false, W2>;
  if (nterms == 2)
    return f16 ? (const void *)&herk_split_grouped_kernel<2, 2, true, W2>
               : (const void *)&herk_split_grouped_kernel<2, 2, false, W2>;
  if (pairs)
    return f16 ? (const void *)&herk_split_grouped_kernel<3, 2, true, 1>
               : (const void *)&herk_split_grouped_kernel<3, 2, false, 1>;
  return f16 ? (const void *)&herk_split_grouped_kernel<3, 2, true, W3>
             : (const void *)&herk_split_grouped_kernel<3, 2, false, W3>;
}

int plan_herk(int form, int nterms, int maxord, int m, int nslices,
              int nbatch, HerkPlan &p) {
  const bool plain = form == MV_FORM_C128 || form == MV_FORM_C64;
  p.ts = plain ? panel_side(form, m) : kSP;
  p.nb = (int)cdiv((int64_t)m, (int64_t)p.ts);
  p.ntiles = p.nb * (p.nb + 1) / 2;
  p.ngroups = panel_groups(p.nb);
  p.kc = plain ? kPK : kSK;
  p.threads = plain ? 256 : 64 * (nterms == 3 ? kGroupWaves<3> : kGroupWaves<2>);
  const int slots =
      kernel_slots(herk_kernel(form, nterms, maxord, p.ts), p.threads);
  if (slots <= 0) return -1;
  p.cfg = SliceCfg{nslices, slots, form_cmax(form, m), plain ? 2 : 4,
                   slice_reach(form, m), form != MV_FORM_SPLIT_BF16};
  const int64_t items = (int64_t)p.ngroups * nslices * nbatch;
  p.grid = (int)(items < slots ? items : slots);
  return 0;
}
}  // namespace

extern "C" int mv_herk_slices(int form, int nterms, int nprod, int m,
                              int nseg, int64_t seg_len, int nslices) {
  const int maxord = mv_herk_tile(form) == kST ? split_maxord(nterms, nprod)
                                               : 0;
  if (mv_herk_tile(form) == 0 || maxord < 0 || m < 1 || nseg < 1 ||
      seg_len < 0 || nslices < 1)
    return MV_ERR_ARG;
  HerkPlan p;
  if (plan_herk(form, nterms, maxord, m, nslices, 1, p))
    return MV_ERR_HIP;
  const int ktiles = (int)(cdiv(seg_len, (int64_t)p.kc) * nseg);
  return active_slices(ktiles, p.ngroups, p.cfg);
}

namespace {
constexpr int kPhaseCompute = 1, kPhaseReduce = 2;

struct PlainLaunch {
  const void *z;
  int m;
  int64_t ldz;
  int nseg;
  int64_t seg_stride, seg_len;
  const int32_t *seg_len_dev;
  double scale;
  double *vacc;
  int64_t ldv;
  int accumulate;
  void *workspace;
  int phases;
  hipStream_t st;
  HerkBatch hb;
};

template <typename T, int P>
int plain_run(const HerkPlan &p, const PlainLaunch &L) {
  PlainProblem<T> Q;
  Q.z = (const cplx<T> *)L.z;
  Q.ldz = L.ldz;
  Q.seg_stride = L.seg_stride;
  Q.part = (cplx<T> *)L.workspace;
  Q.m = L.m;
  Q.n = p.nb;
  Q.ngroups = p.ngroups;
  Q.npairs = p.ntiles;
  Q.wide = plain_wide(Q, L.nseg) &&
           L.hb.z_stride * 2 * (int64_t)sizeof(T) % 16 == 0;
  if (L.phases & kPhaseCompute) {
    herk_plain_kernel<T, P>
        <<<p.grid, 256, 0, L.st>>>(Q, L.nseg, L.seg_len, L.seg_len_dev, p.cfg,
                                   L.hb);
    if (int e = check_launch("mv_herk/plain")) return e;
  }
  if (!(L.phases & kPhaseReduce)) return MV_OK;
  herk_reduce_kernel<T>
      <<<reduce_grid<T>(p.ts, p.ntiles, L.hb.n), 256, 0, L.st>>>(
          (const cplx<T> *)L.workspace, nullptr, p.ntiles, p.ngroups, p.nb,
          p.ts, L.seg_len, L.seg_len_dev, L.nseg, p.kc, p.cfg, L.hb, L.scale,
          (cplx<double> *)L.vacc, L.ldv, L.accumulate);
  return check_launch("mv_herk/reduce");
}

// Validation shared by every phase, then the compute kernel (partial tiles
// into the workspace) and/or the reduce kernel (workspace into Vacc).
int herk_run(int phases, int form, int nterms, int nprod, const void *z0,
             const void *z1, const void *z2, int m, int64_t ldz, int nseg,
             int64_t seg_stride, int64_t seg_len, const int32_t *seg_len_dev,
             int nslices, double scale, double *vacc, int64_t ldv,
             int accumulate, void *workspace, size_t ws_bytes,
             mv_stream_t stream, HerkBatch hb = {1, 0, 0, 0, nullptr}) {
  const int ts = mv_herk_tile(form);
  MV_REQUIRE(ts > 0, "mv_herk: unknown form %d", form);
  MV_REQUIRE(z0 && vacc && workspace, "mv_herk: null pointer");
  MV_REQUIRE(m >= 1 && nseg >= 1 && seg_len >= 0 && nslices >= 1,
             "mv_herk: bad sizes m=%d nseg=%d seg_len=%lld nslices=%d", m,
             nseg, (long long)seg_len, nslices);
  MV_REQUIRE(nseg == 1 || seg_stride >= seg_len,
             "mv_herk: segments overlap (seg_stride %lld < seg_len %lld)",
             (long long)seg_stride, (long long)seg_len);
  MV_REQUIRE(ldz >= (form == MV_FORM_C128 || form == MV_FORM_C64
                         ? (int64_t)(nseg - 1) * seg_stride + seg_len
                         : (int64_t)m),
             "mv_herk: ldz %lld too small", (long long)ldz);
  MV_REQUIRE(cdiv(seg_len, (int64_t)16) * nseg < (int64_t)INT32_MAX / 2,
             "mv_herk: K too large");
  const int64_t nb = cdiv((int64_t)m, (int64_t)ts);
  const int64_t ntiles = nb * (nb + 1) / 2;
  MV_REQUIRE(ldv >= nb * ts, "mv_herk: ldv %lld < %lld (tile-padded m)",
             (long long)ldv, (long long)(nb * ts));
  MV_REQUIRE(ntiles * nslices * hb.n < (int64_t)INT32_MAX / 2,
             "mv_herk: too many work items");
  const size_t ws_one = mv_herk_workspace_bytes(form, m, nslices);
  MV_REQUIRE(ws_bytes / hb.n >= ws_one,
             "mv_herk: workspace too small (%zu < %d x %zu)", ws_bytes, hb.n,
             ws_one);
  hb.ws_stride = (int64_t)ws_one;
  const bool plain = form == MV_FORM_C128 || form == MV_FORM_C64;
  const int maxord = plain ? 0 : split_maxord(nterms, nprod);
  if (plain)
    MV_REQUIRE(nterms == 1, "mv_herk: plain forms take nterms=1");
  MV_REQUIRE(maxord >= 0,
             "mv_herk: unsupported split (nterms=%d, nprod=%d); supported: "
             "(2,3) (2,4) (3,6)",
             nterms, nprod);
  HerkPlan p;
  if (plan_herk(form, nterms, maxord, m, nslices, hb.n, p)) {
    set_error(MV_ERR_HIP, "mv_herk: occupancy query failed");
    return MV_ERR_HIP;
  }
  hipStream_t st = as_stream(stream);
  if (plain) {
    const PlainLaunch L = {z0,      m,      ldz,  nseg, seg_stride, seg_len,
                           seg_len_dev, scale, vacc, ldv,  accumulate,
                           workspace, phases, st, hb};
    if (form == MV_FORM_C128) return plain_run<double, 32>(p, L);
    return p.ts == 64 ? plain_run<float, 64>(p, L) : plain_run<float, 32>(p, L);
  }
  MV_REQUIRE(z1 && (nterms < 3 || z2), "mv_herk: missing term arrays");
  MV_REQUIRE(((uintptr_t)z0 | (uintptr_t)z1 | (uintptr_t)(z2 ? z2 : z0)) %
                     16 == 0,
             "mv_herk: split terms must be 16-byte aligned");
  const int64_t padded = cdiv(seg_len, (int64_t)kSK) * kSK;
  MV_REQUIRE(nseg == 1 || (seg_stride % kSK == 0 && seg_stride >= padded),
             "mv_herk: split terms need segments of whole %d-column K tiles "
             "(seg_stride %lld, seg_len %lld)",
             kSK, (long long)seg_stride, (long long)seg_len);
  const bool f16 = form == MV_FORM_SPLIT_F16;
  double *dpart = (double *)((char *)workspace + split_partial_bytes(m, nslices));
  SplitProblem P;
  P.t[0] = (const uint32_t *)z0;
  P.t[1] = (const uint32_t *)z1;
  P.t[2] = (const uint32_t *)z2;
  P.ldz = ldz;
  P.seg_stride = seg_stride;
  P.seg_len_host = seg_len;
  P.seg_len_dev = seg_len_dev;
  P.part = (cplx<float> *)workspace;
  P.dpart = dpart;
  P.vacc = (cplx<double> *)vacc;
  P.ldv = ldv;
  P.scale = scale;
  P.m = m;
  P.nseg = nseg;
  P.nb = p.nb;
  P.ntiles = p.ntiles;
  P.ngroups = p.ngroups;
  P.accumulate = accumulate;
#define MV_SPLIT_LAUNCH(NT, MO, F)                                           \
  herk_split_kernel<NT, MO, F><<<p.grid, p.threads, 0, st>>>(P, p.cfg, hb)
  if (phases & kPhaseCompute) {
    if (nterms == 2 && maxord == 1) {
      if (f16) MV_SPLIT_LAUNCH(2, 1, true);
      else MV_SPLIT_LAUNCH(2, 1, false);
    } else if (nterms == 2) {
      if (f16) MV_SPLIT_LAUNCH(2, 2, true);
      else MV_SPLIT_LAUNCH(2, 2, false);
    } else {
      if (f16) MV_SPLIT_LAUNCH(3, 2, true);
      else MV_SPLIT_LAUNCH(3, 2, false);
    }
    if (int e = check_launch("mv_herk/split")) return e;
  }
#undef MV_SPLIT_LAUNCH
  if (!(phases & kPhaseReduce)) return MV_OK;
  herk_reduce_kernel<float>
      <<<reduce_grid<float>(p.ts, p.ntiles, hb.n), 256, 0, st>>>(
          (const cplx<float> *)workspace, dpart, p.ntiles, p.ngroups, p.nb,
          p.ts, seg_len, seg_len_dev, nseg, p.kc, p.cfg, hb, scale,
          (cplx<double> *)vacc, ldv, accumulate);
  return check_launch("mv_herk/reduce");
}

}  // namespace

#define MV_HERK_ARGS                                                        \
  int form, int nterms, int nprod, const void *z0, const void *z1,          \
      const void *z2, int m, int64_t ldz, int nseg, int64_t seg_stride,     \
      int64_t seg_len, const int32_t *seg_len_dev, int nslices,             \
      double scale, double *vacc, int64_t ldv, int accumulate,              \
      void *workspace, size_t ws_bytes, mv_stream_t stream
#define MV_HERK_PASS                                                        \
  form, nterms, nprod, z0, z1, z2, m, ldz, nseg, seg_stride, seg_len,       \
      seg_len_dev, nslices, scale, vacc, ldv, accumulate, workspace,        \
      ws_bytes, stream

extern "C" int mv_herk(MV_HERK_ARGS) {
  return herk_run(kPhaseCompute | kPhaseReduce, MV_HERK_PASS);
}
extern "C" int mv_herk_compute(MV_HERK_ARGS) {
  return herk_run(kPhaseCompute, MV_HERK_PASS);
}
extern "C" int mv_herk_reduce(MV_HERK_ARGS) {
  return herk_run(kPhaseReduce, MV_HERK_PASS);
}
#undef MV_HERK_ARGS
#undef MV_HERK_PASS

extern "C" int mv_herk_batch(int phases, int form, int nterms, int nprod,
                             const void *z0, const void *z1, const void *z2,
                             int64_t z_stride, int nbatch, int m, int64_t ldz,
                             int nseg, int64_t seg_stride, int64_t seg_len,
                             const int32_t *seg_len_dev, int nslices,
                             const double *scales, double *vacc, int64_t ldv,
                             int64_t vacc_stride, int accumulate,
                             void *workspace, size_t ws_bytes,
                             mv_stream_t stream) {
  MV_REQUIRE(phases >= 1 && phases <= 3, "mv_herk_batch: phases 1, 2 or 3");
  MV_REQUIRE(nbatch >= 1 && nbatch <= 65535 && z_stride >= 0,
             "mv_herk_batch: bad batch");
  MV_REQUIRE(form == MV_FORM_C128 || form == MV_FORM_C64 || z_stride % 4 == 0,
             "mv_herk_batch: split terms must be 16-byte aligned");
  MV_REQUIRE(nbatch == 1 || vacc_stride >= ldv * ldv,
             "mv_herk_batch: accumulators overlap");
  return herk_run(phases, form, nterms, nprod, z0, z1, z2, m, ldz, nseg,
                  seg_stride, seg_len, seg_len_dev, nslices, 1.0, vacc, ldv,
                  accumulate, workspace, ws_bytes, stream,
                  HerkBatch{nbatch, z_stride, 0, vacc_stride, scales});
}

// ------------------------------------------------------------ no-alloc entry

namespace {
// The split-K partials of mv_herk_noalloc: device memory the library holds
// from load until the process ends, one copy on each device it runs on
// (128 MiB: room for 48 slices of the 350-antenna polarized split form,
// more than its accuracy cap of 192 K tiles a slice needs at 100k sources).
// A sum that would take more slices than fit runs longer ones than form_cmax:
// the 31 of complex128 at m = 700 hold 241 K tiles each of 2 x 59.7k columns.
// Host code uses the per-device address from hipGetSymbolAddress, never the
// array's name.  Every call on a device shares that device's copy and
// leaves its partials in it; nothing in it needs clearing (each call's
// kernels write every partial they later read).
constexpr size_t kScratchBytes = size_t(128) << 20;
}  // namespace

static __device__ __align__(256) char scratch[kScratchBytes];

namespace {
std::mutex g_scratch_mu;
std::map<int, void *> g_scratch_ptr;

// The address of this device's scratch copy (looked up once per device).
int scratch_address(void **out) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess)
    return set_error(MV_ERR_HIP, "mv_herk_noalloc: hipGetDevice failed");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  auto f = g_scratch_ptr.find(dev);
  if (f != g_scratch_ptr.end()) {
    *out = f->second;
    return MV_OK;
  }
  void *ptr = nullptr;
  const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !ptr)
    return set_error(MV_ERR_HIP,
                     "mv_herk_noalloc: hipGetSymbolAddress(scratch): %s",
                     hipGetErrorString(e));
  g_scratch_ptr[dev] = ptr;
  *out = ptr;
  return MV_OK;
}
}  // namespace

extern "C" int mv_herk_noalloc(int form, int nterms, int nprod,
                               const void *z0, const void *z1, const void *z2,
                               int m, int64_t ldz, int nseg,
                               int64_t seg_stride, int64_t seg_len,
                               const int32_t *seg_len_dev, double scale,
                               double *vacc, int64_t ldv, int accumulate,
                               mv_stream_t stream) {
  const int ts = mv_herk_tile(form);
  MV_REQUIRE(ts > 0, "mv_herk_noalloc: unknown form %d", form);
  MV_REQUIRE(m >= 1 && nseg >= 1 && seg_len >= 0,
             "mv_herk_noalloc: bad sizes m=%d nseg=%d seg_len=%lld", m, nseg,
             (long long)seg_len);
  // the slices the scratch holds, at most what mv_herk would size for
  const size_t one = mv_herk_workspace_bytes(form, m, 1);
  if (one == 0 || one > kScratchBytes)
    return set_error(MV_ERR_CAPACITY,
                     "mv_herk_noalloc: m=%d needs %zu bytes of partials for "
                     "one K-slice, more than the %zu-byte scratch",
                     m, one, kScratchBytes);
  int ns = mv_herk_max_slices(form, m, (int64_t)nseg * seg_len);
  const int fit = (int)(kScratchBytes / one);
  ns = ns < 1 ? 1 : (ns > fit ? fit : ns);
  void *ws = nullptr;
  if (int e = scratch_address(&ws)) return e;
  return herk_run(kPhaseCompute | kPhaseReduce, form, nterms, nprod, z0, z1,
                  z2, m, ldz, nseg, seg_stride, seg_len, seg_len_dev, ns,
                  scale, vacc, ldv, accumulate, ws,
                  mv_herk_workspace_bytes(form, m, ns), stream);
}

// ------------------------------------------------------------ grouped API

namespace {
int64_t align256(int64_t b) { return (b + 255) / 256 * 256; }

// Head of a grouped workspace: internal descriptors, then the plan arrays;
// the partial areas follow at `parts`.
struct GroupLayout {
  int64_t probs, ns, item_off, tile_off, parts, total;
};

// Bytes per partial element and whether FP64 row norms are kept, per form.
bool is_split_form(int form) {
  return form == MV_FORM_SPLIT_BF16 || form == MV_FORM_SPLIT_F16;
}
int part_bytes(int form) { return form == MV_FORM_C128 ? 16 : 8; }

// Panel side of a grouped launch.
int group_side(int form, const mv_herk_problem *q, int nprob) {
  int m = 0;
  for (int i = 0; i < nprob; ++i) m = q[i].m > m ? q[i].m : m;
  return is_split_form(form) ? kSP : panel_side(form, m);
}

// The partial areas are those of the plan kernel: slices of panel pairs.
GroupLayout group_layout(int form, const mv_herk_problem *q, int nprob) {
  const int ts = group_side(form, q, nprob);
  GroupLayout g;
  g.probs = 0;
  g.ns = align256((int64_t)nprob * sizeof(SplitProblem));
  g.item_off = g.ns + align256((int64_t)nprob * 4);
  g.tile_off = g.item_off + align256((int64_t)(nprob + 1) * 8);
  g.parts = g.tile_off + align256((int64_t)(nprob + 1) * 4);
  int64_t bytes = 0;
  for (int i = 0; i < nprob; ++i) {
    const int64_t nb = cdiv((int64_t)q[i].m, (int64_t)ts);
    const int64_t pairs = nb * (nb + 1) / 2;
    bytes += (int64_t)q[i].nslices *
             (pairs * ts * ts * part_bytes(form) +
              (is_split_form(form) ? nb * ts * 8 : 0));
  }
  g.total = g.parts + bytes;
  return g;
}
}  // namespace

extern "C" size_t mv_herk_problem_bytes(void) {
  return sizeof(mv_herk_problem);
}

namespace {
bool group_tile_ok(int form, int tile) {
  return is_split_form(form) ? (tile == 64 || tile == kST)
                             : ((form == MV_FORM_C128 || form == MV_FORM_C64) &&
                                tile == kPT);
}
}  // namespace

extern "C" size_t mv_herk_grouped_workspace_bytes(
    int form, int tile, const mv_herk_problem *problems, int nprob) {
  if (!group_tile_ok(form, tile) || !problems || nprob < 1) return 0;
  return (size_t)group_layout(form, problems, nprob).total;
}

extern "C" int mv_herk_grouped(int form, int nterms, int nprod, int tile,
                               const mv_herk_problem *problems_host,
                               const mv_herk_problem *problems_dev, int nprob,
                               void *workspace, size_t ws_bytes,
                               mv_stream_t stream) {
  const bool split = is_split_form(form);
  MV_REQUIRE(split || form == MV_FORM_C128 || form == MV_FORM_C64,
             "mv_herk_grouped: unknown form %d", form);
  MV_REQUIRE(group_tile_ok(form, tile),
             "mv_herk_grouped: tile %d (split forms: 64 or %d; plain: %d)",
             tile, kST, kPT);
  const int maxord = split ? split_maxord(nterms, nprod) : 0;
  MV_REQUIRE(split ? maxord >= 0 : nterms == 1,
             "mv_herk_grouped: unsupported terms (nterms=%d, nprod=%d)",
             nterms, nprod);
  MV_REQUIRE(problems_host && problems_dev && workspace && nprob >= 1,
             "mv_herk_grouped: null pointer or no problems");
  int64_t total_tiles = 0, max_items = 0;
  for (int i = 0; i < nprob; ++i) {
    const mv_herk_problem &q = problems_host[i];
    MV_REQUIRE(q.m >= 1 && q.nseg >= 1 && q.seg_len >= 0 &&
                   q.nslices >= 1 && q.kchain >= 0,
               "mv_herk_grouped: problem %d: bad sizes m=%d nseg=%d "
               "seg_len=%lld nslices=%d kchain=%d", i, q.m, q.nseg,
               (long long)q.seg_len, q.nslices, q.kchain);
    MV_REQUIRE(q.z[0] && (!split || q.z[1]) && (nterms < 3 || q.z[2]) &&
                   q.vacc,
               "mv_herk_grouped: problem %d: null pointer", i);
    if (split) {
      const int64_t padded = cdiv(q.seg_len, (int64_t)kSK) * kSK;
      MV_REQUIRE(((q.z[0] | q.z[1] | (q.z[2] ? q.z[2] : q.z[0])) % 16) == 0,
                 "mv_herk_grouped: problem %d: terms must be 16-byte "
                 "aligned", i);
      MV_REQUIRE((q.nseg == 1 ||
                  (q.seg_stride % kSK == 0 && q.seg_stride >= padded)) &&
                     q.ldz >= q.m,
                 "mv_herk_grouped: problem %d: split terms need segments of "
                 "whole %d-column K tiles and ldz >= m", i, kSK);
    } else {
      MV_REQUIRE((q.nseg == 1 || q.seg_stride >= q.seg_len) &&
                     q.ldz >= (int64_t)(q.nseg - 1) * q.seg_stride + q.seg_len,
                 "mv_herk_grouped: problem %d: segments overlap or ldz too "
                 "small", i);
    }
    const int64_t nb = cdiv((int64_t)q.m, (int64_t)tile);
    MV_REQUIRE(q.ldv >= nb * tile,
               "mv_herk_grouped: problem %d: ldv %lld < %lld", i,
               (long long)q.ldv, (long long)(nb * tile));
    total_tiles += nb * (nb + 1) / 2;
    max_items += nb * (nb + 1) / 2 * q.nslices;
  }
  MV_REQUIRE(total_tiles < 65536 && max_items < (int64_t)INT32_MAX / 2,
             "mv_herk_grouped: too many tiles (%lld) or items",
             (long long)total_tiles);
  const GroupLayout g = group_layout(form, problems_host, nprob);
  MV_REQUIRE(ws_bytes >= (size_t)g.total,
             "mv_herk_grouped: workspace too small (%zu < %lld)", ws_bytes,
             (long long)g.total);
  const bool f16 = form == MV_FORM_SPLIT_F16;
  const int side = group_side(form, problems_host, nprob);
  const bool by_wave = split && wave_pairs(nterms, tile);
  const void *kernel =
      split ? grouped_kernel(f16, nterms, maxord, by_wave)
      : form == MV_FORM_C128
          ? (const void *)&herk_plain_grouped_kernel<double, 32>
      : side == 64 ? (const void *)&herk_plain_grouped_kernel<float, 64>
                   : (const void *)&herk_plain_grouped_kernel<float, 32>;
  const int threads =
      !split       ? 256
      : by_wave    ? 64
                   : 64 * (nterms == 3 ? kGroupWaves<3> : kGroupWaves<2>);
  const int slots = kernel_slots(kernel, threads);
  if (slots <= 0) {
    set_error(MV_ERR_HIP, "mv_herk_grouped: occupancy query failed");
    return MV_ERR_HIP;
  }
  char *ws = (char *)workspace;
  SplitProblem *probs = (SplitProblem *)(ws + g.probs);
  GroupPlan plan{(int32_t *)(ws + g.ns), (int64_t *)(ws + g.item_off),
                 (int32_t *)(ws + g.tile_off)};
  hipStream_t st = as_stream(stream);
  // slices of a problem that names no chain: kGroupChain K tiles; plain forms
  // take slices of 64 K tiles (1024 columns) for parallelism
  herk_group_plan_kernel<<<1, 256, 0, st>>>(
      problems_dev, nprob, side, by_wave ? 0 : 1,
      split ? kSK : kPK,
      split ? form_cmax(form, 0) : 64, split ? kGroupChain : 64,
      part_bytes(form), split ? 1 : 0, probs, ws + g.parts, plan);
  if (int e = check_launch("mv_herk_grouped/plan")) return e;
  const int grid = (int)(max_items < slots ? max_items : slots);
  // the reduce runs over panel pairs, of which there are more than tiles
  int64_t pairs = 0;
  for (int i = 0; i < nprob; ++i) {
    const int64_t n = cdiv((int64_t)problems_host[i].m, (int64_t)side);
    pairs += n * (n + 1) / 2;
  }
  if (!split) {
    if (form == MV_FORM_C128)
      herk_plain_grouped_kernel<double, 32><<<grid, 256, 0, st>>>(probs, nprob,
                                                                  plan);
    else if (side == 64)
      herk_plain_grouped_kernel<float, 64><<<grid, 256, 0, st>>>(probs, nprob,
                                                                 plan);
    else
      herk_plain_grouped_kernel<float, 32><<<grid, 256, 0, st>>>(probs, nprob,
                                                                 plan);
    if (int e = check_launch("mv_herk_grouped/plain")) return e;
    if (form == MV_FORM_C128)
      herk_group_reduce_kernel<double>
          <<<reduce_grid<double>(side, pairs), 256, 0, st>>>(probs, nprob,
                                                             side, plan);
    else
      herk_group_reduce_kernel<float>
          <<<reduce_grid<float>(side, pairs), 256, 0, st>>>(probs, nprob, side,
                                                            plan);
    return check_launch("mv_herk_grouped/reduce");
  }
#define MV_GROUP_LAUNCH(NT, MO, W)                                           \
  do {                                                                       \
    if (f16)                                                                 \
      herk_split_grouped_kernel<NT, MO, true, W>                             \
          <<<grid, threads, 0, st>>>(probs, nprob, plan);                    \
    else                                                                     \
      herk_split_grouped_kernel<NT, MO, false, W>                            \
          <<<grid, threads, 0, st>>>(probs, nprob, plan);                    \
  } while (0)
  if (nterms == 2 && maxord == 1) MV_GROUP_LAUNCH(2, 1, kGroupWaves<2>);
  else if (nterms == 2) MV_GROUP_LAUNCH(2, 2, kGroupWaves<2>);
  else if (by_wave) MV_GROUP_LAUNCH(3, 2, 1);
  else MV_GROUP_LAUNCH(3, 2, kGroupWaves<3>);
#undef MV_GROUP_LAUNCH
  if (int e = check_launch("mv_herk_grouped/split")) return e;
  herk_group_reduce_kernel<float>
      <<<reduce_grid<float>(side, pairs), 256, 0, st>>>(probs, nprob, side,
                                                        plan);
  return check_launch("mv_herk_grouped/reduce");
}

extern "C" int mv_vacc_sum(const double *src, int nsrc_v, int64_t stride,
                           double *dst, int64_t count, mv_stream_t stream) {
  MV_REQUIRE(src && dst, "mv_vacc_sum: null pointer");
  MV_REQUIRE(nsrc_v >= 1 && count >= 0 && stride >= count,
             "mv_vacc_sum: bad sizes");
  if (count == 0) return MV_OK;
  vacc_sum_kernel<<<(unsigned)cdiv(count, (int64_t)256), 256, 0,
                    as_stream(stream)>>>(src, nsrc_v, stride, dst, count);
  return check_launch("mv_vacc_sum");
}

extern "C" int mv_vis_expand_batch(const double *vacc, int64_t ldv,
                                   int64_t vacc_stride, int nbatch, int tile,
                                   int nant, int nfeed, const int32_t *pairs,
                                   int64_t npairs, void *out, int out_is_f64,
                                   int64_t out_stride, mv_stream_t stream) {
  MV_REQUIRE(vacc && out, "mv_vis_expand: null pointer");
  MV_REQUIRE(tile > 0 && nant >= 1 && (nfeed == 1 || nfeed == 2) &&
                 npairs >= 0 && ldv >= (int64_t)nant * nfeed,
             "mv_vis_expand: bad sizes");
  MV_REQUIRE(nbatch >= 1 && nbatch <= 65535 && vacc_stride >= 0 &&
                 (nbatch == 1 || out_stride >= npairs * nfeed * nfeed),
             "mv_vis_expand: bad batch");
  const int64_t total = npairs * nfeed * nfeed;
  if (total == 0) return MV_OK;
  dim3 g((unsigned)cdiv(total, (int64_t)256), (unsigned)nbatch);
  hipStream_t st = as_stream(stream);
  if (out_is_f64)
    expand_kernel<double><<<g, 256, 0, st>>>(
        (const cplx<double> *)vacc, ldv, nant, nfeed, pairs, npairs,
        (cplx<double> *)out, vacc_stride, out_stride);
  else
    expand_kernel<float><<<g, 256, 0, st>>>(
        (const cplx<double> *)vacc, ldv, nant, nfeed, pairs, npairs,
        (cplx<float> *)out, vacc_stride, out_stride);
  return check_launch("mv_vis_expand");
}

extern "C" int mv_vis_expand(const double *vacc, int64_t ldv, int tile,
                             int nant, int nfeed, const int32_t *pairs,
                             int64_t npairs, void *out, int out_is_f64,
                             mv_stream_t stream) {
  return mv_vis_expand_batch(vacc, ldv, 0, 1, tile, nant, nfeed, pairs, npairs,
                             out, out_is_f64, 0, stream);
}

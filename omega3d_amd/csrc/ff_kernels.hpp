// ff_kernels.hpp -- factored far field for the point->point sums with velocity
// gradient, Rosenhead-Moore and compact-exponential cores (CoreFunc.h:65-71,
// 225-236), on the gfx950 matrix cores.
//
// The sums are the same direct sums over every pair (Kernels.h:155-193); only
// their arithmetic is reorganised for pairs of a target block and a source tile
// that are well separated.  Relative to the block centre c, with t' = t - c,
// s' = s - c, d = t' - s', m = alpha x s', and
//   RM:          r2 = |d|^2 + ss^2 + st^2,   K = r2^-3/2,  Bp = r2^-5/2
//   EXP (q>16):  r2 = |d|^2,                 K = r2^-3/2,  Bp = r2^-5/2
// every pair has K = Bp r2 = Bp (a - 2 t'.s' + b) with a = |t'|^2 + st^2 and
// b = |s'|^2 + ss^2 (no core terms for EXP).  Hence, summing over the tile,
//   W   = sum K alpha     = a P - 2 t'_l R_l + U
//   M   = sum K m         = a Q - 2 t'_l S_l + V
//   u   = sum K alpha x d = W x t' - M
//   D_ji = sum Bp d_j (alpha x d)_i = t'_j (P x t')_i - t'_j Q_i - (R_j x t')_i + S_ji
// with 29 moment sums, all of the form sum_k Bp_k f(source k):
//   P = sum Bp alpha (3), Q = sum Bp m (3), R_lk = sum Bp s'_l alpha_k (9),
//   S_lk = sum Bp s'_l m_k (8: s'.m = 0 so S_22 = -S_00 - S_11),
//   U = sum Bp b alpha (3), V = sum Bp b m (3).
// That is a product of the pair matrix Bp (sources x targets) with a per-source
// moment table (29 columns padded to 32) on the matrix cores; the squared distances
// are a matrix product too, which leaves one v_rsq_f32, three products and the split of
// the weight into two FP16 values per pair on the vector ALUs.  Two rings, compensated,
// far field of one call, before and after the pipelined form of k_ff_far, its slices and
// its cheaper staging: 65,536 particles 1.67 -> 1.32 ms, 131,072 5.7 -> 4.9, 262,144
// 21.6 -> 19.8, 1,048,576 323 -> 311.  By counter the last takes 303 ms now (3.55e12 pairs/s
// at 2.14 GHz): 7.2 vector instructions per pair, the vector units active 89% of the time
// and the matrix cores 41%.
//
// Separation: a tile is "far" for a block when the gap between their bounding
// spheres is at least one block radius (then every term above is at most
// (1+1/1)^2 = 4 times the pair's own contribution; measured on the two-ring
// workload, gaps of 1 and 2 radii give the same error, 1.5e-7, against FP64,
// and 0.5 radii 2.1e-7, with hardly fewer near pairs) and,
// for EXP, when that gap guarantees q = rho^3/(ss^3+st^3) > 16 for every pair,
// i.e. the reference's far branch (CoreFunc.h:121,169).  Other tiles go through
// the direct per-pair code in original coordinates, so near pairs keep exact
// differences t - s.
//
// The centre may be any point: a tile that is smaller than the block and one of its own
// radii away is far as well, with its own centre in place of the block's (the same bound
// by symmetry).  It is then summed by itself, and its gap is at least a third of the
// block's radius, so that the block's weights, scaled for the nearest target, keep their
// 22 bits at the farthest ((1 / 7)^5 of 2^13 is above 2^-3).  Few targets, wide blocks:
// pairs left near 21 -> 11% for 524,288 particles on 20,480 panels, 15 -> 8% for 65,537
// points in a box around two rings of 100,002 (whole calls 5.13 -> 4.58 and 2.16 -> 2.00 ms).
//
// Nor may a block be so much smaller than the tile, or the core terms (RM and WL: part of
// r2, V2: beside its square) so unlike each other, that one scale leaves a weight too few
// bits: the largest r2 that a pair of the tile and the block can have is at most FF_RANGE
// times the least, from which the scale is taken, cores included (a gap alone, beside cores
// ten times as wide, left weights of 1e-5 times the scale, and fewer bits with each).
//
// Particles are sorted along a Hilbert curve first (keys on a 10-bit grid per axis) so
// that blocks and tiles are compact; the decision per (block, tile) is computed
// once into a bit mask read by both kernels.  The curve has no jumps: in Morton order a
// block across a jump has nearly every tile near.  Pairs left near, Morton and Hilbert:
// two rings of 131,070 7.6 and 6.4%, of 262,144 5.3 and 4.4%; 65,537 points in a box
// around two rings of 100,002 25 and 15%; 20,480 panels on 524,288 points 13 and 7.6%.
#pragma once
#include "p2p_kernels.hpp"

#include <algorithm>
#include <type_traits>

// the far field's schedule of one phase (k_ff_far): n matrix products, each followed by
// its share (tr, va) of the phase's vector work, the quarter-rate square roots first
#define FF_SCHED(n, tr, va)                                                  \
  _Pragma("unroll") for (int q_ = 0; q_ < (n); ++q_) {                   \
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                       \
    __builtin_amdgcn_sched_group_barrier(0x400, (tr), 0);                    \
    __builtin_amdgcn_sched_group_barrier(0x002, (va), 0);                    \
  }                                                                          \
  __builtin_amdgcn_sched_barrier(0)

namespace o3d {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// the singular kernel of panel points: K = r^-3, Bp = r^-5, no core terms; the core term
// of a row is the distance from there beyond which a pair is a plain point pair
constexpr int CORE_SING = 0;
constexpr int FF_TB = 256;          // targets per workgroup: 4 waves x 64
constexpr float FF_KAPPA = 1.0f;    // minimum gap, in radii of the block or the tile, whichever is smaller
constexpr float FF_SPREAD = 1.0f / 3.0f;   // and in block radii, so that one scale serves the block's weights
constexpr float FF_RANGE = 81.0f;   // largest to least r2: 9 to the fifth is 2^16, of a weight's 2^13 and 24 bits below
// near field, compensated: sources per FP32 partial.  Gradient error against FP64 on two
// rings: EXP, 1,048,576 particles, 5.9e-8 at 32 and 5.0e-8 at 16 (near field 30.3 and
// 31.5 ms); RM, 262,144, 4.5e-8 and 4.3e-8, with the near field 6% slower at 16; WL,
// 131,070, 5.6e-8 at 32, 5.2e-8 at 16, 4.9e-8 at 8 (the call 0 and 1% slower)
template <int CORE, bool GRAD>
constexpr int ff_fold() { return !GRAD || CORE == CORE_WL ? 8 : CORE == CORE_RM ? 32 : 16; }
constexpr int FF_M0 = 4;            // near field: fewest tiles per work item
constexpr int FF_FAR_THREADS = 256; // far field: 4 waves of 64 targets per block
constexpr int FF_TP = 264;          // far field: LDS row of the FP16 moment tables (halves, tile <= 256)
constexpr int FF_SL = 40;           // far field: LDS row of a source's BF16 r2 slots (32 used, 80 bytes)
// far field: most consecutive tiles per fold into FP64.  Two rings, 262,144 particles, RM:
// velocity error 4.5e-8 at 8 tiles, 4.2e-8 at 4; far field 20.2 and 20.5 ms.
// Cores that the direct kernel sums otherwise (4.6e-8): 2
template <int CORE, bool GRAD>
constexpr int ff_merge() { return GRAD && (CORE == CORE_RM || CORE == CORE_EXP || CORE == CORE_SING) ? 4 : 2; }
// RM and EXP with gradient, compensated, of fewer points: both are finer, so that such a call
// is no further from FP64 than the direct sum, which serves it below AUTO's line.  Normwise
// errors of velocity and gradient, two rings of RM: 30,100 particles direct 3.6e-8 3.9e-8, as
// above 4.1e-8 5.0e-8, with 2 tiles and 8 sources 3.5e-8 3.3e-8; 60,000 3.5e-8 3.5e-8, 3.8e-8
// 4.2e-8, 3.4e-8 3.1e-8; EXP 24,600 4.2e-8 1.1e-7, 4.3e-8 1.1e-7, 3.9e-8 0.9e-7.  It costs 3.5%
// (65,536 RM 1.64 and 1.70 ms), and at 1,048,576 EXP 2.6%; from FF_FINE_BELOW targets and
// sources, where single calls have always come here, the coarser ones stay.
constexpr int64_t FF_FINE_BELOW = 65536;
constexpr int FF_FINE_MERGE = 2, FF_FINE_FOLD = 8;
template <int CORE, bool GRAD>
constexpr bool ff_sized() { return GRAD && (CORE == CORE_RM || CORE == CORE_EXP); }

struct FFArgs {
  const float4* sp;    // sorted sources {x, y, z, core_term}, up to a whole tile: the last one again
  const float4* sa;    // sorted sources {ax, ay, az, q}, up to a whole tile: zeros (q: source strength of panels, or 0)
  const float4* tq;    // sorted targets {x, y, z, core_term or 0 for point targets}
  const int* tperm;    // sorted target -> original target index
  const float4* tsph;  // per source tile: bounding sphere {cx, cy, cz, r}
  const float4* tlim;  // per source tile and target block: FFBounds::lim
  const float4* bsph;  // per target block: bounding sphere
  const float4* blim;
  const unsigned* mask;  // far bit per (block, tile), mwords words per block
  double* farv;        // per slice and target, sorted: far-field velocity and gradient, 12 (3) (FFSum)
  const int* tinv;     // original target -> sorted target
  int32_t nslice;      // slices of the far field: slice y takes tiles [y * tslice, (y + 1) * tslice)
  int32_t tslice;
  const int* nn;       // near tiles per block
  const int* items;    // near-field work items per block
  const int* ioff;     // exclusive scan of items
  const int* mfold;    // near tiles per item
  unsigned* ctr;       // work-queue counter
  double* part;        // per item and target of the block: 12 (3) partial sums (FFSum)
  int32_t rows;        // a target's sums lie in a row
  SrcView s;           // original sources (self-pair exclusion)
  TgtView t;           // original targets (outputs, accumulated)
  int64_t ns, nt;
  int32_t tile;        // sources per tile: 64, 128 or 256
  int32_t mwords;
  int32_t ntiles;
  int32_t self_excl;
  int32_t merge, fold;   // ff_sized: far tiles per fold, near sources per partial
};

// NOUT sums of one target: in a row, or each a whole array of n targets apart.  k_ff_combine
// gathers rows and reads and writes the 12 output arrays in order; from arrays it scatters a
// float of each to a line of its own, which costs where the outputs do not stay in the
// caches: 524,288 targets 206 us, the call 4.82 ms, with rows 4.68; 262,144 alike, 65,536
// with 16 slices 1.66 and 1.69
constexpr int64_t FF_ROWS_MIN = 393216;
template <int NOUT>
__device__ __forceinline__ void ff_sum_store(double* base, int64_t n, int64_t i, bool rows, const double* v) {
  if (rows) {
#pragma unroll
    for (int k = 0; k < NOUT; ++k) base[i * NOUT + k] = v[k];
  } else {
#pragma unroll
    for (int k = 0; k < NOUT; ++k) base[k * n + i] = v[k];
  }
}
template <int NOUT>
__device__ __forceinline__ void ff_sum_add(const double* base, int64_t n, int64_t i, bool rows, double* v) {
  if (rows) {
#pragma unroll
    for (int k = 0; k < NOUT; ++k) v[k] += base[i * NOUT + k];
  } else {
#pragma unroll
    for (int k = 0; k < NOUT; ++k) v[k] += base[k * n + i];
  }
}

// ---- order-preserving float <-> uint (for atomic min / max of floats) ---------
__device__ __forceinline__ unsigned fenc(float f) {
  const unsigned b = __float_as_uint(f);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float fdec(unsigned e) {
  return __uint_as_float((e & 0x80000000u) ? (e & 0x7fffffffu) : ~e);
}

static __global__ void k_ff_bbox_init(unsigned* bb) {
  if (threadIdx.x < 3) bb[threadIdx.x] = 0xffffffffu;
  else if (threadIdx.x < 6) bb[threadIdx.x] = 0u;
}

// bounding box of one or two point sets (x, y, z SoA) into bb[0..5] (encoded).
// Each workgroup reduces its strided share through shuffles and LDS and then
// issues 6 atomics, so a launch of FF_BBOX_GRID workgroups makes few atomics on
// the 6 shared words (one per wave took ~0.5 ms at N = 1M).
constexpr unsigned FF_BBOX_GRID = 512;
static __global__ __launch_bounds__(256) void k_ff_bbox(const float* x, const float* y, const float* z, int64_t n,
                                                 unsigned* bb) {
  __shared__ float red[4][6];
  float lo[3] = {__builtin_huge_valf(), __builtin_huge_valf(), __builtin_huge_valf()};
  float hi[3] = {-__builtin_huge_valf(), -__builtin_huge_valf(), -__builtin_huge_valf()};
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const float v[3] = {x[i], y[i], z[i]};
#pragma unroll
    for (int d = 0; d < 3; ++d) { lo[d] = fminf(lo[d], v[d]); hi[d] = fmaxf(hi[d], v[d]); }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      lo[d] = fminf(lo[d], __shfl_xor(lo[d], off));
      hi[d] = fmaxf(hi[d], __shfl_xor(hi[d], off));
    }
  }
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
#pragma unroll
    for (int d = 0; d < 3; ++d) { red[w][d] = lo[d]; red[w][3 + d] = hi[d]; }
  }
  __syncthreads();
  if (threadIdx.x < 6) {
    const int d = threadIdx.x;
    const int nw = (int)(blockDim.x >> 6);
    float v = red[0][d];
    for (int k = 1; k < nw; ++k) v = d < 3 ? fminf(v, red[k][d]) : fmaxf(v, red[k][d]);
    if (d < 3) atomicMin(&bb[d], fenc(v));
    else atomicMax(&bb[d], fenc(v));
  }
}

__device__ __forceinline__ unsigned spread10(unsigned v) {
  v &= 1023u;
  v = (v | (v << 16)) & 0x030000FFu;
  v = (v | (v << 8)) & 0x0300F00Fu;
  v = (v | (v << 4)) & 0x030C30C3u;
  v = (v | (v << 2)) & 0x09249249u;
  return v;
}

// position of a point of the 2^10 grid along the Hilbert curve: coordinates turned and
// mirrored bit by bit from the top (Skilling, "Programming the Hilbert curve", AIP Conf.
// Proc. 707, 2004), then Gray-decoded
__device__ __forceinline__ unsigned hilbert30(unsigned x, unsigned y, unsigned z) {
  unsigned c[3] = {x, y, z};
#pragma unroll
  for (int b = 9; b >= 1; --b) {
    const unsigned low = (1u << b) - 1u;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      if ((c[d] >> b) & 1u) {
        c[0] ^= low;
      } else {
        const unsigned t = (c[0] ^ c[d]) & low;
        c[0] ^= t;
        c[d] ^= t;
      }
    }
  }
  c[1] ^= c[0];
  c[2] ^= c[1];
  unsigned t = 0;
#pragma unroll
  for (int b = 9; b >= 1; --b)
    if ((c[2] >> b) & 1u) t ^= (1u << b) - 1u;
  return (spread10(c[0] ^ t) << 2) | (spread10(c[1] ^ t) << 1) | spread10(c[2] ^ t);
}

// 30-bit Morton keys on the common bounding box, and the identity permutation
static __global__ __launch_bounds__(256) void k_ff_keys(const float* x, const float* y, const float* z, int64_t n,
                                                 const unsigned* bb, unsigned* keys, int* idx) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float lx = fdec(bb[0]), ly = fdec(bb[1]), lz = fdec(bb[2]);
  const float ext = fmaxf(fmaxf(fdec(bb[3]) - lx, fdec(bb[4]) - ly), fdec(bb[5]) - lz);
  const float sc = ext > 0.0f ? 1023.0f / ext : 0.0f;
  const float q[3] = {(x[i] - lx) * sc, (y[i] - ly) * sc, (z[i] - lz) * sc};
  unsigned k = 0;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const float c = fminf(fmaxf(q[d], 0.0f), 1023.0f);   // NaN -> 0
    k |= spread10((unsigned)c) << d;
  }
  keys[i] = k;
  if (idx) idx[i] = (int)i;
}

// ---- the factored calls' preparation ------------------------------------------------
// Sources and targets (one set where they are the same collection) are sorted in one go,
// the set as the top bit of the key, and each step is one launch for both: box, keys,
// the sort's passes, rows and bounds, far bits, plan.  A small call waits for its launches,
// about 4 us each.  Two sets of 2,048 and 5,120: 40 launches before, 14 now.
struct FFSets {
  const float *x[2], *y[2], *z[2];
  int64_t n[2];          // n[1] = 0: one set
  const uint32_t* idx;   // set `pan` is panels: three node indices each, x, y, z the nodes
  int32_t pan;
};
__device__ __forceinline__ void ff_position(const FFSets& s, int set, int64_t i, float* p) {
  if (s.idx && set == s.pan) {   // about the centroid: it only decides the order
    const uint32_t a = s.idx[3 * i], b = s.idx[3 * i + 1], c = s.idx[3 * i + 2];
    p[0] = (s.x[set][a] + s.x[set][b] + s.x[set][c]) * (1.0f / 3.0f);
    p[1] = (s.y[set][a] + s.y[set][b] + s.y[set][c]) * (1.0f / 3.0f);
    p[2] = (s.z[set][a] + s.z[set][b] + s.z[set][c]) * (1.0f / 3.0f);
  } else {
    p[0] = s.x[set][i]; p[1] = s.y[set][i]; p[2] = s.z[set][i];
  }
}

// largest of each of N values over the workgroup's four waves, in every thread
template <int N>
__device__ __forceinline__ void wg_max_n(float* v) {
  __shared__ float red[4][N];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
#pragma unroll
    for (int k = 0; k < N; ++k) v[k] = fmaxf(v[k], __shfl_xor(v[k], off));
  __syncthreads();
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int k = 0; k < N; ++k) red[threadIdx.x >> 6][k] = v[k];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < N; ++k) v[k] = fmaxf(fmaxf(red[0][k], red[1][k]), fmaxf(red[2][k], red[3][k]));
}

// middle one of a wave's values (no NaN), in every lane: the largest that at most half
// are below
__device__ __forceinline__ float wave_median(float x) {
  int below = 0;
#pragma unroll
  for (int j = 0; j < 64; ++j) below += __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(x), j)) < x;
  float m = below <= 32 ? x : -__builtin_huge_valf();
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
  return m;
}

// Each workgroup's boxes {-lo, hi} of both sets over its strided share of them; and, one
// workgroup per set beside these, where its points are: of 64 of them, per axis, the median
// and the median distance from it, {median 3, distance 3} in `where`
constexpr int FF_BOX_GRID = 256;
constexpr int FF_BOX_FLOATS = 12 * FF_BOX_GRID + 12;   // boxes, then where
static __global__ __launch_bounds__(256) void k_ff_box(FFSets s, float* part, int nparts, float* where) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if ((int)blockIdx.x >= nparts) {
    const int set = (int)blockIdx.x - nparts;
    if (w > 2) return;
    float p[3] = {0.0f, 0.0f, 0.0f};
    if (s.n[set] > 0) ff_position(s, set, s.n[set] * lane / 64, p);
    const float x = w == 0 ? p[0] : w == 1 ? p[1] : p[2];
    const float m = wave_median(x == x ? x : 0.0f);
    const float r = wave_median(x == x ? fabsf(x - m) : 0.0f);
    if (lane == 0) { where[6 * set + w] = m; where[6 * set + 3 + w] = r; }
    return;
  }
  float v[12];
#pragma unroll
  for (int d = 0; d < 12; ++d) v[d] = -__builtin_huge_valf();
#pragma unroll
  for (int set = 0; set < 2; ++set)
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < s.n[set]; i += (int64_t)nparts * 256) {
      float p[3];
      ff_position(s, set, i, p);
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        v[6 * set + d] = fmaxf(v[6 * set + d], -p[d]);
        v[6 * set + 3 + d] = fmaxf(v[6 * set + 3 + d], p[d]);
      }
    }
  wg_max_n<12>(v);
  if (threadIdx.x == 0)
#pragma unroll
    for (int d = 0; d < 12; ++d) part[12 * blockIdx.x + d] = v[d];
}

// Where a set's box says little about where its points are (a few particles that have left,
// a dense collection in a wide field), a grid of 2^8 or 2^10 cells per axis has the collection
// in a few cells and its blocks in no order.  So each axis is laid out about the median,
// linear up to twice the points' spread (the median distance from it, of the widest axis)
// and logarithmic beyond; a box within FF_WIDE spreads, as of any collection that fills its
// box somehow, stays linear.  Ring pairs, RM with gradient, one particle in 10,000 100 radii
// away: of 100,000 7.2 ms without and 3.7 with (3.7 without such particles), of 300,000 63
// and 29.6 (28.5); a tenth of 100,000 WL particles 300 radii away 9.9 and 6.2
constexpr float FF_WIDE = 8.0f;
struct FFAxes {
  float mid[3], lo[3], sc;
  float core;   // half the width of the linear part, 0: linear throughout
  __device__ __forceinline__ float at(int d, float x) const {
    if (core == 0.0f) return x;
    const float u = x - mid[d], a = fabsf(u);
    return copysignf(a <= core ? a : core * (1.0f + 0.69314718f * __builtin_amdgcn_logf(a / core)), u);
  }
  // v: the set's box {-lo, hi}
  __device__ __forceinline__ FFAxes(const float* v, const float* where) {
    float far = 0.0f, ext = 0.0f;
    core = 0.0f;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      mid[d] = where[d];
      core = fmaxf(core, 2.0f * where[3 + d]);
      far = fmaxf(far, fmaxf(v[3 + d] - mid[d], v[d] + mid[d]));
    }
    if (!(far > 0.5f * FF_WIDE * core && far < __builtin_huge_valf())) core = 0.0f;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      lo[d] = -at(d, -v[d]);
      ext = fmaxf(ext, at(d, v[3 + d]) + lo[d]);
    }
    sc = ext > 0.0f ? 1023.0f / ext : 0.0f;
  }
};

// the top `bits` bits of the 30-bit Hilbert keys, each set's on a grid of its own (they are
// sorted apart, so nothing has to match), below the set's bit, and each set's identity
// permutation
static __global__ __launch_bounds__(256) void k_ff_hkeys(FFSets s, const float* part, int nparts, const float* where,
                                                  int bits, unsigned* keys, int* idx) {
  float v[12];
#pragma unroll
  for (int d = 0; d < 12; ++d) v[d] = -__builtin_huge_valf();
  for (int k = threadIdx.x; k < nparts; k += 256)
#pragma unroll
    for (int d = 0; d < 12; ++d) v[d] = fmaxf(v[d], part[12 * k + d]);
  if (s.n[1] > 0) wg_max_n<12>(v);
  else wg_max_n<6>(v);
#pragma unroll
  for (int set = 0; set < 2; ++set) {
    if (s.n[set] == 0) continue;
    const FFAxes ax(v + 6 * set, where + 6 * set);
    for (int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x; j < s.n[set]; j += (int64_t)gridDim.x * 256) {
      float p[3];
      ff_position(s, set, j, p);
      unsigned c[3];
#pragma unroll
      for (int d = 0; d < 3; ++d)
        c[d] = (unsigned)fminf(fmaxf((ax.at(d, p[d]) + ax.lo[d]) * ax.sc, 0.0f), 1023.0f);   // NaN -> 0
      const int64_t i = set ? s.n[0] + j : j;
      keys[i] = ((unsigned)set << bits) | (hilbert30(c[0], c[1], c[2]) >> (30 - bits));
      idx[i] = (int)j;
    }
  }
}

// sources as rows in a given order (the direct EXP kernel's)
template <int CORE>
__global__ __launch_bounds__(256) void k_ff_gather_src(SrcView s, const int* perm, int64_t n, float4* sp, float4* sa) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int j = perm[i];
  sp[i] = make_float4(s.x[j], s.y[j], s.z[j], core_term<CORE>(s.r[j]));
  sa[i] = make_float4(s.ax[j], s.ay[j], s.az[j], 0.0f);
}

// workgroup-wide reductions over 256 threads (4 waves), result in every thread
__device__ __forceinline__ float wg_max(float v, float* red) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off));
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}
__device__ __forceinline__ float wg_min(float v, float* red) { return -wg_max(-v, red); }

// bounding sphere (bbox centre, largest distance) and largest core term of each group of
// `group` consecutive sorted points; one workgroup per group
static __global__ __launch_bounds__(256) void k_ff_bounds(const float4* p, int64_t n, int group, float4* sph, float* cs) {
  __shared__ float red[4];
  const int64_t b0 = (int64_t)blockIdx.x * group;
  const int64_t b1 = (b0 + group) < n ? (b0 + group) : n;
  float lo[3] = {__builtin_huge_valf(), __builtin_huge_valf(), __builtin_huge_valf()};
  float hi[3] = {-__builtin_huge_valf(), -__builtin_huge_valf(), -__builtin_huge_valf()};
  float cmax = 0.0f;
  for (int64_t i = b0 + threadIdx.x; i < b1; i += blockDim.x) {
    const float4 q = p[i];
    lo[0] = fminf(lo[0], q.x); hi[0] = fmaxf(hi[0], q.x);
    lo[1] = fminf(lo[1], q.y); hi[1] = fmaxf(hi[1], q.y);
    lo[2] = fminf(lo[2], q.z); hi[2] = fmaxf(hi[2], q.z);
    cmax = fmaxf(cmax, q.w);
  }
  float c[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const float l = wg_min(lo[d], red);
    const float h = wg_max(hi[d], red);
    c[d] = 0.5f * l + 0.5f * h;
  }
  cmax = wg_max(cmax, red);
  float r2 = 0.0f;
  for (int64_t i = b0 + threadIdx.x; i < b1; i += blockDim.x) {
    const float4 q = p[i];
    const float dx = q.x - c[0], dy = q.y - c[1], dz = q.z - c[2];
    r2 = fmaxf(r2, fmaf(dz, dz, fmaf(dy, dy, dx * dx)));
  }
  r2 = wg_max(r2, red);
  if (threadIdx.x == 0) {
    // margin for the rounding of the distances above
    sph[blockIdx.x] = make_float4(c[0], c[1], c[2], __fsqrt_rn(r2) * 1.00001f + 1e-30f);
    cs[blockIdx.x] = cmax;
  }
}

// where a group's bounds go: sphere (bbox centre, largest distance), and {largest and least
// core term, of sources a bound of |alpha| and |q|, and the sign of the first nonzero strength
// (0: none), by its first nonzero component}
struct FFBounds {
  float4 *sph, *lim;
};
// the bounds of the workgroup's points, N per thread (valid: this thread has some) with
// core terms p.w; strengths a, of sources
template <int N>
__device__ __forceinline__ void ff_group_bounds(bool valid, const float4* p, const float4* a, const FFBounds& out,
                                                int64_t g) {
  const float inf = __builtin_huge_valf();
  float v[8] = {-inf, -inf, -inf, -inf, -inf, -inf, 0.0f, -inf};
  if (valid)
#pragma unroll
    for (int k = 0; k < N; ++k) {
      const float q[3] = {p[k].x, p[k].y, p[k].z};
#pragma unroll
      for (int d = 0; d < 3; ++d) { v[d] = fmaxf(v[d], -q[d]); v[3 + d] = fmaxf(v[3 + d], q[d]); }
      v[6] = fmaxf(v[6], p[k].w);
      v[7] = fmaxf(v[7], -p[k].w);
    }
  wg_max_n<8>(v);
  const float c[3] = {0.5f * v[3] - 0.5f * v[0], 0.5f * v[4] - 0.5f * v[1], 0.5f * v[5] - 0.5f * v[2]};
  float w[3] = {0.0f, 0.0f, -inf};   // squared radius, largest component, -(2 i + negative) of the first strength
  if (valid)
#pragma unroll
    for (int k = 0; k < N; ++k) {
      const float dx = p[k].x - c[0], dy = p[k].y - c[1], dz = p[k].z - c[2];
      w[0] = fmaxf(w[0], fmaf(dz, dz, fmaf(dy, dy, dx * dx)));
      if (a) {   // no square that could leave the range
        // one that is no number counts as infinite
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const float m = fabsf(c == 0 ? a[k].x : c == 1 ? a[k].y : c == 2 ? a[k].z : a[k].w);
          w[1] = m <= w[1] ? w[1] : m < inf ? m : inf;
        }
        const float f = a[k].x != 0.0f ? a[k].x : a[k].y != 0.0f ? a[k].y : a[k].z != 0.0f ? a[k].z : a[k].w;
        if (f != 0.0f) w[2] = fmaxf(w[2], -(float)(2 * (N * (int)threadIdx.x + k) + (f < 0.0f ? 1 : 0)));
      }
    }
  wg_max_n<3>(w);
  if (threadIdx.x != 0) return;
  // margin for the rounding of the distances above
  out.sph[g] = make_float4(c[0], c[1], c[2], __fsqrt_rn(w[0]) * 1.00001f + 1e-30f);
  // w[1] times sqrt 3, rounded up
  out.lim[g] = make_float4(v[6], -v[7], w[1] * 1.7321f, w[2] == -inf ? 0.0f : ((int)-w[2] & 1) ? -1.0f : 1.0f);
}

// rows and bounds, one workgroup per source tile and then one per target block: sources up
// to a whole tile (the rest: the last one's place with no strength) and targets; the
// blocks' near counts are cleared for k_ff_classify
template <int CORE, bool THICK>
__global__ __launch_bounds__(256) void k_ff_rows(SrcView s, TgtView t, const int* sperm, const int* tperm, int64_t ns,
                                                 int64_t nt, int tile, int ntiles, float4* sp, float4* sa, float4* tq,
                                                 FFBounds sb, FFBounds tb, int* nn, int* tinv) {
  const int tid = threadIdx.x;
  if ((int)blockIdx.x < ntiles) {
    const int64_t i = (int64_t)blockIdx.x * tile + tid;
    float4 p{}, a{};
    if (tid < tile) {
      const int j = sperm[i < ns ? i : ns - 1];
      p = make_float4(s.x[j], s.y[j], s.z[j], core_term<CORE>(s.r[j]));
      if (i < ns) a = make_float4(s.ax[j], s.ay[j], s.az[j], 0.0f);
      sp[i] = p;
      sa[i] = a;
    }
    ff_group_bounds<1>(tid < tile, &p, &a, sb, blockIdx.x);
  } else {
    const int64_t b = (int64_t)blockIdx.x - ntiles, i = b * FF_TB + tid;
    float4 p{};
    if (i < nt) {
      const int j = tperm[i];
      p = make_float4(t.x[j], t.y[j], t.z[j], THICK ? core_term<CORE>(t.r[j]) : 0.0f);
      tq[i] = p;
      if (tinv) tinv[j] = (int)i;
    }
    ff_group_bounds<1>(i < nt, &p, nullptr, tb, b);
    if (tid == 0) nn[b] = 0;
  }
}

// r2 at a distance of d with core terms c, as the far field's weights take it
template <int CORE>
__device__ __forceinline__ float ff_r2_with(float d, float c) {
  const float d2 = d * d;
  if (CORE == CORE_RM || CORE == CORE_WL) return d2 + c;
  if (CORE == CORE_V2) return fmaxf(d2, __fsqrt_rn(fmaf(d2, d2, c)));
  return d2;
}

// far bit of every (target block, source tile), and the near tiles counted into nn (cleared
// before): one thread per 32 tiles of a block.  A tile with a strength that is infinite or no
// number is near, as its products would leave nothing of the finite components, and so is one
// whose r2 can leave the range
template <int CORE>
__global__ __launch_bounds__(256) void k_ff_classify(FFBounds bb, int64_t nb, FFBounds tb, int ntiles, int mwords,
                                                     unsigned* mask, int* nn) {
  constexpr bool CORES = CORE == CORE_RM || CORE == CORE_WL || CORE == CORE_V2;   // part of the weights
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= nb * mwords) return;
  const int64_t b = g / mwords;
  const int w = (int)(g - b * mwords);
  const float4 cb = bb.sph[b], lb = bb.lim[b];
  unsigned bits = 0u;
  const int left = ntiles - 32 * w < 32 ? ntiles - 32 * w : 32;
#pragma unroll 8
  for (int k = 0; k < left; ++k) {
    const float4 ct = tb.sph[32 * w + k], lt = tb.lim[32 * w + k];
    const float dx = cb.x - ct.x, dy = cb.y - ct.y, dz = cb.z - ct.z;
    const float gap = __fsqrt_rn(fmaf(dz, dz, fmaf(dy, dy, dx * dx))) - cb.w - ct.w;
    const float most = ff_r2_with<CORE>(gap + 2.0f * (cb.w + ct.w), lb.x + lt.x);
    const float least = ff_r2_with<CORE>(gap, CORES ? lb.y + lt.y : 0.0f);
    // no branches: the loads of the next tiles go ahead
    bool far = gap > 0.0f;
    far &= gap > FF_KAPPA * fmaxf(fminf(cb.w, ct.w), FF_SPREAD * cb.w);
    far &= most <= FF_RANGE * least;
    far &= fmaxf(most, lt.z) < __builtin_huge_valf();
    if (CORE == CORE_EXP) far &= gap * gap > exp_threshold(lb.x + lt.x);
    if (CORE == CORE_SING) far &= gap > fmaxf(lb.x, lt.x);
    if (far) bits |= 1u << k;
  }
  mask[g] = bits;
  atomicAdd(&nn[b], left - __popc(bits));
}

// velocity and gradient (ug order, g = -3 D + skew(W)) of one target from its 32
// moment sums c[] and its offset t from the block centre; al = |t|^2 + st^2 (RM)
__device__ __forceinline__ void ff_epilogue(const double* c, double tx, double ty, double tz, double al,
                                            double* out) {
  const double P[3] = {c[0], c[1], c[2]};
  const double Q[3] = {c[3], c[4], c[5]};
  double R[3][3], S[3][3];
#pragma unroll
  for (int l = 0; l < 3; ++l)
#pragma unroll
    for (int k = 0; k < 3; ++k) R[l][k] = c[6 + 3 * l + k];
#pragma unroll
  for (int e = 0; e < 8; ++e) S[e / 3][e % 3] = c[15 + e];
  S[2][2] = -S[0][0] - S[1][1];
  const double U[3] = {c[23], c[24], c[25]};
  const double V[3] = {c[26], c[27], c[28]};
  const double t[3] = {tx, ty, tz};
  double W[3], M[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    W[k] = al * P[k] - 2.0 * (t[0] * R[0][k] + t[1] * R[1][k] + t[2] * R[2][k]) + U[k];
    M[k] = al * Q[k] - 2.0 * (t[0] * S[0][k] + t[1] * S[1][k] + t[2] * S[2][k]) + V[k];
  }
  out[0] = W[1] * t[2] - W[2] * t[1] - M[0];
  out[1] = W[2] * t[0] - W[0] * t[2] - M[1];
  out[2] = W[0] * t[1] - W[1] * t[0] - M[2];
  const double Px[3] = {P[1] * t[2] - P[2] * t[1], P[2] * t[0] - P[0] * t[2], P[0] * t[1] - P[1] * t[0]};
  double a[NACC];   // a[3 + 3j + i] = D_ji for 3j + i < 8 (D_22 = -D_00 - D_11)
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const double Rx[3] = {R[j][1] * t[2] - R[j][2] * t[1], R[j][2] * t[0] - R[j][0] * t[2],
                          R[j][0] * t[1] - R[j][1] * t[0]};
#pragma unroll
    for (int i = 0; i < 3; ++i)
      if (3 * j + i < 8) a[3 + 3 * j + i] = t[j] * Px[i] - t[j] * Q[i] - Rx[i] + S[j][i];
  }
  a[11] = W[0]; a[12] = W[1]; a[13] = W[2];
  grad_from<double>(a, out + 3);
}

// the same from the sums of K (k: alpha 0-2, m 3-5) and, with the gradient, of Bp (c:
// the first 23 columns)
template <bool GRAD>
__device__ __forceinline__ void ff_epilogue_k(const double* k, const double* c, double tx, double ty, double tz,
                                              double* out) {
  out[0] = k[1] * tz - k[2] * ty - k[3];
  out[1] = k[2] * tx - k[0] * tz - k[4];
  out[2] = k[0] * ty - k[1] * tx - k[5];
  if (!GRAD) return;
  const double t[3] = {tx, ty, tz};
  const double Px[3] = {c[1] * tz - c[2] * ty - c[3], c[2] * tx - c[0] * tz - c[4], c[0] * ty - c[1] * tx - c[5]};
  double a[NACC];
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const double* R = c + 6 + 3 * j;
    const double Rx[3] = {R[1] * tz - R[2] * ty, R[2] * tx - R[0] * tz, R[0] * ty - R[1] * tx};
#pragma unroll
    for (int i = 0; i < 3; ++i)
      if (3 * j + i < 8) a[3 + 3 * j + i] = t[j] * Px[i] - Rx[i] + c[15 + 3 * j + i];
  }
  a[11] = k[0]; a[12] = k[1]; a[13] = k[2];
  grad_from<double>(a, out + 3);
}

// ... and for panels with source strengths q: K sums of alpha 0-2, m 3-5, q 6, q s' 7-9,
// Bp sums of these and of s' x alpha 10-18, s' x m 19-26, q s' s' 27-31 (00, 01, 02, 11,
// 12).  With X_ij = sum Bp q d_i d_j, whose trace is sum K q: u += sum K q d and
// g_ji += -3 X_ji + delta_ji sum K q
template <bool GRAD>
__device__ __forceinline__ void ff_epilogue_sheet(const double* k, const double* c, double tx, double ty, double tz,
                                                  double* out) {
  const double t[3] = {tx, ty, tz};
  if (GRAD) {
    double p[23];   // the vortex part's own columns
#pragma unroll
    for (int i = 0; i < 23; ++i) p[i] = c[i < 6 ? i : i + 4];
    ff_epilogue_k<true>(k, p, tx, ty, tz, out);
    const double X00 = t[0] * t[0] * c[6] - 2.0 * t[0] * c[7] + c[27];
    const double X01 = t[0] * t[1] * c[6] - t[0] * c[8] - t[1] * c[7] + c[28];
    const double X02 = t[0] * t[2] * c[6] - t[0] * c[9] - t[2] * c[7] + c[29];
    const double X11 = t[1] * t[1] * c[6] - 2.0 * t[1] * c[8] + c[30];
    const double X12 = t[1] * t[2] * c[6] - t[1] * c[9] - t[2] * c[8] + c[31];
    const double X22 = k[6] - X00 - X11;
    out[3] += k[6] - 3.0 * X00; out[4] -= 3.0 * X01; out[5] -= 3.0 * X02;
    out[6] -= 3.0 * X01; out[7] += k[6] - 3.0 * X11; out[8] -= 3.0 * X12;
    out[9] -= 3.0 * X02; out[10] -= 3.0 * X12; out[11] += k[6] - 3.0 * X22;
  } else {
    ff_epilogue_k<false>(k, c, tx, ty, tz, out);
  }
#pragma unroll
  for (int d = 0; d < 3; ++d) out[d] += k[6] * t[d] - k[7 + d];
}

// ---- far field: the three forms ------------------------------------------------
// FF_B: one weight per pair, Bp; K comes back as Bp r2 (RM and EXP with gradient).
// FF_K: one weight, K, and the velocity alone.
// FF_KB: both weights, for the cores whose K is no product of Bp with r2 (WL, V2), and for
// panels with source strengths (SHEET), whose moments fill the 32 rows with K beside them.
enum { FF_B = 0, FF_K = 1, FF_KB = 2 };
template <int CORE, bool GRAD, bool SHEET>
constexpr int ff_form() {
  return !GRAD ? FF_K : SHEET || CORE == CORE_WL || CORE == CORE_V2 ? FF_KB : FF_B;
}
// columns of the moment table (rows of the matrix product):
//   FF_B   alpha 0-2, m 3-5, s' x alpha 6-14, s' x m 15-22, b alpha 23-25, b m 26-28
//   FF_KB  the first 23 (K multiplies alpha and m, Bp all of them); SHEET: ff_epilogue_sheet
//   FF_K   what K multiplies, in 16 rows of leading parts and 16 rows of remainders
template <int FORM, bool SHEET>
constexpr int ff_cols() { return FORM == FF_B ? 29 : FORM == FF_KB ? (SHEET ? 32 : 23) : (SHEET ? 10 : 6); }
template <int FORM>
constexpr int ff_rows() { return FORM == FF_K ? 16 : 32; }

// moment column -> scale group: alpha and q (0), m, s' alpha and q s' (1), s' m and q s' s'
// (2), b alpha (3), b m (4); padding columns hold zeros
template <bool SHEET>
__host__ __device__ constexpr int ff_group(int col) {
  if (SHEET) return col < 3 || col == 6 ? 0 : col < 19 ? 1 : 2;
  return col < 3 ? 0 : col < 15 ? 1 : col < 23 ? 2 : col < 26 ? 3 : 4;
}

// column c of one source: alpha a, q, s' s, m = alpha x s', b
template <bool SHEET>
__device__ __forceinline__ float ff_column(int c, const float* a, float q, const float* s, const float* m, float b) {
  if (c < 3) return a[c];
  if (c < 6) return m[c - 3];
  if (SHEET) {
    if (c == 6) return q;
    if (c < 10) return q * s[c - 7];
    if (c < 19) return s[(c - 10) / 3] * a[(c - 10) % 3];
    if (c < 27) return s[(c - 19) / 3] * m[(c - 19) % 3];
    return q * s[c < 30 ? 0 : 1] * s[c < 30 ? c - 27 : c - 29];
  }
  if (c < 15) return s[(c - 6) / 3] * a[(c - 6) % 3];
  if (c < 23) return s[(c - 15) / 3] * m[(c - 15) % 3];
  if (c < 26) return b * a[c - 23];
  if (c < 29) return b * m[c - 26];
  return 0.0f;
}

// FP16 hi + lo split of two FP32 values (|x| < 2^16) into elements e, e + 1: hi is x
// rounded to nearest, so that lo = x - hi (exact in FP32) has either sign and the
// dropped product of two los averages out over the sources instead of adding up
// (with hi truncated every los' product has the sign of the pair's own term); lo is
// truncated, the sum of both has about 22 significant bits.  One packed conversion
// each and one mixed-precision FMA per value: 4.5 cycles per wave instruction, where
// an FMA that rounds its own result to FP16 (v_fma_mixlo/mixhi_f16) takes 8.3.
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void split16x2(float x0, float x1, f16x8& hv, f16x8& lv, int e) {
  const f16x2 h = __builtin_convertvector(f32x2{x0, x1}, f16x2);
  const auto l = __builtin_amdgcn_cvt_pkrtz(x0 - (float)h[0], x1 - (float)h[1]);
  hv[e] = h[0];
  hv[e + 1] = h[1];
  lv[e] = (_Float16)l[0];
  lv[e + 1] = (_Float16)l[1];
}

// BF16 three-way split x = hi + mid + lo (about 24 significant bits): hi and mid
// take the leading bits, each remainder is exact in FP32
__device__ __forceinline__ void split_bf3(float x, __bf16& hi, __bf16& mid, __bf16& lo) {
  hi = (__bf16)x;
  const float r = x - (float)hi;
  mid = (__bf16)r;
  lo = (__bf16)(r - (float)mid);
}

// squared distances on the matrix cores: r2 = sum_c S_c T_c over the five terms
// S = (-2 s'x, -2 s'y, -2 s'z, b, 1) (per source) and T = (t'x, t'y, t'z, 1, a) (per
// target), both pre-scaled by the tile's r2 scale, each split into BF16 hi/mid/lo
// and multiplied as hi lo + lo hi + mid mid + hi mid + mid hi + hi hi (about 24 bits: the
// accuracy of the FP32 expression it replaces).  Slot q < 30 of the K = 32 product
// holds term q / 5 of component q % 5, the small terms first: a product of the first 16
// slots has no large term, against which the matrix cores would cut the small ones off
// (large terms first: an error of 4e-8 in K that the targets' own parts decide, the
// same for all far sources).  The parts taken per term:
__device__ __forceinline__ int ff_src_part(int term) { return term == 1 ? 2 : (term == 2 || term == 4 ? 1 : 0); }
__device__ __forceinline__ int ff_tgt_part(int term) { return term == 0 ? 2 : (term == 2 || term == 3 ? 1 : 0); }

// source position of tile slot p in the FP16 moment tables: inside each group of 16
// sources, slot 16g + 8h + e holds source 16g + 4h + (e % 4) + 8 (e / 4), so that the
// squared distances a lane gets from the r2 product (rows 8(r/4) + 4h + r%4) are, in
// register order, the sources of its contiguous 8 K-slots in the moment product.
// Four consecutive sources 4q .. 4q + 3 so take four consecutive slots, from here:
__device__ __forceinline__ int ff_quad_slot(int q) { return 16 * (q >> 2) + 8 * (q & 1) + 4 * ((q >> 1) & 1); }

// the pair weights of one scaled squared distance r (RM, WL: core terms included);
// tau (WL, V2): the pair's scaled core term, of WL 2.5 times
template <int CORE, int FORM>
__device__ __forceinline__ void ff_weights(float r, float tau, float& K, float& Bp) {
  if (CORE == CORE_RM || CORE == CORE_EXP || CORE == CORE_SING) {
    const float ir = frsq(r);
    const float ir2 = ir * ir;
    if (FORM != FF_B) K = ir2 * ir;
    if (FORM == FF_KB) Bp = K * ir2;
    if (FORM == FF_B) Bp = (ir2 * ir2) * ir;
  } else if (CORE == CORE_WL) {     // CoreFunc.h:265-274 with D = rho^2 + tau = r
    const float ir = frsq(r);
    const float ir2 = ir * ir;
    const float i5 = (ir2 * ir2) * ir;
    K = i5 * fmaf(0.6f, tau, r);    // tau: 2.5 times the core term
    if (FORM == FF_KB) Bp = i5 * fmaf(tau, ir2, 1.0f);
  } else {                          // CoreFunc.h:317-328
    const float rs = frsq(fmaf(r, r, tau));
    K = rs * fsqrt(rs);
    if (FORM == FF_KB) Bp = K * rs;
  }
}

// Relative errors with a mean, which a sum over many pairs keeps while the rest of them
// averages out; the folds take it out of the sums of Bp and of K.  v_rsq_f32: -6.98e-9
// over all mantissas of two octaves weighted by 1 / x (rms 2.6e-8, largest 9.4e-8);
// v_sqrt_f32: -1.43e-8 likewise; the squared distance: -1.97e-8, as the matrix cores cut
// off what does not fit the sum (from K of far clouds of particles in FP64).
constexpr double FF_RSQ_MEAN = -6.98e-9, FF_SQRT_MEAN = -1.43e-8, FF_R2_MEAN = -1.97e-8;
template <int CORE>
constexpr double ff_mean_b() {
  return 1.0 - (CORE == CORE_V2 ? 2.5 * FF_RSQ_MEAN + FF_SQRT_MEAN : 5.0 * FF_RSQ_MEAN) + 2.5 * FF_R2_MEAN;
}
template <int CORE>
constexpr double ff_mean_k() {
  return 1.0 - (CORE == CORE_V2 ? 1.5 * FF_RSQ_MEAN + FF_SQRT_MEAN : (CORE == CORE_WL ? 5.0 : 3.0) * FF_RSQ_MEAN) +
         1.5 * FF_R2_MEAN;
}

// 16 bytes per lane from memory to LDS without a register: lane l's from src to dst + l
// (dst the same in every lane); done when the wave's loads are
__device__ __forceinline__ void ff_load_lds16(const float4* src, float4* dst) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                   (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}

// Far field: one workgroup per 256 sorted targets (4 waves of 64); lane l of wave w
// owns target w*64 + l at the end, and during the sums works for targets
// w*64 + (l & 31) (set 0) and w*64 + 32 + (l & 31) (set 1).  Per chunk of 32 sources
// and set: two BF16 products give the 32 x 32 squared distances (lane l: target
// l & 31, 16 sources), the lane turns its 16 into pair weights split into FP16
// hi + lo, and FP16 products (two 16-source K blocks, three split terms each; the K
// weight of the two-weight form takes leading parts and remainders of its columns
// as rows of one operand, two products) add the weights times the moment columns.
//
// The moment products keep about 22 significant bits per product (hi hi + lo hi +
// hi lo), the accuracy of the FP32 products they replace.  Weights are scaled by
// powers of 2^(1/2): r2 -> r2 2^-jw through the staged source terms and the targets'
// a, so Bp takes 2^(5 jw / 2) and K 2^(3 jw / 2) (from Bp <= 3.5 r^-5 at the least r of the
// gap and the cores), and each moment
// group by 2^eg (from the tile's largest |alpha| and source distance), so that every
// FP16 factor stays below 2^16.  Consecutive tiles keep the scales of the first as
// long as they fit (ff_merge tiles at most) and share one fold into FP64, where the
// scales are removed.  All strengths are taken times the sign of the first nonzero one
// (in sorted order, its first nonzero component) and the result times that sign again:
// the matrix cores do not round a product and its negative alike, and so negating
// every strength negates the result exactly.
//
// 32x32x16 FP16/BF16 matrix operand layout (A: 32 x 16, B: 16 x 32, D: 32 x 32):
//   A[i][k] in lane i + 32 (k / 8), element k % 8;  B[k][j] in lane j + 32 (k / 8),
//   element k % 8;  D[i][j] in lane j + 32 ((i / 4) % 2), register (i % 4) + 4 (i / 8).
// r2 product: A = source slots (row = source), B = target slots, D = r2.
// Moment product: A = moment table transposed (row = column), B = weights (source, target).
// LDS: r2 source slots [source][FF_SL] BF16 (rows of 80 bytes), the scaled moments as
// FP16 hi and lo tables [column][FF_TP], rows of 264 halves, so that the 16-byte reads
// of 16 lanes cover all 64 banks, the rows of the next tile, and (WL, V2) the scaled
// core term per source.
//
// The loop over chunks is a pipeline: while the weights of one set and half are formed on
// the vector ALUs, the matrix cores take the moment products of the half before and the
// next squared distances.  A wave issues in order, so each product is followed by its share of the
// vector work (FF_SCHED).  Measured cycles per wave instruction with two waves per SIMD:
// product 32; add, multiply, fmac 2.3; conversions and v_fma_mix_f32 4.5; v_rsq_f32 and
// v_fma_mixlo/mixhi_f16 8.3.  A product beside 2 rsq, 6 multiplies and 4 conversions
// takes 64.5, the twelve alone 57: this loop runs at 69.  The tile's tables cost about
// 200 vector instructions per wave, the loop 1,700; what a run (ff_fold and the target
// slots) costs is shared by ff_merge tiles.
template <int CORE, bool GRAD, bool SHEET = false>
__global__ __launch_bounds__(FF_FAR_THREADS, 2) void k_ff_far(FFArgs a) {
  constexpr int FORM = ff_form<CORE, GRAD, SHEET>();
  constexpr int ROWS = ff_rows<FORM>(), COLS = ff_cols<FORM, SHEET>();
  constexpr int KCOLS = SHEET ? 10 : 6;   // of them, the first KCOLS take K
  constexpr bool HASB = FORM != FF_K, HASK = FORM != FF_B;
  constexpr bool TAU = CORE == CORE_WL || CORE == CORE_V2;
  constexpr bool COREA = CORE == CORE_RM || CORE == CORE_WL;   // core terms are part of r2
  constexpr int NG = FORM == FF_B ? 5 : FORM == FF_KB ? 3 : 2;
  constexpr int NOUT = GRAD ? 12 : 3;
  constexpr int TP = FF_TP;
  extern __shared__ float4 sh[];
  const int T = a.tile;
  __bf16* sl = reinterpret_cast<__bf16*>(sh);
  _Float16* mh = reinterpret_cast<_Float16*>(sl + 256 * FF_SL);
  _Float16* ml = mh + ROWS * TP;
  float4* raw = reinterpret_cast<float4*>(ml + ROWS * TP);   // the tile's rows: 256 of sp, 256 of sa
  float* tc = reinterpret_cast<float*>(raw + 512);
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5, col = lane & 31;
  const int64_t blk = blockIdx.x;
  const int64_t base = blk * FF_TB + w * 64;
  const float4 cb = a.bsph[blk];
  float sgn = a.tlim[0].w;   // of the first nonzero strength of all
  for (int t = 1; sgn == 0.0f && t < a.ntiles; ++t) sgn = a.tlim[t].w;
  sgn = sgn < 0.0f ? -1.0f : 1.0f;

  // targets; and the current run's centre, the block's or its one tile's
  float qx[2], qy[2], qz[2], tt[2];
  float cx = cb.x, cy = cb.y, cz = cb.z;
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    int64_t i = base + 32 * s + col;
    i = i < a.nt ? i : a.nt - 1;
    const float4 q = a.tq[i];
    qx[s] = q.x; qy[s] = q.y; qz[s] = q.z;
    tt[s] = COREA || TAU ? q.w : 0.0f;
  }
  f32x16 accB[2], accK[2], accR[2];
  double sum[NOUT];
#pragma unroll
  for (int k = 0; k < NOUT; ++k) sum[k] = 0.0;
  const int64_t own = base + lane;

  const unsigned* mrow = a.mask + blk * a.mwords;
  int jw = 0, eg[NG];
  bf16x8 tb[2][2] = {};
  float tts[2] = {0.0f, 0.0f};
  // fold: one v_permlane32_swap per register exchanges the upper 32 lanes of acc[0][r]
  // with the lower 32 of acc[1][r], after which every lane holds its own target's rows
  // of half 0 in the one and of half 1 in the other (row of register r in half h:
  // 8 (r / 4) + 4 h + r % 4); the scales are removed and the epilogue adds the run's
  // velocity and gradient in FP64.  Lane l < 32 owns target w*64 + l (set 0), lane
  // l >= 32 target w*64 + l (set 1).
  auto rows_of = [&](f32x16* acc, double* c) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[0][r]), __float_as_uint(acc[1][r]),
                                                       false, false);
      const int i0 = 8 * (r / 4) + (r % 4);
      c[i0] = (double)__uint_as_float(sw[0]);
      c[i0 + 4] = (double)__uint_as_float(sw[1]);
    }
  };
  auto fold = [&]() {
    const double ox = (half ? qx[1] : qx[0]) - cx, oy = (half ? qy[1] : qy[0]) - cy, oz = (half ? qz[1] : qz[0]) - cz;
    const double oa = ox * ox + oy * oy + oz * oz + (COREA ? (double)(half ? tt[1] : tt[0]) : 0.0);
    double sc[NG];
#pragma unroll
    for (int g = 0; g < NG; ++g) sc[g] = ldexp((double)sgn, -eg[g]);
    double c[32], ck[32], out[12];
    if (HASB) {
      // 2^(-5 jw / 2)
      const double wb = ldexp(jw & 1 ? 0.70710678118654752440 : 1.0, -2 * jw - (jw >> 1)) * ff_mean_b<CORE>();
      if (FORM == FF_B)
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
          for (int r = 0; r < 16; ++r) accB[s][r] += accR[s][r];
      rows_of(accB, c);
#pragma unroll
      for (int i = 0; i < COLS; ++i) c[i] *= sc[ff_group<SHEET>(i)] * wb;
    }
    if (HASK) {
      // 2^(-3 jw / 2)
      const double wk = ldexp(jw & 1 ? 0.70710678118654752440 : 1.0, -jw - (jw >> 1)) * ff_mean_k<CORE>();
      rows_of(accK, ck);
#pragma unroll
      for (int i = 0; i < KCOLS; ++i) ck[i] = (ck[i] + ck[16 + i]) * (sc[ff_group<SHEET>(i)] * wk);
    }
    if constexpr (SHEET) ff_epilogue_sheet<GRAD>(ck, c, ox, oy, oz, out);
    else if constexpr (FORM == FF_B) ff_epilogue(c, ox, oy, oz, oa, out);
    else ff_epilogue_k<GRAD>(ck, c, ox, oy, oz, out);
#pragma unroll
    for (int k = 0; k < NOUT; ++k) sum[k] += out[k];
  };
  // one chunk of 32 sources: its slots and moment operands (two halves of 16 sources) of
  // this lane, its squared distances per set, and the weights of two consecutive halves
  struct Frag {
    f16x8 bh, bl, kh, kl;
  };
  bf16x8 sa[2];
  f16x8 mb[2][2], mk[2];
  f32x16 r2[2];
  Frag f[2];
  auto load_slots = [&](int k0, int part) {
    sa[part] = *reinterpret_cast<const bf16x8*>(sl + (k0 + col) * FF_SL + 8 * half + 16 * part);
  };
  auto load_moments = [&](int k0, int kb) {
    const int pbase = k0 + 16 * kb + 8 * half;
    if (HASB) {
      mb[kb][0] = *reinterpret_cast<const f16x8*>(mh + col * TP + pbase);
      mb[kb][1] = *reinterpret_cast<const f16x8*>(ml + col * TP + pbase);
    }
    // rows 0-15 the leading parts of the first 16 columns, rows 16-31 their remainders
    if (HASK) mk[kb] = *reinterpret_cast<const f16x8*>((col < 16 ? mh + col * TP : ml + (col - 16) * TP) + pbase);
  };
  // squared distances of the 32 sources of sa to this lane's target of set s, in two parts
  auto dist = [&](int s, int part) {
    const f32x16 z = {};
    r2[s] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(sa[part], tb[s][part], part == 0 ? z : r2[s], 0, 0, 0);
  };
  // scaled core terms of the 8 sources that the lane weighs next
  float tau[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  auto load_tau = [&](int k0, int kb) {
    if (TAU) {
      const float4 t0 = *reinterpret_cast<const float4*>(tc + k0 + 16 * kb + 4 * half);
      const float4 t1 = *reinterpret_cast<const float4*>(tc + k0 + 16 * kb + 8 + 4 * half);
      tau[0] = t0.x; tau[1] = t0.y; tau[2] = t0.z; tau[3] = t0.w;
      tau[4] = t1.x; tau[5] = t1.y; tau[6] = t1.z; tau[7] = t1.w;
    }
  };
  auto weigh = [&](int s, int kb) {
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
      float K0, K1, B0, B1;
      ff_weights<CORE, FORM>(r2[s][8 * kb + e], tau[e] + tts[s], K0, B0);
      ff_weights<CORE, FORM>(r2[s][8 * kb + e + 1], tau[e + 1] + tts[s], K1, B1);
      if (HASB) split16x2(B0, B1, f[kb].bh, f[kb].bl, e);
      if (HASK) split16x2(K0, K1, f[kb].kh, f[kb].kl, e);
    }
  };
  auto moments = [&](int s, int kb) {
    if (HASB) {
      accB[s] = __builtin_amdgcn_mfma_f32_32x32x16_f16(mb[kb][0], f[kb].bh, accB[s], 0, 0, 0);
      // the products with a remainder in sums of their own (FF_B: there are registers for
      // it): the matrix cores cut off every sum they add to, so the large one is cut once
      // per 16 sources instead of three times (far clouds of particles, RM and EXP with
      // gradient: error 7.4e-8 -> 4.5e-8)
      f32x16& rest = FORM == FF_B ? accR[s] : accB[s];
      rest = __builtin_amdgcn_mfma_f32_32x32x16_f16(mb[kb][0], f[kb].bl, rest, 0, 0, 0);
      rest = __builtin_amdgcn_mfma_f32_32x32x16_f16(mb[kb][1], f[kb].bh, rest, 0, 0, 0);
    }
    if (HASK) {
      accK[s] = __builtin_amdgcn_mfma_f32_32x32x16_f16(mk[kb], f[kb].kh, accK[s], 0, 0, 0);
      accK[s] = __builtin_amdgcn_mfma_f32_32x32x16_f16(mk[kb], f[kb].kl, accK[s], 0, 0, 0);
    }
  };
  // nothing pending: zero weights (and operands) for the moments of a chunk before the first
  auto none_pending = [&]() {
    const f16x8 z = {};
    if (HASB) { f[1].bh = z; f[1].bl = z; mb[1][0] = z; mb[1][1] = z; }
    if (HASK) { f[1].kh = z; f[1].kl = z; mk[1] = z; }
  };
  // the next far tile of this slice of the block (-1: none).  A mask word at a time, lane
  // l works out the scales that tile l of the word wants: the largest weight and moment
  // of each group below 2^13 (2^11 where a core adds up to 3.5 times), the logarithms'
  // error being far below the margin.
  const int first_tile = (int)blockIdx.y * a.tslice;
  const int end_tile = first_tile + a.tslice < a.ntiles ? first_tile + a.tslice : a.ntiles;
  int word = (first_tile >> 5) - 1;
  unsigned bits = 0u;
  int pk0 = 0, pk1 = 0;   // lane l: jw and eg[0..1], eg[2..4] wanted by tile l of the word
  auto next_tile = [&]() {
    while (bits == 0u) {
      if (32 * ++word >= end_tile) return -1;
      bits = __builtin_amdgcn_readfirstlane(mrow[word]);
      if (32 * word < first_tile) bits &= ~0u << (first_tile & 31);
      if (32 * word + 32 > end_tile) bits &= (1u << (end_tile & 31)) - 1u;
      if (bits == 0u) continue;
      const int t = word * 32 + col < a.ntiles ? word * 32 + col : a.ntiles - 1;
      const float4 ct = a.tsph[t], lt = a.tlim[t];
      const float ddx = cb.x - ct.x, ddy = cb.y - ct.y, ddz = cb.z - ct.z;
      const float dc = __fsqrt_rn(fmaf(ddz, ddz, fmaf(ddy, ddy, ddx * ddx)));
      const float gap = dc - cb.w - ct.w;   // > 0 for a far tile
      float lr = __builtin_amdgcn_logf(fmaxf(gap, 1e-37f));   // of the least distance that the weights see
      if (COREA || TAU) lr = fmaxf(lr, 0.5f * __builtin_amdgcn_logf(ff_r2_with<CORE>(gap, a.blim[blk].y + lt.y)));
      const bool own = !(gap > FF_KAPPA * cb.w);   // a tile nearer than the block is wide: its own centre
      const float rs = own ? fmaxf(ct.w, gap * 0x1p-12f) : dc + ct.w;   // |s'| bound
      const float lrs = __builtin_amdgcn_logf(rs);
      // strengths by exponent and mantissa, so that scaling all by a power of two moves the
      // scales by just that and the results with them, exactly
      int ea;
      const float lam = __builtin_amdgcn_logf(fmaxf(frexpf(lt.z, &ea), 0.5f));
      const float lbm = __builtin_amdgcn_logf(fmaf(rs, rs, COREA ? lt.x : 0.0f));
      const float top = (TAU ? 11.0f : 13.0f) * (HASB ? 1.0f / 5.0f : 1.0f / 3.0f);
      const float lg[5] = {lam, lam + lrs, lam + 2.0f * lrs, lam + lbm, lam + lbm + lrs};
      int wg[5];
#pragma unroll
      for (int g = 0; g < 5; ++g) wg[g] = (int)fminf(fmaxf(floorf(13.0f - lg[g]) - (float)ea, -126.0f), 126.0f) & 255;
      pk0 = ((int)floorf(2.0f * (lr + top)) << 16) | (wg[1] << 8) | wg[0];
      pk1 = (own ? 1 << 24 : 0) | (wg[4] << 16) | (wg[3] << 8) | wg[2];
    }
    const int t = __builtin_ctz(bits);
    bits &= bits - 1u;
    return word * 32 + t;
  };
  // a tile's rows on their way to LDS, straight from memory, while the tile before is
  // summed; and the scales it wants
  int wj = 0, wg[5] = {0, 0, 0, 0, 0};
  bool wown = false;
  auto fetch = [&](int t) {
    const int p0 = __builtin_amdgcn_readlane(pk0, t & 31), p1 = __builtin_amdgcn_readlane(pk1, t & 31);
    wj = p0 >> 16;
    wg[0] = (int8_t)p0; wg[1] = (int8_t)(p0 >> 8);
    wg[2] = (int8_t)p1; wg[3] = (int8_t)(p1 >> 8); wg[4] = (int8_t)(p1 >> 16);
    wown = (p1 >> 24) != 0;
    if (w * 64 < T) {
      const int i = w * 64 + lane, q4 = T / 4;   // slot i: source 4 (i mod T/4) + i / (T/4)
      const int64_t g = (int64_t)t * T + 4 * (i & (q4 - 1)) + i / q4;
      ff_load_lds16(a.sp + g, raw + w * 64);
      ff_load_lds16(a.sa + g, raw + 256 + w * 64);
    }
  };
  bool slots = false;   // tb holds slots about the block's centre, scaled by jw
  int ti = next_tile();
  if (ti >= 0) fetch(ti);
  while (ti >= 0) {
    // a run: consecutive tiles summed under the scales of the first, its scale of r2 and its
    // centre, and with them the targets' slots, those of the run before where they serve
    const bool own = wown;
    const bool keep = slots && !own && (unsigned)(jw - wj + 1) <= 2u;
    slots = !own;
    if (!keep) {
      const float4 c = own ? a.tsph[ti] : cb;
      cx = c.x; cy = c.y; cz = c.z;
      jw = wj;
    }
#pragma unroll
    for (int g = 0; g < NG; ++g) eg[g] = wg[g];
    const float rsc = ldexpf(1.0f, -jw);
    float gs[NG];
#pragma unroll
    for (int g = 0; g < NG; ++g) gs[g] = ldexpf(sgn, eg[g]);
    if (!keep) {
      // this lane's target slots for both sets and both r2 products (K slots 8 half + e
      // and 16 + 8 half + e)
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const float tx = qx[s] - cx, ty = qy[s] - cy, tz = qz[s] - cz;
        const float al = fmaf(tz, tz, fmaf(ty, ty, fmaf(tx, tx, COREA ? tt[s] : 0.0f)));
        const float tv[5] = {tx, ty, tz, 1.0f, al * rsc};
        __bf16 part[3][5];
#pragma unroll
        for (int c = 0; c < 5; ++c) split_bf3(tv[c], part[0][c], part[1][c], part[2][c]);
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const int q0 = 16 * m + e, q1 = 16 * m + 8 + e;     // slot for half 0 / half 1
            const __bf16 v0 = q0 < 30 ? part[ff_tgt_part(q0 / 5)][q0 % 5] : (__bf16)0.0f;
            const __bf16 v1 = q1 < 30 ? part[ff_tgt_part(q1 / 5)][q1 % 5] : (__bf16)0.0f;
            tb[s][m][e] = half ? v1 : v0;
          }
        if (TAU) tts[s] = tt[s] * rsc * (CORE == CORE_V2 ? rsc : 2.5f);
      }
    }
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int r = 0; r < 16; ++r) { accB[s][r] = 0.0f; accK[s][r] = 0.0f; accR[s][r] = 0.0f; }
    none_pending();
    int run = 0;
    bool more;
    do {
    // every wave's rows have arrived and the tables are free
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    // moment tables: a lane takes four consecutive sources (one 8-byte store per column
    // and table) and a wave a quarter of the columns
    constexpr int CW = ROWS / 4;
    auto stage = [&](auto wave) {
      constexpr int C0 = decltype(wave)::value * CW;
      if constexpr (C0 < COLS) {
        if (4 * lane < T) {
          float cv[CW][4];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const float4 P = raw[u * (T / 4) + lane];   // source 4 lane + u
            const float4 A = raw[256 + u * (T / 4) + lane];
            const float s[3] = {P.x - cx, P.y - cy, P.z - cz};
            const float b = fmaf(s[2], s[2], fmaf(s[1], s[1], fmaf(s[0], s[0], COREA ? P.w : 0.0f)));
            // strengths take their group's power of two first: exact, one product per group and component
            float al3[NG][3], m[NG][3], qs[NG];
#pragma unroll
            for (int g = 0; g < NG; ++g) {
              const float ax = A.x * gs[g], ay = A.y * gs[g], az = A.z * gs[g];
              qs[g] = SHEET ? A.w * gs[g] : 0.0f;
              al3[g][0] = ax; al3[g][1] = ay; al3[g][2] = az;
              m[g][0] = fmaf(ay, s[2], -az * s[1]);
              m[g][1] = fmaf(az, s[0], -ax * s[2]);
              m[g][2] = fmaf(ax, s[1], -ay * s[0]);
            }
#pragma unroll
            for (int c = 0; c < CW; ++c) {
              constexpr int last = COLS - 1;
              const int cc = C0 + c < COLS ? C0 + c : last, g = ff_group<SHEET>(cc);
              cv[c][u] = C0 + c < COLS ? ff_column<SHEET>(cc, al3[g], qs[g], s, m[g], b) : 0.0f;
            }
          }
          const int pos = ff_quad_slot(lane);
#pragma unroll
          for (int c = 0; c < CW; ++c) {
            if (C0 + c >= COLS) break;
            f16x8 hv, lv;
            split16x2(cv[c][0], cv[c][1], hv, lv, 0);
            split16x2(cv[c][2], cv[c][3], hv, lv, 2);
            typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
            *reinterpret_cast<f16x4*>(mh + (C0 + c) * TP + pos) = f16x4{hv[0], hv[1], hv[2], hv[3]};
            *reinterpret_cast<f16x4*>(ml + (C0 + c) * TP + pos) = f16x4{lv[0], lv[1], lv[2], lv[3]};
          }
        }
      }
    };
    if (w == 0) stage(std::integral_constant<int, 0>{});
    else if (w == 1) stage(std::integral_constant<int, 1>{});
    else if (w == 2) stage(std::integral_constant<int, 2>{});
    else stage(std::integral_constant<int, 3>{});
    // r2 slots (and core terms) of one source per lane
    if (tid < T) {
      const float4 P = raw[(tid & 3) * (T / 4) + (tid >> 2)];
      const float sx = P.x - cx, sy = P.y - cy, sz = P.z - cz;
      const float b = fmaf(sz, sz, fmaf(sy, sy, fmaf(sx, sx, COREA ? P.w : 0.0f)));
      const float sv5[5] = {-2.0f * sx * rsc, -2.0f * sy * rsc, -2.0f * sz * rsc, b * rsc, 1.0f};   // exact scalings
      __bf16 part[3][5];
#pragma unroll
      for (int c = 0; c < 5; ++c) split_bf3(sv5[c], part[0][c], part[1][c], part[2][c]);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        bf16x8 row;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int q = 8 * v + e;
          row[e] = q < 30 ? part[ff_src_part(q / 5)][q % 5] : (__bf16)0.0f;
        }
        *reinterpret_cast<bf16x8*>(sl + tid * FF_SL + 8 * v) = row;
      }
      if (TAU) tc[tid] = P.w * rsc * (CORE == CORE_V2 ? rsc : 2.5f);
    }
    __syncthreads();
    ti = next_tile();
    if (ti >= 0) fetch(ti);

    // Four phases per chunk of 32 sources, one per set and half: while a half is weighed,
    // the matrix cores take the moments of the half before (in the first phase: of the
    // chunk or tile before, or zeros) and half of the distances that the phase after next
    // needs.
    constexpr int NM = (HASB ? 3 : 0) + (HASK ? 2 : 0) + 1;
    constexpr int TR = FORM == FF_K || CORE == CORE_V2 ? 3 : 2;
    constexpr int VA = FORM == FF_B ? 10 : FORM == FF_K ? (CORE == CORE_WL ? 16 : 12) : CORE == CORE_WL ? 18 : 12;
    load_slots(0, 0);
    load_slots(0, 1);
    load_tau(0, 0);
    dist(0, 0);
    dist(0, 1);
    for (int k0 = 0; k0 < T; k0 += 32) {
      const int kn = k0 + 32 < T ? k0 + 32 : 0;   // after the last chunk: distances that nothing uses
      __builtin_amdgcn_sched_barrier(0);
      dist(1, 0);
      moments(1, 1);
      weigh(0, 0);
      load_tau(k0, 1);
      load_moments(k0, 0);
      FF_SCHED(NM, TR, VA);
      dist(1, 1);
      moments(0, 0);
      weigh(0, 1);
      load_tau(k0, 0);
      load_moments(k0, 1);
      load_slots(kn, 0);
      FF_SCHED(NM, TR, VA);
      dist(0, 0);
      moments(0, 1);
      weigh(1, 0);
      load_tau(k0, 1);
      load_slots(kn, 1);
      FF_SCHED(NM, TR, VA);
      dist(0, 1);
      moments(1, 0);
      weigh(1, 1);
      load_tau(kn, 0);
      FF_SCHED(NM, TR, VA);
    }
    // the run's scales fit a further tile when no factor passes 2^16 and none loses more
    // than 4 of its leading bits
    more = ti >= 0 && !own && !wown && ++run < (ff_sized<CORE, GRAD>() ? a.merge : ff_merge<CORE, GRAD>()) && (unsigned)(jw - wj + 1) <= 2u;
#pragma unroll
    for (int g = 0; g < NG; ++g) more = more && (unsigned)(eg[g] - wg[g] + 4) <= 6u;
    } while (more);
    moments(1, 1);
    fold();
  }
  if (own < a.nt) ff_sum_store<NOUT>(a.farv + (int64_t)blockIdx.y * NOUT * a.nt, a.nt, own, a.rows, sum);
}

// ---- near field -------------------------------------------------------------
// The near tiles of a block are split into items of at most M tiles (M chosen on
// the device so that there are at most `split` + 1 items per block on average), so that
// a block that has most tiles near (a few targets far apart) is spread over many
// workgroups, and few blocks still make several rounds of them.  Items are taken from a
// queue by a persistent kernel and write FP64 partial sums; the combine kernel
// adds a block's partials in item order, so results do not depend on scheduling.

// The plan, by one workgroup: M = max(ceil(total / (split nb)), FF_M0, or fewer while that
// makes less than 2,048 items), the item count of every block (at most (split + 1) nb items
// in all) and its exclusive scan; the counters of the kernels that follow cleared
constexpr int FF_PLAN_THREADS = 1024;
static __global__ __launch_bounds__(FF_PLAN_THREADS) void k_ff_plan(const int* nn, int64_t nb, int split, int* items,
                                                             int* ioff, int* mfold, unsigned* ctr, unsigned* count) {
  __shared__ long long sh[FF_PLAN_THREADS / 64];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  // inclusive scan over the workgroup; every thread also gets the sum
  auto scan = [&](long long x, long long* all) {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const long long y = __shfl_up(x, o, 64);
      if (lane >= o) x += y;
    }
    __syncthreads();
    if (lane == 63) sh[w] = x;
    __syncthreads();
    long long before = 0, sum = 0;
    for (int k = 0; k < FF_PLAN_THREADS / 64; ++k) {
      before += k < w ? sh[k] : 0;
      sum += sh[k];
    }
    *all = sum;
    return before + x;
  };
  long long mine = 0, total;
  for (int64_t b = tid; b < nb; b += FF_PLAN_THREADS) mine += nn[b];
  (void)scan(mine, &total);
  long long m = (total + split * nb - 1) / (split * nb);
  const long long m0 = (total + 2047) / 2048 < FF_M0 ? (total + 2047) / 2048 : FF_M0;
  m = m < m0 ? m0 : m;
  m = m < 1 ? 1 : m;
  if (tid == 0) {
    *mfold = (int)m;
    *ctr = 0u;
    if (count) *count = 0u;
  }
  long long carry = 0;
  for (int64_t b0 = 0; b0 < nb; b0 += FF_PLAN_THREADS) {
    const int64_t b = b0 + tid;
    const int it = b < nb ? (int)((nn[b] + m - 1) / m) : 0;
    long long sum;
    const long long incl = scan(it, &sum);
    if (b < nb) {
      items[b] = it;
      ioff[b] = (int)(carry + incl - it);
    }
    carry += sum;
  }
}

// per-target partial of one item: near tiles of rank [r0, r1) among block b's
template <int CORE, bool GRAD, int PREC>
__device__ __forceinline__ void near_item(const FFArgs& a, int64_t b, int r0, int r1, float4* sh, double* r) {
  const int T = a.tile;
  const int tid = threadIdx.x;
  const int64_t i = b * FF_TB + tid;
  const int64_t ic = i < a.nt ? i : a.nt - 1;
  const float4 q = a.tq[ic];
  float tx[1] = {q.x}, ty[1] = {q.y}, tz[1] = {q.z}, tt[1] = {q.w};
  float acc[1][NACC];
  float hi[3] = {0.f, 0.f, 0.f}, lo[3] = {0.f, 0.f, 0.f};
  double gr[NACC];
#pragma unroll
  for (int c = 0; c < NACC; ++c) { acc[0][c] = 0.0f; gr[c] = 0.0; }

  const unsigned* mrow = a.mask + b * a.mwords;
  int rank = 0;
  for (int w = 0; w < a.mwords && rank < r1; ++w) {
    const int base = w * 32;
    const unsigned valid = (a.ntiles - base) >= 32 ? 0xffffffffu : ((1u << (a.ntiles - base)) - 1u);
    unsigned near = ~mrow[w] & valid;
    const int c = __popc(near);
    if (rank + c <= r0) { rank += c; continue; }
    while (near && rank < r1) {
      const int ti = base + __builtin_ctz(near);
      near &= near - 1u;
      if (rank++ < r0) continue;
      const int64_t s0 = (int64_t)ti * T;
      const int cnt = (int)((a.ns - s0) < T ? (a.ns - s0) : T);
      __syncthreads();
      for (int j = tid; j < cnt; j += FF_TB) {
        sh[2 * j] = a.sp[s0 + j];
        sh[2 * j + 1] = a.sa[s0 + j];
      }
      __syncthreads();
      float thr[1] = {CORE == CORE_EXP ? exp_threshold(a.tlim[ti].x + tt[0]) : 0.0f};
      if (PREC == PREC_COMP) {
        // In this order a near tile holds the target's closest sources, whose large
        // terms cancel; the FP32 partials are therefore folded every ff_fold sources, the
        // gradient's into FP64 and the velocity's into its TwoSum pair (the velocity
        // once per tile: error against FP64 on 65,536-131,072 particles in two rings
        // 9.1e-8 to 1.2e-7 instead of 4.8e-8 to 6.0e-8, near field 0-1% faster).
        const int every = ff_sized<CORE, GRAD>() ? a.fold : ff_fold<CORE, GRAD>();
        for (int j0 = 0; j0 < cnt; j0 += every) {
          const int j1 = j0 + every < cnt ? j0 + every : cnt;
          for (int j = j0; j < j1; ++j)
            source_acc<CORE, GRAD, 1>(tx, ty, tz, tt, thr, sh[2 * j], sh[2 * j + 1], acc);
          if (GRAD) fold_grad_raw(acc[0], gr);
          fold_vel_comp(acc[0], hi, lo);
        }
      } else {
        for (int j = 0; j < cnt; ++j)
          source_acc<CORE, GRAD, 1>(tx, ty, tz, tt, thr, sh[2 * j], sh[2 * j + 1], acc);
      }
    }
  }
  if (PREC == PREC_COMP) {
    r[0] = (double)hi[0] + (double)lo[0];
    r[1] = (double)hi[1] + (double)lo[1];
    r[2] = (double)hi[2] + (double)lo[2];
    if (GRAD) grad_from<double>(gr, r + 3);
  } else {
    r[0] = acc[0][0]; r[1] = acc[0][1]; r[2] = acc[0][2];
    if (GRAD) {
      float g[9];
      grad_from<float>(acc[0], g);
#pragma unroll
      for (int c = 0; c < 9; ++c) r[3 + c] = g[c];
    }
  }
}

// persistent: every workgroup takes items from the queue until none is left
template <int CORE, bool GRAD, int PREC>
__global__ __launch_bounds__(256) void k_ff_near(FFArgs a) {
  extern __shared__ float4 sh[];
  __shared__ int s_item;
  const int64_t nb = (a.nt + FF_TB - 1) / FF_TB;
  const int total = a.ioff[nb - 1] + a.items[nb - 1];
  const int m = *a.mfold;
  for (;;) {
    __syncthreads();
    if (threadIdx.x == 0) s_item = (int)atomicAdd(a.ctr, 1u);
    __syncthreads();
    const int item = s_item;
    if (item >= total) break;
    // block b: the last with ioff[b] <= item (blocks without items share the offset
    // of the next block, so the last of a run of equal offsets owns the items)
    int64_t lo = 0, hi = nb;
    while (hi - lo > 1) {
      const int64_t mid = (lo + hi) / 2;
      if (a.ioff[mid] <= item) lo = mid; else hi = mid;
    }
    const int64_t b = lo;
    const int k = item - a.ioff[b];
    const int r0 = k * m;
    const int nnb = a.nn[b];
    const int r1 = r0 + m < nnb ? r0 + m : nnb;
    double r[12];
    near_item<CORE, GRAD, PREC>(a, b, r0, r1, sh, r);
    constexpr int NOUT = GRAD ? 12 : 3;
    ff_sum_store<NOUT>(a.part + (int64_t)item * NOUT * FF_TB, FF_TB, threadIdx.x, a.rows, r);
  }
}

// per target (original order with ROWS, else sorted): far part by slice, near partials in
// item order, self-pair exclusion, accumulated into the caller's arrays
template <int CORE, bool GRAD, bool ROWS>
__global__ __launch_bounds__(256) void k_ff_combine(FFArgs a) {
  constexpr int NOUT = GRAD ? 12 : 3;
  const int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (g >= a.nt) return;
  const int64_t i = ROWS ? a.tinv[g] : g, io = ROWS ? g : a.tperm[g];
  const int64_t b = i / FF_TB;
  double r[NOUT] = {};
#pragma unroll 2
  for (int y = 0; y < a.nslice; ++y) ff_sum_add<NOUT>(a.farv + (int64_t)y * NOUT * a.nt, a.nt, i, ROWS, r);
  const int n_it = a.items[b], off = a.ioff[b];
#pragma unroll 2
  for (int k = 0; k < n_it; ++k)
    ff_sum_add<NOUT>(a.part + (int64_t)(off + k) * NOUT * FF_TB, FF_TB, i % FF_TB, ROWS, r);
  a.t.u[io] = (float)((double)a.t.u[io] + r[0]);
  a.t.v[io] = (float)((double)a.t.v[io] + r[1]);
  a.t.w[io] = (float)((double)a.t.w[io] + r[2]);
  if constexpr (GRAD) {
    if (a.self_excl) {
      // the self pair entered only W (velocity and dyad vanish at d = 0)
      float ks, Bp;
      kb<CORE>(0.0f, core_term<CORE>(a.s.r[io]) + a.tq[i].w, 0.0f, ks, Bp);
      const double kx = (double)ks * a.s.ax[io], ky = (double)ks * a.s.ay[io], kz = (double)ks * a.s.az[io];
      r[4] -= kz; r[5] += ky; r[6] += kz; r[8] -= kx; r[9] -= ky; r[10] += kx;
    }
#pragma unroll
    for (int c = 0; c < 9; ++c) a.t.g[c][io] = (float)((double)a.t.g[c][io] + r[3 + c]);
  }
}

// number of (target, source) pairs the far-field kernel takes: one thread per block
static __global__ __launch_bounds__(256) void k_ff_count(const unsigned* mask, int64_t nb, int mwords, int ntiles, int T,
                                                  int64_t ns, int64_t nt, unsigned long long* out) {
  const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nb) return;
  const int64_t bt = (nt - b * FF_TB) < FF_TB ? (nt - b * FF_TB) : FF_TB;
  unsigned long long sum = 0;
  for (int w = 0; w < mwords; ++w) {
    unsigned bits = mask[b * mwords + w];
    while (bits) {
      const int ti = w * 32 + __builtin_ctz(bits);
      bits &= bits - 1u;
      const int64_t cnt = (ns - (int64_t)ti * T) < T ? (ns - (int64_t)ti * T) : T;
      if (ti < ntiles) sum += (unsigned long long)(cnt * bt);
    }
  }
  atomicAdd(out, sum);
}

static __global__ void k_ff_zero_u64(unsigned long long* p) {
  if (threadIdx.x == 0) *p = 0ull;
}

// ---- host side shared by the factored calls ----------------------------------------

// Key bits, the set's bit included, of n points in all: up to 131,072 points 24, which sort
// in three passes (2^8 cells per axis, or one bit less: a block of 256 is many cells even in
// a ring), then all 30 or 31 in four, which collections of parts far apart need.  With 24 and
// 30 bits: two RM rings of 150,000 each 300 radii apart 49.0 and 30.2 ms, of 50,000 5.5 and
// 3.7; near each other 28.4 and 28.5, 3.74 and 3.77; 165,540 points of two sets 1,766 and
// 1,781 us, 544,768 4.51 and 4.54 ms; 30,000 EXP particles 693 and 712 us
inline int key_bits(int64_t n, bool two_sets) { return n <= 131072 ? 24 : two_sets ? 31 : 30; }

// sequential sub-allocation of a workspace, 256-byte aligned
struct Carve {
  char* base;
  size_t off = 0;
  template <class T>
  T* take(size_t count) {
    T* p = base ? reinterpret_cast<T*>(base + off) : nullptr;
    off += (count * sizeof(T) + 255) & ~(size_t)255;
    return p;
  }
};

inline unsigned grid_of(int64_t n, int per) { return (unsigned)std::max<int64_t>(1, (n + per - 1) / per); }

// LDS of the far-field kernel: r2 slots, moment tables, a tile's rows, core terms
template <int CORE, bool GRAD, bool SHEET = false>
constexpr size_t ff_far_lds() {
  return (size_t)256 * FF_SL * sizeof(__bf16) +
         (size_t)2 * ff_rows<ff_form<CORE, GRAD, SHEET>()>() * FF_TP * sizeof(_Float16) + 512 * sizeof(float4) +
         (CORE == CORE_WL || CORE == CORE_V2 ? 256 * sizeof(float) : 0);
}

// Near-field items per block: about 4,096 in all, three rounds of the workgroups that the
// GPU holds (an item of FF_M0 tiles is 262,144 pairs), and at least 2 per block; 2,048 in
// all where there are few blocks, but no more per block than it has tiles
inline int near_split(int64_t nb, int64_t ntiles) {
  return (int)std::max<int64_t>(2, std::min<int64_t>(std::max<int64_t>(std::min<int64_t>(16, 4096 / nb), 2048 / nb),
                                                     ntiles));
}

// Slices of the far field: blocks x slices workgroups, at least about eight rounds of those
// that a CU holds (three of the velocity form, two else), so that the last round is short
// beside the whole, of eight tiles or more each.  With four rounds of two, in words of 32
// tiles, 65,537 points and 391 tiles made 1,799 workgroups, 2.3 rounds; us then, and with
// 4, 8 and 16 rounds: 1,877 and 1,803, 1,758, 1,745; 524,288 particles on 20,480 panels 3,917
// and 3,646, 3,596, 3,594; WL 131,071 9,209 and 9,199, 8,960, 9,077; RM 65,536 1,611 and
// 1,609, 1,583, 1,583
inline int far_slices(int64_t nb, int64_t ntiles, int per_cu, int cus) {
  const int64_t want = (8 * (int64_t)per_cu * cus + nb - 1) / nb;
  return (int)std::max<int64_t>(1, std::min<int64_t>({want, ntiles / 8, 64}));
}

// (ff.hip) the order of one or two sets along the curve, in the caller's scratch: *perm gets
// the first set's permutation and the second's after it
int factored_order(const FFSets& s, float* box, unsigned* ka, int* va, unsigned* kb, int* vb, void* tmp, hipStream_t st,
                   const int** perm);

}  // namespace o3d

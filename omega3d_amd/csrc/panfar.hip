// panfar.hip -- the panel sums with their separated pairs on the matrix cores.
//
// A panel far from a target is one singular point (recursive rule, pan_kernels.hpp; the
// roles reversed for particles -> panels, ptpan.hip) or seven of them (7-point rule,
// pan_g7.hpp).  Panels and points are sorted along a Hilbert curve, and a block of 256 targets
// takes the tiles of sources that lie a block radius away, and beyond every distance at
// which one of the pairs would not be plain, through k_ff_far (ff_kernels.hpp).  The
// other tiles go through the code of the direct kernels, tile by tile in work items of a
// queue: each item leaves its sums per target, and lists the targets that have pairs
// which need the recursion (or the closed form); a second kernel takes those pairs entry
// by entry and adds to the item's sums.  All decisions per pair are the direct kernels'.
//
// The direct kernels are bound by the issue of about 40 vector instructions per pair (35
// per point of the 7-point rule); a far pair takes one square root, three products and the
// weight's split beside the matrix products (2.5e12 pairs/s with 128 panels per tile).
// Compensated: 20,480 panels on 524,288 points, velocity and gradient 12.1 -> 6.2 ms (far
// 3.74, items 1.49, walks 0.91); 5,120 panels with source strengths on 200,003 points,
// 7-point rule 7.7 -> 4.3 ms (2.74, 1.28, 0.32); 524,288 particles on 20,480 panels 6.4 ->
// 5.7 ms (2.31, 2.54, 1.06); with Hilbert blocks, tiles' own centres and the node stack
// 5.0, 4.0 and 4.0 ms.  Errors against FP64 as before or smaller (1.2e-7 -> 0.9e-7).
#include "ff_kernels.hpp"
#include "o3d_api_internal.hpp"
#include "pan_g7.hpp"
#include "panfar.hpp"
#include "ptpan_kernels.hpp"

namespace o3d {
namespace {

constexpr int PF_FOLD = 64;   // panels or particles per FP32 partial of the compensated sums: half the direct tile, near terms being the large ones

struct PanFarArgs {
  FFArgs f;            // targets: points (PANFAR_POINTS7: too) or panels
  PanArgs p;           // panels as sources
  PtPanArgs t;         // panels as targets
  float4* rec;         // records of the panels in sorted order (targets: rows of tq are enough)
  float4* cen;         // panels as sources: what the near test needs first
  unsigned* list;      // entries (item * 256 + target of the block) with pairs to walk
  unsigned* count;
  int* iblk;           // block of every item
  int64_t units;       // panels or particles that are sources
  int32_t unit;        // of them, per tile
};

// what makes a pair of a panel with a point plain: the distance of the point from the
// panel's centroid, with a margin far above the rounding of the distances compared; a
// limit that is no number keeps the panel out of the far field
__device__ __forceinline__ float plain_limit(float lim) { return lim >= 0.0f ? lim * 1.00001f : __builtin_huge_valf(); }

// rows, records and bounds, one workgroup per tile of sources and then one per block of
// targets (ff_kernels.hpp: k_ff_rows): source rows up to a whole tile, the panels' records
// and near-test rows, and targets: points, or panels' centroids with their limit
template <int RULE>
__global__ __launch_bounds__(256) void k_pf_rows(PanFarArgs a, const int* sperm, float4* sp, float4* sa, float4* tq,
                                                 FFBounds sb, FFBounds tb, int* nn, int* tinv) {
  constexpr int N = RULE == PANFAR_POINTS7 ? 7 : 1;
  const int tid = threadIdx.x;
  if ((int)blockIdx.x >= a.f.ntiles) {
    const int64_t b = (int64_t)blockIdx.x - a.f.ntiles, i = b * FF_TB + tid;
    float4 p{};
    if (i < a.f.nt) {
      const int j = a.f.tperm[i];
      if (RULE == PANFAR_PARTICLES) {
        float4 s[PAN_F4];
        ptpan_record(a.t, j, s);
        p = make_float4(s[3].x, s[3].y, s[3].z, plain_limit(s[4].z * 4.0f));
      } else {
        p = make_float4(a.p.tx[j], a.p.ty[j], a.p.tz[j], 0.0f);
      }
      tq[i] = p;
      if (tinv) tinv[j] = (int)i;
    }
    ff_group_bounds<1>(i < a.f.nt, &p, nullptr, tb, b);
    if (tid == 0) nn[b] = 0;
    return;
  }
  const int64_t t = blockIdx.x, i = t * a.unit + tid;
  const bool has = tid < a.unit, real = has && i < a.units;
  float4 p[N] = {}, q[N] = {};
  if (has) {
    const int64_t j = sperm[real ? i : a.units - 1];
    if constexpr (RULE == PANFAR_PARTICLES) {
      p[0] = make_float4(a.t.sx[j], a.t.sy[j], a.t.sz[j], 0.0f);
      if (real) q[0] = make_float4(a.t.ax[j], a.t.ay[j], a.t.az[j], 0.0f);
    } else if constexpr (RULE == PANFAR_POINTS) {
      float4 s[PAN_F4];
      panel_record(a.p, j, s);
      p[0] = make_float4(s[3].x, s[3].y, s[3].z, plain_limit(s[4].z * 4.0f));
      if (real) {
        q[0] = s[2];
#pragma unroll
        for (int k = 0; k < PAN_F4; ++k) a.rec[PAN_F4 * i + k] = s[k];
        a.cen[i] = s[3];
      }
    } else {
      float4 s[G7_F4];
      g7_record(a.p, j, s);
      const float lim = plain_limit(sqrtf(s[7].x));
      const float pt[21] = {s[0].x, s[0].y, s[0].z, s[0].w, s[1].x, s[1].y, s[1].z, s[1].w, s[2].x, s[2].y, s[2].z,
                            s[2].w, s[3].x, s[3].y, s[3].z, s[3].w, s[4].x, s[4].y, s[4].z, s[4].w, s[5].x};
#pragma unroll
      for (int k = 0; k < 7; ++k) {
        const float w = (float)g7_weight(k);
        p[k] = make_float4(pt[3 * k], pt[3 * k + 1], pt[3 * k + 2], lim);
        if (real) q[k] = make_float4(w * s[6].x, w * s[6].y, w * s[6].z, w * s[6].w);
      }
      if (real) {
#pragma unroll
        for (int k = 0; k < G7_F4; ++k) a.rec[G7_F4 * i + k] = s[k];
        a.cen[i] = make_float4(s[5].y, s[5].z, s[5].w, s[7].x);
      }
    }
    const int64_t row = t * a.f.tile + N * tid;
#pragma unroll
    for (int k = 0; k < N; ++k) { sp[row + k] = p[k]; sa[row + k] = q[k]; }
    if (N > 1 && tid == a.unit - 1)   // the last panel of a tile fills it up
      for (int k = N * a.unit; k < a.f.tile; ++k) {
        sp[t * a.f.tile + k] = p[0];
        sa[t * a.f.tile + k] = make_float4(0.f, 0.f, 0.f, 0.f);
      }
  }
  ff_group_bounds<N>(has, p, q, sb, t);
}

// block b's near tiles of rank [r0, r1), in order: next() gives -1 after the last
struct NearTiles {
  const unsigned* mrow;
  int mwords, ntiles, r0, r1, w = -1, rank = 0;
  unsigned bits = 0u;
  __device__ __forceinline__ NearTiles(const FFArgs& f, int64_t b, int r0_, int r1_)
      : mrow(f.mask + b * f.mwords), mwords(f.mwords), ntiles(f.ntiles), r0(r0_), r1(r1_) {}
  __device__ __forceinline__ int next() {
    for (;;) {
      while (bits == 0u) {
        if (rank >= r1 || ++w >= mwords) return -1;
        const int left = ntiles - 32 * w;
        bits = ~mrow[w] & (left >= 32 ? 0xffffffffu : (1u << left) - 1u);
        const int c = __popc(bits);
        if (rank + c <= r0) { rank += c; bits = 0u; }
      }
      const int t = 32 * w + __builtin_ctz(bits);
      bits &= bits - 1u;
      if (rank++ < r0) continue;
      return rank <= r1 ? t : -1;
    }
  }
};

// one item: the pairs of a block with some of its near tiles, as the direct kernel takes
// them (k_pan, k_pan_g7, k_ptpan)
template <int RULE, bool GRAD, int PREC>
__device__ __forceinline__ void pf_item(const PanFarArgs& a, int64_t b, int item, int r0, int r1, float4* sh) {
  constexpr int NOUT = GRAD ? 12 : 3;
  constexpr int F4 = RULE == PANFAR_POINTS ? PAN_F4 : RULE == PANFAR_POINTS7 ? G7_F4 : 2;
  const int tid = threadIdx.x;
  const int64_t i = b * FF_TB + tid;
  const bool active = i < a.f.nt;
  const int64_t ic = active ? i : a.f.nt - 1;
  const float4 q = a.f.tq[ic];
  float4 s[PAN_F4] = {};
  if (RULE == PANFAR_PARTICLES) ptpan_record(a.t, a.f.tperm[ic], s);
  const PtRoot<float> root(s);
  float acc[16];
  float hi[3] = {0.f, 0.f, 0.f}, lo[3] = {0.f, 0.f, 0.f};
  double gd[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  bool has_near = false;
#pragma unroll
  for (int c = 0; c < 16; ++c) acc[c] = 0.0f;
  NearTiles tiles(a.f, b, r0, r1);
  for (int t = tiles.next(); t >= 0; t = tiles.next()) {
    const int64_t p0 = (int64_t)t * a.unit;
    const int cnt = (int)(a.units - p0 < a.unit ? a.units - p0 : a.unit);
    __syncthreads();
    if (RULE == PANFAR_PARTICLES) {
      for (int j = tid; j < cnt; j += FF_TB) {
        sh[2 * j] = a.f.sp[p0 + j];
        sh[2 * j + 1] = a.f.sa[p0 + j];
      }
    } else {
      for (int j = tid; j < F4 * cnt; j += FF_TB) sh[j] = a.rec[F4 * p0 + j];
    }
    __syncthreads();
    for (int j0 = 0; j0 < cnt; j0 += PF_FOLD) {
      const int n = cnt - j0 < PF_FOLD ? cnt - j0 : PF_FOLD;
      const float4* w = sh + F4 * j0;
      if constexpr (RULE == PANFAR_POINTS) {
        pan_root_tile<float, GRAD>(w, n, q.x, q.y, q.z, a.p.maxlev, active, acc, has_near);
      } else if constexpr (RULE == PANFAR_POINTS7) {
        for (int j = 0; j < n; ++j) {
          const bool near = g7_is_near(q.x, q.y, q.z, w + G7_F4 * j);
          has_near |= near;
          g7_far_pair<float, GRAD>(q.x, q.y, q.z, w + G7_F4 * j, near ? 0.0f : 1.0f, acc);
        }
      } else {
        int nnear = 0;
        ptpan_root_tile<PREC, false>(w, n, p0 + j0, root, a.t.maxlev, active, acc, nullptr, nnear);
        has_near |= nnear > 0;
      }
      if (PREC == PREC_COMP) {
        two_sum(hi[0], lo[0], acc[0]);
        two_sum(hi[1], lo[1], acc[1]);
        two_sum(hi[2], lo[2], acc[2]);
        if (GRAD) {
          float g[9];
          if (RULE == PANFAR_POINTS7) {
#pragma unroll
            for (int k = 0; k < 9; ++k) g[k] = acc[3 + k];
          } else {
            grad_of<float>(acc, g);
          }
#pragma unroll
          for (int k = 0; k < 9; ++k) gd[k] += (double)g[k];
        }
#pragma unroll
        for (int c = 0; c < 16; ++c) acc[c] = 0.0f;
      }
    }
  }
  // particles -> panels: the pairs were summed with the roles reversed
  const double sg = RULE == PANFAR_PARTICLES ? -1.0 : 1.0;
  double r[NOUT];
#pragma unroll
  for (int d = 0; d < 3; ++d)
    r[d] = sg * (PREC == PREC_COMP ? (double)hi[d] + (double)lo[d] : (double)acc[d]);
  if (GRAD) {
    float g[9];
    if (PREC != PREC_COMP) {
      if (RULE == PANFAR_POINTS7) {
#pragma unroll
        for (int k = 0; k < 9; ++k) g[k] = acc[3 + k];
      } else {
        grad_of<float>(acc, g);
      }
    }
#pragma unroll
    for (int k = 0; k < 9; ++k) r[3 + k] = PREC == PREC_COMP ? gd[k] : (double)g[k];
  }
  ff_sum_store<NOUT>(a.f.part + (int64_t)item * NOUT * FF_TB, FF_TB, tid, a.f.rows, r);
  if (has_near && active) a.list[atomicAdd(a.count, 1u)] = (unsigned)item * FF_TB + tid;
}

// persistent: every workgroup takes items from the queue until none is left
template <int RULE, bool GRAD, int PREC>
__global__ __launch_bounds__(FF_TB) void k_pf_items(PanFarArgs a) {
  extern __shared__ float4 sh[];
  __shared__ int s_item;
  const int64_t nb = (a.f.nt + FF_TB - 1) / FF_TB;
  const int total = a.f.ioff[nb - 1] + a.f.items[nb - 1];
  const int m = *a.f.mfold;
  for (;;) {
    __syncthreads();
    if (threadIdx.x == 0) s_item = (int)atomicAdd(a.f.ctr, 1u);
    __syncthreads();
    const int item = s_item;
    if (item >= total) break;
    // block b: the last with ioff[b] <= item (blocks without items share the offset of the next)
    int64_t lo = 0, hi = nb;
    while (hi - lo > 1) {
      const int64_t mid = (lo + hi) / 2;
      if (a.f.ioff[mid] <= item) lo = mid; else hi = mid;
    }
    if (threadIdx.x == 0) a.iblk[item] = (int)lo;
    const int r0 = (item - a.f.ioff[lo]) * m;
    const int nnb = a.f.nn[lo];
    pf_item<RULE, GRAD, PREC>(a, lo, item, r0, r0 + m < nnb ? r0 + m : nnb, sh);
  }
}

// an entry's block, item, target row and tiles
struct PfEntry {
  int64_t b;
  int item, tid, r0, r1;
  __device__ __forceinline__ PfEntry(const PanFarArgs& a, unsigned e) : item((int)(e / FF_TB)), tid((int)(e % FF_TB)) {
    b = a.iblk[item];
    const int m = *a.f.mfold;
    r0 = (item - a.f.ioff[b]) * m;
    r1 = r0 + m < a.f.nn[b] ? r0 + m : a.f.nn[b];
  }
};

// The listed entries' pairs that need the recursion: one wave per entry, whose lanes test
// the item's panels (particles) in turn and split the near ones' nodes together
// (NodeStack).  A fixed butterfly adds the lanes' sums in FP64; the order in which entries
// were listed decides nothing.
template <int RULE, bool GRAD, int PREC>
__global__ __launch_bounds__(BLOCK) void k_pf_walk(PanFarArgs a) {
  constexpr int NOUT = GRAD ? 12 : 3;
  constexpr bool PART = RULE == PANFAR_PARTICLES;
  extern __shared__ int2 shn[];
  const int maxlev = PART ? a.t.maxlev : a.p.maxlev;
  NodeStack stack{shn + (threadIdx.x >> 6) * node_cap(maxlev), 0, node_cap(maxlev)};
  const int lane = threadIdx.x & 63;
  const int64_t wave = ((int64_t)blockIdx.x * BLOCK + threadIdx.x) >> 6;
  const int64_t nwaves = ((int64_t)gridDim.x * BLOCK) >> 6;
  const int64_t listed = *a.count;
  for (int64_t e = wave; e < listed; e += nwaves) {
    const PfEntry n(a, a.list[e]);
    const float4 q = a.f.tq[n.b * FF_TB + n.tid];
    float4 s[PAN_F4] = {};
    if (PART) ptpan_record(a.t, a.f.tperm[n.b * FF_TB + n.tid], s);
    const PtRoot<float> root(s);
    float acc[16];
#pragma unroll
    for (int c = 0; c < 16; ++c) acc[c] = 0.0f;
    auto split = [&]() {
      int2 node;
      const bool has = stack.pop(node);
      const int64_t p = has ? node.x : 0;
      if constexpr (PART) {
        const float4 P = a.f.sp[p];
        ptpan_strength<PREC>(s, a.f.sa[p]);
        split_node<float, false>(has, node, P.x, P.y, P.z, s, maxlev, acc, stack);
      } else {
        split_node<float, GRAD>(has, node, q.x, q.y, q.z, a.rec + PAN_F4 * p, maxlev, acc, stack);
      }
    };
    NearTiles tiles(a.f, n.b, n.r0, n.r1);
    for (int t = tiles.next(); t >= 0; t = tiles.next()) {
      const int64_t p0 = (int64_t)t * a.unit;
      const int cnt = (int)(a.units - p0 < a.unit ? a.units - p0 : a.unit);
      for (int j0 = 0; j0 < cnt; j0 += 64) {
        const int64_t p = p0 + j0 + lane;
        bool near = j0 + lane < cnt;
        const float4 c = PART ? a.f.sp[near ? p : 0] : a.cen[near ? p : 0];
        const float4 P = PART ? c : q;
        if constexpr (PART) {
          near = near && !root_leaf<float>(P.x, P.y, P.z, root.cx, root.cy, root.cz, root.lim, root.rl, maxlev, near);
        } else {
          const float ex = P.x - c.x, ey = P.y - c.y, ez = P.z - c.z;
          near = near && !(fmaf(ez, ez, fmaf(ey, ey, ex * ex)) > c.w);
          if (near) {
            float gx, gy, gz, gs, cx0, cy0, cz0, lim;
            RootLim rl;
            panel_root<float>(a.rec + PAN_F4 * p, gx, gy, gz, gs, cx0, cy0, cz0, lim, rl);
            near = !root_leaf<float>(P.x, P.y, P.z, cx0, cy0, cz0, lim, rl, maxlev, true);
          }
        }
        stack.push(near, (int)p, 0u);
        while (stack.n >= 64) split();
      }
    }
    while (stack.n > 0) split();
    double* slot = a.f.part + (int64_t)n.item * NOUT * FF_TB + (a.f.rows ? n.tid * NOUT : n.tid);
    const int step = a.f.rows ? 1 : FF_TB;
    double u[3], g[9];
#pragma unroll
    for (int d = 0; d < 3; ++d) u[d] = wave_sum((PART ? -1.0 : 1.0) * (double)acc[d]);
    if (GRAD) {
      float gl[9];
      grad_of<float>(acc, gl);
#pragma unroll
      for (int k = 0; k < 9; ++k) g[k] = wave_sum((double)gl[k]);
    }
    if (lane != 0) continue;
#pragma unroll
    for (int d = 0; d < 3; ++d) slot[d * step] += u[d];
    if (GRAD) {
#pragma unroll
      for (int k = 0; k < 9; ++k) slot[(3 + k) * step] += g[k];
    }
  }
}

// The 7-point rule's near pairs in closed form, FP64.  Each quarter of a wave takes an
// entry: its 16 lanes test the item's panels in turn, queue those that are near and
// evaluate them when 16 are there or none is left, hit h in lane h mod 16.  Summed as above.
template <bool GRAD>
__global__ __launch_bounds__(BLOCK) void k_pf_near7(PanFarArgs a) {
  constexpr int NOUT = GRAD ? 12 : 3;
  __shared__ int ring[BLOCK / 16][32];
  const int lane = threadIdx.x & 63, ql = lane & 15, q0 = lane & 48;
  int* mine = ring[threadIdx.x >> 4];
  const int64_t wave = ((int64_t)blockIdx.x * BLOCK + threadIdx.x) >> 6;
  const int64_t nwaves = ((int64_t)gridDim.x * BLOCK) >> 6;
  const int64_t listed = *a.count;
  for (int64_t e = wave; 4 * e < listed; e += nwaves) {
    const int64_t li = 4 * e + (lane >> 4);
    const bool has = li < listed;
    const PfEntry n(a, a.list[has ? li : 4 * e]);
    const float4 q = a.f.tq[n.b * FF_TB + n.tid];
    double u[3] = {0, 0, 0}, g[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    int head = 0, tail = 0;   // hits evaluated and found, alike in the quarter's lanes
    auto drain = [&]() {
      const int h = head + ((ql - head) & 15);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      if (h < tail) {
        const float4* r = a.rec + G7_F4 * (int64_t)mine[h & 31];
        const float4 f6 = r[6], f7 = r[7], f8 = r[8], f9 = r[9];
        const float v[9] = {f7.y, f7.z, f7.w, f8.x, f8.y, f8.z, f8.w, f9.x, f9.y};
        const float ts[3] = {f6.x, f6.y, f6.z};
        g7_near_pair<GRAD>(q.x, q.y, q.z, v, ts, f9.z, f9.w, u, g);
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      head = head + 16 < tail ? head + 16 : tail;
    };
    NearTiles tiles(a.f, n.b, n.r0, has ? n.r1 : n.r0);
    for (int t = tiles.next(); wave_any(t >= 0); t = t >= 0 ? tiles.next() : -1) {
      const int64_t p0 = (int64_t)t * a.unit;
      const int cnt = t < 0 ? 0 : (int)(a.units - p0 < a.unit ? a.units - p0 : a.unit);
      for (int j0 = 0; j0 < a.unit; j0 += 16) {
        const int j = j0 + ql;
        const float4 c = a.cen[j < cnt ? p0 + j : 0];
        float d2;
        {
#pragma clang fp contract(off)
          const float ex = q.x - c.x, ey = q.y - c.y, ez = q.z - c.z;
          d2 = ex * ex + ey * ey + ez * ez;
        }
        const bool near = j < cnt && d2 < c.w;
        const unsigned hits = (unsigned)(__builtin_amdgcn_ballot_w64(near) >> q0) & 0xffffu;
        if (near) mine[(tail + __popc(hits & ((1u << ql) - 1u))) & 31] = (int)(p0 + j);
        tail += __popc(hits);
        while (wave_any(tail - head >= 16)) drain();
      }
    }
    while (wave_any(head < tail)) drain();
    double* slot = a.f.part + (int64_t)n.item * NOUT * FF_TB + (a.f.rows ? n.tid * NOUT : n.tid);
    const int step = a.f.rows ? 1 : FF_TB;
#pragma unroll
    for (int d = 0; d < 3; ++d) u[d] = quarter_sum(u[d]);
    if (GRAD) {
#pragma unroll
      for (int k = 0; k < 9; ++k) g[k] = quarter_sum(g[k]);
    }
    if (ql != 0 || !has) continue;
#pragma unroll
    for (int d = 0; d < 3; ++d) slot[d * step] += u[d];
    if (GRAD) {
#pragma unroll
      for (int k = 0; k < 9; ++k) slot[(3 + k) * step] += g[k];
    }
  }
}

struct PanFarLayout {
  unsigned *k_in, *k_out, *mask, *ctr, *list, *count;
  int *i_in, *i_out, *tinv, *nn, *items, *ioff, *mfold, *iblk;
  void* tmp;
  float* box;
  float4 *sp, *sa, *tq, *tsph, *tlim, *bsph, *blim, *rec, *cen;
  double *farv, *part;
  size_t bytes;
};

// sources per tile and panels per tile.  A tile of fewer panels is smaller, but its tables
// are made for fewer pairs.  5,120 panels on 262,144 points: 1.44 ms with 256 and 1.34 with
// 128; 20,480 panels on 524,288 4.96 and 5.00, on 2,048 0.38 and 0.44
int tile_of(int rule, int64_t units) { return rule == PANFAR_POINTS && units < 8192 ? 128 : 256; }
int unit_of(int rule, int64_t units) { return rule == PANFAR_POINTS7 ? tile_of(rule, units) / 7 : tile_of(rule, units); }

PanFarLayout layout(char* base, int rule, int64_t units, int64_t nt, int nout) {
  const int T = tile_of(rule, units), U = unit_of(rule, units);
  const int64_t nb = (nt + FF_TB - 1) / FF_TB;
  const int64_t ntiles = (units + U - 1) / U;
  const int64_t mwords = (ntiles + 31) / 32;
  const int64_t maxitems = (near_split(nb, ntiles) + 1) * nb;
  const int f4 = rule == PANFAR_POINTS ? PAN_F4 : rule == PANFAR_POINTS7 ? G7_F4 : 0;
  Carve cv{base};
  PanFarLayout L{};
  L.box = cv.take<float>(FF_BOX_FLOATS);
  L.k_in = cv.take<unsigned>(units + nt);
  L.k_out = cv.take<unsigned>(units + nt);
  L.i_in = cv.take<int>(units + nt);
  L.i_out = cv.take<int>(units + nt);
  L.tinv = cv.take<int>(nt);
  L.tmp = cv.take<char>(radix_tmp_bytes(units + nt));
  L.sp = cv.take<float4>((size_t)ntiles * T);
  L.sa = cv.take<float4>((size_t)ntiles * T);
  L.rec = cv.take<float4>((size_t)f4 * units);
  L.cen = cv.take<float4>(f4 ? units : 0);
  L.tq = cv.take<float4>(nt);
  L.tsph = cv.take<float4>(ntiles);
  L.tlim = cv.take<float4>(ntiles);
  L.bsph = cv.take<float4>(nb);
  L.blim = cv.take<float4>(nb);
  L.mask = cv.take<unsigned>((size_t)(nb * mwords));
  L.farv = cv.take<double>((size_t)nout * far_slices(nb, ntiles, nout == 3 ? 3 : 2, num_cus()) * nt);
  L.nn = cv.take<int>(nb);
  L.items = cv.take<int>(nb);
  L.ioff = cv.take<int>(nb);
  L.mfold = cv.take<int>(1);
  L.ctr = cv.take<unsigned>(1);
  L.count = cv.take<unsigned>(1);
  L.iblk = cv.take<int>(maxitems);
  L.list = cv.take<unsigned>((size_t)maxitems * FF_TB);
  L.part = cv.take<double>((size_t)maxitems * nout * FF_TB);
  L.bytes = cv.off;
  return L;
}

template <int RULE, bool GRAD, int PREC>
int64_t items_grid(size_t lds) {
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_pf_items<RULE, GRAD, PREC>, FF_TB, lds) != hipSuccess ||
      per_cu < 1)
    per_cu = 1;
  return (int64_t)per_cu * num_cus();
}

template <int RULE, bool GRAD, bool SHEET, int PREC>
int run(const PanArgs* p, const PtPanArgs* t, void* ws, hipStream_t st) {
  constexpr bool PART = RULE == PANFAR_PARTICLES;
  PanFarArgs a{};
  if (p) a.p = *p;
  if (t) a.t = *t;
  const int64_t units = PART ? t->ns : p->np, nt = PART ? t->np : p->nt;
  const int T = tile_of(RULE, units), U = unit_of(RULE, units);
  const int64_t nb = (nt + FF_TB - 1) / FF_TB;
  const int ntiles = (int)((units + U - 1) / U), mwords = (ntiles + 31) / 32;
  const PanFarLayout L = layout(static_cast<char*>(ws), RULE, units, nt, GRAD ? 12 : 3);
  FFArgs& f = a.f;
  f.sp = L.sp; f.sa = L.sa; f.tq = L.tq;
  f.tsph = L.tsph; f.tlim = L.tlim; f.bsph = L.bsph; f.blim = L.blim;
  f.mask = L.mask; f.farv = L.farv;
  f.nn = L.nn; f.items = L.items; f.ioff = L.ioff; f.mfold = L.mfold; f.ctr = L.ctr; f.part = L.part;
  f.nt = nt; f.ns = (int64_t)ntiles * T;
  f.tile = T; f.mwords = mwords; f.ntiles = ntiles;
  f.t.u = (float*)(PART ? t->u : p->u); f.t.v = (float*)(PART ? t->v : p->v); f.t.w = (float*)(PART ? t->w : p->w);
  for (int k = 0; k < 9; ++k) f.t.g[k] = GRAD ? (float*)p->g[k] : nullptr;
  a.rec = L.rec; a.cen = L.cen; a.list = L.list; a.count = L.count; a.iblk = L.iblk;
  a.units = units; a.unit = U;

  FFSets sets{};
  const int pan = PART ? 1 : 0, pts = 1 - pan;   // sources first
  sets.x[pan] = PART ? t->nx : p->nx; sets.y[pan] = PART ? t->ny : p->ny; sets.z[pan] = PART ? t->nz : p->nz;
  sets.x[pts] = PART ? t->sx : p->tx; sets.y[pts] = PART ? t->sy : p->ty; sets.z[pts] = PART ? t->sz : p->tz;
  sets.n[0] = units; sets.n[1] = nt;
  sets.idx = PART ? t->idx : p->idx;
  sets.pan = pan;
  const int* perm = nullptr;
  const int rc = factored_order(sets, L.box, L.k_in, L.i_in, L.k_out, L.i_out, L.tmp, st, &perm);
  if (rc != O3D_OK) return rc;
  f.tperm = perm + units;
  f.tinv = L.tinv;
  f.rows = nt >= FF_ROWS_MIN;
  const FFBounds tb{L.tsph, L.tlim}, bb{L.bsph, L.blim};
  hipLaunchKernelGGL((k_pf_rows<RULE>), dim3((unsigned)(ntiles + nb)), dim3(256), 0, st, a, perm, L.sp, L.sa, L.tq, tb, bb,
                     L.nn, nt >= FF_ROWS_MIN ? L.tinv : nullptr);
  hipLaunchKernelGGL((k_ff_classify<CORE_SING>), dim3(grid_of(nb * mwords, 256)), dim3(256), 0, st, bb, nb, tb, ntiles,
                     mwords, L.mask, L.nn);
  hipLaunchKernelGGL(k_ff_plan, dim3(1), dim3(FF_PLAN_THREADS), 0, st, L.nn, nb, near_split(nb, ntiles), L.items, L.ioff,
                     L.mfold, L.ctr, L.count);
  HIPCHK(hipGetLastError());

  const int nslice = far_slices(nb, ntiles, GRAD ? 2 : 3, num_cus());
  f.tslice = (ntiles + nslice - 1) / nslice;
  f.nslice = (ntiles + f.tslice - 1) / f.tslice;
  hipLaunchKernelGGL((k_ff_far<CORE_SING, GRAD, SHEET>), dim3((unsigned)nb, (unsigned)f.nslice), dim3(FF_FAR_THREADS),
                     (ff_far_lds<CORE_SING, GRAD, SHEET>()), st, f);
  HIPCHK(hipGetLastError());
  const size_t lds = (size_t)U * (RULE == PANFAR_POINTS ? PAN_F4 : RULE == PANFAR_POINTS7 ? G7_F4 : 2) * sizeof(float4);
  const int64_t maxitems = (near_split(nb, ntiles) + 1) * nb;
  const unsigned gitems = (unsigned)std::min<int64_t>(maxitems, items_grid<RULE, GRAD, PREC>(lds));
  hipLaunchKernelGGL((k_pf_items<RULE, GRAD, PREC>), dim3(gitems), dim3(FF_TB), lds, st, a);
  HIPCHK(hipGetLastError());
  // at most 16 waves per CU
  const unsigned gwalk = (unsigned)std::min<int64_t>((maxitems * FF_TB + 15) / 16, 4 * (int64_t)num_cus());
  if constexpr (RULE == PANFAR_POINTS7)
    hipLaunchKernelGGL((k_pf_near7<GRAD>), dim3(gwalk), dim3(BLOCK), 0, st, a);
  else
    hipLaunchKernelGGL((k_pf_walk<RULE, GRAD, PREC>), dim3(gwalk), dim3(BLOCK), node_lds(PART ? t->maxlev : p->maxlev), st, a);
  HIPCHK(hipGetLastError());
  if (f.rows) hipLaunchKernelGGL((k_ff_combine<CORE_SING, GRAD, true>), dim3((unsigned)nb), dim3(FF_TB), 0, st, f);
  else hipLaunchKernelGGL((k_ff_combine<CORE_SING, GRAD, false>), dim3((unsigned)nb), dim3(FF_TB), 0, st, f);
  HIPCHK(hipGetLastError());
  return O3D_OK;
}

template <int RULE, bool GRAD>
int run_points(const PanArgs& p, int prec, void* ws, hipStream_t st) {
  if (prec == PREC_COMP)
    return p.ss ? run<RULE, GRAD, true, PREC_COMP>(&p, nullptr, ws, st) : run<RULE, GRAD, false, PREC_COMP>(&p, nullptr, ws, st);
  return p.ss ? run<RULE, GRAD, true, PREC_FP32>(&p, nullptr, ws, st) : run<RULE, GRAD, false, PREC_FP32>(&p, nullptr, ws, st);
}

}  // namespace

// Where the far field pays, compensated, direct against here, spheres and points in a shell
// around them.  Panels on points, recursive: the direct kernel takes 0.14 us per panel with
// few points, here 0.2 ms: 960 panels on 2,048 points 233 and 211 us, 5,120 panels on 32
// points 690 and 218, 20,480 on 2,048 points 3.2 and 0.44 ms.  With many points the near
// field of few, coarse panels decides: 1,280 panels on 16,384 points 333 and 318 us, on
// 65,536 449 and 553; 1,600 panels (a patch) on 16,384 282 and 295; 2,560 on 262,144 0.90
// and 0.89 ms; 3,600 on 262,144 1.30 and 1.11, 5,120 1.89 and 1.33.  7-point rule: 960
// panels on 1,024 points 511 and 212 us, 1,280 on 131,072 1.45 and 1.03 ms (velocity alone
// 0.87 and 0.77); 640 panels on 65,536 520 and 498 us (311 and 429), 320 on 524,288 points
// 4.86 and 2.57 ms.  Both rules gain alike in plain FP32
// (5,120 panels on 100,000 points 848 and 506 us, 7-point rule 3,426 and 2,077), with errors
// against FP64 that are no larger (7.1e-7 and 3.6e-7).
//
// Particles on panels: the direct kernel keeps eight near particles per panel and slice and
// scans a slice with more again, so the particles per panel decide for few panels, and the
// pairs for many; how near the particles lie decides as much and is not known here.  us direct
// and here of whole spheres, particles in the shells 1.01-2.5, 1.005-1.1, 1.02-1.5 and 1.5-4:
//   320 panels,  32,768 particles    192  214     686   359     457   254      80  184
//   320         100,000              488  359   2,002   652   1,300   464     185  238
//   1,280       180,000              409  463   1,781 1,058     617   626     407  350
//   1,280       262,144              425  585   2,765 1,372   1,604   821     398  409
//   1,280       400,000              626  729   4,280 1,992   2,438 1,112     583  508
//   5,120       262,144              760  759   3,822 1,435     847   954     769  620
//   5,120       400,000                         6,489 1,944   1,470 1,297   1,096  820
//   20,480       65,536              715  680     783   842     731   751     695  551
//   20,480      131,072            1,327  999   1,660 1,307   1,371 1,182   1,318  888
// With 8,192 particles 20 panels take 183 and 160, 80 panels 189 and 171; from 512 panels on
// the launches are worth 200 particles per panel instead of 100 (640 and 131,072 270 354,
// 1,239 625, 410 456, 275 278).  A call that names its method or a tile is the direct kernels'.
bool panfar_pays(int rule, int64_t units, int64_t nt, int method, int tile, int prec) {
  if (method != O3D_METHOD_AUTO || tile > 0 || prec == PREC_FP64 || units > (1 << 26) || nt > (1 << 26)) return false;
  if (rule == PANFAR_PARTICLES) {
    return units >= 8192 && (units >= (nt < 512 ? 100 : 200) * nt || units * nt >= 1800000000LL);
  }
  if (nt < 32) return false;
  if (rule == PANFAR_POINTS7) return units >= 1024 || units * nt >= 160000000LL;
  return units >= 3072 || (units >= 1024 && nt <= 8 * units);
}

size_t panfar_bytes(int rule, int64_t units, int64_t nt, bool grad) {
  return layout(nullptr, rule, units, nt, grad ? 12 : 3).bytes;
}

bool panfar_scratch(size_t bytes, hipStream_t st, void** ws) {
  if (stream_capturing(st) && !stream_workspace_fits(st, bytes)) return false;
  if (stream_workspace(st, bytes, ws) == O3D_OK) return true;
  clear_error();
  (void)hipGetLastError();
  return false;
}

int panfar_points(const PanArgs& p, int rule, bool grad, int prec, void* ws, hipStream_t st) {
  if (rule == PANFAR_POINTS7)
    return grad ? run_points<PANFAR_POINTS7, true>(p, prec, ws, st) : run_points<PANFAR_POINTS7, false>(p, prec, ws, st);
  return grad ? run_points<PANFAR_POINTS, true>(p, prec, ws, st) : run_points<PANFAR_POINTS, false>(p, prec, ws, st);
}

int panfar_particles(const PtPanArgs& t, int prec, void* ws, hipStream_t st) {
  return prec == PREC_COMP ? run<PANFAR_PARTICLES, false, false, PREC_COMP>(nullptr, &t, ws, st)
                           : run<PANFAR_PARTICLES, false, false, PREC_FP32>(nullptr, &t, ws, st);
}

}  // namespace o3d

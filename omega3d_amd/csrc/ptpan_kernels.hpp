// ptpan_kernels.hpp -- particles -> panels: what k_ptpan (ptpan.hip) and the factored form
// (panfar.hip) share: a target panel's record, a particle's strength on it and the root
// pairs of staged particles (Influence.h:1196-1210).
#pragma once
#include "pan_kernels.hpp"

namespace o3d {

struct PtPanArgs {
  const float* sx; const float* sy; const float* sz;    // particles
  const float* ax; const float* ay; const float* az;
  int64_t ns;
  const float* nx; const float* ny; const float* nz;    // panel nodes
  const uint32_t* idx;
  const float* area;
  int64_t np;
  void* u; void* v; void* w;   // float (decremented in place) or double (FP64: zeroed scratch)
  int32_t tile;
  int32_t maxlev;
  int32_t* near_list;          // panels with a pair that needs the recursion
  unsigned int* near_count;
  double* part;                // per slice: 3 sums per panel
  int32_t* cnt;                // [panel][slice]: particles that need the recursion
  int32_t* ent;                // [panel][slice][PTPAN_CAP]: the first of them, ascending
  int64_t slen;                // particles per slice
  int32_t nslice;
};

// particles kept per (slice, panel) for the near kernel; a slice with more is
// scanned again there
constexpr int PTPAN_CAP = 8;

// this lane's panel in the staged-panel layout of pan_kernels.hpp (the strength
// fields are filled per particle)
__device__ __forceinline__ void ptpan_record(const PtPanArgs& a, int64_t i, float4* s) {
  const uint32_t i0 = a.idx[3 * i], i1 = a.idx[3 * i + 1], i2 = a.idx[3 * i + 2];
  const float x0 = a.nx[i0], y0 = a.ny[i0], z0 = a.nz[i0];
  const float x1 = a.nx[i1], y1 = a.ny[i1], z1 = a.nz[i1];
  const float x2 = a.nx[i2], y2 = a.ny[i2], z2 = a.nz[i2];
  const float ar = a.area[i];
  float cx, cy, cz;
  centroid_exact(x0, y0, z0, x1, y1, z1, x2, y2, z2, cx, cy, cz);
  s[0] = make_float4(x0, y0, z0, x1);
  s[1] = make_float4(y1, z1, x2, y2);
  s[2] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  float far2, near2;
  root_bands(sqrtf(ar), far2, near2);
  s[3] = make_float4(cx, cy, cz, far2);
  s[4] = make_float4(z2, ar, sqrtf(ar), near2);
  s[5] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
}

// particle j's strength on panel record s at level 0.  FP64: the walk forms
// (alpha / area) * area in double from s[5].  FP32 and compensated: alpha itself;
// the reference's float round trip (alpha / area) * area (Influence.h:1198,
// Kernels.h:1136-1146) moves it by at most one float ulp and costs three IEEE
// divisions per pair.
template <int PREC>
__device__ __forceinline__ void ptpan_strength(float4* s, float4 A) {
  if (PREC == PREC_FP64) s[5] = make_float4(A.x, A.y, A.z, 0.0f);
  else { s[2].x = A.x; s[2].y = A.y; s[2].z = A.z; }
}

constexpr int PTPAN_UNROLL = 4;   // particles per step of the separated-pair loop

// what the root decision of a target panel needs of its record
template <class R>
struct PtRoot {
  R cx, cy, cz, lim;
  RootLim rl;
  float area;
  __device__ __forceinline__ explicit PtRoot(const float4* s) : area(s[4].y) {
    R gx, gy, gz, gs;
    panel_root<R>(s, gx, gy, gz, gs, cx, cy, cz, lim, rl);
  }
};

// the staged particles 0 .. cnt - 1 ({x, y, z}, {alpha} in turn; numbered from p0) on this
// lane's panel: the pairs that are leaves at the root are added to sums, the
// particles of the others counted in listed and, with LIST, the first PTPAN_CAP noted in ent
template <int PREC, bool LIST, class R>
__device__ __forceinline__ void ptpan_root_tile(const float4* shs, int cnt, int64_t p0, const PtRoot<R>& t, int maxlev,
                                                bool active, R* sums, int32_t* ent, int& listed) {
  R acc[3] = {sums[0], sums[1], sums[2]};   // local copies stay in registers
  int nnear = listed;
  // the root decision of particle j of the tile: a leaf is evaluated, a recursed
  // pair listed
  auto pair = [&](const float4 P, const float4 A, int j) {
    if (root_leaf<R>(P.x, P.y, P.z, t.cx, t.cy, t.cz, t.lim, t.rl, maxlev, active)) {
      if (!active) return;
      R ax, ay, az;
      if (PREC == PREC_FP64) {
#pragma clang fp contract(off)
        const R ar = t.area;
        ax = (R(A.x) / ar) * ar; ay = (R(A.y) / ar) * ar; az = (R(A.z) / ar) * ar;
      } else {
        ax = A.x; ay = A.y; az = A.z;
      }
      leaf_acc<R, false>(P.x, P.y, P.z, t.cx, t.cy, t.cz, ax, ay, az, R(0), acc);
    } else if (active) {
      if (LIST && nnear < PTPAN_CAP) ent[nnear] = (int32_t)(p0 + j);
      ++nnear;
    }
  };
  int j = 0;
  if constexpr (sizeof(R) == 4) {
    // PTPAN_UNROLL particles at a time while they are surely beyond every lane's
    // far band: one scalar branch on the OR of the ballots, the leaves with no
    // per-pair mask, the LDS address in a vector register (made so by an opaque
    // zero); the same leaves in the same order as the per-pair path, and an idle
    // lane's sums are dropped
    int vz;
    asm volatile("v_mov_b32 %0, 0" : "=v"(vz));
    const float4* q = shs + vz;
    for (; j + PTPAN_UNROLL <= cnt; j += PTPAN_UNROLL, q += 2 * PTPAN_UNROLL) {
      float4 P[PTPAN_UNROLL], A[PTPAN_UNROLL];
      uint64_t near = 0;
#pragma unroll
      for (int u = 0; u < PTPAN_UNROLL; ++u) {
        P[u] = q[2 * u];
        A[u] = q[2 * u + 1];
        const float ex = P[u].x - t.cx, ey = P[u].y - t.cy, ez = P[u].z - t.cz;
        near |= __builtin_amdgcn_ballot_w64(!(fmaf(ez, ez, fmaf(ey, ey, ex * ex)) > t.rl.far2));
      }
      if (near == 0) {
#pragma unroll
        for (int u = 0; u < PTPAN_UNROLL; ++u)
          leaf_acc<R, false>(P[u].x, P[u].y, P[u].z, t.cx, t.cy, t.cz, A[u].x, A[u].y, A[u].z, R(0), acc);
      } else {
#pragma unroll
        for (int u = 0; u < PTPAN_UNROLL; ++u) pair(P[u], A[u], j + u);
      }
    }
  }
  for (; j < cnt; ++j) pair(shs[2 * j], shs[2 * j + 1], j);
  sums[0] = acc[0]; sums[1] = acc[1]; sums[2] = acc[2];
  listed = nnear;
}

}  // namespace o3d

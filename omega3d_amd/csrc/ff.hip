// ff.hip -- host side of the factored far-field evaluation (method "factored").
//
// One call enqueues, on the caller's stream and without synchronising:
//   bounding boxes and medians -> Hilbert keys -> radix sort (sort.hip) of sources (and of
//   targets when they are a different collection) -> sorted float4 rows, bounding spheres
//   and limits of source tiles and target blocks -> far/near bit per (block, tile) ->
//   near-field plan -> far-field kernel (matrix cores) -> near-field kernel -> combine, which
//   adds the parts and accumulates into the caller's arrays.
// Scratch lives in one device workspace per stream (calls on one stream are
// ordered, so they can share it); it grows when a larger call comes, after the
// stream has drained.  A caller that owns its scratch (a batch) passes it in
// instead, sized by ff_workspace_bytes.
#include "ff_kernels.hpp"
#include "o3d_api_internal.hpp"

#include <algorithm>
#include <climits>
#include <map>
#include <mutex>

namespace o3d {
namespace {

struct Work {
  void* p = nullptr;
  size_t bytes = 0;
};
std::mutex g_ws_mu;
std::map<hipStream_t, Work> g_ws;

// workgroups of the persistent near-field kernel: every slot of every CU
template <int CORE, bool GRAD, int PREC>
int64_t near_grid(size_t lds) {
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_ff_near<CORE, GRAD, PREC>, FF_TB, lds) != hipSuccess ||
      per_cu < 1)
    per_cu = 1;
  return (int64_t)per_cu * num_cus();
}

// RAII pair of events for the optional stage timing
struct Ev {
  hipEvent_t e = nullptr;
  ~Ev() { if (e) (void)hipEventDestroy(e); }
};

bool same_points(const o3d_points* src, const o3d_points* targ) {
  return src->n == targ->n && src->x[0] == targ->x[0] && src->x[1] == targ->x[1] && src->x[2] == targ->x[2];
}

// scratch of the radix sort of one call
size_t lib_tmp_bytes(int64_t ns, int64_t nt, bool same) { return radix_tmp_bytes(same ? ns : ns + nt); }

// the workspace's sub-arrays in order; with base == nullptr only .bytes is meaningful
struct Layout {
  unsigned *k_in, *k_out, *mask, *ctr;
  int *i_in, *i_out, *tinv, *nn, *items, *ioff, *mfold;
  void* tmp;
  float4 *sp, *sa, *tq, *tsph, *tlim, *bsph, *blim;
  float* box;
  double *farv, *part;
  unsigned long long* npair;
  size_t bytes;
};

Layout layout(char* base, int64_t ns, int64_t nt, bool same, int T, size_t tmp_bytes, int nout) {
  const int64_t nb = (nt + FF_TB - 1) / FF_TB;
  const int64_t ntiles = (ns + T - 1) / T;
  const int64_t mwords = (ntiles + 31) / 32;
  Carve cv{base};
  Layout L{};
  const int64_t n = same ? ns : ns + nt;
  L.box = cv.take<float>(FF_BOX_FLOATS);
  L.k_in = cv.take<unsigned>(n);
  L.k_out = cv.take<unsigned>(n);
  L.i_in = cv.take<int>(n);
  L.i_out = cv.take<int>(n);
  L.tinv = cv.take<int>(nt);
  L.tmp = cv.take<char>(tmp_bytes);
  L.sp = cv.take<float4>((size_t)ntiles * T);
  L.sa = cv.take<float4>((size_t)ntiles * T);
  L.tq = cv.take<float4>(nt);
  L.tsph = cv.take<float4>(ntiles);
  L.tlim = cv.take<float4>(ntiles);
  L.bsph = cv.take<float4>(nb);
  L.blim = cv.take<float4>(nb);
  L.mask = cv.take<unsigned>((size_t)(nb * mwords));
  L.farv = cv.take<double>((size_t)nout * far_slices(nb, ntiles, nout == 3 ? 3 : 2, num_cus()) * nt);
  L.npair = cv.take<unsigned long long>(1);
  L.nn = cv.take<int>(nb);
  L.items = cv.take<int>(nb);
  L.ioff = cv.take<int>(nb);
  L.mfold = cv.take<int>(1);
  L.ctr = cv.take<unsigned>(1);
  L.part = cv.take<double>((size_t)(near_split(nb, ntiles) + 1) * nb * nout * FF_TB);
  L.bytes = cv.off;
  return L;
}

// ws == nullptr: the stream's own workspace (caller holds g_ws_mu); otherwise the
// caller's, of ws_bytes
template <int CORE, bool THICK, bool GRAD, int PREC>
int run(const o3d_points* src, o3d_points* targ, bool self_excl, int T, hipStream_t st, o3d_factored_profile* prof,
        void* ws, size_t ws_bytes) {
  const int64_t ns = src->n, nt = targ->n;
  const bool same = same_points(src, targ);
  const int64_t nb = (nt + FF_TB - 1) / FF_TB;
  const int ntiles = (int)((ns + T - 1) / T);
  const int mwords = (ntiles + 31) / 32;

  const size_t tmp_bytes = lib_tmp_bytes(ns, nt, same);

  Layout L = layout(nullptr, ns, nt, same, T, tmp_bytes, GRAD ? 12 : 3);
  char* base = static_cast<char*>(ws);
  if (ws) {
    if (ws_bytes < L.bytes) return fail(O3D_EINVAL, "factored path: workspace of %zu bytes, %zu needed", ws_bytes, L.bytes);
  } else {
    void* p = nullptr;
    int rc = stream_workspace(st, L.bytes, &p);
    if (rc != O3D_OK) return rc;
    base = static_cast<char*>(p);
  }
  L = layout(base, ns, nt, same, T, tmp_bytes, GRAD ? 12 : 3);

  SrcView sv{src->x[0], src->x[1], src->x[2], src->r, src->s[0], src->s[1], src->s[2]};
  TgtView tv{};
  tv.x = targ->x[0]; tv.y = targ->x[1]; tv.z = targ->x[2]; tv.r = targ->r;
  tv.u = targ->u[0]; tv.v = targ->u[1]; tv.w = targ->u[2];
  for (int k = 0; k < 9; ++k) tv.g[k] = GRAD ? targ->ug[k] : nullptr;

  Ev ev[4];
  if (prof) {
    for (auto& e : ev) HIPCHK(hipEventCreate(&e.e));
    HIPCHK(hipEventRecord(ev[0].e, st));
  }
  FFSets sets{};
  sets.x[0] = sv.x; sets.y[0] = sv.y; sets.z[0] = sv.z; sets.n[0] = ns;
  sets.x[1] = tv.x; sets.y[1] = tv.y; sets.z[1] = tv.z; sets.n[1] = same ? 0 : nt;
  const int* perm = nullptr;
  int rc = factored_order(sets, L.box, L.k_in, L.i_in, L.k_out, L.i_out, L.tmp, st, &perm);
  if (rc != O3D_OK) return rc;
  const int *sperm = perm, *tperm = same ? perm : perm + ns;
  const FFBounds tb{L.tsph, L.tlim}, bb{L.bsph, L.blim};
  hipLaunchKernelGGL((k_ff_rows<CORE, THICK>), dim3((unsigned)(ntiles + nb)), dim3(256), 0, st, sv, tv, sperm, tperm, ns,
                     nt, T, ntiles, L.sp, L.sa, L.tq, tb, bb, L.nn, nt >= FF_ROWS_MIN ? L.tinv : nullptr);
  hipLaunchKernelGGL((k_ff_classify<CORE>), dim3(grid_of(nb * mwords, 256)), dim3(256), 0, st, bb, nb, tb, ntiles, mwords,
                     L.mask, L.nn);
  hipLaunchKernelGGL(k_ff_plan, dim3(1), dim3(FF_PLAN_THREADS), 0, st, L.nn, nb, near_split(nb, ntiles), L.items, L.ioff,
                     L.mfold, L.ctr, (unsigned*)nullptr);
  HIPCHK(hipGetLastError());

  FFArgs a{};
  a.sp = L.sp; a.sa = L.sa; a.tq = L.tq; a.tperm = tperm; a.tinv = L.tinv; a.rows = nt >= FF_ROWS_MIN;
  a.tsph = L.tsph; a.tlim = L.tlim; a.bsph = L.bsph; a.blim = L.blim;
  a.mask = L.mask; a.farv = L.farv;
  a.nn = L.nn; a.items = L.items; a.ioff = L.ioff; a.mfold = L.mfold; a.ctr = L.ctr; a.part = L.part;
  a.s = sv; a.t = tv;
  a.ns = ns; a.nt = nt;
  a.tile = T; a.mwords = mwords; a.ntiles = ntiles;
  a.self_excl = self_excl ? 1 : 0;
  const bool fine = PREC == PREC_COMP && (a.ns < FF_FINE_BELOW || a.nt < FF_FINE_BELOW);
  a.merge = fine ? FF_FINE_MERGE : ff_merge<CORE, GRAD>();
  a.fold = fine ? FF_FINE_FOLD : ff_fold<CORE, GRAD>();
  const int nslice = far_slices(nb, ntiles, GRAD ? 2 : 3, num_cus());
  a.tslice = (ntiles + nslice - 1) / nslice;
  a.nslice = (ntiles + a.tslice - 1) / a.tslice;
  const size_t lds_far = ff_far_lds<CORE, GRAD>();
  if (prof) HIPCHK(hipEventRecord(ev[1].e, st));
  hipLaunchKernelGGL((k_ff_far<CORE, GRAD>), dim3((unsigned)nb, (unsigned)a.nslice), dim3(FF_FAR_THREADS), lds_far, st, a);
  HIPCHK(hipGetLastError());
  if (prof) HIPCHK(hipEventRecord(ev[2].e, st));
  const size_t lds_near = (size_t)T * 2 * sizeof(float4);
  const unsigned gnear = (unsigned)std::min<int64_t>((near_split(nb, ntiles) + 1) * nb, near_grid<CORE, GRAD, PREC>(lds_near));
  hipLaunchKernelGGL((k_ff_near<CORE, GRAD, PREC>), dim3(gnear), dim3(FF_TB), lds_near, st, a);
  HIPCHK(hipGetLastError());
  if (a.rows) hipLaunchKernelGGL((k_ff_combine<CORE, GRAD, true>), dim3((unsigned)nb), dim3(FF_TB), 0, st, a);
  else hipLaunchKernelGGL((k_ff_combine<CORE, GRAD, false>), dim3((unsigned)nb), dim3(FF_TB), 0, st, a);
  HIPCHK(hipGetLastError());
  if (prof) {
    HIPCHK(hipEventRecord(ev[3].e, st));
    hipLaunchKernelGGL(k_ff_zero_u64, dim3(1), dim3(64), 0, st, L.npair);
    hipLaunchKernelGGL(k_ff_count, dim3(grid_of(nb, 256)), dim3(256), 0, st, L.mask, nb, mwords, ntiles, T, ns, nt,
                       L.npair);
    HIPCHK(hipGetLastError());
    unsigned long long far_pairs = 0;
    HIPCHK(hipMemcpyAsync(&far_pairs, L.npair, sizeof far_pairs, hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    float ms[3];
    for (int k = 0; k < 3; ++k) HIPCHK(hipEventElapsedTime(&ms[k], ev[k].e, ev[k + 1].e));
    prof->prep_ms = ms[0];
    prof->far_ms = ms[1];
    prof->near_ms = ms[2];
    prof->total_ms = (double)ms[0] + ms[1] + ms[2];
    prof->far_pairs = (double)far_pairs;
    prof->pairs = (double)ns * (double)nt;
    prof->far_tile_fraction = 0.0;
    if (nb > 0 && ntiles > 0) prof->far_tile_fraction = prof->far_pairs / prof->pairs;
  }
  return O3D_OK;
}

// plain FP32 sums come here for the cores and results that the method FACTORED serves;
// the others only in compensated precision
template <int CORE, bool GRAD>
int run_core(const o3d_points* src, o3d_points* targ, bool thick, int prec, bool self_excl, int T, hipStream_t st,
             o3d_factored_profile* prof, void* ws, size_t wsb) {
  if (prec == PREC_COMP)
    return thick ? run<CORE, true, GRAD, PREC_COMP>(src, targ, self_excl, T, st, prof, ws, wsb)
                 : run<CORE, false, GRAD, PREC_COMP>(src, targ, self_excl, T, st, prof, ws, wsb);
  if constexpr (GRAD && (CORE == CORE_RM || CORE == CORE_EXP))
    return thick ? run<CORE, true, GRAD, PREC_FP32>(src, targ, self_excl, T, st, prof, ws, wsb)
                 : run<CORE, false, GRAD, PREC_FP32>(src, targ, self_excl, T, st, prof, ws, wsb);
  return fail(O3D_EINVAL, "internal: plain FP32 sums of core %d routed to the factored path", CORE);
}

}  // namespace

// the order of one or two sets along the curve: *perm gets the first set's permutation and
// the second's after it.  box, keys and indices in the caller's scratch
int factored_order(const FFSets& s, float* box, unsigned* ka, int* va, unsigned* kb, int* vb, void* tmp, hipStream_t st,
                   const int** perm) {
  const int64_t n = s.n[0] + s.n[1];
  const int bits = key_bits(n, s.n[1] > 0);
  const unsigned g = std::min<unsigned>(FF_BOX_GRID, grid_of(n, 1024));
  float* where = box + 12 * FF_BOX_GRID;
  hipLaunchKernelGGL(k_ff_box, dim3(g + 2), dim3(256), 0, st, s, box, (int)g, where);
  hipLaunchKernelGGL(k_ff_hkeys, dim3(std::min(1024u, grid_of(n, 256))), dim3(256), 0, st, s, box, (int)g, where,
                     s.n[1] > 0 ? bits - 1 : bits, ka, va);
  HIPCHK(hipGetLastError());
  unsigned* keys = nullptr;
  int* vals = nullptr;
  const int rc = radix_sort_pairs(ka, va, kb, vb, n, bits, tmp, st, &keys, &vals);
  *perm = vals;
  return rc;
}

// Morton order of n points (the direct kernel's target order): workspace bytes,
// and the order itself, written into ws (bounding box, keys, indices and the
// sort's scratch; *perm points into ws)
size_t point_order_bytes(int64_t n) {
  const size_t a = (sizeof(int32_t) * (size_t)n + 255) & ~(size_t)255;
  return 256 + 4 * a + ((radix_tmp_bytes(n) + 255) & ~(size_t)255);
}

int point_order(const float* x, const float* y, const float* z, int64_t n, void* ws, hipStream_t st,
                const int32_t** perm, const unsigned** keys) {
  const size_t a = (sizeof(int32_t) * (size_t)n + 255) & ~(size_t)255;
  char* p = (char*)ws;
  unsigned* bb = (unsigned*)p;
  unsigned* kin = (unsigned*)(p + 256);
  unsigned* kout = (unsigned*)(p + 256 + a);
  int* iin = (int*)(p + 256 + 2 * a);
  int* iout = (int*)(p + 256 + 3 * a);
  void* tmp = p + 256 + 4 * a;
  hipLaunchKernelGGL(k_ff_bbox_init, dim3(1), dim3(64), 0, st, bb);
  hipLaunchKernelGGL(k_ff_bbox, dim3(std::min(grid_of(n, 256), FF_BBOX_GRID)), dim3(256), 0, st, x, y, z, n, bb);
  hipLaunchKernelGGL(k_ff_keys, dim3(grid_of(n, 256)), dim3(256), 0, st, x, y, z, n, bb, kin, iin);
  HIPCHK(hipGetLastError());
  unsigned* sk = nullptr;
  int* sp = nullptr;
  const int rc = radix_sort_pairs(kin, iin, kout, iout, n, 30, tmp, st, &sk, &sp);
  if (rc != O3D_OK) return rc;
  *perm = sp;
  if (keys) *keys = sk;
  return O3D_OK;
}

bool ff_same_points(const o3d_points* src, const o3d_points* targ) { return same_points(src, targ); }

// Sources of a direct EXP call as rows sorted by perm (the targets' Morton order of
// the same collection), and each tile's bounding sphere and largest core term, in
// ws (sorted_sources_bytes) after the point order's own point_order_bytes(n)
size_t sorted_sources_bytes(int64_t n, int tile) {
  const size_t ntiles = (size_t)((n + tile - 1) / tile);
  const auto r = [](size_t b) { return (b + 255) & ~(size_t)255; };
  return 2 * r(sizeof(float4) * (size_t)n) + r(sizeof(float4) * ntiles) + r(sizeof(float) * ntiles);
}

int sorted_sources(const o3d_points* src, const int32_t* perm, int tile, void* ws, hipStream_t st, P2PArgs* a) {
  const int64_t n = src->n;
  const int ntiles = (int)((n + tile - 1) / tile);
  const auto r = [](size_t b) { return (b + 255) & ~(size_t)255; };
  char* p = (char*)ws;
  float4* sp = (float4*)p;
  float4* sa = (float4*)(p + r(sizeof(float4) * (size_t)n));
  float4* sph = (float4*)(p + 2 * r(sizeof(float4) * (size_t)n));
  float* cs = (float*)(p + 2 * r(sizeof(float4) * (size_t)n) + r(sizeof(float4) * (size_t)ntiles));
  const SrcView sv{src->x[0], src->x[1], src->x[2], src->r, src->s[0], src->s[1], src->s[2]};
  hipLaunchKernelGGL((k_ff_gather_src<CORE_EXP>), dim3(grid_of(n, 256)), dim3(256), 0, st, sv, perm, n, sp, sa);
  hipLaunchKernelGGL(k_ff_bounds, dim3((unsigned)ntiles), dim3(256), 0, st, (const float4*)sp, n, tile, sph, cs);
  HIPCHK(hipGetLastError());
  a->sp = sp;
  a->sa = sa;
  a->tsph = sph;
  a->tcs = cs;
  return O3D_OK;
}

std::mutex& stream_ws_mutex() { return g_ws_mu; }

// caller holds stream_ws_mutex() for the whole enqueue, so that no other thread
// frees or grows this stream's workspace between its sizing and the last launch
// using it; a larger request waits for the stream to drain, then reallocates.  A
// stream being captured into a graph cannot do that: the workspace must already
// be large enough (a call of the same size outside the capture sizes it).
bool stream_capturing(hipStream_t st) {
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  return hipStreamIsCapturing(st, &cs) == hipSuccess && cs != hipStreamCaptureStatusNone;
}

bool stream_workspace_fits(hipStream_t st, size_t bytes) {
  auto it = g_ws.find(st);
  return it != g_ws.end() && it->second.bytes >= bytes;
}

void release_stream_workspace(hipStream_t st) {
  std::lock_guard<std::mutex> lk(g_ws_mu);
  auto it = g_ws.find(st);
  if (it == g_ws.end()) return;
  if (it->second.p) {
    (void)hipStreamSynchronize(st);
    (void)hipFree(it->second.p);
  }
  g_ws.erase(it);
}

int stream_workspace(hipStream_t st, size_t bytes, void** out) {
  Work& w = g_ws[st];
  if (w.bytes < bytes) {
    if (stream_capturing(st))
      return fail(O3D_EINVAL, "the stream is being captured and its device workspace would have to grow to %zu "
                              "bytes; make the same call once outside the capture first", bytes);
    if (w.p) {
      HIPCHK(hipStreamSynchronize(st));
      HIPCHK(hipFree(w.p));
      w.p = nullptr;
      w.bytes = 0;
    }
    const size_t want = bytes + bytes / 4;
    if (hipMalloc(&w.p, want) != hipSuccess) {
      w.p = nullptr;
      return fail(O3D_ENOMEM, "device workspace of %zu bytes: allocation failed", want);
    }
    w.bytes = want;
  }
  *out = w.p;
  return O3D_OK;
}

bool ff_supported(int core, bool grad, int prec) {
  return (core == CORE_RM || core == CORE_EXP) && grad && (prec == PREC_FP32 || prec == PREC_COMP);
}

// AUTO also sends compensated sums of the other cores and of velocities alone.  The line is
// drawn in pairs, where both methods' times cross, us direct and factored on one or two
// rings (particles that fill a cube cross later, having more near tiles: RM 30,100 720-770 and
// 841, 40,000 1,161 and 1,116; EXP velocity alone and WL about 5% at their lines): EXP 24,576
// particles 600-630 and 505; RM 24,576 452 and 468, 32,768 750 and 570-645; WL (V2 alike) 32,768 829 and 798-869, 49,152 1,833 and 1,573-1,641; velocity alone: EXP
// 24,576 376-396 and 410-420, 32,768 675 and 493-562, RM 32,768 441 and 456-504, 49,152 980
// and 830-884, WL 49,152 1,105 and 1,063-1,125, 65,536 faster.  100,000 particles on 16,384
// field points and 8,192 on 262,144 fall on the same lines (less the preparation's recent
// 0.07 ms: RM 1,134 and 1,064, 1,416 and 1,235; WL 1,235 and 1,402, 1,561 and 1,667), 2,048
// on 262,144 not (EXP 631 and 645), nor do fewer targets.  Below FF_FEW_TARGETS the far kernel's
// blocks are few, and a single ring crosses at 1.5 to 1.75 times the pairs: EXP 80,000 on 8,500
// 583 and 596, 150,000 1,028 and 956; WL 240,000 1,571 and 1,670; velocity alone: RM 260,000 927
// and 951, 400,000 1,386 and 1,391, EXP 120,000 520 and 581, 240,000 1,038 and 998.  RM with
// gradient keeps its line there: 110,000 on 9,000 720 and 774 from one ring, 722 and 685 from two
constexpr int64_t FF_FEW_TARGETS = 16384;
// Plain FP32 sums from here on only: below, the far field is faster (RM 40,000 particles 1,162
// and 796 us, EXP 28,672 1,227 and 584), but its near tiles are one FP32 sum where the direct
// kernel adds slices: rms error of the velocity on one ring RM 30,100 0.99e-7 and 1.7e-7, 49,152
// 1.6e-7 and 2.1e-7, 65,000 2.2e-7 and 2.3e-7; EXP 28,672 1.0e-7 and 2.0e-7; 40,000 EXP
// particles on as many points in a box five times as wide 1.8e-7 and 3.0e-7
constexpr int64_t FF_FP32_MIN = 65536;
bool ff_auto_pays(int core, bool grad, int prec, int64_t ns, int64_t nt) {
  if (!(prec == PREC_COMP || ff_supported(core, grad, prec))) return false;
  if (ns < 8192 || nt < 8192 || ns > INT_MAX || nt > INT_MAX) return false;
  if (prec == PREC_FP32) return ns >= FF_FP32_MIN && nt >= FF_FP32_MIN;
  const double least = core == CORE_EXP ? (grad ? 6.0e8 : 1.0e9) : core == CORE_RM ? (grad ? 9.0e8 : 2.2e9)
                                                                                 : (grad ? 2.0e9 : 3.0e9);
  return (double)ns * (double)nt >= (nt < FF_FEW_TARGETS && !(core == CORE_RM && grad) ? 1.75 * least : least);
}

namespace {
int check_factored(const o3d_points* src, const o3d_points* targ, const o3d_opts* o, int* T) {
  const bool grad = o->results == O3D_VELANDGRAD;
  if (o->method == O3D_METHOD_FACTORED && !ff_supported(o->core, grad, o->precision))
    return fail(O3D_EINVAL, "factored method: needs the RM or EXP core, velocity and gradient, and FP32 or "
                            "compensated precision");
  if (src->n > INT_MAX || targ->n > INT_MAX)
    return fail(O3D_EINVAL, "factored method: at most %d sources and %d targets", INT_MAX, INT_MAX);
  *T = o->tile > 0 ? o->tile : 256;
  if (*T != 64 && *T != 128 && *T != 256) return fail(O3D_EINVAL, "factored method: tile must be 0, 64, 128 or 256");
  return O3D_OK;
}

template <bool GRAD>
int dispatch_grad(const o3d_points* src, o3d_points* targ, const o3d_opts* o, int T, hipStream_t st,
                  o3d_factored_profile* prof, void* ws, size_t wsb) {
  const bool thick = targ->r != nullptr;
  const bool self_excl = o->self_term == O3D_SELF_EXCLUDE;
  switch (o->core) {
    case CORE_RM: return run_core<CORE_RM, GRAD>(src, targ, thick, o->precision, self_excl, T, st, prof, ws, wsb);
    case CORE_WL: return run_core<CORE_WL, GRAD>(src, targ, thick, o->precision, self_excl, T, st, prof, ws, wsb);
    case CORE_EXP: return run_core<CORE_EXP, GRAD>(src, targ, thick, o->precision, self_excl, T, st, prof, ws, wsb);
    default: return run_core<CORE_V2, GRAD>(src, targ, thick, o->precision, self_excl, T, st, prof, ws, wsb);
  }
}

int dispatch(const o3d_points* src, o3d_points* targ, const o3d_opts* o, int T, hipStream_t st,
             o3d_factored_profile* prof, void* ws, size_t wsb) {
  return o->results == O3D_VELANDGRAD ? dispatch_grad<true>(src, targ, o, T, st, prof, ws, wsb)
                                      : dispatch_grad<false>(src, targ, o, T, st, prof, ws, wsb);
}
}  // namespace

// device-pointer point->point by the factored far field; arguments already checked
int p2p_factored(const o3d_points* src, o3d_points* targ, const o3d_opts* o, hipStream_t st,
                 o3d_factored_profile* prof) {
  int T = 0, rc = check_factored(src, targ, o, &T);
  if (rc != O3D_OK) return rc;
  std::lock_guard<std::mutex> lk(g_ws_mu);
  return dispatch(src, targ, o, T, st, prof, nullptr, 0);
}

// the same on scratch the caller owns (ws_bytes >= ff_workspace_bytes of this shape);
// nothing is allocated and no lock is taken
int p2p_factored_ws(const o3d_points* src, o3d_points* targ, const o3d_opts* o, hipStream_t st, void* ws,
                    size_t ws_bytes) {
  int T = 0, rc = check_factored(src, targ, o, &T);
  if (rc != O3D_OK) return rc;
  if (!ws) return fail(O3D_EINVAL, "factored method: NULL workspace");
  return dispatch(src, targ, o, T, st, nullptr, ws, ws_bytes);
}

size_t ff_workspace_bytes(int64_t ns, int64_t nt, bool same, int tile, bool grad) {
  const int T = tile > 0 ? tile : 256;
  return layout(nullptr, ns, nt, same, T, lib_tmp_bytes(ns, nt, same), grad ? 12 : 3).bytes;
}

}  // namespace o3d

extern "C" int o3d_morton_order_dev(const float* x, const float* y, const float* z, int64_t n, uint32_t* keys,
                                    int32_t* perm, void* stream) {
  using namespace o3d;
  clear_error();
  int rc = ensure_init();
  if (rc != O3D_OK) return rc;
  if (n < 0 || n > INT32_MAX) return fail(O3D_EINVAL, "morton order: n %lld out of range", (long long)n);
  if (n == 0) return O3D_OK;
  if (!x || !y || !z || !keys || !perm) return fail(O3D_EINVAL, "morton order: NULL array");
  hipStream_t st = (hipStream_t)stream;
  std::lock_guard<std::mutex> lk(g_ws_mu);
  void* ws = nullptr;
  if ((rc = stream_workspace(st, point_order_bytes(n), &ws)) != O3D_OK) return rc;
  const int32_t* p = nullptr;
  if ((rc = point_order(x, y, z, n, ws, st, &p)) != O3D_OK) return rc;
  HIPCHK(hipMemcpyAsync(perm, p, sizeof(int32_t) * (size_t)n, hipMemcpyDeviceToDevice, st));
  // the keys in index order, from the same box (point_order left it at the workspace's start)
  hipLaunchKernelGGL(k_ff_keys, dim3(grid_of(n, 256)), dim3(256), 0, st, x, y, z, n, (const unsigned*)ws,
                     (unsigned*)keys, (int*)nullptr);
  HIPCHK(hipGetLastError());
  return O3D_OK;
}

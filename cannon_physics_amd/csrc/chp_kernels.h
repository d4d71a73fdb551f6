// chp_kernels.h -- the kernels of libcannon_hip.so.  The narrowphase resolvers, which take most of
// the compile time, are instantiated in chp_narrow_kernels.hip (one object per precision); every
// other kernel in chp_api.hip.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "../../include/cannon_hip.h"
#include "chp_build.h"
#include "chp_stages.h"
#include "chp_events.h"
#include "chp_query.h"
#include "chp_split.h"

namespace chp {

// One kernel per stage, one workgroup per listed world.  The batched path launches each stage
// once over every world of the batch; the plain path launches them for one world at a time.
#define CHP_WORLD_PROLOGUE                                          \
  const DevWorld<R>& W = worlds[list[blockIdx.x]];                  \
  if (block_bcast(W.counters[C_STATUS], sh) != 0) return;

// gravity / solve mass / AABBs, broadphase and the collideConnected filter.  One kernel per
// broadphase kind (each holds only its code and registers), each skipping the other kind's
// worlds.  Dynamic LDS holds the broadphase data of worlds of at most lds_nb bodies.  The pairs
// are then counted by narrowphase class (qw: the queue's words; null: the Broadphase slot, the
// pairs alone).
template <typename R, bool SAP>
__global__ __launch_bounds__(1024) void k_bp(const DevWorld<R>* __restrict__ worlds, const int* __restrict__ list,
                                             int lds_nb, int* __restrict__ qw, int wcc) {
  __shared__ int sh[32];
  extern __shared__ float4 lds_bp[];
  const DevWorld<R>& W = worlds[list[blockIdx.x]];
  if (qw && block_bcast(W.counters[C_STATUS], sh) != 0) return;
  if ((W.broadphase == CHP_BROADPHASE_SAP) != SAP) return;
  if (qw && threadIdx.x == 0) {
    W.counters[C_STAGING] = 0;
    if (W.ev_mask) W.ev_ctl[EV_JT] = 0;
  }
  if (W.nb > lds_nb) return;  // the grid-wide kernels below take large worlds
  if (qw) {
    st_prestep<R, SAP>(W);
  } else if (SAP) {
    for (int i = threadIdx.x; i < W.nb; i += blockDim.x)
      if (W.flags[i] & BF_AABB_DIRTY) { body_aabb(W, i); W.flags[i] &= ~BF_AABB_DIRTY; }
  }
  __syncthreads();
  BpLds<R> L;
  L.carve(lds_bp, lds_nb, SAP);
  bool ok;
  if constexpr (SAP) ok = st_bp_sap(W, sh, L);
  else ok = st_bp_naive(W, sh, L);
  if (!ok || !qw) return;
  st_filter(W);
  st_narrow_count(W, qw, (int)blockIdx.x, wcc != 0, sh);
}

// large worlds (at least BP_BIG bodies): prestep, SAP sort and pair passes over the grid.
// spans: (list index, first row) per BP_SPAN rows; tiles: (list index, first position) per
// SAP_TILE keys of the SAP worlds; bigw: list indices of the large worlds.
#define CHP_SPAN_PROLOGUE(tab)                                      \
  const int2 sp = tab[blockIdx.x];                                  \
  const DevWorld<R>& W = worlds[list[sp.x]];                        \
  if (W.counters[C_STATUS] != 0) return;

template <typename R>
__global__ __launch_bounds__(64) void k_big_prestep(const DevWorld<R>* __restrict__ worlds, const int* __restrict__ list,
                                                    const int2* __restrict__ spans) {
  CHP_SPAN_PROLOGUE(spans)
  const int i = sp.y + threadIdx.x;
  if (i < W.nb) prestep_body(W, i);
}
template <typename R>
__global__ __launch_bounds__(256) void k_sap_tile(const DevWorld<R>* __restrict__ worlds, const int* __restrict__ list,
                                                  const int2* __restrict__ tiles, int apply) {
  __shared__ unsigned long long lk[SAP_TILE];
  __shared__ int lord[SAP_TILE];
  CHP_SPAN_PROLOGUE(tiles)
  sap_tile(W, sp.y, lk, lord, apply != 0);
}
template <typename R>
__global__ __launch_bounds__(64) void k_sap_merge(const DevWorld<R>* __restrict__ worlds, const int* __restrict__ list,
                                                  const int2* __restrict__ spans, int w, int src, int apply) {
  CHP_SPAN_PROLOGUE(spans)
  const int g = sp.y + threadIdx.x;
  if (W.broadphase == CHP_BROADPHASE_SAP && g < W.nb) sap_merge(W, g, w, src, apply != 0);
}
// pass 0 counts the pairs of each row into cnt; pass 1 writes them from the scanned offsets.
// Four workgroups per span, BP_ROWS rows each, one wave per row.
constexpr int BP_ROWS = BP_SPAN / 4;
template <typename R>
__global__ __launch_bounds__(256) void k_big_rows(const DevWorld<R>* __restrict__ worlds, const int* __restrict__ list,
                                                  const int2* __restrict__ spans, int emit) {
  const int2 sp = spans[blockIdx.x >> 2];
  const DevWorld<R>& W = worlds[list[sp.x]];
  if (W.counters[C_STATUS] != 0) return;
  const int r0 = sp.y + BP_ROWS * (int)(blockIdx.x & 3), end = min(r0 + BP_ROWS, W.nb);
  for (int k = r0 + (int)(threadIdx.x >> 6); k < end; k += 4) {
    if (emit) {
      big_row(W, k, true, W.cnt[k]);
    } else {
      int c = big_row(W, k, false, 0);
      if ((threadIdx.x & 63) == 0) W.cnt[k] = c;
    }
  }
}
template <typename R>
__global__ __launch_bounds__(1024) void k_big_scan(const DevWorld<R>* __restrict__ worlds, const int* __restrict__ list,
                                                   const int* __restrict__ bigw) {
  __shared__ int sh[1024];
  const DevWorld<R>& W = worlds[list[bigw[blockIdx.x]]];
  if (block_bcast(W.counters[C_STATUS], sh) != 0) return;
  const int P = array_exscan(W.cnt, W.nb, sh);
  if (threadIdx.x == 0) {
    W.counters[C_PAIRS] = P;
    if (P > W.pair_cap) ws_fail(W.counters, WS_PAIRS);
  }
}

// narrowphase class counts and queue placement of a large world's pairs: the world's spans are
// its K workers, worker k takes pairs k * 256 + t, stride K * 256.  Counts add into the class
// totals; placement reserves each class range per workgroup.
template <typename R>
__device__ __forceinline__ void big_pair_classes(const DevWorld<R>& W, int2 sp, int* sh, bool wcc, bool mark_filtered) {
  const int K = (W.nb + BP_SPAN - 1) / BP_SPAN, k = sp.y / BP_SPAN, P = W.counters[C_PAIRS];
  for (int p = k * 256 + (int)threadIdx.x; p < P; p += K * 256) {
    int bi = W.pair_i[p], bj = W.pair_j[p];
    if (bi < 0) {
      if (mark_filtered) pair_counts(W, p, 0, 0);
      continue;
    }
    atomicAdd(&sh[pair_class(W, bi, bj, wcc)], 1);
  }
}
template <typename R>
__global__ __launch_bounds__(256) void k_big_ncount(const DevWorld<R>* __restrict__ worlds, const int* __restrict__ list,
                                                    const int2* __restrict__ spans, int* __restrict__ qw, int wcc) {
  __shared__ int sh[NP_NCLS];
  CHP_SPAN_PROLOGUE(spans)
  if (threadIdx.x < NP_NCLS) sh[threadIdx.x] = 0;
  __syncthreads();
  big_pair_classes(W, sp, sh, wcc != 0, true);
  __syncthreads();
  if (threadIdx.x < NP_NCLS && sh[threadIdx.x]) atomicAdd(&qw[QW_TOT + threadIdx.x], sh[threadIdx.x]);
}
template <typename R>
__global__ __launch_bounds__(256) void k_big_nplace(const DevWorld<R>* __restrict__ worlds, const int* __restrict__ list,
                                                    const int2* __restrict__ spans, int* __restrict__ qw,
                                                    int2* __restrict__ q, int wcc) {
  __shared__ int sh[NP_NCLS];
  CHP_SPAN_PROLOGUE(spans)
  if (threadIdx.x < NP_NCLS) sh[threadIdx.x] = 0;
  __syncthreads();
  big_pair_classes(W, sp, sh, wcc != 0, false);
  __syncthreads();
  if (threadIdx.x < NP_NCLS)
    sh[threadIdx.x] = sh[threadIdx.x] ? queue_base(qw) + atomicAdd(&qw[QW_CUR + threadIdx.x], sh[threadIdx.x]) : 0;
  __syncthreads();
  const int K = (W.nb + BP_SPAN - 1) / BP_SPAN, k = sp.y / BP_SPAN, P = W.counters[C_PAIRS], wid = list[sp.x];
  for (int p = k * 256 + (int)threadIdx.x; p < P; p += K * 256) {
    int bi = W.pair_i[p], bj = W.pair_j[p];
    if (bi < 0) continue;
    q[atomicAdd(&sh[pair_class(W, bi, bj, wcc)], 1)] = make_int2(wid, p);
  }
}

// rows of a large world: the offsets and counters in one workgroup per world, then the rows of
// its pairs and constraints over its spans (worker k of K as above)
template <typename R>
__global__ __launch_bounds__(1024) void k_big_rowscan(const DevWorld<R>* __restrict__ worlds, const int* __restrict__ list,
                                                      const int* __restrict__ bigw) {
  __shared__ int sh[1024];
  const DevWorld<R>& W = worlds[list[bigw[blockIdx.x]]];
  if (block_bcast(W.counters[C_STATUS], sh) != 0) return;
  const int P = W.counters[C_PAIRS];
  const int F = array_exscan(W.pf_cnt, P, sh);
  const int C = array_exscan(W.pc_off, P, sh);
  const int E = F + C + W.ncrows;
  if (threadIdx.x == 0) {
    if (E > W.row_cap) {
      W.counters[C_ROWS] = E;
      ws_fail(W.counters, WS_ROWS);
    } else {
      rows_done(W, P, F, C, E);
    }
  }
}


// integration of a large world's bodies over its spans; a non-finite pose is noted in
// C_POSTFAIL and raised by k_post, which also advances the step counter
template <typename R>
__global__ __launch_bounds__(64) void k_big_post(const DevWorld<R>* __restrict__ worlds, const int* __restrict__ list,
                                                 const int2* __restrict__ spans, double dt) {
  CHP_SPAN_PROLOGUE(spans)
  const int i = sp.y + threadIdx.x;
  if (i < W.nb && !post_body(W, i, (R)dt, W.counters[C_ROWS], post_qn(W))) W.counters[C_POSTFAIL] = 1;
}

// narrowphase: the pairs placed in the queue by class (the counts are the broadphase's), then one
// pair per thread over the thread classes and one pair per wave over the wave class, each
// grid-wide over the whole batch.
template <typename R>
__global__ __launch_bounds__(256) void k_narrow(const DevWorld<R>* __restrict__ worlds, const int* __restrict__ list,
                                                int* __restrict__ qw, int2* __restrict__ q, int wcc) {
  __shared__ int sh[64];
  if (blockIdx.x == 0) queue_bounds(qw);
  CHP_WORLD_PROLOGUE
  if (W.nb >= BP_BIG) return;  // k_big_nplace
  st_narrow_place(W, list[blockIdx.x], qw, (int)blockIdx.x, wcc != 0, q, sh);
}
// LDS of the 64 lanes of a thread class, in f3: the clip polygons of convex-convex (and the mixed
// class), the side vectors of sphere-box
constexpr int cls_lds(int c) { return c == NP_CC || c == NP_OTHER ? 2 * CLIP_THREAD * 64 : c == NP_SB ? 6 * 64 : 1; }
template <typename R, int CLS>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void k_narrow_cls(const DevWorld<R>* __restrict__ worlds, const int2* __restrict__ q,
                                                   const int* __restrict__ bounds, double dt) {
  __shared__ f3 cb[cls_lds(CLS)];
  st_narrow_class<R, CLS>(worlds, q, bounds, (R)dt, cb);
}
template <typename R>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void k_narrow_threads(const DevWorld<R>* __restrict__ worlds,
                                                     const int2* __restrict__ q, const int* __restrict__ bounds, double dt) {
  __shared__ f3 cb[cls_lds(NP_SB)];
  st_narrow_threads<R>(worlds, q, bounds, (R)dt, cb);
}
template <typename R, int CLS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_narrow_wave(const DevWorld<R>* __restrict__ worlds, const int2* __restrict__ q,
                                                     int* __restrict__ bounds, double dt, int clip_cap) {
  __shared__ f3 ws[4][NPCtx<R, true>::WS_F3];            // one LDS workspace per wave
  __shared__ ContactRec<R> loc[4][WAVE_KMAX];             // and one contact buffer
  constexpr unsigned kinds = CLS == NP_WHC ? (NK_CC | NK_HC | NK_SH) : NK_ALL;
  st_narrow_wave<R, kinds>(worlds, q + bounds[CLS], bounds[CLS + 1] - bounds[CLS], bounds + NP_NCLS + 1 + (CLS - NP_WHC),
                           (R)dt, ws[threadIdx.x >> 6],
                           loc[threadIdx.x >> 6], WAVE_KMAX, clip_cap);
}


// equations: the row offsets per world (large worlds: k_big_rowscan), then the friction and
// contact rows of every queued pair (one pair per thread over the whole batch), then the joint
// rows (one workgroup per world)
template <typename R>
__global__ __launch_bounds__(128) void k_rows(const DevWorld<R>* __restrict__ worlds, const int* __restrict__ list,
                                              int* __restrict__ qw) {
  __shared__ int sh[128];
  if (blockIdx.x == 0 && threadIdx.x < 2 * NP_NCLS) qw[QW_TOT + threadIdx.x] = 0;   // totals and cursors of the next step
  CHP_WORLD_PROLOGUE
  if (W.nb >= BP_BIG) return;
  st_rowscan(W, sh);
}
// MODE ROWS_AB: the rows' body pairs only (before the level schedule); ROWS_GS: the rows
// themselves, as GS records at their level-order positions (after it)
template <typename R, int MODE>
__global__ __launch_bounds__(64) void k_pair_rows(const DevWorld<R>* __restrict__ worlds, const int2* __restrict__ q,
                                                  const int* __restrict__ bounds, double dt, int keep) {
  const int n = bounds[NP_NCLS];
  const int g = (int)(blockIdx.x * blockDim.x + threadIdx.x), ng = (int)(gridDim.x * blockDim.x);
  for (int i = g; i < n; i += ng) {
    const int2 e = q[i];
    const DevWorld<R>& W = worlds[e.x];
    if (W.counters[C_STATUS] != 0) continue;
    pair_rows<R, MODE>(W, e.y, W.counters[C_FROWS], (R)dt, keep != 0);
  }
}
template <typename R, int MODE>
__global__ __launch_bounds__(64) void k_joint_rows(const DevWorld<R>* __restrict__ worlds, const int* __restrict__ list,
                                                   double dt, int keep) {
  const DevWorld<R>& W = worlds[list[blockIdx.x]];
  if (W.ncons == 0 || W.counters[C_STATUS] != 0) return;
  const int F = W.counters[C_FROWS], C = W.counters[C_CROWS];
  for (int c = threadIdx.x; c < W.ncons; c += blockDim.x)
    constraint_rows<R, MODE>(W, c, F + C + W.c_row_off[c], (R)dt, keep != 0);
}

// GS sweeps.  Worlds of at most GS_WAVE_NB bodies run one per wave, four to a workgroup; those of
// at most GS_SUB_MAX_NB one per workgroup of four waves, all of them in one launch; larger ones
// one per workgroup of their own launch.  vlambda / wlambda and the step tables live in LDS where
// they fit.
// Worlds of at most GS_ONE_NB join the second launch while there is a CU for each of its workgroups:
// a list on both sides of GS_SUB_MAX_NB then waits for one launch, not two in turn (24 terrains of
// 16 to 1024 bodies 287 us for 333 + 213), and four waves wait less at a step's barrier than eight
// (600 bodies 137 -> 110 us, 900 159 -> 140, 1000 in double 678 -> 474, a 3000-body pile 914 -> 668;
// of a lattice of 3000 spheres, whose levels are wide, 1186 -> 1230).  At 16,384 bodies, whose
// velocities are not in LDS, eight are better (3.5 ms, four 3.9).
constexpr int GS_SUB_MAX_NB = 512, GS_WAVE_NB = 128, GS_ONE_NB = 4096, GS_ONE_WGS = 256;
constexpr int GS_SS_WAVE = 1024, GS_SS_SUB = 2048, GS_SS_BIG = 4096;   // step table entries in LDS
// ring depth: FP32 4, 6 and 8 measured 1188, 1165 and 1186 us on 1024 chains, 338, 329 and 324 us
// on half a batch of 2048 piles, 60, 62 and 66 us on one 217-body world; FP64 2, 3 and 4 measured
// 251, 211 and 213 us on a 157-body world, 474, 397 and 398 us on 1000 bodies, 645, 398 and 395 us
// on half a batch of 512 piles
template <typename R> constexpr int gs_depth() { return sizeof(R) == 4 ? 6 : 4; }

// the list positions of a list sorted by body count (largest first): [0, blk) over
// GS_SUB_MAX_NB bodies, [blk, wave) a workgroup each, [wave, n) a wave each; and the largest body
// count of the last two; one: the worlds over GS_ONE_NB, nb_one: the next world's body count
struct GsSegs {
  int blk = 0, wave = 0, one = 0;
  int nb_sub = 0, nb_wave = 0, nb_one = 0;
};
// nb(k): body count of the k-th of n worlds
template <class NB> static GsSegs gs_segs(int n, NB nb) {
  auto lead = [&](int nb_over) {
    int k = 0;
    while (k < n && nb(k) > nb_over) k++;
    return k;
  };
  GsSegs g;
  g.one = lead(GS_ONE_NB);
  g.blk = lead(GS_SUB_MAX_NB);
  g.wave = lead(GS_WAVE_NB);
  g.nb_one = g.one < n ? nb(g.one) : 0;
  g.nb_sub = g.wave > g.blk ? nb(g.blk) : 0;
  g.nb_wave = g.wave < n ? nb(g.wave) : 0;
  return g;
}
static size_t lds_gs_sub(const GsSegs& g) {
  const size_t sub = (size_t)(g.nb_sub + 1) * 8 * sizeof(float) + GS_SS_SUB * sizeof(int);
  const size_t wave = (size_t)(g.nb_wave + 1) * 8 * sizeof(float) + GS_SS_WAVE * sizeof(int);
  return std::max(g.nb_sub ? sub : 0, g.nb_wave ? 4 * wave : 0);
}
// bodies of a world over GS_SUB_MAX_NB whose velocities fit in LDS beside the step table and the
// static arrays (4 KiB kept free), up to the launch's largest world
static int big_lds_cap(int max_nb, size_t max_lds) {
  const int most = (int)((max_lds - 4096 - GS_SS_BIG * sizeof(int)) / (8 * sizeof(float))) - 1;
  return std::min(max_nb, most);
}

// GS dependency levels of the step's rows.  Worlds of at most GS_WAVE_NB bodies run one per wave,
// those of at most GS_SUB_MAX_NB one per workgroup, all in one launch and with their rows in LDS
// (up to LV_ROWS_WAVE / LV_ROWS_SUB rows: 217 bodies 31 -> 12 us, half a batch of 2048 worlds
// 149 -> 51 us); larger ones in a workgroup of 1024 threads of their own launch, whose passes over
// the rows are what takes the time (16,384 bodies 2.35 -> 0.75 ms, with 256 threads before).
constexpr int LV_ROWS_WAVE = 1024, LV_ROWS_SUB = 6144, LV_TB_SUB = 512, LV_TB_BIG = 1024;
constexpr int LV_HIST_BIG = 4096;                // of a large world's level histogram in LDS
static size_t lds_levels_sub(const GsSegs& g, int bd) {
  return std::max(g.nb_sub ? lev_lds_bytes(g.nb_sub, LV_TB_SUB, LV_ROWS_SUB) : 0,
                  g.nb_wave ? (bd / 64) * lev_lds_bytes(GS_WAVE_NB, GS_WAVE_NB, LV_ROWS_WAVE) : 0);
}
template <typename R>
__global__ __launch_bounds__(256) void k_levels_sub(const DevWorld<R>* __restrict__ worlds, const int* __restrict__ list,
                                                    GsSegs g, int n) {
  __shared__ int sh[8];
  extern __shared__ float4 lds_f4[];
  const int b = (int)blockIdx.x, nsub = g.wave - g.blk;
  if (b < nsub) {
    const DevWorld<R>& W = worlds[list[g.blk + b]];
    if (W.counters[C_STATUS] != 0 || W.solver_kind == CHP_SOLVER_SPLIT) return;   // k_split_prep orders its rows
    if (W.counters[C_ROWS] <= LV_ROWS_SUB) {
      st_levels_lds<R>(W, GBlock(), sh, lds_f4, g.nb_sub, LV_TB_SUB, LV_ROWS_SUB);
    } else {
      unsigned long long* tb = (unsigned long long*)lds_f4;
      int* last = (int*)(tb + LV_TB_SUB);
      st_levels<R, GBlock, true>(W, GBlock(), sh, last, last + g.nb_sub, LV_ROWS_SUB, tb, LV_TB_SUB);
    }
  } else {
    const int wave = uni((int)(threadIdx.x >> 6)), idx = g.wave + (b - nsub) * (int)(blockDim.x >> 6) + wave;
    if (idx >= n) return;
    const DevWorld<R>& W = worlds[list[idx]];
    if (W.counters[C_STATUS] != 0 || W.solver_kind == CHP_SOLVER_SPLIT) return;
    char* lds = (char*)lds_f4 + wave * lev_lds_bytes(GS_WAVE_NB, GS_WAVE_NB, LV_ROWS_WAVE);
    if (W.counters[C_ROWS] <= LV_ROWS_WAVE) {
      st_levels_lds<R>(W, GWave(), sh, lds, GS_WAVE_NB, GS_WAVE_NB, LV_ROWS_WAVE);
    } else {
      unsigned long long* tb = (unsigned long long*)lds;
      int* last = (int*)(tb + GS_WAVE_NB);
      st_levels<R, GWave, true>(W, GWave(), sh, last, last + GS_WAVE_NB, LV_ROWS_WAVE, tb, GS_WAVE_NB);
    }
  }
}
// big_cap: bodies whose last levels fit in the launch's LDS
template <typename R>
__global__ __launch_bounds__(1024) void k_levels(const DevWorld<R>* __restrict__ worlds, const int* __restrict__ list,
                                                 int big_cap) {
  __shared__ int sh[32];
  extern __shared__ float4 lds_f4[];
  const DevWorld<R>& W = worlds[list[blockIdx.x]];
  if (W.counters[C_STATUS] != 0 || W.solver_kind == CHP_SOLVER_SPLIT) return;
  unsigned long long* tb = (unsigned long long*)lds_f4;
  int* hist = (int*)(tb + LV_TB_BIG);
  if (W.nb <= big_cap) st_levels<R, GBlock, true>(W, GBlock(), sh, hist + LV_HIST_BIG, hist, LV_HIST_BIG, tb, LV_TB_BIG);
  else st_levels<R, GBlock, false>(W, GBlock(), sh, W.tmp, hist, LV_HIST_BIG, tb, LV_TB_BIG);
}
// bd: workgroup size of k_levels_sub, and a quarter of k_levels'
template <typename R>
static void launch_levels(const DevWorld<R>* dw, const int* d_list, int n, const GsSegs& g, int max_nb, size_t max_lds, int bd,
                          hipStream_t st) {
  if (g.blk) {
    const size_t fixed = LV_TB_BIG * 8 + LV_HIST_BIG * 4;
    const int cap = std::min(max_nb, (int)((max_lds - 4096 - fixed) / sizeof(int)));
    k_levels<R><<<g.blk, 4 * bd, fixed + (size_t)cap * sizeof(int), st>>>(dw, d_list, cap);
  }
  const int nsub = (g.wave - g.blk) + (n - g.wave + bd / 64 - 1) / (bd / 64);
  if (nsub) k_levels_sub<R><<<nsub, bd, lds_levels_sub(g, bd), st>>>(dw, d_list, g, n);
}

template <typename R, int NW, bool SELF>
__device__ __forceinline__ void gs_sub_run(const DevWorld<R>& W, float* vw, int nb_cap, double* shd, int* sh, int keep) {
  constexpr int D = gs_depth<R>();
  if (W.counters[C_STATUS] != 0 || W.solver_kind == CHP_SOLVER_SPLIT) return;   // k_split_gs solves its islands
  const int E = uni(W.counters[C_ROWS]), steps = gs_steps(uni(W.counters[C_LEVELS]), E, 16 * NW, D);
  int* ss = (int*)(vw + 8 * (nb_cap + 1));
  if (steps < (NW == 1 ? GS_SS_WAVE : GS_SS_SUB) && E <= gs_narrow_rows<R>())
    st_gs<R, NW, D, true, SELF, false>(W, vw, ss, shd, sh, keep != 0);
  else
    st_gs<R, NW, 2, true, SELF, true>(W, vw, (int*)W.last_level, shd, sh, keep != 0);
}
template <typename R, bool SELF>
__global__ __launch_bounds__(256) void k_gs_sub(const DevWorld<R>* __restrict__ worlds, const int* __restrict__ list,
                                                GsSegs g, int n, int keep) {
  __shared__ int sh[4];
  __shared__ double shd[4];
  extern __shared__ float4 lds_f4[];
  float* lds = (float*)lds_f4;
  const int b = (int)blockIdx.x, nsub = g.wave - g.blk;
  if (b < nsub) {
    gs_sub_run<R, 4, SELF>(worlds[list[g.blk + b]], lds, g.nb_sub, shd, sh, keep);
  } else {
    const int wave = uni((int)(threadIdx.x >> 6)), idx = g.wave + (b - nsub) * 4 + wave;
    if (idx >= n) return;
    gs_sub_run<R, 1, SELF>(worlds[list[idx]], lds + wave * (8 * (g.nb_wave + 1) + GS_SS_WAVE), g.nb_wave, shd, sh, keep);
  }
}
// the worlds over GS_SUB_MAX_NB bodies; big_cap: body velocities that fit in the launch's LDS
template <typename R, int NW, bool SELF>
__global__ __launch_bounds__(64 * NW) void k_gs(const DevWorld<R>* __restrict__ worlds, const int* __restrict__ list,
                                                int big_cap, int keep) {
  __shared__ int sh[1];
  __shared__ double shd[NW];
  extern __shared__ float4 lds_f4[];
  constexpr int D = NW == 16 ? 2 : gs_depth<R>();   // 16 waves: at most 128 registers a lane
  const DevWorld<R>& W = worlds[list[blockIdx.x]];
  if (W.counters[C_STATUS] != 0 || W.solver_kind == CHP_SOLVER_SPLIT) return;
  int* ss = (int*)lds_f4;
  float* vw = (float*)(ss + GS_SS_BIG);
  const int E = uni(W.counters[C_ROWS]), steps = gs_steps(uni(W.counters[C_LEVELS]), E, 16 * NW, D);
  if (steps >= GS_SS_BIG || E > gs_narrow_rows<R>())
    st_gs<R, NW, 2, false, SELF, true>(W, W.vw, (int*)W.last_level, shd, sh, keep != 0);
  else if (W.nb <= big_cap)
    st_gs<R, NW, D, true, SELF, false>(W, vw, ss, shd, sh, keep != 0);
  else
    st_gs<R, NW, D, false, SELF, false>(W, W.vw, ss, shd, sh, keep != 0);
}

// the segments the sweeps are launched by: worlds of at most GS_ONE_NB bodies join the small ones'
// launch by the rule above.  What is left in [0, blk) is what launch_gs' `rows` applies to
static GsSegs gs_launch_segs(GsSegs g, int n, size_t max_lds) {
  if (g.blk > g.one && (g.wave - g.one) + (n - g.wave + 3) / 4 <= GS_ONE_WGS &&
      (size_t)(g.nb_one + 1) * 8 * sizeof(float) + GS_SS_SUB * sizeof(int) + 4096 <= max_lds) {
    g.blk = g.one;
    g.nb_sub = g.nb_one;
  }
  return g;
}
// the GS stage of a list (the level schedule and the GS records are in place).  rows: rows a
// large world runs at a time (64, 128 or 256: four lanes each).  SELF: the rows may hold one whose
// two bodies are one (the Solver slot)
template <typename R, bool SELF = false>
static void launch_gs(const DevWorld<R>* dw, const int* d_list, int n, const GsSegs& segs, int max_nb, size_t max_lds, int rows,
                      int keep, hipStream_t st) {
  const GsSegs g = gs_launch_segs(segs, n, max_lds);
  if (g.blk) {
    const int cap = big_lds_cap(max_nb, max_lds);
    const size_t lds = GS_SS_BIG * sizeof(int) + (size_t)(cap + 1) * 8 * sizeof(float);
    if (rows == 64) k_gs<R, 4, SELF><<<g.blk, 256, lds, st>>>(dw, d_list, cap, keep);
    else if (rows == 128) k_gs<R, 8, SELF><<<g.blk, 512, lds, st>>>(dw, d_list, cap, keep);
    else k_gs<R, 16, SELF><<<g.blk, 1024, lds, st>>>(dw, d_list, cap, keep);
  }
  const int nsub = (g.wave - g.blk) + (n - g.wave + 3) / 4;
  if (nsub) k_gs_sub<R, SELF><<<nsub, 256, lds_gs_sub(g), st>>>(dw, d_list, g, n, keep);
}

// World.step(dt, timeSinceLastCalled): the interpolated poses and World.time += the elapsed time
template <typename R>
__global__ __launch_bounds__(256) void k_interp(const DevWorld<R>* __restrict__ worlds, int id, double t, double elapsed) {
  const DevWorld<R>& W = worlds[id];
  const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (i == 0) W.wtime[0] += elapsed;
  if (i < W.nb) interp_body(W, i, (R)t);
}

// queries: the preparation (AABBs, SAP axis list), the AABB query, the ray passes
template <typename R>
__global__ __launch_bounds__(1024) void k_query_prep(const DevWorld<R>* __restrict__ worlds, int id) {
  st_query_prep(worlds[id]);
}
template <typename R>
__global__ __launch_bounds__(1024) void k_aabb_query(const DevWorld<R>* __restrict__ worlds, int id, f3 lo, f3 hi,
                                                     int* __restrict__ out, int cap, int* __restrict__ total) {
  __shared__ int sh[1024];
  const DevWorld<R>& W = worlds[id];
  int carry = 0;
  for (int k0 = 0; k0 < W.nb; k0 += blockDim.x) {
    const int k = k0 + (int)threadIdx.x;
    const int b = k < W.nb ? query_body(W, k) : 0;
    const int hit = (k < W.nb && aabb_overlaps(F3<R>(W.aabb_lo, b), F3<R>(W.aabb_hi, b), lo, hi)) ? 1 : 0;
    int t;
    const int r = tile_exscan(hit, sh, &t);
    if (hit && carry + r < cap) out[carry + r] = b;
    carry += t;
  }
  if (threadIdx.x == 0) *total = carry;
}
template <typename R, int PASS>
__global__ __launch_bounds__(256) void k_rays(const DevWorld<R>* __restrict__ worlds, int id, const chp_ray* __restrict__ rays,
                                              int nr, int4* __restrict__ probe, int* __restrict__ cnt,
                                              const int* __restrict__ off, chp_ray_hit* __restrict__ one,
                                              chp_ray_hit* __restrict__ out, int cap) {
  __shared__ int list[4][RAY_LIST];
  const int wave = uni((int)(threadIdx.x >> 6));
  for (int r = (int)blockIdx.x * 4 + wave; r < nr; r += (int)gridDim.x * 4) {
    if (PASS == 2 && rays[r].mode != CHP_RAY_ALL) continue;
    wave_ray<R, PASS>(worlds[id], rays[r], r, list[wave], probe, cnt, off, one, out, cap);
  }
}
// the rays' counts become offsets, with their total
static __global__ __launch_bounds__(1024) void k_ray_scan(int* __restrict__ cnt, int nr, long long* __restrict__ total) {
  __shared__ int sh[32];
  __shared__ long long big[16];
  long long s = 0;   // the offsets are ints: a total beyond them is told apart here
  for (int r = (int)threadIdx.x; r < nr; r += 1024) s += cnt[r];
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  if ((threadIdx.x & 63) == 0) big[threadIdx.x >> 6] = s;
  __syncthreads();
  s = 0;
  for (int w = 0; w < 16; w++) s += big[w];
  if (threadIdx.x == 0) *total = s;
  if (s <= 0x7fffffffLL) array_exscan(cnt, nr, sh);
}
// the one hit of each closest / any ray to its place
static __global__ __launch_bounds__(256) void k_ray_hits(const chp_ray* __restrict__ rays, int nr, const int* __restrict__ off,
                                                         const long long* __restrict__ total,
                                                         const chp_ray_hit* __restrict__ one, chp_ray_hit* __restrict__ out,
                                                         int cap) {
  const int r = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (r >= nr || rays[r].mode == CHP_RAY_ALL) return;
  const long long end = r + 1 < nr ? (long long)off[r + 1] : *total;
  if (off[r] < end && off[r] < cap) out[off[r]] = one[r];
}

// SplitSolver: ids, islands and row positions (after the rows' body pairs), then the islands'
// Gauss-Seidel (after the rows)
template <typename R>
__global__ __launch_bounds__(1024) void k_split_prep(const DevWorld<R>* __restrict__ worlds, const int* __restrict__ list) {
  __shared__ int sh[1024];
  CHP_WORLD_PROLOGUE
  if (W.solver_kind != CHP_SOLVER_SPLIT) return;
  st_split_prep(W, sh);
}
template <typename R>
__global__ __launch_bounds__(256) void k_split_gs(const DevWorld<R>* __restrict__ worlds, const int* __restrict__ list,
                                                  int keep) {
  __shared__ int sh[256];
  CHP_WORLD_PROLOGUE
  if (W.solver_kind != CHP_SOLVER_SPLIT) return;
  st_split_gs(W, keep != 0);
}

// contact-event bookkeeping after the narrowphase (worlds with events on); seed: only the key
// sets, from the contacts the slab holds
template <typename R>
__global__ __launch_bounds__(1024) void k_events(const DevWorld<R>* __restrict__ worlds, const int* __restrict__ list,
                                                 int seed) {
  __shared__ int sh[32];
  __shared__ u64 lk[EV_LDS];
  CHP_WORLD_PROLOGUE
  if (!W.ev_mask) return;
  st_events(W, seed != 0, sh, lk);
}

// the wake-up pass after the narrowphase (worlds that may hold sleeping bodies)
template <typename R>
__global__ __launch_bounds__(256) void k_wake(const DevWorld<R>* __restrict__ worlds, const int* __restrict__ list) {
  __shared__ int sh[256];
  CHP_WORLD_PROLOGUE
  st_wake(W);
}

// velocities, damping, integration, clearForces
template <typename R>
__global__ __launch_bounds__(256) void k_post(const DevWorld<R>* __restrict__ worlds, const int* __restrict__ list,
                                              double dt) {
  __shared__ int sh[256];
  CHP_WORLD_PROLOGUE
  if (W.nb >= BP_BIG) {  // k_big_post integrated the bodies
    if (threadIdx.x == 0) {
      if (W.counters[C_POSTFAIL]) {
        W.counters[C_POSTFAIL] = 0;
        ws_fail(W.counters, WS_NONFINITE);
      }
      step_done(W, dt);
    }
    return;
  }
  st_post(W, dt);
}

// Narrowphase slot: the given pairs (in the pair slab) queued by class, for the class kernels; then
// the offsets of their equations, then the equations.  One workgroup of one world each, the
// equations over the grid.
template <typename R>
__global__ __launch_bounds__(1024) void k_np_queue(const DevWorld<R>* __restrict__ worlds, int id, int np,
                                                   int* __restrict__ qw, int2* __restrict__ q, int wcc) {
  __shared__ int sh[16];
  const DevWorld<R>& W = worlds[id];
  if (threadIdx.x == 0) {
    W.counters[C_PAIRS] = np;
    W.counters[C_STATUS] = W.counters[C_STAGING] = W.counters[C_ROWS] = 0;
  }
  __threadfence_block();
  __syncthreads();
  st_narrow_count(W, qw, 0, wcc != 0, sh);
  __threadfence();
  __syncthreads();
  queue_bounds(qw);
  st_narrow_place(W, id, qw, 0, wcc != 0, q, sh);
  __syncthreads();
  if (threadIdx.x < 2 * NP_NCLS) qw[QW_TOT + threadIdx.x] = 0;
}
template <typename R>
__global__ __launch_bounds__(1024) void k_np_offsets(const DevWorld<R>* __restrict__ worlds, int id, int cap) {
  __shared__ int sh[32];
  st_equation_offsets(worlds[id], cap, sh);
}
template <typename R>
__global__ __launch_bounds__(64) void k_np_equations(const DevWorld<R>* __restrict__ worlds, int id, double dt,
                                                     chp_equation* __restrict__ out) {
  const DevWorld<R>& W = worlds[id];
  if (W.counters[C_STATUS] & WS_ROWS) return;
  const int P = W.counters[C_PAIRS];
  for (int p = (int)(blockIdx.x * blockDim.x + threadIdx.x); p < P; p += (int)(gridDim.x * blockDim.x))
    pair_equations(W, p, (R)dt, out);
}

// Solver slot: the bodies' solve masses, rows from the given equations, their GS records at the
// schedule's positions (after k_levels), and at the end the velocity update and the multipliers
// (Equation.multiplier = lambda / dt, gs_solver.dart:124-129)
template <typename R>
__global__ __launch_bounds__(256) void k_solve_bodies(const DevWorld<R>* __restrict__ worlds, int id, int n) {
  const DevWorld<R>& W = worlds[id];
  const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (i < W.nb) solve_body(W, i);
  if (i == 0) { W.counters[C_ROWS] = n; W.counters[C_STATUS] = 0; }
}
template <typename R>
__global__ __launch_bounds__(64) void k_solve_rows(const DevWorld<R>* __restrict__ worlds, int id,
                                                   const chp_equation* __restrict__ eq, int n, double dt) {
  const int r = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (r < n) solve_row(worlds[id], eq, r, (R)dt);
}
template <typename R>
__global__ __launch_bounds__(64) void k_solve_records(const DevWorld<R>* __restrict__ worlds, int id, int n) {
  const DevWorld<R>& W = worlds[id];
  const int r = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (r >= n) return;
  const int k = W.rpos[r];
  const int2 x = ((const int2*)W.row_ab)[r];
  gs_store<R>((typename GsWord<R>::T*)W.gsr, k, W.rows[r], (unsigned)x.x, (unsigned)x.y);
  W.glam[2 * (size_t)k] = (R)0;
}
template <typename R>
__global__ __launch_bounds__(256) void k_solve_finish(const DevWorld<R>* __restrict__ worlds, int id, int n, double dt,
                                                      double* __restrict__ mult) {
  const DevWorld<R>& W = worlds[id];
  const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (i < W.nb && n > 0) solve_finish_body(W, i);
  if (i < n && mult) {
    const R invDt = (R)1 / (R)dt;
    mult[i] = (double)(W.glam[2 * (size_t)W.rpos[i]] * invDt);
  }
}

// the kernels instantiated in chp_narrow_kernels.hip
#define CHP_NARROW_KERNELS(X, R)                                                                       \
  X void k_narrow_threads<R>(const DevWorld<R>*, const int2*, const int*, double);                     \
  X void k_narrow_cls<R, NP_SS>(const DevWorld<R>*, const int2*, const int*, double);                  \
  X void k_narrow_cls<R, NP_SP>(const DevWorld<R>*, const int2*, const int*, double);                  \
  X void k_narrow_cls<R, NP_SB>(const DevWorld<R>*, const int2*, const int*, double);                  \
  X void k_narrow_cls<R, NP_SC>(const DevWorld<R>*, const int2*, const int*, double);                  \
  X void k_narrow_cls<R, NP_PC>(const DevWorld<R>*, const int2*, const int*, double);                  \
  X void k_narrow_cls<R, NP_CC>(const DevWorld<R>*, const int2*, const int*, double);                  \
  X void k_narrow_cls<R, NP_OTHER>(const DevWorld<R>*, const int2*, const int*, double);               \
  X void k_narrow_wave<R, NP_WHC>(const DevWorld<R>*, const int2*, int*, double, int);                      \
  X void k_narrow_wave<R, NP_WAVE>(const DevWorld<R>*, const int2*, int*, double, int);

}  // namespace chp

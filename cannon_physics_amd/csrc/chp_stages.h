// chp_stages.h -- the stages of World.internalStep (world_class.dart:433-701) as device
// functions.  Per-world stages run on the workgroup (or wave) that owns a world; per-pair and
// per-body stages of the whole batch, and of large worlds, run over the grid.  The kernels in
// chp_api.hip launch each stage once over every listed world.
#pragma once
#include <type_traits>

#include "chp_narrow.h"

namespace chp {

#define CHP_KMAX 8

enum { C_STATUS = 0, C_PAIRS = 1, C_CONTACTS = 2, C_ROWS = 3, C_ITERS = 4, C_LEVELS = 5, C_STAGING = 6,
       C_STEP = 7, C_FROWS = 8, C_CROWS = 9, C_SUM_PAIRS = 10, C_SUM_ROWS = 11, C_SUM_CONTACTS = 12,
       C_POSTFAIL = 13,
       C_COUNT = 16 };

__device__ __forceinline__ void ws_fail(int* counters, int bit) { atomicOr(&counters[C_STATUS], bit); }

__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }

// in-place exclusive scan of data[0..n); returns the total (same value in every thread).  Each
// wave scans a contiguous segment in coalesced rounds of 64 (a shuffle scan per round, a
// running carry); a pass of wave sums ahead gives every segment its offset.  sh needs
// blockDim.x / 64 + 1 ints; blockDim.x is a multiple of 64.
__device__ __forceinline__ int wave_incl_scan(int v) {
  const int lane = (int)(threadIdx.x & 63);
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int x = __shfl_up(v, off, 64);
    if (lane >= off) v += x;
  }
  return v;
}
// exclusive scan of one value per thread over the workgroup (blockDim.x a multiple of 64); sh
// needs blockDim.x / 64 ints
__device__ __forceinline__ int tile_exscan(int v, int* sh, int* total) {
  const int lane = (int)(threadIdx.x & 63), wv = (int)(threadIdx.x >> 6), nw = (int)(blockDim.x >> 6);
  const int inc = wave_incl_scan(v);
  if (lane == 63) sh[wv] = inc;
  __syncthreads();
  int before = 0, tot = 0;
  for (int w = 0; w < nw; w++) {
    const int x = sh[w];
    before += w < wv ? x : 0;
    tot += x;
  }
  __syncthreads();
  *total = tot;
  return before + inc - v;
}
__device__ __forceinline__ int array_exscan(int* data, int n, int* sh) {
  const int nw = (int)(blockDim.x >> 6), wv = (int)(threadIdx.x >> 6), lane = (int)(threadIdx.x & 63);
  const int seg = (((n + nw - 1) / nw) + 63) & ~63;
  const int b = min(n, wv * seg), e = min(n, b + seg);
  int s = 0;
  for (int i = b + lane; i < e; i += 64) s += data[i];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  if (lane == 0) sh[wv] = s;
  __syncthreads();
  int carry = 0, tot = 0;
  for (int w = 0; w < nw; w++) {
    const int x = sh[w];
    carry += w < wv ? x : 0;
    tot += x;
  }
  for (int i0 = b; i0 < e; i0 += 64) {
    const int i = i0 + lane;
    const int v = i < e ? data[i] : 0;
    const int inc = wave_incl_scan(v);
    if (i < e) data[i] = carry + inc - v;
    carry += __shfl(inc, 63, 64);
  }
  __syncthreads();
  return tot;
}
// flag bits of the body indices in the solver's row records
enum : unsigned { GS_DYN = 0x80000000u, GS_IDX = 0x3fffffffu };

// barrier that orders LDS only: outstanding global loads (prefetches) stay in flight
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}
// value written by thread 0 of the block, read by all
__device__ __forceinline__ int block_bcast(int v, int* sh) {
  __syncthreads();
  if (threadIdx.x == 0) sh[0] = v;
  __syncthreads();
  int r = sh[0];
  __syncthreads();
  return r;
}

template <typename R> __device__ __forceinline__ f3 F3(const float* a, int i) { return ((const f3*)a)[i]; }
template <typename R> __device__ __forceinline__ void S3(float* a, int i, f3 v) { ((f3*)a)[i] = v; }

// ---- gravity, solve mass, AABBs ------------------------------------------------------------
// world_class.dart:459-471 (f += m g for dynamic bodies; kept in feff so that an aborted step
// leaves Body.force untouched), Body.updateSolveMassProperties (rigid_body.dart:303-314),
// SAPBroadphase.sortList's lazy Body.updateAABB (sap_broadphase.dart:168-180)
template <typename R> __device__ void body_aabb(const DevWorld<R>& W, int i) {
  f3 pos = F3<R>(W.pos, i);
  f4 q = ((const f4*)W.quat)[i];
  f3 lo = mk3(0.f, 0.f, 0.f), hi = lo;
  for (int k = 0; k < W.shape_count[i]; k++) {
    int s = W.shape_first[i] + k;
    f3 off = add3<double>(qrot<double>(q, F3<R>(W.si_off, s)), pos);
    f4 ori = qmul<double>(q, ((const f4*)W.si_ori)[s]);
    int h = W.si_hull[s];
    const f3* hv = (W.si_type[s] == CHP_SHAPE_CONVEX) ? ((const f3*)W.h_verts + W.h_vstart[h]) : nullptr;
    int hn = (W.si_type[s] == CHP_SHAPE_CONVEX) ? W.h_vcount[h] : 0;
    f3 a, b;
    shape_aabb(W.si_type[s], (double)W.si_radius[s], F3<R>(W.si_half, s), hv, hn, off, ori, a, b);
    if (k == 0) { lo = a; hi = b; }
    else {
      lo.x = min_dart(lo.x, a.x); hi.x = max_dart(hi.x, b.x);
      lo.y = min_dart(lo.y, a.y); hi.y = max_dart(hi.y, b.y);
      lo.z = min_dart(lo.z, a.z); hi.z = max_dart(hi.z, b.z);
    }
  }
  if (W.shape_count[i] > 0) { S3<R>(W.aabb_lo, i, lo); S3<R>(W.aabb_hi, i, hi); }
}

// World.internalStep before the broadphase for body i (world_class.dart:459-471): gravity into
// the effective force, the solve masses, cleared velocity deltas, the SAP AABB refresh
// SAP: the world may be a SAP world (its dirty AABBs are refreshed); else the code is left out
// a body the broadphase treats as fixed: static, or asleep (broadphase.dart:54-60)
template <typename R> __device__ __forceinline__ bool bp_passive(const DevWorld<R>& W, int i) {
  return W.type[i] == CHP_BODY_STATIC || W.sleep_state[i] == CHP_SLEEP_SLEEPING;
}
// a body whose solve mass is zero: kinematic, or asleep (Body.updateSolveMassProperties,
// rigid_body.dart:302-314)
template <typename R> __device__ __forceinline__ bool solve_massless(const DevWorld<R>& W, int i) {
  return W.type[i] == CHP_BODY_KINEMATIC || W.sleep_state[i] == CHP_SLEEP_SLEEPING;
}

template <typename R, bool SAP = true> __device__ __forceinline__ void prestep_body(const DevWorld<R>& W, int i) {
  int ty = W.type[i];
  f3 f = F3<R>(W.force, i);
  if (ty == CHP_BODY_DYNAMIC) {
    R m = W.mass[i];
    f = set3<R>(ld<R>(f.x) + m * (R)W.gravity[0], ld<R>(f.y) + m * (R)W.gravity[1], ld<R>(f.z) + m * (R)W.gravity[2]);
  }
  S3<R>(W.feff, i, f);
  const bool kin = solve_massless(W, i);
  W.ims[i] = kin ? (R)0 : W.inv_mass[i];
  for (int k = 0; k < 9; k++) W.iiws[9 * i + k] = kin ? 0.f : W.iiw[9 * i + k];
  S3<R>(W.vl, i, mk3(0.f, 0.f, 0.f));
  S3<R>(W.wl, i, mk3(0.f, 0.f, 0.f));
  if constexpr (SAP) {
    if (W.broadphase == CHP_BROADPHASE_SAP && (W.flags[i] & BF_AABB_DIRTY)) {
      body_aabb(W, i);
      W.flags[i] &= ~BF_AABB_DIRTY;
    }
  }
}
template <typename R, bool SAP = true> __device__ void st_prestep(const DevWorld<R>& W) {
  for (int i = threadIdx.x; i < W.nb; i += blockDim.x) prestep_body<R, SAP>(W, i);
}

// ---- broadphase -------------------------------------------------------------------------------
// Broadphase.needBroadphaseCollision (broadphase.dart:44-63) + doBoundingSphereBroadphase
// (:77-86), FP64 predicate
template <typename R> __device__ __forceinline__ bool bp_need(const DevWorld<R>& W, int a, int b) {
  if ((W.group[a] & W.mask[b]) == 0 || (W.group[b] & W.mask[a]) == 0) return false;
  if (bp_passive(W, a) && bp_passive(W, b)) return false;
  return true;
}
__device__ __forceinline__ bool bp_sphere_at(f3 pa, double ra, f3 pb, double rb) {
  f3 r = sub3<double>(pb, pa);
  double s = ra + rb;
  return len2<double>(r) < s * s;
}
template <typename R> __device__ __forceinline__ bool bp_sphere(const DevWorld<R>& W, int a, int b) {
  return bp_sphere_at(F3<R>(W.pos, a), (double)W.brad[a], F3<R>(W.pos, b), (double)W.brad[b]);
}
__device__ __forceinline__ float axis_of(f3 v, int ax) { return ax == 0 ? v.x : (ax == 1 ? v.y : v.z); }

// The bounding-sphere predicate of bp_sphere_at decided in FP32 where the margin allows: 1 it
// holds, 0 it does not, -1 undecided.  The difference of two FP32 coordinates rounded to FP32 is
// the same through FP64 (twice the precision and two bits), so l2 and s2 are off their FP64 values
// by a few FP32 roundings; the margin of 1e-5 is forty times that, and 1e-30 covers underflow.  An
// infinite s2 (a plane's radius) holds for every finite l2, as it does in FP64.
__device__ __forceinline__ int bp_screen(float4 a, float4 b) {
  const float dx = b.x - a.x, dy = b.y - a.y, dz = b.z - a.z, s = a.w + b.w;
  const float l2 = dx * dx + dy * dy + dz * dz, s2 = s * s;
  if (l2 < s2 * 0.99999f - 1e-30f) return 1;
  return l2 > s2 * 1.00001f + 1e-30f ? 0 : -1;
}

// The broadphase data of a world of fewer than BP_BIG bodies, in LDS: position and radius (FP32),
// filter group / mask / static-or-asleep flag / body, the radius in R when that is FP64, and the
// naive pass's ballot masks or the SAP pass's sort keys.
// Naive masks: row i has ceil(i / 64) words, those of rows 0..i-1 take bp_chunks(i).
__host__ __device__ __forceinline__ int bp_chunks(int i) {
  if (i <= 1) return 0;
  const int a = (i - 1) >> 6, b = (i - 1) & 63;
  return (a + 1) * (32 * a + b);
}
__host__ __device__ __forceinline__ int bp_pow2(int n) {
  int p = 1;
  while (p < n) p <<= 1;
  return p;
}
template <typename R> struct BpLds {
  float4* P;
  int4* F;
  unsigned long long* words;   // naive: bp_chunks(n); SAP: the keys, a power of two
  R* rad;                      // FP64 only
  int* cnt;                    // SAP: old positions, then pairs per row
  static __host__ __device__ size_t bytes(int n, bool sap) {
    return (size_t)n * (sizeof(float4) + sizeof(int4) + (sizeof(R) == 8 ? sizeof(R) : 0) + (sap ? sizeof(int) : 0)) +
           (size_t)(sap ? bp_pow2(n) : bp_chunks(n)) * sizeof(unsigned long long);
  }
  __device__ void carve(void* base, int n, bool sap) {
    P = (float4*)base;
    F = (int4*)(P + n);
    words = (unsigned long long*)(F + n);
    rad = (R*)(words + (sap ? bp_pow2(n) : bp_chunks(n)));
    cnt = (int*)(sizeof(R) == 8 ? rad + n : rad);
  }
  __device__ __forceinline__ double radius(int k) const {
    if constexpr (sizeof(R) == 8) return (double)rad[k];
    else return (double)P[k].w;
  }
  // body b's data at k
  __device__ __forceinline__ void put(const DevWorld<R>& W, int k, int b) const {
    const f3 p = F3<R>(W.pos, b);
    const R r = W.brad[b];
    P[k] = make_float4(p.x, p.y, p.z, (float)r);
    F[k] = make_int4(W.group[b], W.mask[b], bp_passive(W, b) ? 1 : 0, b);
    if constexpr (sizeof(R) == 8) rad[k] = r;
  }
  // needBroadphaseCollision of records x, y
  static __device__ __forceinline__ bool need(int4 x, int4 y) {
    return (x.x & y.y) != 0 && (y.x & x.y) != 0 && !(x.z && y.z);
  }
};

// NaiveBroadphase.collisionPairs (naive_broadphase.dart:14-33): pairs (i, j), j < i, in i-major
// order.  A wave keeps 64 bodies j in registers and walks the rows i dealt to it, each row's data
// read once for all 64 from LDS: 14 FP32 instructions screen a row, and only where one of its 64
// spheres is near are the filters (and, undecided, the FP64 predicate) looked at.  The ballots
// of a row's hits stay in LDS; in row order their set bits are the pairs in the reference's
// order, so a scan of the population counts places them.
template <typename R> __device__ bool st_bp_naive(const DevWorld<R>& W, int* sh, const BpLds<R>& L) {
  const int n = W.nb, tid = (int)threadIdx.x, bd = (int)blockDim.x;
  const int lane = tid & 63, wave = uni(tid >> 6), nwave = bd >> 6, nw = bp_chunks(n);
  for (int i = tid; i < n; i += bd) L.put(W, i, i);
  for (int w = tid; w < nw; w += bd) L.words[w] = 0ull;
  __syncthreads();
  for (int j0 = 0; j0 < n - 1; j0 += 64) {
    const int j = j0 + lane;
    const float4 pj = L.P[min(j, n - 1)];
    const int4 fj = L.F[min(j, n - 1)];
    int i = j0 + 1 + wave;
    float4 pn = L.P[min(i, n - 1)];
    for (; i < n; i += nwave) {
      const float4 pi = pn;
      pn = L.P[min(i + nwave, n - 1)];
      const int scr = bp_screen(pi, pj);
      if (!__any(j < i && scr != 0)) continue;
      bool hit = j < i && scr != 0 && BpLds<R>::need(L.F[i], fj);
      if (__any(hit && scr < 0)) {
        const bool exact = bp_sphere_at(mk3(pi.x, pi.y, pi.z), L.radius(i), mk3(pj.x, pj.y, pj.z), L.radius(min(j, n - 1)));
        hit = hit && (scr > 0 || exact);
      }
      const unsigned long long m = __ballot(hit);
      if (lane == 0 && m) L.words[bp_chunks(i) + (j0 >> 6)] = m;
    }
  }
  __syncthreads();
  const int K = (nw + bd - 1) / bd, w0 = min(nw, tid * K), w1 = min(nw, w0 + K);
  int c = 0;
  for (int w = w0; w < w1; w++) c += __popcll(L.words[w]);
  int P;
  int o = tile_exscan(c, sh, &P);
  if (P > W.pair_cap) {
    if (tid == 0) { W.counters[C_PAIRS] = P; ws_fail(W.counters, WS_PAIRS); }
    return false;
  }
  if (c) {
    int lo = 1, hi = n - 1;   // the row of word w0: the last i with bp_chunks(i) <= w0
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (bp_chunks(mid) <= w0) lo = mid;
      else hi = mid - 1;
    }
    int i = lo, next = bp_chunks(i + 1), j0 = 64 * (w0 - bp_chunks(i));
    for (int w = w0; w < w1; w++) {
      if (w == next) {
        i++;
        next = bp_chunks(i + 1);
        j0 = 0;
      }
      for (unsigned long long m = L.words[w]; m; m &= m - 1) {
        W.pair_i[o] = i;
        W.pair_j[o] = j0 + __builtin_ctzll(m);
        o++;
      }
      j0 += 64;
    }
  }
  if (tid == 0) W.counters[C_PAIRS] = P;
  __syncthreads();
  return true;
}

// FP32 sort key with -0 folded onto +0 (the insertion sort compares with <=)
__device__ __forceinline__ unsigned int order_key(float f) {
  unsigned int u = __float_as_uint(f == 0.f ? 0.f : f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// SAPBroadphase.collisionPairs (sap_broadphase.dart:138-190): the persistent axis list is
// re-sorted by aabb.lowerBound[axis]; ties keep the previous order (the insertion sort is
// stable), so sorting (key, previous position) reproduces it exactly.  Then the sweep with
// its `continue` on filtered pairs and `break` on checkBounds (:41-63).
// SAPBroadphase.sortList's insertion sort (sap_broadphase.dart:168-189) on one workgroup: the
// axis list stably re-sorted by aabb.lowerBound[axis] (a bitonic sort of (key, position) pairs)
template <typename R> __device__ void sap_sort(const DevWorld<R>& W) {
  int n = W.nb, ax = W.sap_axis;
  int np2 = 1;
  while (np2 < n) np2 <<= 1;
  unsigned long long* key = W.sort_keys;
  for (int k = threadIdx.x; k < np2; k += blockDim.x) {
    if (k < n) {
      int b = W.order[k];
      key[k] = ((unsigned long long)order_key(axis_of(F3<R>(W.aabb_lo, b), ax)) << 32) | (unsigned)k;
      W.tmp[k] = b;
    } else {
      key[k] = ~0ull;
    }
  }
  __syncthreads();
  for (int size = 2; size <= np2; size <<= 1)
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int t = threadIdx.x; t < np2 / 2; t += blockDim.x) {
        int lo = 2 * stride * (t / stride) + (t % stride);
        int hi = lo + stride;
        bool up = ((lo & size) == 0);
        unsigned long long a = key[lo], b = key[hi];
        if ((a > b) == up) { key[lo] = b; key[hi] = a; }
      }
      __syncthreads();
    }
  for (int k = threadIdx.x; k < n; k += blockDim.x) W.order[k] = W.tmp[(int)(key[k] & 0xffffffffu)];
  __syncthreads();
}
// The whole of it for a world of fewer than BP_BIG bodies, from LDS: the bitonic sort, then one
// wave per row over the sorted records, 64 candidates at a time, once to count and once to write.
template <typename R> __device__ bool st_bp_sap(const DevWorld<R>& W, int* sh, const BpLds<R>& L) {
  const int n = W.nb, ax = W.sap_axis, np2 = bp_pow2(n), tid = (int)threadIdx.x, bd = (int)blockDim.x;
  const int lane = tid & 63, wave = uni(tid >> 6), nwave = bd >> 6;
  for (int k = tid; k < np2; k += bd) {
    unsigned long long key = ~0ull;
    if (k < n) {
      const int b = W.order[k];
      key = ((unsigned long long)order_key(axis_of(F3<R>(W.aabb_lo, b), ax)) << 32) | (unsigned)k;
      L.cnt[k] = b;
    }
    L.words[k] = key;
  }
  __syncthreads();
  for (int size = 2; size <= np2; size <<= 1)
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int t = tid; t < np2 / 2; t += bd) {
        const int lo = ((t & ~(stride - 1)) << 1) | (t & (stride - 1)), hi = lo + stride;
        const unsigned long long a = L.words[lo], b = L.words[hi];
        if ((a > b) == ((lo & size) == 0)) { L.words[lo] = b; L.words[hi] = a; }
      }
      __syncthreads();
    }
  for (int k = tid; k < n; k += bd) {
    const int b = L.cnt[(int)(L.words[k] & 0xffffffffu)];
    W.order[k] = b;
    L.put(W, k, b);
  }
  __syncthreads();
  int P = 0;
  for (int pass = 0; pass < 2; pass++) {
    for (int k = wave; k < n; k += nwave) {
      const float4 p4 = L.P[k];
      const int4 gi = L.F[k];
      const f3 pi = mk3(p4.x, p4.y, p4.z);
      const double ri = L.radius(k), A2 = (double)axis_of(pi, ax) + ri;
      int o = pass ? L.cnt[k] : 0;
      for (int m0 = k + 1; m0 < n; m0 += 64) {
        const int m = min(m0 + lane, n - 1);
        const float4 q4 = L.P[m];
        const int4 gj = L.F[m];
        const f3 pj = mk3(q4.x, q4.y, q4.z);
        const double rj = L.radius(m);
        const bool need = m0 + lane < n && BpLds<R>::need(gi, gj);
        const bool brk = need && !((double)axis_of(pj, ax) - rj < A2);
        const bool hit = need && !brk && bp_sphere_at(pi, ri, pj, rj);
        const unsigned long long bm = __ballot(brk);
        unsigned long long hm = __ballot(hit);
        if (bm) hm &= (1ull << __builtin_ctzll(bm)) - 1ull;
        if (pass && ((hm >> lane) & 1ull)) {
          const int r = o + __popcll(hm & ((1ull << lane) - 1ull));
          W.pair_i[r] = gi.w;
          W.pair_j[r] = gj.w;
        }
        o += __popcll(hm);
        if (bm) break;
      }
      if (!pass && lane == 0) L.cnt[k] = o;
    }
    __syncthreads();
    if (!pass) {
      P = array_exscan(L.cnt, n, sh);
      if (P > W.pair_cap) {
        if (tid == 0) { W.counters[C_PAIRS] = P; ws_fail(W.counters, WS_PAIRS); }
        return false;
      }
    }
  }
  if (tid == 0) W.counters[C_PAIRS] = P;
  __syncthreads();
  return true;
}

// pairs of constraints with collideConnected == false are dropped (world_class.dart:487-499);
// dropped pairs are marked with -1 so the surviving order is unchanged
template <typename R> __device__ void st_filter(const DevWorld<R>& W) {
  if (!W.has_filtered_constraints) return;
  int P = W.counters[C_PAIRS];
  for (int p = threadIdx.x; p < P; p += blockDim.x) {
    int a = W.pair_i[p], b = W.pair_j[p];
    for (int c = 0; c < W.ncons; c++) {
      if (W.c_collide[c]) continue;
      int ca = W.c_a[c], cb = W.c_b[c];
      if ((ca == a && cb == b) || (cb == a && ca == b)) { W.pair_i[p] = -1; break; }
    }
  }
  __syncthreads();
}

// ---- broadphase of large worlds, spread over the grid -----------------------------------------
// A world of at least BP_BIG bodies is not left to one workgroup.  Its rows are dealt out in spans
// of BP_SPAN (one workgroup per span, one wave per row); the SAP axis list is sorted in tiles of
// SAP_TILE keys (bitonic sort in LDS, one workgroup per tile) that are then merged pairwise by
// rank, and the pairs are counted, scanned and written in three grid-wide passes.  Sort order,
// pair order and the collideConnected filter are those of the workgroup path above.
constexpr int BP_BIG = 512, BP_SPAN = 64, SAP_TILE = 4096;

template <typename R> __device__ __forceinline__ bool bp_filtered(const DevWorld<R>& W, int a, int b) {
  for (int c = 0; c < W.ncons; c++) {
    if (W.c_collide[c]) continue;
    int ca = W.c_a[c], cb = W.c_b[c];
    if ((ca == a && cb == b) || (cb == a && ca == b)) return true;
  }
  return false;
}

// the sweep record of body b at axis-list position k
template <typename R> __device__ __forceinline__ void sap_record(const DevWorld<R>& W, int k, int b) {
  const f3 p = F3<R>(W.pos, b);
  ((float4*)W.sbp)[k] = make_float4(p.x, p.y, p.z, __int_as_float(b));
  ((int4*)W.sgm)[k] = make_int4(W.group[b], W.mask[b], bp_passive(W, b) ? 1 : 0, 0);
  W.sbr[k] = W.brad[b];
}

// SAP candidates m0..m0+63 of the row body (filter gi, position pi, radius ri, upper bound A2 on
// the axis), read from the sweep records: the hits before the first break (a pair that passes
// needBroadphaseCollision and fails checkBounds); *stop when the row's sweep ends in this chunk
template <typename R>
__device__ __forceinline__ unsigned long long sap_chunk(const DevWorld<R>& W, int4 gi, f3 pi, double ri, double A2,
                                                        int m0, int* bj, bool* stop) {
  const int n = W.nb, m = m0 + (int)(threadIdx.x & 63);
  float4 pj = make_float4(0.f, 0.f, 0.f, 0.f);
  int4 gj = make_int4(0, 0, 0, 0);
  double rj = 0.0;
  if (m < n) {
    pj = ((const float4*)W.sbp)[m];
    gj = ((const int4*)W.sgm)[m];
    rj = (double)W.sbr[m];
  }
  const f3 pv = mk3(pj.x, pj.y, pj.z);
  bool need = m < n && (gi.x & gj.y) != 0 && (gj.x & gi.y) != 0 && !(gi.z && gj.z);
  bool brk = need && !((double)axis_of(pv, W.sap_axis) - rj < A2);
  bool hit = need && !brk && bp_sphere_at(pi, ri, pv, rj);
  unsigned long long bm = __ballot(brk), hm = __ballot(hit);
  if (bm) hm &= (1ull << __builtin_ctzll(bm)) - 1ull;
  *stop = bm != 0 || m0 + 64 >= n;
  *bj = __float_as_int(pj.w);
  return hm;
}

// row k of a large world (wave-uniform k): SAP, the body at sorted position k against the ones
// after it; naive, body k against the bodies before it.  emit: write the pairs from offset o,
// else return their number.
template <typename R> __device__ int big_row(const DevWorld<R>& W, int k, bool emit, int o) {
  const int lane = threadIdx.x & 63;
  const bool filt = W.has_filtered_constraints;
  int c = 0;
  auto put = [&](unsigned long long m, int a, int b) {
    if (emit && ((m >> lane) & 1ull)) {
      int p = o + c + __popcll(m & ((1ull << lane) - 1ull));
      W.pair_i[p] = (filt && bp_filtered(W, a, b)) ? -1 : a;
      W.pair_j[p] = b;
    }
    c += __popcll(m);
  };
  if (W.broadphase == CHP_BROADPHASE_SAP) {
    const float4 p4 = ((const float4*)W.sbp)[k];
    const int4 gi = ((const int4*)W.sgm)[k];
    const int bi = __float_as_int(p4.w);
    const f3 pi = mk3(p4.x, p4.y, p4.z);
    const double ri = (double)W.sbr[k];
    const double A2 = (double)axis_of(pi, W.sap_axis) + ri;
    for (int m0 = k + 1; m0 < W.nb; m0 += 64) {
      int bj;
      bool stop;
      unsigned long long m = sap_chunk(W, gi, pi, ri, A2, m0, &bj, &stop);
      put(m, bi, bj);
      if (stop) break;
    }
  } else {
    for (int j0 = 0; j0 < k; j0 += 64) {
      const int j = j0 + lane;
      put(__ballot(j < k && bp_need(W, k, j) && bp_sphere(W, k, j)), k, j);
    }
  }
  return c;
}

// one SAP tile: keys (order key of aabb.lowerBound[axis], position) of positions s0.. sorted in
// LDS.  apply (the world is one tile): the new axis list is written at once; else the sorted run
// goes to sort_keys and the old list to tmp for the merges.
template <typename R>
__device__ void sap_tile(const DevWorld<R>& W, int s0, unsigned long long* lk, int* lord, bool apply) {
  const int cnt = min(SAP_TILE, W.nb - s0), ax = W.sap_axis;
  for (int k = threadIdx.x; k < SAP_TILE; k += blockDim.x) {
    unsigned long long key = ~0ull;
    if (k < cnt) {
      int g = s0 + k, b = W.order[g];
      key = ((unsigned long long)order_key(axis_of(F3<R>(W.aabb_lo, b), ax)) << 32) | (unsigned)g;
      if (apply) lord[k] = b;
      else W.tmp[g] = b;
    }
    lk[k] = key;
  }
  __syncthreads();
  for (int size = 2; size <= SAP_TILE; size <<= 1)
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int t = threadIdx.x; t < SAP_TILE / 2; t += blockDim.x) {
        int lo = ((t & ~(stride - 1)) << 1) | (t & (stride - 1)), hi = lo + stride;
        bool up = (lo & size) == 0;
        unsigned long long a = lk[lo], b = lk[hi];
        if ((a > b) == up) { lk[lo] = b; lk[hi] = a; }
      }
      __syncthreads();
    }
  for (int k = threadIdx.x; k < cnt; k += blockDim.x) {
    if (apply) {
      const int b = lord[(int)(lk[k] & 0xffffffffu) - s0];
      W.order[s0 + k] = b;
      sap_record(W, s0 + k, b);
    } else {
      W.sort_keys[s0 + k] = lk[k];
    }
  }
}

// merge round of run width w: the key at g goes to its run's start plus its index in the run plus
// the number of keys below it in the partner run (keys are unique).  src selects the half of
// sort_keys read; apply (last round) writes the new axis list.
template <typename R> __device__ void sap_merge(const DevWorld<R>& W, int g, int w, int src, bool apply) {
  const int n = W.nb;
  const unsigned long long* a = W.sort_keys + (src ? n : 0);
  unsigned long long* d = W.sort_keys + (src ? 0 : n);
  const unsigned long long x = a[g];
  const int run = g / w, base = run * w, pb = (run ^ 1) * w;
  int out = g;
  if (pb < n) {
    int lo = pb, hi = min(pb + w, n);
    while (lo < hi) {
      int mid = (lo + hi) >> 1;
      if (a[mid] < x) lo = mid + 1;
      else hi = mid;
    }
    out = min(base, pb) + (g - base) + (lo - pb);
  }
  d[out] = x;
  if (apply) {
    const int b = W.tmp[(int)(x & 0xffffffffu)];
    W.order[out] = b;
    sap_record(W, out, b);
  }
}

// ---- narrowphase ------------------------------------------------------------------------------
// Pairs whose separating-axis search is large (more than WAVE_AXES axes: convex hulls without
// unique axes, anything against heightfield pillars) or whose clip polygon may outgrow the
// thread path's CLIP_THREAD points run one pair per wave, the axes over the lanes; every other
// pair runs one pair per thread.
constexpr int WAVE_AXES = 96;
template <typename R> __device__ __forceinline__ bool wave_pair(const DevWorld<R>& W, int bi, int bj) {
  for (int a = 0; a < W.shape_count[bi]; a++)
    for (int b = 0; b < W.shape_count[bj]; b++) {
      int sa = W.shape_first[bi] + a, sb = W.shape_first[bj] + b;
      int ta = W.si_type[sa], tb = W.si_type[sb];
      bool ca = ta == CHP_SHAPE_BOX || ta == CHP_SHAPE_CONVEX, cb = tb == CHP_SHAPE_BOX || tb == CHP_SHAPE_CONVEX;
      if ((ca && tb == CHP_SHAPE_HEIGHTFIELD) || (cb && ta == CHP_SHAPE_HEIGHTFIELD)) return true;
      if (ca && cb) {
        int ha = W.si_hull[sa], hb = W.si_hull[sb];
        int axes = (W.h_axes[ha] ? W.h_fcount[ha] : 0) + (W.h_axes[hb] ? W.h_fcount[hb] : 0) +
                   W.h_ecount[ha] * W.h_ecount[hb];
        if (axes > WAVE_AXES || W.h_maxface[ha] + W.h_maxface[hb] > CLIP_THREAD) return true;
      }
    }
  return false;
}

// records a pair's contacts: staging slot, per-pair counts (pc_cnt / pc_base / pf_cnt / pc_off)
template <typename R> __device__ __forceinline__ void pair_counts(const DevWorld<R>& W, int p, int n, int base) {
  int nf = 0, nc = 0;
  for (int k = 0; k < n; k++) {
    int fl = W.contacts[base + k].flags;
    if (fl & 1) { nc++; if (fl & 2) nf += 2; }
  }
  W.pc_cnt[p] = n;
  W.pc_base[p] = base;
  W.pf_cnt[p] = nf;
  W.pc_off[p] = nc;
}

// one pair on one thread: contacts into the staging slab, per-pair counts.  KINDS: the
// resolvers compiled in.  Buffered (DIRECT false): up to KMAX contacts are buffered locally and
// then copied to a reserved range (a pair with more runs again straight into the slab).
// DIRECT: the resolver (planeConvex, convexConvex: one call per pair) reserves its range
// itself and writes there, with no local buffer.  cb: the wave's LDS clip-polygon area
// (2 * CLIP_THREAD * 64 f3), needed when convexConvex is compiled in.
template <typename R, unsigned KINDS = NK_ALL, int KMAX = CHP_KMAX, bool DIRECT = false>
__device__ __forceinline__ void narrow_pair(const DevWorld<R>& W, int p, R dt, f3* cb) {
  int bi = W.pair_i[p], bj = W.pair_j[p];
  int n = 0, base = 0;
  if (bi < 0) {
    pair_counts(W, p, 0, 0);
    return;
  }
  if constexpr (DIRECT) {
    Sink<R> s{W.contacts, W.contact_cap, 0, 0};
    s.slot = &W.counters[C_STAGING];
    NPCtx<R, false, KINDS> ctx(W, dt, &s, nullptr, cb);
    ctx.pair(bi, bj);
    if (ctx.status) ws_fail(W.counters, ctx.status);
    if (s.overflow) {
      ws_fail(W.counters, WS_CONTACTS);
      s.n = s.nf = s.nc = 0;
    }
    W.pc_cnt[p] = s.n;
    W.pc_base[p] = s.base;
    W.pf_cnt[p] = s.nf;
    W.pc_off[p] = s.nc;
    return;
  } else {
    ContactRec<R> loc[KMAX];
    Sink<R> s{loc, KMAX, 0, 0};
    NPCtx<R, false, KINDS> ctx(W, dt, &s, nullptr, cb);
    ctx.pair(bi, bj);
    if (ctx.status) ws_fail(W.counters, ctx.status);
    n = s.n;
    if (n > 0) {
      base = atomicAdd(&W.counters[C_STAGING], n);
      if (base + n > W.contact_cap) {
        ws_fail(W.counters, WS_CONTACTS);
        n = 0;
      } else if (n <= KMAX) {
        for (int k = 0; k < n; k++) W.contacts[base + k] = loc[k];
      } else {  // more contacts than the local buffer: run the pair again into the slab
        Sink<R> s2{W.contacts + base, n, 0, 0};
        NPCtx<R, false, KINDS> ctx2(W, dt, &s2, nullptr, cb);
        ctx2.pair(bi, bj);
      }
    }
  }
  pair_counts(W, p, n, base);
}

// The batched narrowphase sorts the pairs of every listed world by resolver class, so that a
// wave of the thread kernel runs one resolver on neighbouring data.  Classes 0..NP_WAVE-1 run one
// pair per thread, class NP_WAVE one pair per wave.
// Wave classes: NP_WHC, single-shape pairs needing a wave (sphere– and convex–heightfield, large
// SAT), compiled with those resolvers only; NP_WAVE, the rest (compound bodies).  NP_SH (sphere–
// heightfield one pair per thread) is left empty by the batched path.
enum { NP_SS = 0, NP_SP, NP_SB, NP_SC, NP_SH, NP_PC, NP_CC, NP_OTHER, NP_WHC, NP_WAVE, NP_NCLS };
// after the class bounds: one pair ticket per wave class (NP_WHC, NP_WAVE)
constexpr int NP_NTICKET = 2;
static_assert(NP_WAVE == NP_WHC + 1, "the tickets follow the wave classes' order");
// wcc: hull pairs of the batch run on the wave path whatever their size (few of them: a pair takes a
// wave a fraction of the time it takes a thread)
template <typename R> __device__ __forceinline__ int pair_class(const DevWorld<R>& W, int bi, int bj, bool wcc) {
  if (W.ev_mask) {   // justTest pairs (narrow_phase.dart:665-668): their overlap probe is on the wave path
    const int ti = W.type[bi], tj = W.type[bj];
    if ((ti == CHP_BODY_KINEMATIC && tj != CHP_BODY_DYNAMIC) || (tj == CHP_BODY_KINEMATIC && ti != CHP_BODY_DYNAMIC))
      return NP_WAVE;
  }
  if (W.shape_count[bi] != 1 || W.shape_count[bj] != 1) return wave_pair(W, bi, bj) ? NP_WAVE : NP_OTHER;
  int ta = W.si_type[W.shape_first[bi]], tb = W.si_type[W.shape_first[bj]];
  int lo = min(ta, tb), hi = max(ta, tb);
  if (lo == CHP_SHAPE_SPHERE) {
    if (hi == CHP_SHAPE_SPHERE) return NP_SS;
    if (hi == CHP_SHAPE_PLANE) return NP_SP;
    if (hi == CHP_SHAPE_BOX) return NP_SB;
    if (hi == CHP_SHAPE_CONVEX) return NP_SC;
    if (hi == CHP_SHAPE_HEIGHTFIELD) return NP_WHC;   // the wave deals the pillars to its lanes
    return NP_OTHER;
  }
  if (lo == CHP_SHAPE_PLANE && (hi == CHP_SHAPE_BOX || hi == CHP_SHAPE_CONVEX)) return NP_PC;
  if (lo == CHP_SHAPE_BOX || lo == CHP_SHAPE_CONVEX) {
    if (hi == CHP_SHAPE_HEIGHTFIELD) return NP_WHC;
    if (hi == CHP_SHAPE_BOX || hi == CHP_SHAPE_CONVEX) return wcc || wave_pair(W, bi, bj) ? NP_WHC : NP_CC;
  }
  return NP_OTHER;
}

// The queue's words: class totals and cursors (zero between steps: k_rows clears them once the
// step's queue is placed), the class bounds (bounds[c] = first entry of class c, bounds[NP_NCLS] =
// total), the wave classes' tickets, then NP_NCLS pair counts per listed world.
constexpr int QW_TOT = 0, QW_CUR = NP_NCLS, QW_BOUNDS = 2 * NP_NCLS, QW_TICKETS = QW_BOUNDS + NP_NCLS + 1,
              QW_COUNTS = QW_TICKETS + NP_NTICKET;
__host__ __device__ constexpr size_t queue_words(size_t nworlds) { return QW_COUNTS + nworlds * NP_NCLS; }

// pass 1 (at the end of the broadphase): the pair counts of the workgroup's world by class, into
// its words and the totals
template <typename R> __device__ void st_narrow_count(const DevWorld<R>& W, int* qw, int idx, bool wcc, int* sh) {
  const int P = W.counters[C_PAIRS];
  if (threadIdx.x < NP_NCLS) sh[threadIdx.x] = 0;
  __syncthreads();
  for (int p = threadIdx.x; p < P; p += blockDim.x) {
    int bi = W.pair_i[p], bj = W.pair_j[p];
    if (bi < 0) { pair_counts(W, p, 0, 0); continue; }
    atomicAdd(&sh[pair_class(W, bi, bj, wcc)], 1);
  }
  __syncthreads();
  if (threadIdx.x < NP_NCLS) {
    const int c = sh[threadIdx.x];
    qw[QW_COUNTS + idx * NP_NCLS + threadIdx.x] = c;
    if (c) atomicAdd(&qw[QW_TOT + threadIdx.x], c);
  }
}
// the first queue entry of this thread's class (threads 0..NP_NCLS-1): the totals of the classes
// before it
__device__ __forceinline__ int queue_base(const int* qw) {
  int base = 0;
  for (int c = 0; c < NP_NCLS; c++) base += c < (int)threadIdx.x ? qw[QW_TOT + c] : 0;
  return base;
}
// the class bounds and the tickets (one workgroup of the placement)
__device__ __forceinline__ void queue_bounds(int* qw) {
  if (threadIdx.x <= NP_NCLS) qw[QW_BOUNDS + threadIdx.x] = queue_base(qw);
  if (threadIdx.x < NP_NTICKET) qw[QW_TICKETS + threadIdx.x] = 0;
}
// pass 2: the world's pairs into the queue, each class in a range reserved by its cursor (the
// order of the worlds within a class is free)
template <typename R>
__device__ void st_narrow_place(const DevWorld<R>& W, int wid, int* qw, int idx, bool wcc, int2* q, int* sh) {
  const int P = W.counters[C_PAIRS];
  if (threadIdx.x < NP_NCLS) {
    const int c = qw[QW_COUNTS + idx * NP_NCLS + threadIdx.x];
    sh[threadIdx.x] = c ? queue_base(qw) + atomicAdd(&qw[QW_CUR + threadIdx.x], c) : 0;
  }
  __syncthreads();
  for (int p = threadIdx.x; p < P; p += blockDim.x) {
    int bi = W.pair_i[p], bj = W.pair_j[p];
    if (bi < 0) continue;
    q[atomicAdd(&sh[pair_class(W, bi, bj, wcc)], 1)] = make_int2(wid, p);
  }
}

// the resolvers of a thread class and the contacts its pairs make at most (sphere classes: one;
// a pair that makes more still comes out right, run a second time into the slab)
constexpr unsigned cls_kinds(int c) {
  return c == NP_SS ? NK_SS : c == NP_SP ? NK_SP : c == NP_SB ? NK_SB : c == NP_SC ? NK_SC :
         c == NP_SH ? NK_SH : c == NP_PC ? NK_PC : c == NP_CC ? NK_CC : NK_ALL;
}
constexpr int cls_kmax(int c) { return c <= NP_SC ? 1 : CHP_KMAX; }
// classes whose single resolver call emits all of a pair's contacts at once write them straight
// into the slab (no local buffer)
constexpr bool cls_direct(int c) { return c == NP_PC || c == NP_CC; }

// one thread class of the queue, one pair per thread (grid-stride); cb: the wave's LDS clip area
template <typename R, int CLS>
__device__ void st_narrow_class(const DevWorld<R>* worlds, const int2* q, const int* bounds, R dt, f3* cb) {
  const int b1 = bounds[CLS + 1];
  const int g = (int)(blockIdx.x * blockDim.x + threadIdx.x), ng = (int)(gridDim.x * blockDim.x);
  for (int i = bounds[CLS] + g; i < b1; i += ng) {
    const int2 e = q[i];
    narrow_pair<R, cls_kinds(CLS), cls_kmax(CLS), cls_direct(CLS)>(worlds[e.x], e.y, dt, cb);
  }
}

// the thread classes without clip polygons in one launch, 64 queue entries of one class at a time
template <typename R>
__device__ void st_narrow_threads(const DevWorld<R>* worlds, const int2* q, const int* bounds, R dt, f3* cb) {
  constexpr int CLS[5] = {NP_SB, NP_SC, NP_PC, NP_SS, NP_SP};   // the longest first
  int first[6];
  first[0] = 0;
#pragma unroll
  for (int k = 0; k < 5; k++) first[k + 1] = first[k] + (bounds[CLS[k] + 1] - bounds[CLS[k]] + 63) / 64;
  for (int b = (int)blockIdx.x; b < first[5]; b += (int)gridDim.x) {
    auto run = [&](auto cls, int k) {
      constexpr int C = decltype(cls)::value;
      const int i = bounds[C] + 64 * (b - first[k]) + (int)threadIdx.x;
      if (i >= bounds[C + 1]) return;
      const int2 e = q[i];
      narrow_pair<R, cls_kinds(C), cls_kmax(C), cls_direct(C)>(worlds[e.x], e.y, dt, cb);
    };
    if (b < first[1]) run(std::integral_constant<int, NP_SB>(), 0);
    else if (b < first[2]) run(std::integral_constant<int, NP_SC>(), 1);
    else if (b < first[3]) run(std::integral_constant<int, NP_PC>(), 2);
    else if (b < first[4]) run(std::integral_constant<int, NP_SS>(), 3);
    else run(std::integral_constant<int, NP_SP>(), 4);
  }
}

// contact records a wave buffers per pair: a heightfield pair touching several pillars has more
// contacts than a thread's pair, and a pair over the buffer runs twice
constexpr int WAVE_KMAX = 64;
// the queued separating-axis pairs, one wave per pair.  A wave takes each pair from a ticket
// counter (zero at the launch) when it is free, so that waves that drew cheap pairs go on to
// the rest while one runs an expensive pair: the costs differ by orders of magnitude (a hull
// falling clear of a heightfield against one resting on a dozen pillars).  Waves numbered at or
// beyond the queue's length leave at once, so an empty or short queue costs few atomics on the
// one counter.
// A pair is a chain of latencies, its instructions among them: a launch of a few hundred pairs
// runs most of its code for the first time.  So each resolver is compiled once (46 KB; 198 KB when
// the retry, the overlap probe and both users of convexConvex had copies of their own), the pair's
// data are uniform, hulls are read from LDS through LDS pointers, and what follows the axis search
// takes a lane per face, vertex, plane and contact (300-body pile 39 -> 19 us, 157 bodies in double
// 48 -> 21 us, 24 terrains of 16 to 1024 bodies 553 -> 448 us a launch).
// (ws: the wave's LDS workspace; loc: its LDS contact buffer of kmax records; clip_cap: points a
// clip polygon may have)
template <typename R, unsigned KINDS>
__device__ __forceinline__ void st_narrow_wave(const DevWorld<R>* worlds, const int2* queue, int cnt, int* ticket, R dt, f3* ws,
                               ContactRec<R>* loc, int kmax, int clip_cap) {
  const int lane = threadIdx.x & 63;
  if ((int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6) >= cnt) return;
  for (;;) {
    int i = 0;
    if (lane == 0) i = atomicAdd(ticket, 1);
    i = uni(i);
    if (i >= cnt) break;
    const int2 q = queue[i];
    const DevWorld<R>& W = worlds[uni(q.x)];
    const int p = uni(q.y);
    const int bi = uni(W.pair_i[p]), bj = uni(W.pair_j[p]);
    Sink<R, true> s{loc, kmax, 0, 0};
    NPCtx<R, true, KINDS> ctx(W, dt, &s, ws);
    ctx.clip_cap = clip_cap;
    int n, base = 0;
    for (;;) {   // (one call, so that the resolvers are compiled once)
      ctx.pair(bi, bj);
      NPCtx<R, true, KINDS>::wave_fence();   // the lanes' records
      n = s.n;
      if (s.buf != loc) break;
      if (lane == 0) {
        if (ctx.status) ws_fail(W.counters, ctx.status);
        if (n > 0) base = atomicAdd(&W.counters[C_STAGING], n);
      }
      base = uni(base);
      if (n > 0 && base + n > W.contact_cap) {
        if (lane == 0) ws_fail(W.counters, WS_CONTACTS);
        n = 0;
      }
      if (n <= kmax) break;
      s = Sink<R, true>{W.contacts + base, n, 0, 0};   // more contacts than the local buffer: again into the slab
    }
    if (n <= kmax) {
      const int* src = (const int*)loc;
      int* dst = (int*)(W.contacts + base);
      for (int w = lane; w < n * (int)(sizeof(ContactRec<R>) / 4); w += 64) dst[w] = src[w];
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");   // (the lanes read each other's records)
    const ContactRec<R>* rec = n > kmax ? (const ContactRec<R>*)W.contacts + base : loc;
    int nc = 0, nf = 0;
    for (int k0 = 0; k0 < n; k0 += 64) {
      const int fl = k0 + lane < n ? rec[k0 + lane].flags : 0;
      nc += __popcll(__ballot(fl & 1));
      nf += 2 * __popcll(__ballot((fl & 3) == 3));
    }
    if (lane == 0) {
      W.pc_cnt[p] = n;
      W.pc_base[p] = base;
      W.pf_cnt[p] = nf;
      W.pc_off[p] = nc;
    }
    // the next pair reuses the workspace and the buffer
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

// ---- equations ----------------------------------------------------------------------------------
// Equation.setSpookParams (equation_class.dart:53-60)
template <typename R> __device__ __forceinline__ void spook(R k, R d, R h, R& a, R& b, R& eps) {
  a = (R)4 / (h * ((R)1 + (R)4 * d));
  b = ((R)4 * d) / ((R)1 + (R)4 * d);
  eps = (R)4 / (h * h * k * ((R)1 + (R)4 * d));
}
// JacobianElement.multiplyVectors
template <typename R> __device__ __forceinline__ R mulvec(f3 s, f3 r, f3 gs, f3 gr) { return dot3<R>(s, gs) + dot3<R>(r, gr); }
// The body state the row builders read (Equation.bi / bj), loaded once per contact or joint and
// shared by its rows: the row stores do not alias it, but the compiler cannot know that.
template <typename R> struct RowBody {
  int i, fl;            // index; with GS_DYN when dynamic and awake (its vlambda moves)
  f3 p, v, w, f, t;     // position, velocity, angular velocity, effective force, torque
  R im;                 // invMassSolve
  float I[9];           // invInertiaWorldSolve
};
template <typename R> __device__ __forceinline__ RowBody<R> row_body(const DevWorld<R>& W, int i) {
  RowBody<R> o;
  o.i = i;
  o.fl = i | (W.type[i] == CHP_BODY_DYNAMIC && W.sleep_state[i] != CHP_SLEEP_SLEEPING ? (int)GS_DYN : 0);
  o.p = F3<R>(W.pos, i);
  o.v = F3<R>(W.vel, i);
  o.w = F3<R>(W.avel, i);
  o.f = F3<R>(W.feff, i);
  o.t = F3<R>(W.torque, i);
  o.im = W.ims[i];
#pragma unroll
  for (int k = 0; k < 9; k++) o.I[k] = W.iiws[9 * i + k];
  return o;
}
// Equation.computeGiMf (equation_class.dart:108-127)
template <typename R> __device__ __forceinline__ R giMf(const RowBody<R>& A, const RowBody<R>& B, f3 sa, f3 ra, f3 sb, f3 rb) {
  f3 fa = scale3<R>(A.f, A.im);
  f3 fb = scale3<R>(B.f, B.im);
  f3 ta = mvmul<R>(A.I, A.t);
  f3 tb = mvmul<R>(B.I, B.t);
  return mulvec<R>(fa, ta, sa, ra) + mulvec<R>(fb, tb, sb, rb);
}
// Equation.computeGW (:82-92)
template <typename R> __device__ __forceinline__ R gwv(const RowBody<R>& A, const RowBody<R>& B, f3 sa, f3 ra, f3 sb, f3 rb) {
  return mulvec<R>(A.v, A.w, sa, ra) + mulvec<R>(B.v, B.w, sb, rb);
}
// Where the row builders put a row r: ROWS_REC, its row record (and body pair); ROWS_AB, only
// its body pair (the level schedule needs no more); ROWS_GS, its GS record, straight at its
// level-order position rpos[r] (plus the row record when keep).
enum : int { ROWS_REC = 0, ROWS_AB = 1, ROWS_GS = 2 };
template <typename R> struct GsWord;
template <typename R>
__device__ __forceinline__ void gs_store(typename GsWord<R>::T* base, int k, const RowRec<R>& r, unsigned fa, unsigned fb);

// stores the row with 1/C (Equation.computeC = computeGiMGt + eps, :130-174)
template <typename R, int MODE = ROWS_REC>
__device__ void put_row(const DevWorld<R>& W, int r, int kind, const RowBody<R>& A, const RowBody<R>& Bd, f3 sa, f3 ra,
                        f3 sb, f3 rb, R B, R eps, R minF, R maxF, bool keep = false) {
  const int fa = A.fl, fb = Bd.fl;
  if constexpr (MODE == ROWS_AB) {
    W.row_ab[2 * r] = fa;
    W.row_ab[2 * r + 1] = fb;
    return;
  }
  RowRec<R> o;
  o.a = A.i; o.b = Bd.i; o.kind = kind; o.pad = 0;
  o.sa = sa; o.ra = ra; o.sb = sb; o.rb = rb;
  R gim = A.im + Bd.im;
  o.ia = mvmul<R>(A.I, ra);
  gim += dot3<R>(o.ia, ra);
  o.ib = mvmul<R>(Bd.I, rb);
  gim += dot3<R>(o.ib, rb);
  o.B = B;
  o.invC = (R)1 / (gim + eps);
  o.eps = eps;
  o.lambda = 0;
  o.minF = minF; o.maxF = maxF;
  o.ima = A.im; o.imb = Bd.im;
  if constexpr (MODE == ROWS_GS) {
    const int k = W.rpos[r];
    gs_store<R>((typename GsWord<R>::T*)W.gsr, k, o, (unsigned)fa, (unsigned)fb);
    W.glam[2 * k] = (R)0;
    if (keep) W.rows[r] = o;
  } else {
    W.rows[r] = o;
    W.row_ab[2 * r] = fa;
    W.row_ab[2 * r + 1] = fb;
  }
}
// ContactEquation.computeB (contact_equation.dart:34-77)
template <typename R, int MODE = ROWS_REC>
__device__ void contact_row(const DevWorld<R>& W, int r, const RowBody<R>& a, const RowBody<R>& b, f3 ri, f3 rj, f3 n,
                            R rest, R sa_, R sb_, R se, R h, R minF, R maxF, bool keep = false) {
  f3 rixn = cross3<R>(ri, n), rjxn = cross3<R>(rj, n);
  f3 gsa = neg3(n), gra = neg3(rixn), gsb = n, grb = rjxn;
  f3 pen = add3<R>(b.p, rj);
  pen = sub3<R>(pen, a.p);
  pen = sub3<R>(pen, ri);
  R g = dot3<R>(n, pen);
  R e1 = rest + (R)1;
  R gw = e1 * dot3<R>(b.v, n) - e1 * dot3<R>(a.v, n) + dot3<R>(b.w, rjxn) - dot3<R>(a.w, rixn);
  R gm = giMf(a, b, gsa, gra, gsb, grb);
  R B = -g * sa_ - gw * sb_ - h * gm;
  put_row<R, MODE>(W, r, CHP_ROW_CONTACT, a, b, gsa, gra, gsb, grb, B, se, minF, maxF, keep);
}
// FrictionEquation.computeB (friction_equation.dart:19-48)
template <typename R, int MODE = ROWS_REC>
__device__ void friction_row(const DevWorld<R>& W, int r, const RowBody<R>& a, const RowBody<R>& b, f3 ri, f3 rj, f3 t,
                             R sb_, R se, R h, R minF, R maxF, bool keep = false) {
  f3 rixt = cross3<R>(ri, t), rjxt = cross3<R>(rj, t);
  f3 gsa = neg3(t), gra = neg3(rixt), gsb = t, grb = rjxt;
  R gw = gwv(a, b, gsa, gra, gsb, grb);
  R gm = giMf(a, b, gsa, gra, gsb, grb);
  R B = -gw * sb_ - h * gm;
  put_row<R, MODE>(W, r, CHP_ROW_FRICTION, a, b, gsa, gra, gsb, grb, B, se, minF, maxF, keep);
}
// RotationalEquation / ConeEquation.computeB (rotational_equation.dart:34-58, cone_equation.dart:34-57)
template <typename R, int MODE = ROWS_REC>
__device__ void rot_row(const DevWorld<R>& W, int r, int kind, const RowBody<R>& a, const RowBody<R>& b, f3 ni, f3 nj,
                        R cosA, R h, R minF, R maxF, R sa_, R sb_, R se, bool keep = false) {
  f3 z = mk3(0.f, 0.f, 0.f);
  f3 gra = cross3<R>(nj, ni), grb = cross3<R>(ni, nj);
  R g = cosA - dot3<R>(ni, nj);
  R gw = gwv(a, b, z, gra, z, grb);
  R gm = giMf(a, b, z, gra, z, grb);
  R B = -g * sa_ - gw * sb_ - h * gm;
  put_row<R, MODE>(W, r, kind, a, b, z, gra, z, grb, B, se, minF, maxF, keep);
}
// RotationalMotorEquation.computeB (rotational_motor_equation.dart:17-33)
template <typename R, int MODE = ROWS_REC>
__device__ void motor_row(const DevWorld<R>& W, int r, const RowBody<R>& a, const RowBody<R>& b, f3 axA, f3 axB,
                          R target, R h, R minF, R maxF, R sb_, R se, bool keep = false) {
  f3 z = mk3(0.f, 0.f, 0.f);
  f3 gra = axA, grb = neg3(axB);
  R gw = gwv(a, b, z, gra, z, grb) - target;
  R gm = giMf(a, b, z, gra, z, grb);
  R B = -gw * sb_ - h * gm;
  put_row<R, MODE>(W, r, CHP_ROW_MOTOR, a, b, z, gra, z, grb, B, se, minF, maxF, keep);
}

// Constraint.update + the rows each joint feeds the solver (lib/constraints/)
template <typename R, int MODE = ROWS_REC>
__device__ void constraint_rows(const DevWorld<R>& W, int c, int row0, R h, bool keep = false) {
  int type = W.c_type[c], ia = W.c_a[c], ib = W.c_b[c], mask = W.c_eq_mask[c];
  if (!mask) return;
  const RowBody<R> a = row_body(W, ia), b = row_body(W, ib);
  const f3* v = (const f3*)W.c_vec + 12 * c;
  const R* eq = W.c_eq + 25 * c;
  f4 qa = ((const f4*)W.quat)[ia], qb = ((const f4*)W.quat)[ib];
  int r = row0;
  const R sa_ = W.c_spook[0], sb_ = W.c_spook[1], se = W.c_spook[2];
  if (type == CHP_CONSTRAINT_DISTANCE) {  // distance_constraint.dart:27-38
    R half = eq[24] * (R)0.5;
    f3 n = normalize3<R>(sub3<R>(b.p, a.p));
    f3 ri = scale3<R>(n, half), rj = scale3<R>(n, -half);
    contact_row<R, MODE>(W, r, a, b, ri, rj, n, (R)0, sa_, sb_, se, h, eq[0], eq[1], keep);
    return;
  }
  // PointToPointConstraint.update (point_to_point_constraint.dart:68-83): three ContactEquations
  f3 ri = qrot<R>(qa, v[0]), rj = qrot<R>(qb, v[1]);
  const f3 axes3[3] = {mk3(1.f, 0.f, 0.f), mk3(0.f, 1.f, 0.f), mk3(0.f, 0.f, 1.f)};
  for (int k = 0; k < 3; k++) contact_row<R, MODE>(W, r++, a, b, ri, rj, axes3[k], (R)0, sa_, sb_, se, h, eq[4 * k], eq[4 * k + 1], keep);
  if (type == CHP_CONSTRAINT_HINGE) {  // hinge_constraint.dart:79-104
    f3 wA = qrot<R>(qa, v[2]), wB = qrot<R>(qb, v[3]);
    f3 t1, t2;
    tangents3<R>(wA, t1, t2);
    rot_row<R, MODE>(W, r++, CHP_ROW_ROTATIONAL, a, b, t1, wB, eq[12 + 2], h, eq[12], eq[13], sa_, sb_, se, keep);
    rot_row<R, MODE>(W, r++, CHP_ROW_ROTATIONAL, a, b, t2, wB, eq[16 + 2], h, eq[16], eq[17], sa_, sb_, se, keep);
    if (mask & 32) motor_row<R, MODE>(W, r++, a, b, qrot<R>(qa, v[2]), qrot<R>(qb, v[3]), eq[20 + 3], h, eq[20], eq[21], sb_, se, keep);
  } else if (type == CHP_CONSTRAINT_LOCK) {  // lock_constraint.dart:70-88
    rot_row<R, MODE>(W, r++, CHP_ROW_ROTATIONAL, a, b, qrot<R>(qa, v[4]), qrot<R>(qb, v[7]), eq[14], h, eq[12], eq[13], sa_, sb_, se, keep);
    rot_row<R, MODE>(W, r++, CHP_ROW_ROTATIONAL, a, b, qrot<R>(qa, v[6]), qrot<R>(qb, v[9]), eq[18], h, eq[16], eq[17], sa_, sb_, se, keep);
    rot_row<R, MODE>(W, r++, CHP_ROW_ROTATIONAL, a, b, qrot<R>(qa, v[8]), qrot<R>(qb, v[5]), eq[22], h, eq[20], eq[21], sa_, sb_, se, keep);
  } else if (type == CHP_CONSTRAINT_CONE_TWIST) {  // cone_twist_constraint.dart:77-96
    f3 cA = qrot<R>(qa, v[2]), cB = qrot<R>(qb, v[3]);
    rot_row<R, MODE>(W, r++, CHP_ROW_CONE, a, b, cA, cB, eq[14], h, eq[12], eq[13], sa_, sb_, se, keep);
    f3 t1, t2, u1, u2;
    tangents3<R>(v[2], t1, t2);   // axisA.tangents(twist.axisA, twist.axisA): the second write wins
    tangents3<R>(v[3], u1, u2);
    rot_row<R, MODE>(W, r++, CHP_ROW_ROTATIONAL, a, b, qrot<R>(qa, t2), qrot<R>(qb, u2), eq[18], h, eq[16], eq[17], sa_, sb_, se, keep);
  }
}

// the friction rows (from the scanned offset pf_cnt[p]) and contact rows (from F + pc_off[p]) of
// pair p's contacts
template <typename R, int MODE = ROWS_REC>
__device__ void pair_rows(const DevWorld<R>& W, int p, int F, R h, bool keep = false) {
  int fo = W.pf_cnt[p], co = F + W.pc_off[p];
  const int n = W.pc_cnt[p];
  if (n == 0) return;
  // a pair's contacts mostly share their body order (a compound pair's may not)
  RowBody<R> A = row_body(W, W.contacts[W.pc_base[p]].bi), B = row_body(W, W.contacts[W.pc_base[p]].bj);
  for (int k = 0; k < n; k++) {
    const ContactRec<R>& c = W.contacts[W.pc_base[p] + k];
    if (!(c.flags & 1)) continue;
    if (c.bi != A.i) A = row_body(W, c.bi);
    if (c.bj != B.i) B = row_body(W, c.bj);
    const R* cm = W.cm_params + 6 * c.cm;
    if (c.flags & 2) {
      R fa, fb, fe;
      spook<R>(cm[4], cm[5], h, fa, fb, fe);
      f3 t1, t2;
      tangents3<R>(c.ni, t1, t2);
      friction_row<R, MODE>(W, fo++, A, B, c.ri, c.rj, t1, fb, fe, h, -c.slip, c.slip, keep);
      friction_row<R, MODE>(W, fo++, A, B, c.ri, c.rj, t2, fb, fe, h, -c.slip, c.slip, keep);
    }
    R ca, cb, ce;
    spook<R>(cm[2], cm[3], h, ca, cb, ce);
    contact_row<R, MODE>(W, co++, A, B, c.ri, c.rj, c.ni, c.restitution, ca, cb, ce, h, (R)0, (R)1e6, keep);
  }
}
// the row counters of a step (thread 0), after the offsets are known
template <typename R> __device__ void rows_done(const DevWorld<R>& W, int P, int F, int C, int E) {
  W.counters[C_ROWS] = E;
  W.counters[C_FROWS] = F;
  W.counters[C_CROWS] = C;
  W.counters[C_CONTACTS] = W.counters[C_STAGING];
  W.counters[C_SUM_PAIRS] += P;
  W.counters[C_SUM_ROWS] += E;
  W.counters[C_SUM_CONTACTS] += W.counters[C_STAGING];
}

// rows in solver order: every friction row, every contact row, then constraint rows
// (world_class.dart:539-635; Solver.addEquation filter, solver.dart:30-34).  The offsets of a
// step: friction rows of pair p from pf_cnt[p], its contact rows from F + pc_off[p], joint rows
// after every contact row; false (WS_ROWS) when the slab is too small
template <typename R> __device__ bool st_rowscan(const DevWorld<R>& W, int* sh) {
  const int P = W.counters[C_PAIRS];
  const int F = array_exscan(W.pf_cnt, P, sh);
  const int C = array_exscan(W.pc_off, P, sh);
  const int E = F + C + W.ncrows;
  if (E > W.row_cap) {
    if (threadIdx.x == 0) { W.counters[C_ROWS] = E; ws_fail(W.counters, WS_ROWS); }
    return false;
  }
  if (threadIdx.x == 0) rows_done(W, P, F, C, E);
  __syncthreads();
  return true;
}

// ---- slot stages ---------------------------------------------------------------------------------
// The equations World.internalStep hands the solver for the world's current pairs (the
// Narrowphase slot with World's row assembly, world_class.dart:539-635, without the joints):
// friction equations then contact equations in generation order, disabled and trigger ones
// dropped, the body-material restitution override applied.  B and 1/C are the solver's.
// The offsets of a pair's equations (one workgroup); false when they outgrow the buffer.
template <typename R> __device__ bool st_equation_offsets(const DevWorld<R>& W, int cap, int* sh) {
  const int P = W.counters[C_PAIRS];
  const int F = array_exscan(W.pf_cnt, P, sh);
  const int C = array_exscan(W.pc_off, P, sh);
  const bool ok = F + C <= cap;
  if (threadIdx.x == 0) {
    W.counters[C_ROWS] = F + C;
    if (ok) { W.counters[C_FROWS] = F; W.counters[C_CROWS] = C; }
    else ws_fail(W.counters, WS_ROWS);
  }
  return ok;
}
// the equations of pair p
template <typename R> __device__ void pair_equations(const DevWorld<R>& W, int p, R h, chp_equation* out) {
  {
    int fo = W.pf_cnt[p], co = W.counters[C_FROWS] + W.pc_off[p];
    for (int k = 0; k < W.pc_cnt[p]; k++) {
      const ContactRec<R>& c = W.contacts[W.pc_base[p] + k];
      if (!(c.flags & 1)) continue;
      const R* cm = W.cm_params + 6 * c.cm;
      chp_equation e;
      memset(&e, 0, sizeof e);
      e.body_i = c.bi; e.body_j = c.bj;
      e.shape_i = e.shape_j = -1;   // FrictionEquation has no shapes
      e.ri[0] = c.ri.x; e.ri[1] = c.ri.y; e.ri[2] = c.ri.z;
      e.rj[0] = c.rj.x; e.rj[1] = c.rj.y; e.rj[2] = c.rj.z;
      if (c.flags & 2) {
        R fa, fb, fe;
        spook<R>(cm[4], cm[5], h, fa, fb, fe);
        f3 t[2];
        tangents3<R>(c.ni, t[0], t[1]);
        e.kind = CHP_ROW_FRICTION;
        e.min_force = (double)-c.slip; e.max_force = (double)c.slip;
        e.a = (double)fa; e.b = (double)fb; e.eps = (double)fe;
        for (int q = 0; q < 2; q++) {
          e.n[0] = t[q].x; e.n[1] = t[q].y; e.n[2] = t[q].z;
          out[fo++] = e;
        }
      }
      R ca, cb, ce;
      spook<R>(cm[2], cm[3], h, ca, cb, ce);
      e.kind = CHP_ROW_CONTACT;
      e.shape_i = W.si_shape[c.si]; e.shape_j = W.si_shape[c.sj];
      e.n[0] = c.ni.x; e.n[1] = c.ni.y; e.n[2] = c.ni.z;
      e.min_force = 0.0; e.max_force = 1e6;
      e.a = (double)ca; e.b = (double)cb; e.eps = (double)ce;
      e.restitution = (double)c.restitution;
      out[co++] = e;
    }
  }
}

// GSSolver.solve's set-up for given equations (gs_solver.dart:27-75): solve masses, the applied
// force as the body holds it (the World added gravity before calling the solver), and each
// equation's B and 1/C from its own spook parameters.
template <typename R> __device__ __forceinline__ void solve_body(const DevWorld<R>& W, int i) {
  S3<R>(W.feff, i, F3<R>(W.force, i));
  const bool kin = solve_massless(W, i);
  W.ims[i] = kin ? (R)0 : W.inv_mass[i];
  for (int k = 0; k < 9; k++) W.iiws[9 * i + k] = kin ? 0.f : W.iiw[9 * i + k];
  S3<R>(W.vl, i, mk3(0.f, 0.f, 0.f));
  S3<R>(W.wl, i, mk3(0.f, 0.f, 0.f));
}
// row r.  One pass per equation kind, each with a single row builder: the builders are not merged
// into one body
template <typename R> __device__ void solve_row(const DevWorld<R>& W, const chp_equation* eq, int r, R h) {
  const chp_equation& e = eq[r];
  const f3 ri = mk3(e.ri[0], e.ri[1], e.ri[2]), rj = mk3(e.rj[0], e.rj[1], e.rj[2]);
  const f3 nn = mk3(e.n[0], e.n[1], e.n[2]);
  const R sa_ = (R)e.a, sb_ = (R)e.b, se = (R)e.eps, mn = (R)e.min_force, mx = (R)e.max_force;
  const int ps = e.kind == CHP_ROW_CONTACT ? 0 : e.kind == CHP_ROW_FRICTION ? 1 : e.kind == CHP_ROW_MOTOR ? 3 : 2;
  for (int pass = 0; pass < 4; pass++) {
    if (ps != pass) continue;
    const RowBody<R> A = row_body(W, e.body_i), B = row_body(W, e.body_j);
    if (pass == 0)
      contact_row(W, r, A, B, ri, rj, nn, (R)e.restitution, sa_, sb_, se, h, mn, mx);
    else if (pass == 1)
      friction_row(W, r, A, B, ri, rj, nn, sb_, se, h, mn, mx);
    else if (pass == 2 && (e.kind == CHP_ROW_ROTATIONAL || e.kind == CHP_ROW_CONE))
      rot_row(W, r, e.kind, A, B, ri, rj, (R)e.angle_cos, h, mn, mx, sa_, sb_, se);
    else if (pass == 3)
      motor_row(W, r, A, B, ri, rj, (R)e.target_velocity, h, mn, mx, sb_, se);
  }
}

// end of GSSolver.solve: v += vlambda * linearFactor, w += wlambda * angularFactor
// (gs_solver.dart:111-121)
template <typename R> __device__ __forceinline__ void solve_finish_body(const DevWorld<R>& W, int i) {
  f3 v = F3<R>(W.vel, i), w = F3<R>(W.avel, i);
  S3<R>(W.vel, i, add3<R>(v, mul3<R>(F3<R>(W.vl, i), F3<R>(W.lin_factor, i))));
  S3<R>(W.avel, i, add3<R>(w, mul3<R>(F3<R>(W.wl, i), F3<R>(W.ang_factor, i))));
}

// ---- Gauss-Seidel -------------------------------------------------------------------------------
// Exact reordering of GSSolver's sequential sweep: a row only reads and writes the vlambda /
// wlambda of its two bodies, and only dynamic bodies ever change them, so a row may run as
// soon as every earlier row touching one of its dynamic bodies has run.  The level of a row is
// its longest-path depth in that dependency graph; rows of one level touch disjoint dynamic
// bodies and run in parallel, and every row sees exactly the values it sees in the
// sequential order.
//
// A world's levels run on one group: a whole workgroup for a large world, a single wave for a small
// one (four small worlds share a workgroup, one per wave, and never meet at a workgroup barrier).

// a whole workgroup on one world
struct GBlock {
  int tid, n;
  __device__ GBlock() : tid(threadIdx.x), n(blockDim.x) {}
  __device__ void sync() const { __syncthreads(); }
  __device__ void lds_sync() const { lds_barrier(); }
  __device__ int imax(int v, int* sh) const {
    __syncthreads();
    if (tid == 0) sh[0] = 0;
    __syncthreads();
    atomicMax(&sh[0], v);
    __syncthreads();
    int r = sh[0];
    __syncthreads();
    return r;
  }
  __device__ int exscan(int* data, int cnt, int* sh) const { return array_exscan(data, cnt, sh); }
};
// one wave on one world: LDS and memory accesses of a wave are issued in program order, so a
// fence that waits for them replaces the barrier
struct GWave {
  int tid, n;
  __device__ GWave() : tid(threadIdx.x & 63), n(64) {}
  __device__ void sync() const { __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup"); }
  __device__ void lds_sync() const { __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront", "local"); }
  __device__ int imax(int v, int*) const {
    for (int off = 32; off > 0; off >>= 1) v = max(v, __shfl_xor(v, off, 64));
    return v;
  }
  __device__ int exscan(int* data, int cnt, int*) const {
    int carry = 0;
    for (int base = 0; base < cnt; base += 64) {
      int i = base + tid;
      int v = i < cnt ? data[i] : 0, incl = v;
      for (int off = 1; off < 64; off <<= 1) {
        int x = __shfl_up(incl, off, 64);
        if (tid >= off) incl += x;
      }
      if (i < cnt) data[i] = carry + incl - v;
      carry += __shfl(incl, 63, 64);
    }
    sync();
    return carry;
  }
};
// GS record: 6 groups of 4 words, row position k at words [k * 24, k * 24 + 24)
//   g0 sa.x sa.y sa.z ima  | g1 ra.x ra.y ra.z B    | g2 rb.x rb.y rb.z invC
//   g3 ia.x ia.y ia.z eps  | g4 ib.x ib.y ib.z minF | g5 a' maxF imb b'
// a' = a | (a dynamic) << 31, b' = b | (b dynamic) << 31, as in row_ab; imb (never negative) has its
// sign set when sb == -sa (else both spatial parts are +0).  The groups are
// what the four lanes of a row load (st_gs): each a Jacobian part and the part its impulse moves
// the velocity along, with one of the row's scalars in the fourth word; and a word each of g5.
template <typename R> struct GsWord;
template <> struct GsWord<float> {
  typedef unsigned int T;
  static __device__ __forceinline__ T put(float v) { return __float_as_uint(v); }
  static __device__ __forceinline__ float get(T w) { return __uint_as_float(w); }
};
template <> struct GsWord<double> {
  typedef unsigned long long T;
  static __device__ __forceinline__ T put(double v) { return (T)__double_as_longlong(v); }
  static __device__ __forceinline__ double get(T w) { return __longlong_as_double((long long)w); }
};
constexpr int GS_GROUPS = 6;

template <typename R> struct GsRow {
  f3 sa, ra, rb, ia, ib;
  R ima, imb, B, invC, eps, minF, maxF;
  unsigned a, b;
  bool neg;   // sb == -sa
};
// the sign bit of a word that holds an R
template <typename R> __device__ __forceinline__ bool flip_top(typename GsWord<R>::T w) { return (w >> (8 * sizeof(R) - 1)) != 0; }

template <typename R> __device__ __forceinline__ void gs_load(const typename GsWord<R>::T* base, int k, GsRow<R>& o) {
  typedef typename GsWord<R>::T T;
  T w[4 * GS_GROUPS];
#pragma unroll
  for (int g = 0; g < GS_GROUPS; g++) {
    const T* p = base + ((size_t)k * GS_GROUPS + g) * 4;
    if constexpr (sizeof(T) == 4) {
      uint4 v = *(const uint4*)p;
      w[4 * g] = v.x; w[4 * g + 1] = v.y; w[4 * g + 2] = v.z; w[4 * g + 3] = v.w;
    } else {
      ulonglong2 v0 = ((const ulonglong2*)p)[0], v1 = ((const ulonglong2*)p)[1];
      w[4 * g] = v0.x; w[4 * g + 1] = v0.y; w[4 * g + 2] = v1.x; w[4 * g + 3] = v1.y;
    }
  }
  auto F = [&](int i) { return (float)GsWord<R>::get(w[i]); };
  auto S = [&](int i) { return GsWord<R>::get(w[i]); };
  o.sa = mk3(F(0), F(1), F(2)); o.ra = mk3(F(4), F(5), F(6)); o.rb = mk3(F(8), F(9), F(10));
  o.ia = mk3(F(12), F(13), F(14)); o.ib = mk3(F(16), F(17), F(18));
  o.neg = flip_top<R>(w[22]);
  o.ima = S(3); o.imb = o.neg ? -S(22) : S(22); o.B = S(7); o.invC = S(11); o.eps = S(15); o.minF = S(19); o.maxF = S(21);
  o.a = (unsigned)w[20]; o.b = (unsigned)w[23];
}

template <typename R> __device__ __forceinline__ void gs_store(typename GsWord<R>::T* base, int k,
                                                               const RowRec<R>& r, unsigned fa, unsigned fb) {
  typedef typename GsWord<R>::T T;
  T w[4 * GS_GROUPS];
  auto P = [&](int i, R v) { w[i] = GsWord<R>::put(v); };
  P(0, r.sa.x); P(1, r.sa.y); P(2, r.sa.z); P(3, r.ima);
  P(4, r.ra.x); P(5, r.ra.y); P(6, r.ra.z); P(7, r.B);
  P(8, r.rb.x); P(9, r.rb.y); P(10, r.rb.z); P(11, r.invC);
  P(12, r.ia.x); P(13, r.ia.y); P(14, r.ia.z); P(15, r.eps);
  P(16, r.ib.x); P(17, r.ib.y); P(18, r.ib.z); P(19, r.minF);
  P(21, r.maxF);
  bool neg = !(r.kind == CHP_ROW_ROTATIONAL || r.kind == CHP_ROW_CONE || r.kind == CHP_ROW_MOTOR);
  P(22, neg ? -r.imb : r.imb);
  w[20] = (T)fa;
  w[23] = (T)fb;
#pragma unroll
  for (int g = 0; g < GS_GROUPS; g++) {
    T* p = base + ((size_t)k * GS_GROUPS + g) * 4;
    if constexpr (sizeof(T) == 4) {
      *(uint4*)p = make_uint4(w[4 * g], w[4 * g + 1], w[4 * g + 2], w[4 * g + 3]);
    } else {
      ((ulonglong2*)p)[0] = make_ulonglong2(w[4 * g], w[4 * g + 1]);
      ((ulonglong2*)p)[1] = make_ulonglong2(w[4 * g + 2], w[4 * g + 3]);
    }
  }
}

// Levels.  Consecutive rows on the same two bodies (a contact's two friction rows, the rows of
// one box-box contact patch, a joint's rows) form a run; inside a run each row depends on the
// one before it and on nothing later outside the run, so the run's rows take consecutive levels
// from the run's start level.  One wave walks the runs in solver order, 64 at a time (lev_walk).
// Rows without a dynamic body depend on nothing and take level 0.  The rows are then
// counting-sorted by level; the row builders write the GS records at the positions rpos this
// leaves.

// The walk of NR runs by the wave of lanes tid < 64.  A run starts one level above the last level
// of each of its dynamic bodies: last[] for the earlier chunks of 64, and inside the chunk the
// latest earlier lane on each body, whose end it waits for (the runs of a body have increasing
// levels, so its latest is its highest).  Those lanes come from a table of 64-bit lane masks by
// body, and the ends are relaxed until they stand; a chunk that is one long chain (joints) is
// finished by the pass over the lanes instead.  A relaxation round is two lane permutes where the
// pass is sixty-three dependent broadcasts, and a chunk of a pile takes three or four rounds.
//   tb: TB masks (a power of two; bodies share an entry when nb > TB), all zero and left so
//   rs(q): first and one past the last row of run q; put(q, v): the start level, -1 when not dynamic
// Returns the lane's part of the number of levels.
template <bool LDS, class RS, class PUT>
__device__ __forceinline__ int lev_walk(const int2* ab, int NR, int nb, int* last, unsigned long long* tb, int TB, RS rs, PUT put) {
  const int lane = (int)threadIdx.x & 63;
  const unsigned long long below = (1ull << lane) - 1ull;
  const bool shared = nb > TB;
  int lmax = 0;
  auto load_rs = [&](int c) { return c + lane < NR ? rs(c + lane) : make_int2(0, 0); };
  auto load_ab = [&](int2 r, int c) { return c + lane < NR ? ab[r.x] : make_int2(0, 0); };
  int2 rs_next = load_rs(0), x_next = load_ab(rs_next, 0), rs_after = load_rs(64);
  for (int c0 = 0; c0 < NR; c0 += 64) {
    const int q = c0 + lane;
    const bool act = q < NR;
    const int2 r = rs_next, x = x_next;
    x_next = load_ab(rs_after, c0 + 64);   // the runs' bounds are loaded two chunks ahead, their bodies one
    rs_next = rs_after;
    rs_after = load_rs(c0 + 128);
    const bool da = act && (x.x & GS_DYN), db = act && (x.y & GS_DYN), dyn = da || db;
    const int a = x.x & GS_IDX, b = x.y & GS_IDX, len = r.y - r.x;
    const int ka = da ? a : -1 - 2 * lane, kb = db ? b : -2 - 2 * lane;   // non-dynamic keys never match
    const int span = dyn ? len : 1;   // levels a run occupies
    unsigned long long *ta = tb + (a & (TB - 1)), *tbb = tb + (b & (TB - 1));
    if (da) atomicOr(ta, 1ull << lane);
    if (db) atomicOr(tbb, 1ull << lane);
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront", "local");
    unsigned long long ma = da ? *ta & below : 0ull, mb = db ? *tbb & below : 0ull;
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront", "local");
    if (da) *ta = 0ull;
    if (db) *tbb = 0ull;
    int lev = 0;
    if constexpr (LDS) {
      if (da) lev = max(lev, last[a] + 1);
      if (db) lev = max(lev, last[b] + 1);
    } else {
      if (da) lev = max(lev, atomicAdd(&last[a], 0) + 1);
      if (db) lev = max(lev, atomicAdd(&last[b], 0) + 1);
    }
    if (shared) {   // drop the lanes of other bodies from the top of the masks
      for (;;) {
        const int ja = ma ? 63 - __clzll(ma) : lane, jb = mb ? 63 - __clzll(mb) : lane;
        const int aa = __shfl(ka, ja, 64), ab_ = __shfl(kb, ja, 64), ba = __shfl(ka, jb, 64), bb = __shfl(kb, jb, 64);
        const bool xa = ma != 0 && aa != a && ab_ != a, xb = mb != 0 && ba != b && bb != b;
        if (xa) ma ^= 1ull << ja;
        if (xb) mb ^= 1ull << jb;
        if (!__any(xa || xb)) break;
      }
    }
    const int pa = ma ? 63 - __clzll(ma) : lane, pb = mb ? 63 - __clzll(mb) : lane;
    bool more = __any(pa != lane || pb != lane);
    for (int round = 0; more && round < 12; round++) {
      const int e = lev + span;   // one past the run's last level
      const int ea = __shfl(e, pa, 64), eb = __shfl(e, pb, 64);
      int nl = lev;
      if (pa != lane) nl = max(nl, ea);
      if (pb != lane) nl = max(nl, eb);
      more = __any(nl != lev);
      lev = nl;
    }
    if (more) {
      const int n = uni(min(64, NR - c0));
      int endv = lev + span - 1;
      for (int j = 0; j < n - 1; j++) {   // branch-free: exec-mask switches would sit on the chain
        const int kaj = __builtin_amdgcn_readlane(ka, j), kbj = __builtin_amdgcn_readlane(kb, j);
        const int endj = __builtin_amdgcn_readlane(endv, j);
        const int hit = (int)(lane > j) & ((int)(ka == kaj) | (int)(ka == kbj) | (int)(kb == kaj) | (int)(kb == kbj));
        lev = max(lev, hit ? endj + 1 : 0);
        endv = lev + span - 1;
      }
    }
    // the chain through a body has increasing levels: the chunk's last run on it wins
    if (da) atomicMax(&last[a], lev + span - 1);
    if (db) atomicMax(&last[b], lev + span - 1);
    if (act) {
      put(q, dyn ? lev : -1);
      lmax = max(lmax, lev + span);
    }
  }
  return lmax;
}

// Rows in LDS: a world of at most `cap` rows keeps its runs, levels and histogram there, so that
// the passes around the walk cost LDS accesses instead of a memory round trip each.
//   lds: lev_lds_bytes(nbcap, TB, cap)
__host__ __device__ constexpr size_t lev_lds_bytes(int nbcap, int TB, int cap) {
  return ((((size_t)TB + cap / 64) * 8 + (size_t)nbcap * 4 + ((size_t)cap + 2) * 6) + 15) & ~(size_t)15;
}
template <typename R, typename G>
__device__ __forceinline__ void st_levels_lds(const DevWorld<R>& W, const G& g, int* sh, void* lds, int nbcap, int TB, int cap) {
  const int E = uni(W.counters[C_ROWS]), nb = W.nb, tid = g.tid, bd = g.n;
  const int lane = tid & 63, wv = uni(tid >> 6), nw = bd >> 6;
  const int2* ab = (const int2*)W.row_ab;
  unsigned long long* tb = (unsigned long long*)lds;
  unsigned long long* first = tb + TB;   // bit r: row r starts a run
  int* last = (int*)(first + cap / 64);
  unsigned short* rid = (unsigned short*)(last + nbcap);   // run of each row, then its level
  unsigned short* rst = rid + cap + 2;                     // first row of each run (+ E at the end)
  unsigned short* rlv = rst + cap + 2;                     // start level of each run, 0xffff: not dynamic
  int* hist = (int*)rst;                                   // after the levels: cap + 2 ints in their place
  for (int k = tid; k < TB; k += bd) tb[k] = 0ull;
  for (int b = tid; b < nb; b += bd) last[b] = -1;
  // runs: a row starts one when its body pair differs from the previous row's.  Each wave takes a
  // contiguous stretch of 64-row words
  const int words = (E + 63) >> 6, per = (words + nw - 1) / nw, w0 = min(words, wv * per), w1 = min(words, w0 + per);
  int c = 0;
  for (int w = w0; w < w1; w++) {
    const int r = 64 * w + lane;
    const int2 x = r < E ? ab[r] : make_int2(0, 0), y = r > 0 && r < E ? ab[r - 1] : make_int2(-1, -1);
    const unsigned long long m = __ballot(r < E && (r == 0 || x.x != y.x || x.y != y.y));
    if (lane == 0) first[w] = m;
    c += __popcll(m);
  }
  int before = 0, NR = c;
  if (nw > 1) {
    if (lane == 0) sh[wv] = c;
    g.lds_sync();
    NR = 0;
    for (int u = 0; u < nw; u++) {
      const int t = sh[u];
      before += u < wv ? t : 0;
      NR += t;
    }
  }
  g.lds_sync();
  NR = uni(NR);
  for (int w = w0; w < w1; w++) {
    const int r = 64 * w + lane;
    const unsigned long long m = first[w];
    const int id = before + __popcll(m & (~0ull >> (63 - lane))) - 1;
    if (r < E) {
      rid[r] = (unsigned short)id;
      if ((m >> lane) & 1ull) rst[id] = (unsigned short)r;
    }
    before += __popcll(m);
  }
  if (tid == 0) rst[NR] = (unsigned short)E;
  g.lds_sync();
  int lmax = 0;
  if (tid < 64)
    lmax = lev_walk<true>(ab, NR, nb, last, tb, TB, [&](int q) { return make_int2(rst[q], rst[q + 1]); },
                          [&](int q, int v) { rlv[q] = (unsigned short)v; });
  const int L = uni(g.imax(lmax, sh));   // (a barrier for the whole group)
  g.lds_sync();
  for (int r = tid; r < E; r += bd) {
    const int id = rid[r], l0 = rlv[id];
    rid[r] = (unsigned short)(l0 == 0xffff ? 0 : l0 + (r - (int)rst[id]));
  }
  g.lds_sync();
  // counting sort by level; the order inside a level is free (its rows are independent)
  for (int l = tid; l <= L; l += bd) hist[l] = 0;
  g.lds_sync();
  for (int r = tid; r < E; r += bd) atomicAdd(&hist[rid[r]], 1);
  g.lds_sync();
  g.exscan(hist, L + 1, sh);
  for (int l = tid; l <= L; l += bd) W.lvl_start[l] = hist[l];
  g.lds_sync();
  for (int r = tid; r < E; r += bd) {
    const int k = atomicAdd(&hist[rid[r]], 1);
    W.sched[k] = r;
    W.rpos[r] = k;
  }
  if (tid == 0) W.counters[C_LEVELS] = L;
}

// Rows in memory (any number of them).
//   last: nb ints (LDS when LDS, else the world's global scratch, read with atomics so that
//         each chunk sees the previous chunk's values)
//   hist: hist_cap ints of LDS for the level histogram (global scratch when L + 1 > hist_cap)
//   tb: TB lane masks in LDS
template <typename R, typename G, bool LDS>
__device__ __forceinline__ void st_levels(const DevWorld<R>& W, const G& g, int* sh, int* last, int* hist, int hist_cap,
                                          unsigned long long* tb, int TB) {
  const int E = uni(W.counters[C_ROWS]), nb = W.nb;
  const int tid = g.tid, bd = g.n;
  const int2* ab = (const int2*)W.row_ab;
  int* runid = W.level;     // run of each row, then its level
  int* rstart = W.rpos;     // first row of each run (+ E at the end), until the sort below
  int* rlev = W.sched;      // start level of each run, until the sort below
  for (int k = tid; k < TB; k += bd) tb[k] = 0ull;
  for (int b = tid; b < nb; b += bd) last[b] = -1;
  // The passes over the rows take LU rows per thread per turn, loading all of them before any
  // store: each turn then waits for one round of loads rather than one per row.
  constexpr int LU = 4;
  // runs: a row starts one when its body pair differs from the previous row's
  for (int r0 = tid; r0 < E; r0 += LU * bd) {
    int2 x[LU], xp[LU];
#pragma unroll
    for (int u = 0; u < LU; u++) {
      const int r = r0 + u * bd;
      x[u] = r < E ? ab[r] : make_int2(0, 0);
      xp[u] = r > 0 && r < E ? ab[r - 1] : make_int2(-1, -1);
    }
#pragma unroll
    for (int u = 0; u < LU; u++) {
      const int r = r0 + u * bd;
      if (r < E) runid[r] = (r == 0 || x[u].x != xp[u].x || x[u].y != xp[u].y) ? 1 : 0;
    }
  }
  g.sync();
  const int NR = uni(g.exscan(runid, E, sh));
  for (int r0 = tid; r0 < E; r0 += LU * bd) {
    int2 x[LU], xp[LU];
    int rid[LU];
#pragma unroll
    for (int u = 0; u < LU; u++) {
      const int r = r0 + u * bd;
      x[u] = r < E ? ab[r] : make_int2(0, 0);
      xp[u] = r > 0 && r < E ? ab[r - 1] : make_int2(-1, -1);
      rid[u] = r < E ? runid[r] : 0;
    }
#pragma unroll
    for (int u = 0; u < LU; u++) {
      const int r = r0 + u * bd;
      if (r < E) {
        const bool first = r == 0 || x[u].x != xp[u].x || x[u].y != xp[u].y;
        const int id = rid[u] + (first ? 1 : 0) - 1;
        runid[r] = id;
        if (first) rstart[id] = r;
      }
    }
  }
  if (tid == 0) rstart[NR] = E;
  g.sync();
  int lmax = 0;
  if (tid < 64)
    lmax = lev_walk<LDS>(ab, NR, nb, last, tb, TB, [&](int q) { return make_int2(rstart[q], rstart[q + 1]); },
                         [&](int q, int v) { rlev[q] = v; });
  const int L = uni(g.imax(lmax, sh));
  g.sync();
  for (int r0 = tid; r0 < E; r0 += LU * bd) {
    int id[LU], l0[LU], rs[LU];
#pragma unroll
    for (int u = 0; u < LU; u++) id[u] = r0 + u * bd < E ? runid[r0 + u * bd] : 0;
#pragma unroll
    for (int u = 0; u < LU; u++) {
      l0[u] = rlev[id[u]];
      rs[u] = rstart[id[u]];
    }
#pragma unroll
    for (int u = 0; u < LU; u++) {
      const int r = r0 + u * bd;
      if (r < E) runid[r] = l0[u] < 0 ? 0 : l0[u] + (r - rs[u]);
    }
  }
  g.sync();
  // counting sort by level; the order inside a level is free (its rows are independent)
  auto sort = [&](int* cnt) {
    for (int l = tid; l <= L; l += bd) cnt[l] = 0;
    g.sync();
    for (int r0 = tid; r0 < E; r0 += LU * bd) {
      int lv[LU];
#pragma unroll
      for (int u = 0; u < LU; u++) lv[u] = r0 + u * bd < E ? W.level[r0 + u * bd] : -1;
#pragma unroll
      for (int u = 0; u < LU; u++)
        if (lv[u] >= 0) atomicAdd(&cnt[lv[u]], 1);
    }
    g.sync();
    g.exscan(cnt, L + 1, sh);
    for (int l = tid; l <= L; l += bd) W.lvl_start[l] = cnt[l];
    g.sync();
    for (int r0 = tid; r0 < E; r0 += LU * bd) {
      int lv[LU];
#pragma unroll
      for (int u = 0; u < LU; u++) lv[u] = r0 + u * bd < E ? W.level[r0 + u * bd] : -1;
#pragma unroll
      for (int u = 0; u < LU; u++)
        if (lv[u] >= 0) {
          const int r = r0 + u * bd;
          const int k = atomicAdd(&cnt[lv[u]], 1);
          W.sched[k] = r;
          W.rpos[r] = k;
        }
    }
    g.sync();
  };
  if (L + 1 <= hist_cap) sort(hist);
  else sort(W.last_level);
  if (tid == 0) W.counters[C_LEVELS] = L;
}

// GSSolver.solve iterations (gs_solver.dart:76-108) + Equation.computeGWlambda /
// addToWlambda (equation_class.dart:95-105, 151-169) over the level schedule.
//
// Early exit: the reference sums |dlambda| in row order and stops once (sum)^2 < tol^2.  Here
// every thread adds its rows' |dlambda| in double and the group adds the partials; the rounding
// error of the sequential R sum is at most gamma_{E-1} * sum (all terms are >= 0), so the
// comparison is decided from the double sum whenever the interval around it does not straddle
// the threshold.  Otherwise one thread repeats the sequential R sum in solver order from the
// stored |dlambda|.  Either way the decision is the reference's, bit for bit.
template <typename R> __device__ __forceinline__ int gs_decide(double D, int n, R tol2) {
  const double u = sizeof(R) == 4 ? 0x1p-24 : 0x1p-53, ud = 0x1p-53;
  double g = (double)n * u / (1.0 - (double)n * u), gd = (double)n * ud / (1.0 - (double)n * ud);
  double slack = 2.0 * (g + gd) + 1e-15;
  double hi = D * (1.0 + slack), lo = D * (1.0 - slack);
  R hiR, loR;
  if constexpr (sizeof(R) == 4) { hiR = __double2float_ru(hi); loR = __double2float_rd(lo); }
  else { hiR = hi; loR = lo; }
  if (hiR * hiR < tol2) return 1;    // exit whatever the rounding of the sequential sum
  if (loR * loR >= tol2) return 0;   // continue whatever it is
  return -1;                         // undecided, or NaN: the sequential sum decides
}

// One row of a sweep by one thread (SplitSolver's islands): computeGWlambda, the clamped
// dlambda, addToWlambda.  lam: the row's lambda and |dlambda|.  Returns |dlambda|.
template <typename R> __device__ __forceinline__ R gs_row(const GsRow<R>& cr, float* vw, R* lam) {
  const int a = cr.a & GS_IDX, b = cr.b & GS_IDX;
  const bool da = cr.a & GS_DYN, db = cr.b & GS_DYN;
  const f3 z = mk3(0.f, 0.f, 0.f);
  const f3 sb = cr.neg ? neg3(cr.sa) : z;
  const R clam = lam[0];
  float4 va4 = ((const float4*)vw)[2 * a], wa4 = ((const float4*)vw)[2 * a + 1];
  float4 vb4 = ((const float4*)vw)[2 * b], wb4 = ((const float4*)vw)[2 * b + 1];
  f3 va = mk3(va4.x, va4.y, va4.z), wa = mk3(wa4.x, wa4.y, wa4.z);
  f3 vb = mk3(vb4.x, vb4.y, vb4.z), wb = mk3(wb4.x, wb4.y, wb4.z);
  R gwl = mulvec<R>(va, wa, cr.sa, cr.ra) + mulvec<R>(vb, wb, sb, cr.rb);
  R dl = cr.invC * (cr.B - gwl - cr.eps * clam);
  const R t = clam + dl;   // the clamp of gs_solver.dart:91-96
  dl = t < cr.minF ? cr.minF - clam : (t > cr.maxF ? cr.maxF - clam : dl);
  R adlv = dl > (R)0 ? dl : -dl;
  lam[0] = clam + dl;
  if (da) {
    va = axpy3<R>(va, cr.ima * dl, cr.sa);
    wa = axpy3<R>(wa, dl, cr.ia);
    ((float4*)vw)[2 * a] = make_float4(va.x, va.y, va.z, 0.f);
    ((float4*)vw)[2 * a + 1] = make_float4(wa.x, wa.y, wa.z, 0.f);
  }
  if (db) {
    if (a == b) { vb = va; wb = wa; }
    vb = axpy3<R>(vb, cr.imb * dl, sb);
    wb = axpy3<R>(wb, dl, cr.ib);
    ((float4*)vw)[2 * b] = make_float4(vb.x, vb.y, vb.z, 0.f);
    ((float4*)vw)[2 * b + 1] = make_float4(wb.x, wb.y, wb.z, 0.f);
  }
  return adlv;
}

// values of the other lanes of a row's four (CTRL: a DPP quad permutation)
template <int CTRL, typename T> __device__ __forceinline__ T quad(T v) { return dpp<CTRL>(v); }
constexpr int QP_SWAP1 = 0xB1, QP_SWAP2 = 0x4E;   // [1,0,3,2] [2,3,0,1]
constexpr int QP_LANE0 = 0x00, QP_LANE1 = 0x55, QP_LANE3 = 0xFF, QP_LANES0033 = 0xF0;   // [0,..] [1,..] [3,..] [0,0,3,3]
// v with its sign flipped where the top bit of m is set
__device__ __forceinline__ float flip_sign(float v, unsigned m) { return __uint_as_float(__float_as_uint(v) ^ m); }
__device__ __forceinline__ double flip_sign(double v, unsigned m) {
  return __longlong_as_double(__double_as_longlong(v) ^ ((long long)m << 32));
}
// one group of four words of a GS record
template <typename R> struct GsQuad {
  typename GsWord<R>::T w[4];
  __device__ __forceinline__ void load(const typename GsWord<R>::T* p) {
    if constexpr (sizeof(R) == 4) {
      const uint4 v = *(const uint4*)p;
      w[0] = v.x; w[1] = v.y; w[2] = v.z; w[3] = v.w;
    } else {
      const ulonglong2 v0 = ((const ulonglong2*)p)[0], v1 = ((const ulonglong2*)p)[1];
      w[0] = v0.x; w[1] = v0.y; w[2] = v1.x; w[3] = v1.y;
    }
  }
  __device__ __forceinline__ R get(int i) const { return GsWord<R>::get(w[i]); }
};

// GSSolver's sweeps over the level schedule by NW waves on one world (NW = 1: one wave, no
// barrier).
//
// Four lanes run a row: lane p of the four holds one of va, wa, vb, wb, does that part's dot
// product and impulse, and the four partial products meet in two DPP additions, in the
// reference's order ((va.sa + wa.ra) + (vb.sb + wb.rb)).  The sweep is a chain of dependent steps
// whose cost is the instructions one wave issues per step; with a lane doing a whole row a step
// was about 160 of them (four body loads and stores, 24 record words), with four it is about
// half that.
//
// A step is at most 16 * NW rows of one level.  ss[t] is the first row position of step t (ss[Lp]
// = E), the sweep is padded to a multiple of the ring depth D with empty steps, and each thread's
// record and lambda are loaded D steps ahead into a ring of registers.  A sweep is at least D
// steps, so a row's lambda is stored before it is loaded again, by the same threads.  A thread
// without a row runs the record at position E, all zeros, whose impulse is zero; its writes, and
// those of bodies that are not dynamic, go to a spare body slot at nb.
//
// Within a step the next step's body velocities are read straight after this step's are written
// (the barrier between them when NW > 1), and the ring's loads are issued while they arrive.
//   vw: 8 floats per body slot (vlambda xyz, pad, wlambda xyz, pad), nb + 1 slots, in LDS when LDS
//   ss: gs_steps + 1 ints (in LDS or global memory)
//   SELF: rows whose two bodies are one may be present (the Solver slot may be given them)
//   WIDE: record offsets may pass 32 bits
// an upper bound of the entries a sweep's step table takes
__host__ __device__ constexpr int gs_steps(int L, int E, int rows_per_step, int D) { return L + E / rows_per_step + D; }
// rows whose record offsets fit 24 x 24 bit multiplications (full rate) and 32 bits
template <typename R> constexpr int gs_narrow_rows() {
  const unsigned k = 0xffffffffu / (4 * GS_GROUPS * sizeof(R)) - 1;
  return (int)(k < 0xffffffu ? k : 0xffffffu);
}
template <typename R, int NW, int D, bool LDS, bool SELF, bool WIDE>
__device__ __forceinline__ void st_gs(const DevWorld<R>& W, float* vw, int* ss, double* shd, int* sh, bool keep) {
  constexpr int T = 64 * NW, RP = 16 * NW;
  const int tid = NW == 1 ? (int)(threadIdx.x & 63) : (int)threadIdx.x, p = tid & 3, row = tid >> 2;
  const int E = uni(W.counters[C_ROWS]), L = uni(W.counters[C_LEVELS]), iters = uni(W.iterations), nb = uni(W.nb);
  const R tol2 = W.tol2;
  typedef typename GsWord<R>::T WT;
  auto sync = [&]() {
    if constexpr (NW == 1) __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    else __syncthreads();
  };
  auto step_sync = [&]() {   // the next step reads what this one wrote
    if constexpr (NW == 1) __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront", "local");
    else if constexpr (LDS) lds_barrier();
    else __syncthreads();
  };
  for (int i = tid; i < 8 * (nb + 1); i += T) vw[i] = 0.f;
  int Lp = 0;
  if (E != 0 && iters > 0) {
    if (tid < 64) {   // the step table: level l is cut into steps of RP rows
      for (int l0 = 0; l0 < L; l0 += 64) {
        const int l = l0 + tid;
        const int a0 = l < L ? W.lvl_start[l] : 0, a1 = l < L ? W.lvl_start[l + 1] : 0;
        const int n = (a1 - a0 + RP - 1) / RP, inc = wave_incl_scan(n);
        for (int j = 0; j < n; j++) ss[Lp + inc - n + j] = a0 + j * RP;
        Lp += __shfl(inc, 63, 64);
      }
      if (NW > 1 && tid == 0) sh[0] = Lp;
    }
    if constexpr (NW > 1) {
      __syncthreads();
      Lp = sh[0];
    }
    Lp = uni(Lp);
  }
  const int Lpad = max(1, (Lp + D - 1) / D) * D;
  for (int t = Lp + tid; t <= Lpad; t += T) ss[t] = E;
  const char* gsr = (const char*)(const WT*)W.gsr;
  char* lam = (char*)(R*)W.glam;
  constexpr unsigned REC = 4 * GS_GROUPS * sizeof(R), LAM = 2 * sizeof(R);   // bytes per row
  if (tid < 4 * GS_GROUPS) ((WT*)(gsr + (size_t)E * REC))[tid] = (WT)0;      // the idle threads' record
  if (tid < 2) ((R*)(lam + (size_t)E * LAM))[tid] = (R)0;
  sync();
  int it = 0;
  if (E != 0 && iters > 0) {
    // this lane's groups of a record, its half of a body slot, the sign of its spatial part
    const unsigned oa = (p == 1 ? 4u : p == 3 ? 8u : 0u) * sizeof(R), ok = (p == 1 ? 12u : p == 3 ? 16u : 0u) * sizeof(R);
    const unsigned negm = p == 2 ? 0x80000000u : 0u, half = (p & 1) * 16u, spare = 32u * nb + half;
    const bool first = p < 2, odd = p & 1;
    char* vb = (char*)vw;
    GsQuad<R> qa[D], qk[D];
    // g5: a word per lane, handed round the four (a quarter of the bytes the loads move, two
    // permutations more), or all of it in each lane.  The word wins where the loads are what the
    // steps wait for and loses where one world's four waves wait for each other: half a batch
    // of 1024 chains 1167 -> 1063 us, of 2048 piles 334 -> 322, a 16,384-body world 4.01 -> 3.74 ms,
    // a 300-body pile in double 290 -> 253, but in single 83 -> 92.  Four waves in single take the
    // whole group however many of their workgroups there are: the word was measured there on one
    // world and on the piles' mixture, not on hundreds of worlds of four waves each
    constexpr bool WORD = sizeof(R) == 8 || NW != 4;
    GsQuad<R> qc[WORD ? 1 : D];
    WT qw[WORD ? D : 1];
    const unsigned oc = (WORD ? 20u + p : 20u) * (unsigned)sizeof(R);
    R ql[D];
    unsigned qr[D];   // the row's position
    int pt = 0, s0, s1;   // the next step to load and its rows
    auto fetch = [&]() { s0 = ss[pt]; s1 = ss[pt + 1]; };
    auto load = [&](int s) {
      const unsigned k = (unsigned)(s0 + row < s1 ? s0 + row : E);
      if constexpr (WIDE) {
        const size_t o = (size_t)k * REC;
        qa[s].load((const WT*)(gsr + (o + oa)));
        qk[s].load((const WT*)(gsr + (o + ok)));
        if constexpr (WORD) qw[s] = *(const WT*)(gsr + (o + oc));
        else qc[s].load((const WT*)(gsr + (o + oc)));
        ql[s] = *(const R*)(lam + (size_t)k * LAM);
      } else {
        qa[s].load((const WT*)(gsr + (__umul24(k, REC) + oa)));
        qk[s].load((const WT*)(gsr + (__umul24(k, REC) + ok)));
        if constexpr (WORD) qw[s] = *(const WT*)(gsr + (__umul24(k, REC) + oc));
        else qc[s].load((const WT*)(gsr + (__umul24(k, REC) + oc)));
        ql[s] = *(const R*)(lam + k * LAM);
      }
      qr[s] = k;
      pt = pt + 1 == Lpad ? 0 : pt + 1;
    };
    // a' or b' of slot s's row; the half of that body's slot this lane reads
    auto word = [&](int s) {
      if constexpr (WORD) return (unsigned)__builtin_amdgcn_update_dpp(0, (int)qw[s], QP_LANES0033, 0xf, 0xf, true);
      else return first ? (unsigned)qc[s].w[0] : (unsigned)qc[s].w[3];
    };
    auto body = [&](int s) { return (word(s) << 5) + half; };
    // The sweeps run in an inner loop whose only memory traffic is the ring's loads and the
    // lambda stores.  The rare undecided early-exit test reads the stored |dlambda| outside
    // it, and the ring then starts again at the first step of the next sweep.
    for (;;) {
      pt = 0;
#pragma unroll
      for (int s = 0; s < D; s++) {
        fetch();
        load(s);
        __builtin_amdgcn_sched_barrier(0);   // the slots' loads stay in slot order
      }
      fetch();
      int step = 0, dec = 0;   // dec, the sweep-end decision: 1 stop, -1 undecided
      double part = 0.0;
      unsigned at = body(0);
      float4 v4 = *(const float4*)(vb + at);
      for (;;) {
#pragma unroll
        for (int s = 0; s < D; s++) {
          // nothing of another slot's step may move into this one: an instruction that reads a
          // slot's row before its own step makes the wave wait for that row's loads, and the
          // ring then hides no latency
          __builtin_amdgcn_sched_barrier(0);
          const unsigned w = word(s);
          WT wi;       // imb: lane 2's
          R maxF;
          if constexpr (WORD) {
            wi = qw[s];
            maxF = quad<QP_LANE1>(GsWord<R>::get(wi));
          } else {
            wi = qc[s].w[2];
            maxF = qc[s].get(1);
          }
          const unsigned neg = (unsigned)(wi >> (8 * sizeof(R) - 32)) & negm;
          const R jx = flip_sign(qa[s].get(0), neg), jy = flip_sign(qa[s].get(1), neg), jz = flip_sign(qa[s].get(2), neg);
          R d = (R)v4.x * jx;
          d += (R)v4.y * jy;
          d += (R)v4.z * jz;
          d += quad<QP_SWAP1>(d);
          const R gwl = d + quad<QP_SWAP2>(d);
          const R own = qa[s].get(3);
          const R B = quad<QP_LANE1>(own), invC = quad<QP_LANE3>(own);
          const R eps = quad<QP_LANE1>(qk[s].get(3)), minF = quad<QP_LANE3>(qk[s].get(3));
          const R clam = ql[s];
          R dl = invC * (B - gwl - eps * clam);
          // the clamp of gs_solver.dart:91-96 as selects; NaN compares false, as in the branches
          const R t = clam + dl;
          dl = t < minF ? minF - clam : (t > maxF ? maxF - clam : dl);
          // va += (ima dl) sa, wa += dl ia, vb += (imb dl) sb, wb += dl ib
          const R c = odd ? (R)1 : (first ? own : (R)fabs(GsWord<R>::get(wi)));
          const R sc = flip_sign(c * dl, neg);
          const R kx = qk[s].get(0), ky = qk[s].get(1), kz = qk[s].get(2);
          float4 o = make_float4((float)((R)v4.x + sc * kx), (float)((R)v4.y + sc * ky), (float)((R)v4.z + sc * kz), 0.f);
          unsigned to = (w & GS_DYN) ? at : spare;
          if constexpr (SELF) {   // one body on both sides: its second impulse follows the first
            const unsigned wa = (unsigned)__builtin_amdgcn_update_dpp(0, (int)w, QP_LANE0, 0xf, 0xf, true);
            const unsigned wb = (unsigned)__builtin_amdgcn_update_dpp(0, (int)w, QP_LANE3, 0xf, 0xf, true);
            const bool same = ((wa ^ wb) & GS_IDX) == 0;
            const float ax = quad<0x44>(o.x), ay = quad<0x44>(o.y), az = quad<0x44>(o.z);   // lanes 0, 1, 0, 1
            if (same && !first && (wa & GS_DYN))
              o = make_float4((float)((R)ax + sc * kx), (float)((R)ay + sc * ky), (float)((R)az + sc * kz), 0.f);
            if (same && first) to = spare;
          }
          *(float4*)(vb + to) = o;
          step_sync();
          at = body((s + 1) % D);
          v4 = *(const float4*)(vb + at);
          __builtin_amdgcn_sched_barrier(0);
          const R adlv = (R)fabs(dl);
          part += (double)adlv;
          R* lp = (R*)(WIDE ? lam + (size_t)qr[s] * LAM : lam + qr[s] * LAM);
          if constexpr (sizeof(R) == 4) *(float2*)lp = make_float2((float)(clam + dl), (float)adlv);
          else *(double2*)lp = make_double2((double)(clam + dl), (double)adlv);
          load(s);   // the slot's next row (D steps on)
          fetch();
        }
        step += D;
        if (step == Lpad) {   // end of a sweep: GSSolver's early-exit test
          step = 0;
          double S = part;
          for (int off = 32; off > 0; off >>= 1) S += __shfl_xor(S, off, 64);
          if constexpr (NW > 1) {
            if ((tid & 63) == 0) shd[tid >> 6] = S;
            lds_barrier();
            S = 0.0;
            for (int u = 0; u < NW; u++) S += shd[u];
            lds_barrier();
          }
          part = 0.0;
          dec = uni(gs_decide<R>(0.25 * S, E, tol2));   // the four lanes of a row add the same |dlambda|
          if (dec != 0) break;
          if (++it == iters) {
            dec = 1;
            break;
          }
        }
      }
      if (dec > 0) break;
      // undecided: the sequential sum in solver order decides (every |dlambda| of the sweep is
      // stored)
      sync();
      int vv = 0;
      if (tid == 0) {
        const int* rpos = W.rpos;
        R tot = 0;
        for (int r = 0; r < E; r++) tot += ((const R*)(lam + (size_t)(unsigned)rpos[r] * LAM))[1];
        vv = tot * tot < tol2 ? 1 : 0;
        if (NW > 1) sh[0] = vv;
      }
      if constexpr (NW > 1) {
        __syncthreads();
        vv = sh[0];
        __syncthreads();
      } else {
        vv = __shfl(vv, 0, 64);
      }
      if (uni(vv) || ++it == iters) break;
      // next sweep: the ring starts again at its first step
    }
    sync();
    // Equation.multiplier and the capture read lambda from the row records (keep)
    if (keep)
      for (int k = tid; k < E; k += T) W.rows[W.sched[k]].lambda = *(const R*)(lam + (size_t)k * LAM);
  }
  // hand the lambda velocities to st_post
  for (int i = tid; i < nb; i += T) {
    const float4 v = ((const float4*)vw)[2 * i], w = ((const float4*)vw)[2 * i + 1];
    S3<R>(W.vl, i, mk3(v.x, v.y, v.z));
    S3<R>(W.wl, i, mk3(w.x, w.y, w.z));
  }
  if (tid == 0) W.counters[C_ITERS] = it;
}

// ---- interpolation (World.step with timeSinceLastCalled, world_class.dart:421-428) ----------------
// Quaternion.slerp (quaternion.dart:118-168)
template <typename R> __device__ __forceinline__ f4 slerp4(f4 a, f4 b, R t) {
  const R ax = a.x, ay = a.y, az = a.z, aw = a.w;
  R bx = b.x, by = b.y, bz = b.z, bw = b.w;
  R cosom = ax * bx + ay * by + az * bz + aw * bw;
  if (cosom < (R)0) {
    cosom = -cosom;
    bx = -bx; by = -by; bz = -bz; bw = -bw;
  }
  R s0, s1;
  if ((R)1 - cosom > (R)0.000001) {
    const R omega = acos(cosom), sinom = sin(omega);
    s0 = sin(((R)1 - t) * omega) / sinom;
    s1 = sin(t * omega) / sinom;
  } else {
    s0 = (R)1 - t;
    s1 = t;
  }
  f4 r;
  r.x = st<R>(s0 * ax + s1 * bx); r.y = st<R>(s0 * ay + s1 * by);
  r.z = st<R>(s0 * az + s1 * bz); r.w = st<R>(s0 * aw + s1 * bw);
  return r;
}
// body i: interpolatedPosition = previousPosition.lerp(position, t), interpolatedQuaternion =
// previousQuaternion.slerp(quaternion, t), then previousQuaternion.normalize()
template <typename R> __device__ void interp_body(const DevWorld<R>& W, int i, R t) {
  ((f3*)W.interp_pos)[i] = lerp3<R>(((const f3*)W.prev_pos)[i], F3<R>(W.pos, i), t);
  f4 a = ((const f4*)W.prev_quat)[i];
  ((f4*)W.interp_quat)[i] = slerp4<R>(a, ((const f4*)W.quat)[i], t);
  const R x = a.x, y = a.y, z = a.z, w = a.w;
  const R l = sqrt((x * x) + (y * y) + (z * z) + (w * w));   // vector_math Quaternion.normalize
  if (l != (R)0) {
    const R d = (R)1 / l;
    a.x = st<R>(x * d); a.y = st<R>(y * d); a.z = st<R>(z * d); a.w = st<R>(w * d);
    ((f4*)W.prev_quat)[i] = a;
  }
}

// ---- sleep ------------------------------------------------------------------------------------
// the wake-up marks of one contact side (world_class.dart:562-590): sleeping dynamic body a,
// allowed to sleep, touched by awake non-static body b whose speed^2 (|v|^2 + |w|^2) is at least
// twice b's sleep speed limit squared
template <typename R> __device__ __forceinline__ bool wake_mark(const DevWorld<R>& W, int a, int b) {
  if (!(W.flags[a] & BF_ALLOW_SLEEP) || W.type[a] != CHP_BODY_DYNAMIC || W.sleep_state[a] != CHP_SLEEP_SLEEPING)
    return false;
  if (W.sleep_state[b] != CHP_SLEEP_AWAKE || W.type[b] == CHP_BODY_STATIC) return false;
  const R s2 = len2<R>(F3<R>(W.vel, b)) + len2<R>(F3<R>(W.avel, b));
  const R lim = W.sleep_speed[b];
  return s2 >= lim * lim * (R)2;
}
// Body.wakeUpAfterNarrowphase over the step's contacts, then the wake-up pass after them
// (world_class.dart:617-624): a woken body is awake and gets its solve mass back before the
// solver reads it.  The marks read only the states from before the pass, so the contacts' order
// does not matter.  One workgroup per world.
template <typename R> __device__ void st_wake(const DevWorld<R>& W) {
  const int nc = W.counters[C_STAGING];
  for (int k = threadIdx.x; k < nc; k += blockDim.x) {
    const int bi = W.contacts[k].bi, bj = W.contacts[k].bj;
    if (wake_mark(W, bi, bj)) atomicOr(&W.flags[bi], (int)BF_WAKE);
    if (wake_mark(W, bj, bi)) atomicOr(&W.flags[bj], (int)BF_WAKE);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < W.nb; i += blockDim.x) {
    const int fl = W.flags[i];
    if (!(fl & BF_WAKE)) continue;
    W.flags[i] = fl & ~BF_WAKE;
    W.sleep_state[i] = CHP_SLEEP_AWAKE;
    W.ims[i] = W.inv_mass[i];   // a dynamic body: Body.updateSolveMassProperties
    for (int k = 0; k < 9; k++) W.iiws[9 * i + k] = W.iiw[9 * i + k];
  }
}
// Body.sleepTick (rigid_body.dart:280-300) at World.time before this step's increment, on the
// velocities the step leaves; Body.sleep() zeroes them
template <typename R> __device__ __forceinline__ void sleep_tick(const DevWorld<R>& W, int i, f3& v, f3& w) {
  const int s = W.sleep_state[i];
  const R s2 = len2<R>(v) + len2<R>(w);
  const R lim = W.sleep_speed[i], l2 = lim * lim;
  const double t = W.wtime[0];
  if (s == CHP_SLEEP_AWAKE && s2 < l2) {
    W.sleep_state[i] = CHP_SLEEP_SLEEPY;
    W.sleep_tls[i] = t;
  } else if (s == CHP_SLEEP_SLEEPY && s2 > l2) {
    W.sleep_state[i] = CHP_SLEEP_AWAKE;
  } else if (s == CHP_SLEEP_SLEEPY && t - W.sleep_tls[i] > W.sleep_time[i]) {
    W.sleep_state[i] = CHP_SLEEP_SLEEPING;
    v = mk3(0.f, 0.f, 0.f);
    w = mk3(0.f, 0.f, 0.f);
  }
}

// body i's velocity update, damping, integration and sleep timer; false when its pose turned
// non-finite
template <typename R> __device__ bool post_body(const DevWorld<R>& W, int i, R dt, int E, bool qn) {
  bool ok = true;
  // Body.integrate saves the pose first, for every body (rigid_body.dart:628-630)
  ((f3*)W.prev_pos)[i] = F3<R>(W.pos, i);
  ((f4*)W.prev_quat)[i] = ((const f4*)W.quat)[i];
  f3 v = F3<R>(W.vel, i), w = F3<R>(W.avel, i);
  f3 lf = F3<R>(W.lin_factor, i), af = F3<R>(W.ang_factor, i);
  if (E != 0 && (W.solver_kind != CHP_SOLVER_SPLIT || (W.flags[i] & BF_SOLVED))) {
    v = add3<R>(v, mul3<R>(F3<R>(W.vl, i), lf));
    w = add3<R>(w, mul3<R>(F3<R>(W.wl, i), af));
  }
  int ty = W.type[i];
  if (ty == CHP_BODY_DYNAMIC) {
    v = scale3<R>(v, W.ldamp[i]);
    w = scale3<R>(w, W.adamp[i]);
  }
  if ((ty == CHP_BODY_DYNAMIC || ty == CHP_BODY_KINEMATIC) && W.sleep_state[i] != CHP_SLEEP_SLEEPING) {
    f3 f = F3<R>(W.feff, i), tq = F3<R>(W.torque, i);
    R iMdt = W.inv_mass[i] * dt;
    v = set3<R>(ld<R>(v.x) + ld<R>(f.x) * iMdt * ld<R>(lf.x), ld<R>(v.y) + ld<R>(f.y) * iMdt * ld<R>(lf.y),
                ld<R>(v.z) + ld<R>(f.z) * iMdt * ld<R>(lf.z));
    const float* e = W.iiw + 9 * i;
    R tx = ld<R>(tq.x) * ld<R>(af.x), ty_ = ld<R>(tq.y) * ld<R>(af.y), tz = ld<R>(tq.z) * ld<R>(af.z);
    w = set3<R>(ld<R>(w.x) + dt * (ld<R>(e[0]) * tx + ld<R>(e[1]) * ty_ + ld<R>(e[2]) * tz),
                ld<R>(w.y) + dt * (ld<R>(e[3]) * tx + ld<R>(e[4]) * ty_ + ld<R>(e[5]) * tz),
                ld<R>(w.z) + dt * (ld<R>(e[6]) * tx + ld<R>(e[7]) * ty_ + ld<R>(e[8]) * tz));
    f3 p = F3<R>(W.pos, i);
    p = set3<R>(ld<R>(p.x) + ld<R>(v.x) * dt, ld<R>(p.y) + ld<R>(v.y) * dt, ld<R>(p.z) + ld<R>(v.z) * dt);
    f4 q = ((const f4*)W.quat)[i];
    {  // Quat.integrate (quaternion.dart:93-111)
      R ax = ld<R>(w.x) * ld<R>(af.x), ay = ld<R>(w.y) * ld<R>(af.y), az = ld<R>(w.z) * ld<R>(af.z);
      R bx = q.x, by = q.y, bz = q.z, bw = q.w;
      R hd = dt * (R)0.5;
      q.x = st<R>(bx + hd * (ax * bw + ay * bz - az * by));
      q.y = st<R>(by + hd * (ay * bw + az * bx - ax * bz));
      q.z = st<R>(bz + hd * (az * bw + ax * by - ay * bx));
      q.w = st<R>(bw + hd * (-ax * bx - ay * by - az * bz));
    }
    if (qn) {
      R x = q.x, y = q.y, z = q.z, ww = q.w;
      if (W.quat_fast) {  // Quat.normalizeFast (quaternion.dart:171-185)
        R f2 = ((R)3 - (x * x + y * y + z * z + ww * ww)) / (R)2;
        if (f2 == (R)0) { q.x = q.y = q.z = q.w = 0.f; }
        else { q.x = st<R>(x * f2); q.y = st<R>(y * f2); q.z = st<R>(z * f2); q.w = st<R>(ww * f2); }
      } else {  // vector_math Quaternion.normalize
        R l = sqrt((x * x) + (y * y) + (z * z) + (ww * ww));
        if (l != (R)0) {
          R d = (R)1 / l;
          q.x = st<R>(x * d); q.y = st<R>(y * d); q.z = st<R>(z * d); q.w = st<R>(ww * d);
        }
      }
    }
    S3<R>(W.pos, i, p);
    ((f4*)W.quat)[i] = q;
    W.flags[i] |= BF_AABB_DIRTY;
    if (!(W.flags[i] & BF_ISOTROPIC)) inertia_world<R>(q, F3<R>(W.inv_inertia, i), W.iiw + 9 * i);
    ok = isfinite(p.x) && isfinite(p.y) && isfinite(p.z) && isfinite(q.w);
  }
  if (W.allow_sleep && (W.flags[i] & BF_ALLOW_SLEEP)) sleep_tick(W, i, v, w);
  S3<R>(W.vel, i, v);
  S3<R>(W.avel, i, w);
  S3<R>(W.force, i, mk3(0.f, 0.f, 0.f));   // World.clearForces
  S3<R>(W.torque, i, mk3(0.f, 0.f, 0.f));
  return ok;
}
// quaternion normalisation this step (World.quatNormalizeSkip)
template <typename R> __device__ __forceinline__ bool post_qn(const DevWorld<R>& W) {
  return W.counters[C_STEP] % (W.quat_skip + 1) == 0;
}

// ---- velocities, damping, integration ---------------------------------------------------------
// gs_solver.dart:157-168, world_class.dart:647-674, Body.integrate (rigid_body.dart:627-680)
// the end of a step: the step counter, World.time += dt (world_class.dart:397-399)
template <typename R> __device__ __forceinline__ void step_done(const DevWorld<R>& W, double dt) {
  W.counters[C_STEP] += 1;
  if (!W.time_frozen) W.wtime[0] += dt;
}
template <typename R> __device__ void st_post(const DevWorld<R>& W, double dt) {
  const int E = W.counters[C_ROWS];
  const bool qn = post_qn(W);
  for (int i = threadIdx.x; i < W.nb; i += blockDim.x)
    if (!post_body(W, i, (R)dt, E, qn)) ws_fail(W.counters, WS_NONFINITE);
  __syncthreads();
  if (threadIdx.x == 0) step_done(W, dt);
  __syncthreads();
}

}  // namespace chp

// Reference-mode kernels: NEXT's FP64 gravity + time-step path on gfx950.
//
// Compiled with -ffp-contract=off: every product and sum is rounded as
// written, in the order NEXT writes it, so the GPU reproduces the reference
// arithmetic operation by operation.
//
// Pipeline of one tree build (positions in `st`):
//   bbox -> root cube (step.h:68-102)
//   keys: each body replays the FP64 node-centre recurrence of
//         octree.h:49-64 for 21 levels -> 63-bit digit key
//   stable radix sort of keys, gather of the state into key order
//   lcp of neighbouring keys -> the one-body-per-leaf octree of
//         octree.h:69-87 in depth-first preorder (children 0..7), built from
//         the rule "an internal node exists for every digit prefix shared by
//         two or more bodies", with skip pointers for stackless traversal
//   upward pass, deepest first, one launch per depth or, in small systems,
//         within units of bodies (octree.h:92-127)
//   walk: one wave per group of consecutive targets; the group decides once
//         what all its targets decide alike, each target walks the rest with
//         its own acceptance test (octree.h:133-179), so every target
//         accumulates the reference's terms.
#include "common.hpp"
#include "layout.hpp"
#include "prims.hpp"
#include "ref_kernels.hpp"
#include "units.hpp"

#include <algorithm>
#include <climits>
#include <type_traits>

namespace nbx {
namespace {

__device__ __forceinline__ void lo_upd(double& lo, double p) { if (p < lo) lo = p; }   // std::min(lo, p)
__device__ __forceinline__ void hi_upd(double& hi, double p) { if (hi < p) hi = p; }   // std::max(hi, p)

// Block-wide min/max of 6 values (3 lows, 3 highs) written as one partial.
__device__ void block_bbox_write(double lo[3], double hi[3], double* part) {
  __shared__ double sm[kBlock / kWave][6];
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      lo_upd(lo[k], __shfl_xor(lo[k], off, kWave));
      hi_upd(hi[k], __shfl_xor(hi[k], off, kWave));
    }
  }
  const int w = threadIdx.x / kWave;
  if (lane_id() == 0) {
    for (int k = 0; k < 3; ++k) { sm[w][k] = lo[k]; sm[w][3 + k] = hi[k]; }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int q = 1; q < kBlock / kWave; ++q)
      for (int k = 0; k < 3; ++k) { lo_upd(lo[k], sm[q][k]); hi_upd(hi[k], sm[q][3 + k]); }
    for (int k = 0; k < 3; ++k) { part[6 * blockIdx.x + k] = lo[k]; part[6 * blockIdx.x + 3 + k] = hi[k]; }
  }
}

__global__ __launch_bounds__(kBlock) void k_fill_scalars(DevScalars* sc, int what) {
  const int t = threadIdx.x;
  if (what & 1) {
    if (t < kMaxDepthSlots) sc->level_count[t] = 0;
    if (t == 0) { sc->collisions = 0; sc->coincident = 0; sc->max_leaf_depth = 0; sc->ndesc = 0; sc->over_depths = 0ull; }
  }
  if ((what & 4) && t == 0) sc->err = 0;
  if ((what & 8) && t == 0) { sc->n_pp = 0ull; sc->n_pc = 0ull; sc->n_open = 0ull; sc->n_iter = 0ull; sc->n_eval = 0ull; }
}

// Start of a captured run: no abort yet, dt log entries from `step` on.
__global__ void k_set_run(DevScalars* sc, int32_t step) {
  sc->abort_flags = 0;
  sc->step_count = step;
}

__global__ __launch_bounds__(kBlock) void k_fill_u32(int64_t n, uint32_t* __restrict__ a, uint32_t v) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) a[i] = v;
}

__global__ __launch_bounds__(kBlock) void k_fill_v2max(SysArrays sy) {
  const int s = blockIdx.x * kBlock + threadIdx.x;
  if (s < sy.nsys) sy.v2max[s] = 0ull;
}

__global__ __launch_bounds__(kBlock) void k_set_dt(SysArrays sy, double dt) {
  const int s = blockIdx.x * kBlock + threadIdx.x;
  if (s < sy.nsys) sy.dt[s] = dt;
}

// Min/max of the bodies [begin, end) of one system (one block).
__global__ __launch_bounds__(kBlock) void k_bbox_partial(StateArrays st, const BoxBlock* __restrict__ blocks,
                                                         double* part) {
  const BoxBlock b = blocks[blockIdx.x];
  double lo[3] = {1e30, 1e30, 1e30}, hi[3] = {-1e30, -1e30, -1e30};
  for (int64_t i = b.begin + threadIdx.x; i < b.end; i += kBlock) {
    const double p[3] = {st.x[i], st.y[i], st.z[i]};
    for (int k = 0; k < 3; ++k) { lo_upd(lo[k], p[k]); hi_upd(hi[k], p[k]); }
  }
  block_bbox_write(lo, hi, part);
}

// Root centre and half-width of each system from its blocks' partials
// (step.h:93-100), one wave per system; min and max are exact, so the
// order does not matter.  clear (may be null): scalars to reset for the
// tree build that follows.
__global__ __launch_bounds__(kWave) void k_bbox_final(const double* __restrict__ part,
                                                      const int32_t* __restrict__ block_off, SysArrays sy,
                                                      DevScalars* clear) {
  const int s = blockIdx.x;
  if (clear && s == 0) {     // a tree build's counts and flags (k_fill_scalars, what = 1 | 4)
    const int t = threadIdx.x;
    clear->level_count[t] = 0;
    if (t == 0) {
      clear->collisions = 0; clear->coincident = 0; clear->max_leaf_depth = 0; clear->err = 0; clear->ndesc = 0;
      clear->over_depths = 0ull;
    }
  }
  if (s >= sy.nsys) return;
  double lo[3] = {1e30, 1e30, 1e30}, hi[3] = {-1e30, -1e30, -1e30};
  for (int b = block_off[s] + (int)threadIdx.x; b < block_off[s + 1]; b += kWave)
    for (int k = 0; k < 3; ++k) { lo_upd(lo[k], part[6 * b + k]); hi_upd(hi[k], part[6 * b + 3 + k]); }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1)
    for (int k = 0; k < 3; ++k) {
      lo_upd(lo[k], __shfl_xor(lo[k], off, kWave));
      hi_upd(hi[k], __shfl_xor(hi[k], off, kWave));
    }
  if (threadIdx.x != 0) return;
  const double cx = (lo[0] + hi[0]) * 0.5;
  const double cy = (lo[1] + hi[1]) * 0.5;
  const double cz = (lo[2] + hi[2]) * 0.5;
  double e = hi[0] - lo[0];
  const double ey = hi[1] - lo[1], ez = hi[2] - lo[2];
  if (e < ey) e = ey;
  if (e < ez) e = ez;
  double h = e * 0.5;
  if (h <= 0.0) h = 1.0;
  double* r = sy.root + 4 * s;
  r[0] = cx; r[1] = cy; r[2] = cz; r[3] = h;
}

// Digits of one body along the node-centre recurrence (octree.h:49-64),
// levels [l0, l1), starting from the root.
__device__ __forceinline__ void key_digits(double px, double py, double pz, const double* root, int l0, int l1,
                                           uint64_t& hi, uint64_t& lo) {
  double cx = root[0], cy = root[1], cz = root[2], s = root[3];
  hi = 0; lo = 0;
  for (int l = 0; l < l1; ++l) {
    const uint32_t o = (px > cx ? 1u : 0u) | (py > cy ? 2u : 0u) | (pz > cz ? 4u : 0u);
    if (l >= l0) {
      if (l < kKeyDigits) hi = (hi << 3) | o; else lo = (lo << 3) | o;
    }
    const double hs = s * 0.5;
    cx = cx + ((o & 1u) ? hs : -hs);
    cy = cy + ((o & 2u) ? hs : -hs);
    cz = cz + ((o & 4u) ? hs : -hs);
    s = hs;
  }
}

// m^0.333333333 (the exponent of octree.h:146) as p (1 + r), from cb =
// cbrt(m), odd in m and 0 at 0.  A softening floor is the quotient of two of
// these, rounded once, so both carry their rounding errors along: the floor is
// within 1.6e-16 of the exact one for masses of 1e-307 to 1e210 (pow of the
// mass ratio: 2.5e-16), and for equal masses it is the half-width's double as
// pow(1) makes it.  In units of a power of eight, g = m / 8^k:
//   g^(1/3) = c (1 + (g - c^3) / (3 g)), the residual formed exactly;
//   the exponents differ by d = 1/3 - 0.333333333, and g^-d = 1 - t + t^2 / 2
//   with t = d ln m < 2.5e-7, so an error of 1e-7 in ln m (log of the mantissa
//   in FP32, the exponent's part in FP64) moves the power by 3e-17.
struct DmPower {
  double p;
  float r;
};

__device__ __forceinline__ DmPower dm_power(double m, double cb) {
  if (m == 0.0) return DmPower{0.0, 0.0f};
  constexpr double kD = 3.3333332390602283e-10;             // 1/3 minus the double nearest 0.333333333
  int e;
  const double f = frexp(fabs(m), &e);
  const int k = e / 3;
  const double g = ldexp(f, e - 3 * k), c = ldexp(fabs(cb), -k);
  const double c2 = c * c, e2 = __builtin_fma(c, c, -c2);
  const double c3 = c2 * c, e3 = __builtin_fma(e2, c, __builtin_fma(c2, c, -c3));
  const float rel = (float)((g - c3) - e3) * __builtin_amdgcn_rcpf(3.0f * (float)g);
  const double t = kD * __builtin_fma(0.6931471805599453, (double)e, (double)__logf((float)f));
  const double w = (double)rel - __builtin_fma(-0.5 * t, t, t);
  const double p = __builtin_fma(c, w, c);
  const double left = __builtin_fma(c, w, c - p);
  return DmPower{copysign(ldexp(p, k), m), (float)left * __builtin_amdgcn_rcpf((float)p)};
}

// The dmk and dmr of a node of half-width `size` and mass power q.
__device__ __forceinline__ void set_floor(RefNode& nd, double size, const DmPower& q) {
  const double s2 = 2.0 * size, k = s2 / q.p;
  nd.dmk = k;
  nd.dmr = (float)(__builtin_fma(-k, q.p, s2) * __builtin_amdgcn_rcp(s2)) - q.r;
}

__device__ __forceinline__ void sys_root(const SysArrays& sy, int32_t s, double root[4]) {
  const double* r = sy.root + 4 * s;
  root[0] = r[0]; root[1] = r[1]; root[2] = r[2]; root[3] = r[3];
}

__global__ __launch_bounds__(kBlock) void k_keys(int64_t n, StateArrays st, SysArrays sy,
                                                 uint64_t* __restrict__ key, uint32_t* __restrict__ idx,
                                                 DevScalars* scw) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const double px = st.x[i], py = st.y[i], pz = st.z[i];
  if (!(__builtin_isfinite(px) && __builtin_isfinite(py) && __builtin_isfinite(pz))) atomicOr(&scw->err, 1);
  double root[4];
  sys_root(sy, st.sys[i], root);
  uint64_t hi, lo;
  key_digits(px, py, pz, root, 0, kKeyDigits, hi, lo);
  key[i] = hi;
  idx[i] = (uint32_t)i;
}

__global__ __launch_bounds__(kBlock) void k_keys2(int64_t n, StateArrays st, SysArrays sy,
                                                  uint64_t* __restrict__ key2) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  double root[4];
  sys_root(sy, st.sys[i], root);
  uint64_t hi, lo;
  key_digits(st.x[i], st.y[i], st.z[i], root, kKeyDigits, kMaxLevels, hi, lo);
  key2[i] = lo;
}

// The sort orders bodies by bits [lo, 63) of the first key word (its top
// digits: enough to separate the bodies of a tree of the last build's depth).
// Bodies of one system whose words agree on those bits sit next to each
// other, in their previous order.  Each such run is sorted in place by the
// whole first word, then the second word (digits 21..41), stably: the order a
// sort by (system, first word, second word) with ties in the previous order
// gives.  The second word is written for the runs' bodies only, the only ones
// whose second word is ever read (where two neighbours' first words are
// equal).  Runs are disjoint and a swap inside one keeps its bits [lo, 63), so
// the run bounds every thread finds do not depend on the others' swaps.
__global__ __launch_bounds__(kBlock) void k_fix_runs(int64_t n, StateArrays st, SysArrays sy, uint64_t* key,
                                                     uint64_t* __restrict__ key2, uint32_t* __restrict__ amag,
                                                     int lo) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const int32_t s = st.sys[i];
  const uint64_t top = key[i] >> lo;
  auto same = [&](int64_t j) { return st.sys[j] == s && (key[j] >> lo) == top; };
  const bool eq_next = i + 1 < n && same(i + 1);
  const bool eq_prev = i > 0 && same(i - 1);
  if (!eq_next || eq_prev) return;                           // not the first body of a run
  int64_t j = i + 1;                                         // the run is [i, j]
  while (j + 1 < n && same(j + 1)) ++j;
  double root[4];
  sys_root(sy, s, root);
  for (int64_t t = i; t <= j; ++t) {
    uint64_t hi, lo2;
    key_digits(st.x[t], st.y[t], st.z[t], root, kKeyDigits, kMaxLevels, hi, lo2);
    key2[t] = lo2;
  }
  for (int64_t t = i + 1; t <= j; ++t)
    for (int64_t u = t; u > i && (key[u - 1] > key[u] || (key[u - 1] == key[u] && key2[u - 1] > key2[u])); --u) {
      const int64_t v = u - 1;
      auto sw_d = [&](double* a) { const double w = a[u]; a[u] = a[v]; a[v] = w; };
      auto sw_i = [&](int32_t* a) { const int32_t w = a[u]; a[u] = a[v]; a[v] = w; };
      auto sw_k = [&](uint64_t* a) { const uint64_t w = a[u]; a[u] = a[v]; a[v] = w; };
      sw_d(st.x); sw_d(st.y); sw_d(st.z); sw_d(st.vx); sw_d(st.vy); sw_d(st.vz); sw_d(st.m);
      sw_i(st.type); sw_i(st.id);
      sw_k(key); sw_k(key2);
      if (amag) { const uint32_t a = amag[u]; amag[u] = amag[v]; amag[v] = a; }
    }
}

__global__ __launch_bounds__(kBlock) void k_keys_export(int64_t n, StateArrays st, SysArrays sy,
                                                        uint64_t* __restrict__ hi_out,
                                                        uint64_t* __restrict__ lo_out) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  double root[4];
  sys_root(sy, st.sys[i], root);
  uint64_t hi, lo;
  key_digits(st.x[i], st.y[i], st.z[i], root, 0, kMaxLevels, hi, lo);
  const int32_t o = st.id[i];
  hi_out[o] = hi;
  lo_out[o] = lo;
}

__global__ __launch_bounds__(kBlock) void k_iota(int64_t n, uint32_t* idx) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) idx[i] = (uint32_t)i;
}

__global__ __launch_bounds__(kBlock) void k_gather_u64(int64_t n, const uint32_t* __restrict__ perm,
                                                       const uint64_t* __restrict__ src, uint64_t* __restrict__ dst) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) dst[i] = src[perm[i]];
}

__global__ __launch_bounds__(kBlock) void k_gather_state(int64_t n, const uint32_t* __restrict__ perm, StateArrays a,
                                                         StateArrays b) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const uint32_t p = perm[i];
  b.x[i] = a.x[p]; b.y[i] = a.y[p]; b.z[i] = a.z[p];
  b.vx[i] = a.vx[p]; b.vy[i] = a.vy[p]; b.vz[i] = a.vz[p];
  b.m[i] = a.m[p]; b.type[i] = a.type[p]; b.id[i] = a.id[p]; b.sys[i] = a.sys[p];
}

// Sort by counting, for small systems: body i's place is the number of keys
// below its own plus the equal keys before it.  One workgroup per 64 bodies,
// each wave counting over its part of the keys (wave-uniform, so by scalar
// loads: a compare and an add with carry per key), then the waves move the
// body arrays to their places.  n^2 / 64 compares of 64 lanes over the whole
// chip in one launch stand against ten launches of the radix sort and the
// gather, whose tiles leave most of the chip idle at these sizes: forces of
// 1,000 bodies 290 -> 215 us, of 12,289 bodies 398 -> 328 us a call.  (34 us at
// 12,289 bodies, 40 at 16,384, growing as n^2: the radix sort takes over there.)
__global__ __launch_bounds__(kRankWaves* kWave) void k_rank_sort(int32_t n, const uint64_t* __restrict__ key,
                                                                  uint64_t* __restrict__ kout, StateArrays a,
                                                                  StateArrays b, const uint32_t* __restrict__ amag,
                                                                  uint32_t* __restrict__ amag_out) {
  __shared__ uint32_t part[kRankWaves][kWave];
  typedef const __attribute__((address_space(4))) uint64_t* kptr;   // scalar loads
  const kptr keys = (kptr)key;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = lane_id();
  const int32_t i0 = (int32_t)blockIdx.x * kWave, i1 = i0 + kWave < n ? i0 + kWave : n;
  const int32_t i = i0 + lane;
  const uint64_t k = key[i < n ? i : n - 1];
  const int32_t per = (n + kRankWaves - 1) / kRankWaves;
  int32_t j = wave * per;
  const int32_t end = j + per < n ? j + per : n;
  uint32_t cnt = 0;
  const int32_t before = end < i0 ? end : i0;               // keys before the block: equal ones count
#pragma unroll 8
  for (; j < before; ++j) cnt += keys[j] <= k ? 1u : 0u;
  const int32_t own = end < i1 ? end : i1;
  for (; j < own; ++j) cnt += (keys[j] < k || (keys[j] == k && j < i)) ? 1u : 0u;
#pragma unroll 8
  for (; j < end; ++j) cnt += keys[j] < k ? 1u : 0u;
  part[wave][lane] = cnt;
  __syncthreads();
  uint32_t r = 0;
#pragma unroll
  for (int w = 0; w < kRankWaves; ++w) r += part[w][lane];
  if (i >= n) return;
  // one array per wave (12 of them)
  auto move = [&](auto* dst, const auto* src) { dst[r] = src[i]; };
  switch (wave) {
    case 0: move(b.x, a.x); break;
    case 1: move(b.y, a.y); break;
    case 2: move(b.z, a.z); break;
    case 3: move(b.vx, a.vx); break;
    case 4: move(b.vy, a.vy); break;
    case 5: move(b.vz, a.vz); break;
    case 6: move(b.m, a.m); break;
    case 7: move(b.type, a.type); break;
    case 8: move(b.id, a.id); break;
    case 9: move(b.sys, a.sys); break;
    case 10: kout[r] = k; break;
    case 11: if (amag) move(amag_out, amag); break;
    default: break;
  }
}

__global__ __launch_bounds__(kBlock) void k_set_ids(int64_t n, int32_t* __restrict__ id, int32_t id0,
                                                    int32_t* __restrict__ sys, int32_t sys_no) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) { id[i] = id0 + (int32_t)i; sys[i] = sys_no; }
}

// inv[id[i] - base] = i for the indices in range.
__global__ __launch_bounds__(kBlock) void k_out_index(int64_t cnt, const int32_t* __restrict__ id, int32_t base,
                                                      uint32_t* __restrict__ inv) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= cnt) return;
  const int64_t j = (int64_t)id[i] - base;
  if (j >= 0 && j < cnt) inv[j] = (uint32_t)i;
}

// The cnt slots hold a permutation exactly when some slot holds each index:
// inv[j] (stale where no slot wrote it) must be a slot that holds j.
__global__ __launch_bounds__(kBlock) void k_out_check(int64_t cnt, const int32_t* __restrict__ id, int32_t base,
                                                      const uint32_t* __restrict__ inv, int32_t* bad) {
  const int64_t j = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (j >= cnt) return;
  const uint32_t i = inv[j];
  if (i >= (uint64_t)cnt || (int64_t)id[i] - base != j) *bad = 1;
}

__global__ __launch_bounds__(kBlock) void k_out_gather(int64_t j0, int64_t len, int64_t cnt,
                                                       const uint32_t* __restrict__ inv, OutArrays src, int m,
                                                       double* __restrict__ dst) {
  const int64_t j = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (j >= len) return;
  const uint32_t i = inv[j0 + j];
  if (i >= (uint64_t)cnt) return;                            // not a permutation (k_out_check)
#pragma unroll
  for (int k = 0; k < kOutArrays; ++k)
    if (k < m) dst[k * len + j] = src.p[k][i];
}

__global__ __launch_bounds__(kBlock) void k_gather_sys(int64_t n, const uint32_t* __restrict__ perm,
                                                       const int32_t* __restrict__ sys, uint32_t* __restrict__ dst) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) dst[i] = (uint32_t)sys[perm[i]];
}

// Map for removing the bodies [cut, cut + len) of one system: slot i of the
// shortened arrays takes old slot perm[i].
__global__ __launch_bounds__(kBlock) void k_remove_map(int64_t n_new, int64_t cut, int64_t len,
                                                       uint32_t* __restrict__ perm) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n_new) perm[i] = (uint32_t)(i < cut ? i : i + len);
}

__global__ __launch_bounds__(kBlock) void k_relabel(int64_t n, int32_t* __restrict__ sys, int32_t removed) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n && sys[i] > removed) sys[i] -= 1;
}

__global__ __launch_bounds__(kBlock) void k_gather_f64(int64_t n, const uint32_t* __restrict__ perm,
                                                       const double* __restrict__ src, double* __restrict__ dst) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) dst[i] = src[perm[i]];
}

// Number of leading octree digits two keys share (0..21 per word).
__device__ __forceinline__ int lcp_word(uint64_t a, uint64_t b) {
  const uint64_t d = a ^ b;
  return d ? (__clzll((long long)d) - 1) / 3 : kKeyDigits;
}

// Bodies of different systems share nothing: -1 separates their trees.
__device__ __forceinline__ int lcp_pair(const uint64_t* key, const uint64_t* key2, const int32_t* sys, int64_t i,
                                        int& equal) {
  equal = 0;
  if (sys[i] != sys[i + 1]) return -1;
  int l = lcp_word(key[i], key[i + 1]);
  if (l == kKeyDigits) {
    if (key2) {
      l += lcp_word(key2[i], key2[i + 1]);
      if (l == kMaxLevels) equal = 1;
    } else {
      equal = 1;
    }
  }
  return l;
}

// lcp[i] = digits shared by sorted bodies i and i+1 (-1 past the end).
// Body i starts the internal nodes at depths (lcp[i-1], lcp[i]] and its leaf;
// it ends the internal nodes at depths (lcp[i], lcp[i-1]].  Each block also
// writes one row of partial counts (internal nodes started and ended per
// depth, deepest leaf, equal-key pairs) for k_lcp_scan: plain stores, no
// global atomics.
__global__ __launch_bounds__(kBlock) void k_lcp_count(int64_t n, const uint64_t* __restrict__ key,
                                                      const uint64_t* __restrict__ key2,
                                                      const int32_t* __restrict__ sys, int32_t* __restrict__ lcp,
                                                      uint32_t* __restrict__ cnt_s, uint32_t* __restrict__ part) {
  __shared__ uint32_t hist[kPartW];
  if (threadIdx.x < kPartW) hist[threadIdx.x] = 0;
  __syncthreads();
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) {
    int eq_i = 0, eq_p = 0;
    const int li = (i + 1 < n) ? lcp_pair(key, key2, sys, i, eq_i) : -1;
    const int lp = (i > 0) ? lcp_pair(key, key2, sys, i - 1, eq_p) : -1;
    lcp[i] = li;
    cnt_s[i] = 1u + (uint32_t)(li > lp ? li - lp : 0);
    for (int d = lp + 1; d <= li; ++d) atomicAdd(&hist[d], 1u);
    for (int d = li + 1; d <= lp; ++d) atomicAdd(&hist[kPartEnds + d], 1u);
    atomicMax(&hist[kPartMaxDepth], (uint32_t)(1 + (li > lp ? li : lp)));
    if (eq_i) atomicAdd(&hist[kPartEqual], 1u);
  }
  __syncthreads();
  if (threadIdx.x < kPartW) part[(int64_t)threadIdx.x * gridDim.x + blockIdx.x] = hist[threadIdx.x];
}

// Column `col` of the partial counts, one block per column: a per-depth
// column becomes its exclusive prefix over the blocks (in place) and its
// total is the node count of that depth; the last two columns reduce to the
// deepest leaf and the equal-key pairs.
__global__ __launch_bounds__(kBlock) void k_lcp_scan(uint32_t* __restrict__ part, int64_t rows, int has_key2,
                                                     DevScalars* sc) {
  __shared__ uint32_t scr[kBlock / kWave + 1];
  const int col = blockIdx.x;
  uint32_t* cp = part + (int64_t)col * rows;
  if (col < kPartMaxDepth) {
    // thread t takes rows [t*per, (t+1)*per) of the column: their sum, one
    // block scan of the sums, then the rows' running prefix
    const int64_t per = (rows + kBlock - 1) / kBlock;
    const int64_t r0 = (int64_t)threadIdx.x * per;
    const int64_t r1 = r0 + per < rows ? r0 + per : rows;
    uint32_t sum = 0;
    for (int64_t r = r0; r < r1; ++r) sum += cp[r];
    uint32_t tot;
    uint32_t run = block_excl_scan_u32<kBlock>(sum, scr, &tot);
    for (int64_t r = r0; r < r1; ++r) {
      const uint32_t v = cp[r];
      cp[r] = run;
      run += v;
    }
    if (threadIdx.x == 0 && col < kPartEnds) sc->level_count[col] = (int32_t)tot;
    return;
  }
  __shared__ uint32_t red[kBlock / kWave];
  const bool is_max = col == kPartMaxDepth;
  uint32_t v = 0;
  for (int64_t r = threadIdx.x; r < rows; r += kBlock) {
    const uint32_t x = cp[r];
    v = is_max ? (x > v ? x : v) : v + x;
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const uint32_t o = __shfl_xor(v, off, kWave);
    v = is_max ? (o > v ? o : v) : v + o;
  }
  if (lane_id() == 0) red[threadIdx.x / kWave] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kBlock / kWave; ++w) v = is_max ? (red[w] > v ? red[w] : v) : v + red[w];
    if (is_max) sc->max_leaf_depth = (int32_t)v;
    else if (has_key2) sc->coincident = (int32_t)v;
    else sc->collisions = (int32_t)v;
  }
}

// Preorder index of each system's root (its first body starts at depth 0)
// and of the node after its tree.
__global__ __launch_bounds__(kBlock) void k_sys_roots(SysArrays sy, const uint32_t* __restrict__ pre_off,
                                                      const DevScalars* __restrict__ sc) {
  const int s = blockIdx.x * kBlock + threadIdx.x;
  if (s >= sy.nsys) return;
  sy.sroot[s] = (int32_t)pre_off[sy.soff[s]];
  sy.send[s] = s + 1 < sy.nsys ? (int32_t)pre_off[sy.soff[s + 1]] : sc->total_nodes;
}

__global__ __launch_bounds__(kBlock) void k_emit(int64_t n, const int32_t* __restrict__ lcp,
                                                 const uint32_t* __restrict__ pre_off,
                                                 const uint32_t* __restrict__ part, StateArrays st, SysArrays sy,
                                                 const DevScalars* __restrict__ sc, RefNode* __restrict__ nodes,
                                                 WalkHead* __restrict__ heads, int32_t* __restrict__ level_list,
                                                 uint32_t* __restrict__ end_list, uint32_t cap_nodes,
                                                 uint32_t cap_int) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  const bool valid = i < n;
  int li = -1, lp = -1;
  uint32_t pre = 0, skipv = 0;
  if (valid) {
    li = lcp[i];
    lp = i > 0 ? lcp[i - 1] : -1;
    pre = pre_off[i];
    skipv = (i + 1 < n) ? pre_off[i + 1] : (uint32_t)sc->total_nodes;
  }
  place_internal_nodes(valid, lp, li, pre, skipv, part, sc, level_list, end_list,
                       cap_int);
  if (!valid) return;
  // One all-zero record after the last node: the walk reads a leaf's
  // quadrupole there.
  if (i == n - 1) {
    const uint32_t z = (uint32_t)sc->total_nodes;
    if (z < cap_nodes) nodes[z] = RefNode{};
  }
  // Internal nodes are written by the upward pass (their records, skip
  // pointers included, come from the node lists placed above).
  const int ns = li > lp ? li - lp : 0;
  if (pre + ns < cap_nodes) {
    const uint32_t p = pre + ns;
    const int d = 1 + (li > lp ? li : lp);
    const double m = st.m[i];
    const double size = ldexp(sy.root[4 * st.sys[i] + 3], -d);
    // Leaves carry no quadrupole; the walk never reads a leaf's Q fields
    // (the first 64 bytes of the record are written, in one piece).
    const double px = st.x[i], py = st.y[i], pz = st.z[i];
    RefNode& nd = nodes[p];
    nd.cx = px; nd.cy = py; nd.cz = pz;
    nd.m = m;
    nd.skip = (int32_t)(p + 1);
    nd.first = (int32_t)i;
    nd.depth = (int16_t)d;
    nd.leaf = 1;
    // softening.h:26-27: size*0.015 + cbrt(m)*0.002, summed before the taper
    const double cm = cbrt(m);
    nd.esum = size * 0.015 + cm * 0.002;
    set_floor(nd, size, dm_power(m, cm));
    // a leaf is accepted whatever its distance: no threshold
    heads[p] = WalkHead{px, py, pz, 0.0f, m == 0.0 ? (int32_t)(p + 1) | kLinkZeroMass : ~(int32_t)i};
  }
}

// A build whose counts stay on the device: each depth's offset in the node
// list, and the abort flag if the tree does not fit the buffers and launches
// sized beforehand (node records, node-list entries, depth levels), needs
// the two-word keys, or has a non-finite position.  One wave.
__global__ __launch_bounds__(kWave) void k_check(DevScalars* sc, int64_t cap_records, int64_t cap_list, int dmax) {
  const int t = threadIdx.x;
  const uint32_t v = (uint32_t)sc->level_count[t];
  const uint32_t inc = wave_incl_scan_u32(v);
  sc->level_off[t] = (int32_t)(inc - v);
  if (t == kWave - 1) {
    int32_t f = 0;
    if ((int64_t)(uint32_t)sc->total_nodes + 1 > cap_records || (int64_t)inc > cap_list) f |= kAbortCapacity;
    if (sc->max_leaf_depth - 1 > dmax) f |= kAbortDepth;
    if (sc->collisions > 0 || sc->coincident > 0) f |= kAbortCollision;
    if (sc->err & 1) f |= kAbortNonFinite;
    if (sc->err & kSortErrTimeout) f |= kAbortSort;
    if (sc->err & kSortErrPatch) f |= kAbortPatch;
    if (f) sc->abort_flags |= f;
  }
}

// Mass, centre of mass and one-level softened quadrupole of an internal node
// of depth d from its children (octree.h:104-126), and the squared-distance
// thresholds of the walk's opening test for this theta: the node's record
// (all of it but the padding) and its walk head.  end: the preorder index after its
// subtree (its skip pointer, from the list of skip targets); the first body
// comes from the first child, the half-width from the system's root.
//
// The unit's nodes keep mass, centre and first body in LDS (36 bytes each).
// 1,856 nodes (a unit of up to 1,152 bodies has about 1,700) so that two units
// fit a CU; with 2,048 one did, and 512 systems of 500 bodies took 80 us instead
// of 59, 262,144 bodies 98 instead of 80.
constexpr int kUnitNodes = 1856;
struct UnitMoments {
  double m[kUnitNodes], x[kUnitNodes], y[kUnitNodes], z[kUnitNodes];
  int32_t first[kUnitNodes];
};

__device__ __forceinline__ void upward_node(const UnitView& v, UnitMoments* lm, int32_t id, int32_t end, int d,
                                            RefNode* __restrict__ nodes, WalkHead* __restrict__ heads,
                                            double inv_theta, double half, const int32_t* __restrict__ sys,
                                            const double* __restrict__ root) {
  // One walk of the child chain (at most 8; the bound also keeps a malformed
  // chain finite) gathers each child's mass and centre into registers; a
  // slot past the last child keeps mass 0, which both sums skip.
  double cmv[8], cxv[8], cyv[8], czv[8];
  int32_t first = 0;
  if (v.lds) {
    int c = v.slot(id) + 1;
    const int e = v.slot(end);
    first = lm->first[c];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      cmv[j] = 0.0; cxv[j] = 0.0; cyv[j] = 0.0; czv[j] = 0.0;
      if (c < e) {
        cmv[j] = lm->m[c]; cxv[j] = lm->x[c]; cyv[j] = lm->y[c]; czv[j] = lm->z[c];
        c = v.skips[c];
      }
    }
  } else {
    int32_t c = id + 1;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      cmv[j] = 0.0; cxv[j] = 0.0; cyv[j] = 0.0; czv[j] = 0.0;
      if (c < end) {
        const RefNode& ch = nodes[c];
        cmv[j] = ch.m; cxv[j] = ch.cx; cyv[j] = ch.cy; czv[j] = ch.cz;
        if (j == 0) first = ch.first;
        c = ch.skip;
      }
    }
  }
  double M = 0.0, sx = 0.0, sy = 0.0, sz = 0.0;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const double cm = cmv[j];
    if (cm == 0.0) continue;
    M = M + cm;
    sx = sx + cxv[j] * cm;
    sy = sy + cyv[j] * cm;
    sz = sz + czv[j] * cm;
  }
  double cx = sx, cy = sy, cz = sz;
  if (M > 0.0) { cx = sx / M; cy = sy / M; cz = sz / M; }
  const double size = ldexp(sys ? root[4 * sys[first] + 3] : half, -d);
  double qxx = 0, qyy = 0, qzz = 0, qxy = 0, qxz = 0, qyz = 0;
  const double soft = size * size * 0.01;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const double mc = cmv[j];
    if (mc == 0.0) continue;
    const double rx = cxv[j] - cx, ry = cyv[j] - cy, rz = czv[j] - cz;
    const double r2 = rx * rx + ry * ry + rz * rz + soft;
    qxx = qxx + mc * (3.0 * rx * rx - r2);
    qyy = qyy + mc * (3.0 * ry * ry - r2);
    qzz = qzz + mc * (3.0 * rz * rz - r2);
    qxy = qxy + mc * (3.0 * rx * ry);
    qxz = qxz + mc * (3.0 * rx * rz);
    qyz = qyz + mc * (3.0 * ry * rz);
  }
  if (v.lds) {
    const int k = v.slot(id);
    lm->m[k] = M; lm->x[k] = cx; lm->y[k] = cy; lm->z[k] = cz;
    lm->first[k] = first;
  }
  const double cb = cbrt(M);
  RefNode& out = nodes[id];                  // the record but its padding
  out.cx = cx; out.cy = cy; out.cz = cz;
  set_floor(out, size, dm_power(M, cb));
  out.m = M;
  out.esum = size * 0.015 + cb * 0.002;
  out.skip = end; out.first = first; out.depth = (int16_t)d; out.leaf = 0;
  out.qxx = qxx; out.qyy = qyy; out.qzz = qzz; out.qxy = qxy; out.qxz = qxz; out.qyz = qyz;
  out.size = size;
  // Upper edge of the opening test's band for r^2 (NEXT tests r^2 + 1e-20,
  // so the 1e-20 is taken off the edge); NaN (a group's test then forms the band
  // in FP64, a target's is exact) beyond FP32's range and where
  // (size/theta)^2 <= 1e-16, where the 1e-20 would eat the band's margin.
  const double q = size * inv_theta;
  const double q2 = q * q;
  const float acc2 =
      (q2 > 1e-16 && q2 < 1e36) ? __double2float_ru(q2 * (1.0 + 2e-6) - 1e-20) : __builtin_nanf("");
  heads[id] = WalkHead{cx, cy, cz, acc2, M == 0.0 ? (end | kLinkZeroMass) : end};
}

// The internal nodes [beg, beg + cnt) of the node list, all of depth d.
__global__ __launch_bounds__(kBlock) void k_upward(const int32_t* __restrict__ level_list,
                                                   const uint32_t* __restrict__ end_list, int64_t beg, int64_t cnt,
                                                   int d, RefNode* __restrict__ nodes, WalkHead* __restrict__ heads,
                                                   double inv_theta, const int32_t* __restrict__ sys,
                                                   const double* __restrict__ root) {
  const int64_t k = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (k >= cnt) return;
  upward_node(UnitView{}, nullptr, level_list[beg + k], (int32_t)end_list[beg + k], d, nodes, heads, inv_theta, 0.0,
              sys, root);
}

// Depths d_lo .. 41 of a build whose counts stay on the device, deepest
// first, in one workgroup (a barrier between depths: the waves share the
// CU's cache, so a depth's results are visible to the next): the deep end
// of a tree holds few nodes, chains mostly, and its depth varies from build
// to build.
__global__ __launch_bounds__(kBlock) void k_upward_tail(int d_lo, const int32_t* __restrict__ level_list,
                                                        const uint32_t* __restrict__ end_list,
                                                        RefNode* __restrict__ nodes, WalkHead* __restrict__ heads,
                                                        double inv_theta, const int32_t* __restrict__ sys,
                                                        const double* __restrict__ root,
                                                        const DevScalars* __restrict__ sc) {
  if (sc->abort_flags) return;
  for (int d = kMaxLevels - 1; d >= d_lo; --d) {
    const int64_t beg = sc->level_off[d], cnt = sc->level_count[d];
    if (cnt == 0) continue;
    for (int64_t k = threadIdx.x; k < cnt; k += kBlock)
      upward_node(UnitView{}, nullptr, level_list[beg + k], (int32_t)end_list[beg + k], d, nodes, heads, inv_theta, 0.0,
              sys, root);
    __syncthreads();
  }
}

// The same for depth d of a build whose counts stay on the device: the
// depth's extent in the node list comes from the scalars (k_check), the grid
// is fixed and strides over it.
__global__ __launch_bounds__(kBlock) void k_upward_level(int d, const int32_t* __restrict__ level_list,
                                                         const uint32_t* __restrict__ end_list,
                                                         RefNode* __restrict__ nodes, WalkHead* __restrict__ heads,
                                                         double inv_theta, const int32_t* __restrict__ sys,
                                                         const double* __restrict__ root,
                                                         const DevScalars* __restrict__ sc) {
  if (sc->abort_flags) return;
  const int64_t beg = sc->level_off[d], cnt = sc->level_count[d];
  for (int64_t k = (int64_t)blockIdx.x * kBlock + threadIdx.x; k < cnt; k += (int64_t)gridDim.x * kBlock)
    upward_node(UnitView{}, nullptr, level_list[beg + k], (int32_t)end_list[beg + k], d, nodes, heads, inv_theta, 0.0,
              sys, root);
}

__global__ __launch_bounds__(kBlock) void k_upward_unit(UnitArgs a, RefNode* __restrict__ nodes,
                                                        WalkHead* __restrict__ heads, double inv_theta,
                                                        const int32_t* __restrict__ sys,
                                                        const double* __restrict__ root) {
  __shared__ UnitMoments lm;
  static_assert(2 * (sizeof(UnitMoments) + unit_lds<kUnitNodes>()) <= 160 * 1024, "two units on a CU");
  const double half = root[3];
  upward_unit<kUnitNodes>(
      a,
      [&](const UnitView& v, int32_t k) {
        const RefNode& nd = nodes[k];
        const int s = v.slot(k);
        lm.m[s] = nd.m; lm.x[s] = nd.cx; lm.y[s] = nd.cy; lm.z[s] = nd.cz;
        lm.first[s] = nd.first;
      },
      [&](const UnitView& v, int32_t id, int32_t end, int d) {
        upward_node(v, &lm, id, end, d, nodes, heads, inv_theta, half, sys, root);
      });
}

__global__ __launch_bounds__(kOverBlock) void k_upward_over(UnitArgs a, SysArrays sy, RefNode* __restrict__ nodes,
                                                            WalkHead* __restrict__ heads, double inv_theta,
                                                            const int32_t* __restrict__ sys) {
  const double half = sy.root[3];
  upward_over(a, sy, [&](const UnitView& v, int32_t id, int32_t end, int d) {
    upward_node(v, nullptr, id, end, d, nodes, heads, inv_theta, half, sys, sy.root);
  });
}

// Blocks are dealt to the 8 XCDs round-robin; remap so that each XCD walks
// one contiguous (spatially coherent) range of targets and its L2 holds
// the part of the tree those targets touch.
__device__ __forceinline__ int64_t xcd_block(int nb) {
  const int per = (nb + 7) / 8;
  return (int64_t)(blockIdx.x % 8) * per + blockIdx.x / 8;
}

// Reciprocal square root and reciprocal: the v_rsq_f64 / v_rcp_f64 estimates
// refined by one Newton step each (the residual formed with an FMA).  v_rsq_f64
// is off by up to 5.2e-8, 1.1e-8 in the root mean square, so rsq_nr by up to
// 4.2e-15, 3.5e-16 in the root mean square, 1.8e-16 too small on average.  The walk's
// arguments are positive, finite and mid-range: r^2 + 1e-20, r^2 + eps^2
// with eps >= 1e-4, and 1 + 10 dist >= 1.
__device__ __forceinline__ double rsq_nr(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = __builtin_fma(-(x * y), y, 1.0);        // 1 - x y^2
  return __builtin_fma(0.5 * y, e, y);
}

__device__ __forceinline__ double rcp_nr(double x) {
  const double y = __builtin_amdgcn_rcp(x);
  const double e = __builtin_fma(-x, y, 1.0);              // 1 - x y
  return __builtin_fma(y, e, y);
}

// Lower edge of the opening test's band from its upper edge acc2 (FP32,
// (size/theta)^2 (1 + 2e-6) - 1e-20 rounded up, for (size/theta)^2 > 1e-16):
// r^2 below it has r^2 + 1e-20 below (size/theta)^2 (1 - 2e-6).  Squared
// distances between the edges are decided by NEXT's expression.
constexpr double kBandLow = (1.0 - 2e-6) / (1.0 + 2.2e-6);

// The walk.  One wave per group of up to 64 targets (fewer targets: 64 / width
// lanes on each), three parts:
//  - Group traversal.  Each lane tests another node against the group's box:
//    a node that every target accepts goes to a list, one that every target
//    opens is descended (the rest of the lane's preorder range handed to idle
//    lanes through a stack in LDS), and a subtree on which the targets may
//    differ goes to a second list.  About 26 wave steps per group of 64.
//  - Nodes the whole group accepts (44 of a target's 174 on the cold sphere
//    of 2^20 bodies): with one lane per target their records come in by
//    scalar loads, every lane busy.
//  - The mixed subtrees: each lane walks them on its own with NEXT's test
//    (192 lane steps for 130 accepted nodes), so the wave's steps are its
//    slowest lane's visits, not the union of all lanes' (725 of which 28 % of
//    lanes decided anything), and nothing waits in a ring.
// Each target's terms are NEXT's; they are added in another order than
// NEXT's recursion: group part first, every list summed from zero and then
// added to the target's total (in one running sum, the 2^20 bodies' median
// error was 7.2e-16; so it is 5.1e-16, NEXT's own order 4.9e-16).  Measured,
// walk per step, against one union traversal per 64 targets with deferred
// evaluation: cold sphere 2^20 1.69 -> 1.31 ms; 200,003 bodies at theta 0.3, a tenth dark matter 2.83 ->
// 0.83; Plummer 16,384 0.37 -> 0.11; 50,021 with a fifth dark matter 0.82 ->
// 0.16.  Bound at 2^20 by the lanes' record loads: the texture units are busy
// 86 % (addresses) and 91 % (data) of the time and a fifth of the vector cache's
// accesses go on to L2 (16 waves of some 80 KB each on 32 KB), VALU 47 %.  Loading the records cooperatively (4
// lanes per record, through LDS, by DMA or registers) cut the accesses by a
// third and was as fast (1.29-1.34), several waves per workgroup and lanes
// kept to windows of the list were slower, and so are 5 or 6 waves per SIMD
// (1.36, 1.43; 6 and more registers spilled) instead of 4.
constexpr int kWalkStack = 64;     // donated node ranges per wave (a full stack only means a lane keeps its range)
constexpr int kWalkCommon = 192;   // nodes the whole group accepts, per flush
constexpr int kWalkMixed = 192;    // subtrees on which the group's targets differ, per flush
static_assert(kWalkCommon > kWave && kWalkMixed > kWave, "a wave step appends up to 64 entries");

// The running sums of a target.
struct Sum3 { double x, y, z; };

// One accepted node on one target (octree.h:139-172, G = 1): products fused
// into FMAs and the square roots and divides as rsq_nr and rcp_nr give them.
// d: node minus target, r2 = |d|^2 as the opening test forms it; dist =
// sqrt(r2 + 1e-20), eps from softening.h:26-36, dinv = 1/sqrt(r2 + eps^2).
// DM: some target is dark matter: its softening floor (octree.h:146-148) is
// 2 size / (m/mi)^p, dmk (1 + dmr) times the target's mass power mip (dm_power;
// 0 for a target that is not dark matter).  QUAD: the quadrupole term
// 0.5 (2 (Q d) inv5 - 5 q inv7 d), q = d.Q.d, as (Q d) inv5 + d (-(2.5 q) inv7).
template <bool DM, bool QUAD>
__device__ __forceinline__ void interact(double dx, double dy, double dz, double r2, double m, double esum,
                                         double dmk, float dmr, const DmPower& mip, double qxx, double qyy,
                                         double qzz, double qxy, double qxz, double qyz, Sum3& a) {
  const double r2e = r2 + 1e-20;
  const double dist = r2e * rsq_nr(r2e);
  double eps = esum * rcp_nr(__builtin_fma(dist, 10.0, 1.0));
  if (eps < 1e-4) eps = 1e-4;
  if (DM) {
    const double alt = __builtin_fma(dmk, mip.p, dmk * mip.p * (double)(dmr + mip.r));
    if (eps < alt) eps = alt;
  }
  const double dinv = rsq_nr(__builtin_fma(eps, eps, r2));
  const double inv2 = dinv * dinv;
  const double inv3 = inv2 * dinv;
  if (QUAD) {
    const double inv5 = inv3 * inv2;
    const double inv7 = inv5 * inv2;
    const double sx = __builtin_fma(qxz, dz, __builtin_fma(qxy, dy, qxx * dx));
    const double sy = __builtin_fma(qyz, dz, __builtin_fma(qyy, dy, qxy * dx));
    const double sz = __builtin_fma(qzz, dz, __builtin_fma(qyz, dy, qxz * dx));
    const double q = __builtin_fma(dz, sz, __builtin_fma(dy, sy, dx * sx));
    const double c = __builtin_fma(-2.5 * q, inv7, m * inv3);
    a.x = __builtin_fma(dx, c, __builtin_fma(sx, inv5, a.x));
    a.y = __builtin_fma(dy, c, __builtin_fma(sy, inv5, a.y));
    a.z = __builtin_fma(dz, c, __builtin_fma(sz, inv5, a.z));
  } else {
    const double c = m * inv3;
    a.x = __builtin_fma(dx, c, a.x);
    a.y = __builtin_fma(dy, c, a.y);
    a.z = __builtin_fma(dz, c, a.z);
  }
}

__device__ __forceinline__ const RefNode& node_at(const RefNode* nodes, uint32_t off) {
  return *reinterpret_cast<const RefNode*>(reinterpret_cast<const char*>(nodes) + off);
}

// Nodes every target of the group accepts (bit 31: a leaf, which carries no
// quadrupole).  One lane per target (parts == 1): the entry is wave-uniform,
// so its record comes in through scalar loads and every lane is busy.  With
// more lanes per target, each part takes every parts-th entry.
template <bool DM>
__device__ __forceinline__ void walk_common(const int32_t* list, int n, int part, int parts,
                                            const RefNode* __restrict__ nodes, uint32_t zoff, double px, double py,
                                            double pz, const DmPower& mip, Sum3& sum) {
  Sum3 a{0.0, 0.0, 0.0};
  if (parts == 1) {
    for (int k = 0; k < n; ++k) {
      const int32_t e = __builtin_amdgcn_readfirstlane(list[k]);
      const RefNode& nd = node_at(nodes, (uint32_t)e << 7);
      const double dx = nd.cx - px, dy = nd.cy - py, dz = nd.cz - pz;
      const double r2 = __builtin_fma(dz, dz, __builtin_fma(dy, dy, dx * dx));
      if (e < 0)
        interact<DM, false>(dx, dy, dz, r2, nd.m, nd.esum, nd.dmk, nd.dmr, mip, 0, 0, 0, 0, 0, 0, a);
      else
        interact<DM, true>(dx, dy, dz, r2, nd.m, nd.esum, nd.dmk, nd.dmr, mip, nd.qxx, nd.qyy, nd.qzz, nd.qxy,
                           nd.qxz, nd.qyz, a);
    }
  } else {
    for (int k = part; k < n; k += parts) {
      const int32_t e = list[k];
      const uint32_t off = (uint32_t)e << 7;
      const RefNode& nd = node_at(nodes, off);
      const RefNode& qn = node_at(nodes, e < 0 ? zoff : off);
      const double dx = nd.cx - px, dy = nd.cy - py, dz = nd.cz - pz;
      const double r2 = __builtin_fma(dz, dz, __builtin_fma(dy, dy, dx * dx));
      interact<DM, true>(dx, dy, dz, r2, nd.m, nd.esum, nd.dmk, nd.dmr, mip, qn.qxx, qn.qyy, qn.qzz, qn.qxy, qn.qxz,
                         qn.qyz, a);
    }
  }
  sum.x += a.x; sum.y += a.y; sum.z += a.z;
}

// Subtrees on which the group's targets differ: every lane walks them on its
// own, with its own target's opening test, and evaluates a node as it
// accepts it.  The next node's head is loaded while the accepted node is
// evaluated.
template <bool DM, bool COUNT>
__device__ __forceinline__ void walk_mixed(const int32_t* list, int n, bool valid, int part, int parts, int32_t self,
                                           const RefNode* __restrict__ nodes, const WalkHead* __restrict__ heads,
                                           uint32_t zoff, double theta, double px, double py, double pz,
                                           const DmPower& mip, Sum3& sum, uint32_t& npp, uint32_t& npc, uint32_t& nop,
                                           uint32_t& nit) {
  Sum3 a{0.0, 0.0, 0.0};
  int k = part;
  bool live = valid && k < n;
  int32_t cur = live ? list[k] : 0, root = cur, end = 0;
  WalkHead h = heads[cur];
  while (live) {
    const bool leaf = h.link < 0;
    int32_t skip = leaf ? cur + 1 : (h.link & ~kLinkZeroMass);
    if (skip <= cur) skip = cur + 1;                         // skip > cur by construction
    if (cur == root) end = skip;
    const double dx = h.cx - px, dy = h.cy - py, dz = h.cz - pz;
    const double r2 = __builtin_fma(dz, dz, __builtin_fma(dy, dy, dx * dx));
    // octree.h:134-135: massless nodes and the target itself
    const bool pass = (h.link >= 0 && (h.link & kLinkZeroMass)) || h.link == self;
    bool accept = leaf;
    if (!leaf) {
      // Against the band edges (about 4e-6 wide) any rounding of r^2 decides
      // alike: FMAs here, NEXT's expression, as NEXT rounds it, inside.
      const double hi = (double)h.acc2;                      // NaN: no fast decision
      accept = r2 > hi;
      if (!accept && !(r2 < hi * kBandLow)) {                // rare
        const double r2e = (dx * dx + dy * dy + dz * dz) + 1e-20;
        accept = (nodes[cur].size / sqrt(r2e)) < theta;
      }
    }
    const bool take = !pass && accept;
    int32_t next = (pass || accept) ? skip : cur + 1;
    if (COUNT) {
      npp += (take && leaf) ? 1u : 0u;
      npc += (take && !leaf) ? 1u : 0u;
      nop += (!pass && !accept) ? 1u : 0u;
      nit += 1u;
    }
    if (next >= end) {                                       // this subtree is done
      k += parts;
      live = k < n;
      next = live ? list[k] : 0;
      root = next;
    }
    const WalkHead hn = heads[next];
    if (take) {
      const uint32_t off = (uint32_t)cur << 7;
      const RefNode& nd = node_at(nodes, off);
      const RefNode& qn = node_at(nodes, leaf ? zoff : off);
      interact<DM, true>(dx, dy, dz, r2, nd.m, nd.esum, nd.dmk, nd.dmr, mip, qn.qxx, qn.qyy, qn.qzz, qn.qxy, qn.qxz,
                         qn.qyz, a);
    }
    cur = next;
    h = hn;
  }
  sum.x += a.x; sum.y += a.y; sum.z += a.z;
}

template <bool KICK, bool COUNT>
__global__ __launch_bounds__(kWave) __attribute__((amdgpu_waves_per_eu(4)))
void k_walk(const Group* __restrict__ groups, int64_t ngroups, const RefNode* __restrict__ nodes,
            const WalkHead* __restrict__ heads, StateArrays st, SysArrays sy, double theta, double* __restrict__ ax,
            double* __restrict__ ay, double* __restrict__ az, DevScalars* sc) {
  __shared__ int32_t stk_b[kWalkStack], stk_e[kWalkStack];   // donated ranges [stk_b, stk_e)
  __shared__ int32_t common[kWalkCommon], mixed[kWalkMixed];
  const int64_t gi = xcd_block(gridDim.x);
  if (gi >= ngroups || sc->abort_flags) return;            // past the end, or an aborted build
  const int lane = threadIdx.x;
  const Group g = groups[gi];
  if (g.count == 0) return;                                // (fills an XCD's part of the table)
  int width = kWave;
  while (width > 1 && (width >> 1) >= g.count) width >>= 1;
  const int parts = kWave / width;
  const int slot = lane & (width - 1), part = lane / width;
  const bool valid = slot < g.count;
  const int64_t i = g.first + (valid ? slot : 0);
  const double px = st.x[i], py = st.y[i], pz = st.z[i], pm = st.m[i];
  const bool dark = valid && st.type[i] == 1;
  const DmPower mip = dark ? dm_power(pm, cbrt(pm)) : DmPower{0.0, 0.0f};
  const bool any_dm = __ballot(dark) != 0;
  const int32_t self = ~(int32_t)i;                          // link of this target's own leaf
  const uint64_t ltmask = lanemask_lt();
  const uint32_t zoff = (uint32_t)sc->total_nodes << 7;      // the all-zero record (k_emit)

  // The group's box.
  double lo[3] = {px, py, pz}, hi[3] = {px, py, pz};
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      lo_upd(lo[k], __shfl_xor(lo[k], off, kWave));
      hi_upd(hi[k], __shfl_xor(hi[k], off, kWave));
    }
  }

  Sum3 a{0.0, 0.0, 0.0};
  uint32_t npp = 0, npc = 0, nop = 0, nit = 0, nev = 0, nlane = 0;
  int nc = 0, nm = 0, sp = 0;
  auto flush_common = [&]() {
    __syncthreads();
    if (any_dm) walk_common<true>(common, nc, part, parts, nodes, zoff, px, py, pz, mip, a);
    else walk_common<false>(common, nc, part, parts, nodes, zoff, px, py, pz, mip, a);
    if (COUNT) nev += (nc + parts - 1) / parts;
    __syncthreads();
    nc = 0;
  };
  auto flush_mixed = [&]() {
    __syncthreads();
    uint32_t steps = 0;
    if (any_dm)
      walk_mixed<true, COUNT>(mixed, nm, valid, part, parts, self, nodes, heads, zoff, theta, px, py, pz, mip, a, npp,
                              npc, nop, steps);
    else
      walk_mixed<false, COUNT>(mixed, nm, valid, part, parts, self, nodes, heads, zoff, theta, px, py, pz, mip, a,
                               npp, npc, nop, steps);
    if (COUNT) {
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) {
        const uint32_t o = __shfl_xor(steps, off, kWave);
        steps = o > steps ? o : steps;
      }
      nlane += steps;
    }
    __syncthreads();
    nm = 0;
  };

  const int32_t root = sy.sroot[g.sys], total = sy.send[g.sys];   // this system's tree
  int32_t cur = lane == 0 ? root : total, end = total;
  for (;;) {
    // idle lanes take ranges from the top of the stack
    const bool idle = cur >= end;
    const uint64_t im = __ballot(idle);
    const int avail = (int)__popcll(im);
    const int give = avail < sp ? avail : sp;
    if (idle) {
      const int r = (int)__popcll(im & ltmask);
      if (r < give) { cur = stk_b[sp - 1 - r]; end = stk_e[sp - 1 - r]; }
    }
    sp -= give;
    const bool busy = cur < end;
    if (!__ballot(busy)) break;
    if (COUNT) ++nit;
    if (nc > kWalkCommon - kWave) flush_common();
    if (nm > kWalkMixed - kWave) flush_mixed();
    bool acc = false, mix = false, donate = false, leaf = false, opened = false;
    int32_t skip = 0;
    if (busy) {
      const WalkHead h = heads[cur];
      leaf = h.link < 0;
      skip = leaf ? cur + 1 : (h.link & ~kLinkZeroMass);
      if (skip <= cur) skip = cur + 1;
      const bool zero = h.link >= 0 && (h.link & kLinkZeroMass);
      if (leaf) {
        const int32_t body = ~h.link;
        mix = body >= g.first && body < g.first + g.count;   // some target's own leaf
        acc = !mix;
      } else if (!zero) {
        // |fl(c - p)| lies between the distances of the box's near and far
        // faces (rounding is monotone), and so does r^2, formed alike: a
        // decision outside the band for both faces is every target's.
        const double nx = fmax(fmax(lo[0] - h.cx, h.cx - hi[0]), 0.0), fx = fmax(h.cx - lo[0], hi[0] - h.cx);
        const double ny = fmax(fmax(lo[1] - h.cy, h.cy - hi[1]), 0.0), fy = fmax(h.cy - lo[1], hi[1] - h.cy);
        const double nz = fmax(fmax(lo[2] - h.cz, h.cz - hi[2]), 0.0), fz = fmax(h.cz - lo[2], hi[2] - h.cz);
        const double r2n = __builtin_fma(nz, nz, __builtin_fma(ny, ny, nx * nx));
        const double r2f = __builtin_fma(fz, fz, __builtin_fma(fy, fy, fx * fx));
        const double e = (double)h.acc2;
        acc = r2n > e;
        opened = r2f < e * kBandLow;
        if (e != e) {                                        // the band lies outside FP32's range
          const double q = nodes[cur].size / theta, q2 = q * q;
          acc = r2n + 1e-20 > q2 * (1.0 + 2e-6);
          opened = r2f + 1e-20 < q2 * (1.0 - 2e-6);
        }
        mix = !acc && !opened;
        donate = opened && skip < end;
      }
    }
    const uint64_t am = __ballot(acc), mm = __ballot(mix), dm = __ballot(donate);
    if (acc) common[nc + (int)__popcll(am & ltmask)] = leaf ? (int32_t)(cur | 0x80000000u) : cur;
    if (mix) mixed[nm + (int)__popcll(mm & ltmask)] = cur;
    nc += (int)__popcll(am);
    nm += (int)__popcll(mm);
    if (COUNT) {
      if (acc) { if (leaf) npp += g.count; else npc += g.count; }
      if (opened) nop += g.count;
    }
    // opened nodes hand [skip, end) to the stack while it has room
    const int room = kWalkStack - sp;
    if (donate) {
      const int r = (int)__popcll(dm & ltmask);
      if (r < room) { stk_b[sp + r] = skip; stk_e[sp + r] = end; end = skip; }
    }
    sp += (int)__popcll(dm) < room ? (int)__popcll(dm) : room;
    if (busy) cur = opened ? cur + 1 : skip;
    __syncthreads();
  }
  if (nc) flush_common();
  if (nm) flush_mixed();
  for (int off = width; off < kWave; off <<= 1) {
    a.x += __shfl_xor(a.x, off, kWave);
    a.y += __shfl_xor(a.y, off, kWave);
    a.z += __shfl_xor(a.z, off, kWave);
  }
  double v2 = 0.0;
  if (valid && part == 0) {
    ax[i] = a.x; ay[i] = a.y; az[i] = a.z;
    if (KICK) {                                             // step.h:171-173
      const double half = sy.dt[g.sys] * 0.5;
      const double vx = st.vx[i] + a.x * half;
      const double vy = st.vy[i] + a.y * half;
      const double vz = st.vz[i] + a.z * half;
      st.vx[i] = vx; st.vy[i] = vy; st.vz[i] = vz;
      v2 = vx * vx + vy * vy + vz * vz;
      if (!(v2 > 0.0)) v2 = 0.0;
    }
  }
  if (KICK) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
      const double o = __shfl_xor(v2, off, kWave);
      if (o > v2) v2 = o;
    }
    if (lane == 0 && v2 > 0.0) atomicMax(&sy.v2max[g.sys], (unsigned long long)__double_as_longlong(v2));
  }
  if (COUNT) {
    const uint32_t sp2 = wave_sum_u32(npp), sc2 = wave_sum_u32(npc), so = wave_sum_u32(nop);
    if (lane == 0) {
      atomicAdd(&sc->n_pp, (unsigned long long)sp2);
      atomicAdd(&sc->n_pc, (unsigned long long)sc2);
      atomicAdd(&sc->n_open, (unsigned long long)so);
      atomicAdd(&sc->n_iter, (unsigned long long)(nit + nlane));
      atomicAdd(&sc->n_eval, (unsigned long long)(nev + nlane));
    }
  }
}

// Opening half kick and drift (step.h:120-122, 141-146), each system with its dt.
// amag (may be null) receives |a| of each body, in FP32, for an opening
// criterion relative to the previous acceleration.
__global__ __launch_bounds__(kBlock) void k_kick_drift(int64_t n, StateArrays st, const double* __restrict__ ax,
                                                       const double* __restrict__ ay, const double* __restrict__ az,
                                                       SysArrays sy, float* __restrict__ amag) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const double dt = sy.dt[st.sys[i]];
  const double half = dt * 0.5;
  const double gx = ax[i], gy = ay[i], gz = az[i];
  const double vx = st.vx[i] + gx * half;
  const double vy = st.vy[i] + gy * half;
  const double vz = st.vz[i] + gz * half;
  st.vx[i] = vx; st.vy[i] = vy; st.vz[i] = vz;
  st.x[i] = st.x[i] + vx * dt;
  st.y[i] = st.y[i] + vy * dt;
  st.z[i] = st.z[i] + vz * dt;
  if (amag) amag[i] = (float)sqrt(gx * gx + gy * gy + gz * gz);
}

// Max |v|^2 per system (adaptive.h:31-37).  Each thread takes kMaxv2Items
// bodies (block-strided), a block whose bodies all belong to one system
// reduces in registers and LDS and makes one atomic; otherwise every body
// makes its own.
constexpr int kMaxv2Items = 4;
__global__ __launch_bounds__(kBlock) void k_maxv2(int64_t n, StateArrays st, SysArrays sy) {
  __shared__ double red[kBlock / kWave];
  const int64_t base = (int64_t)blockIdx.x * kBlock * kMaxv2Items;
  const int64_t last = base + (int64_t)kBlock * kMaxv2Items - 1 < n ? base + (int64_t)kBlock * kMaxv2Items - 1 : n - 1;
  const int32_t s0 = st.sys[base];
  const bool one = st.sys[last] == s0;                    // sorted by system within the block's range
  double v2 = 0.0;
  for (int k = 0; k < kMaxv2Items; ++k) {
    const int64_t i = base + (int64_t)k * kBlock + threadIdx.x;
    if (i >= n) break;
    double w = st.vx[i] * st.vx[i] + st.vy[i] * st.vy[i] + st.vz[i] * st.vz[i];
    if (!(w > 0.0)) w = 0.0;
    if (one) {
      if (w > v2) v2 = w;
    } else if (w > 0.0) {
      atomicMax(&sy.v2max[st.sys[i]], (unsigned long long)__double_as_longlong(w));
    }
  }
  if (!one) return;                                        // block-uniform
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const double o = __shfl_xor(v2, off, kWave);
    if (o > v2) v2 = o;
  }
  if (lane_id() == 0) red[threadIdx.x / kWave] = v2;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kBlock / kWave; ++w) v2 = red[w] > v2 ? red[w] : v2;
    if (v2 > 0.0) atomicMax(&sy.v2max[s0], (unsigned long long)__double_as_longlong(v2));
  }
}

// computeAdaptiveDt (adaptive.h:38-51) for each system from its max |v|^2;
// dts (may be null) receives system 0's value for `step`.
__global__ __launch_bounds__(kBlock) void k_dt(SysArrays sy, double base, double* dts, int64_t step,
                                               DevScalars* sc) {
  const int s = blockIdx.x * kBlock + threadIdx.x;
  if (s >= sy.nsys) return;
  const double v2 = __longlong_as_double((long long)sy.v2max[s]);
  sy.v2max[s] = 0ull;   // read once: the next kicks gather the next step's maximum
  double v = sqrt(v2);
  if (1e4 < v) v = 1e4;
  double dt;
  if (v < 1e-8) {
    dt = base;
  } else {
    dt = base / (1.0 + v);
    if (dt < base * 0.01) dt = base * 0.01;
    if (base * 1.0 < dt) dt = base * 1.0;
  }
  sy.dt[s] = dt;
  if (dts && s == 0) {
    // step < 0: the entry comes from the device's step counter (captured runs)
    const int64_t at = step >= 0 ? step : (int64_t)(sc->step_count++);
    dts[at] = dt;
  }
}

__device__ __forceinline__ uint32_t digit_at(const uint64_t* key, const uint64_t* key2, int32_t f, int l) {
  if (l < kKeyDigits) return (uint32_t)(key[f] >> (3 * (kKeyDigits - 1 - l))) & 7u;
  return key2 ? (uint32_t)(key2[f] >> (3 * (kMaxLevels - 1 - l))) & 7u : 0u;
}

__global__ __launch_bounds__(kBlock) void k_export(int64_t total, const RefNode* __restrict__ nodes,
                                                   const uint64_t* __restrict__ key, const uint64_t* __restrict__ key2,
                                                   const int32_t* __restrict__ id, SysArrays sy,
                                                   int32_t* depth, int32_t* leaf, int32_t* body, int32_t* cmask,
                                                   double* geo4, double* mass, double* com3, double* q6) {
  const int64_t k = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (k >= total) return;
  const RefNode nd = nodes[k];
  depth[k] = nd.depth;
  leaf[k] = nd.leaf;
  body[k] = nd.leaf ? id[nd.first] : -1;
  double cx = sy.root[0], cy = sy.root[1], cz = sy.root[2], s = sy.root[3];
  for (int l = 0; l < nd.depth; ++l) {
    const uint32_t o = digit_at(key, key2, nd.first, l);
    const double hs = s * 0.5;
    cx = cx + ((o & 1u) ? hs : -hs);
    cy = cy + ((o & 2u) ? hs : -hs);
    cz = cz + ((o & 4u) ? hs : -hs);
    s = hs;
  }
  geo4[4 * k] = cx; geo4[4 * k + 1] = cy; geo4[4 * k + 2] = cz; geo4[4 * k + 3] = s;
  int32_t mask = 0;
  if (!nd.leaf)
    for (int32_t c = (int32_t)k + 1, it = 0; it < 8 && c < nd.skip; ++it, c = nodes[c].skip)
      mask |= 1 << digit_at(key, key2, nodes[c].first, nd.depth);
  cmask[k] = mask;
  mass[k] = nd.m;
  com3[3 * k] = nd.cx; com3[3 * k + 1] = nd.cy; com3[3 * k + 2] = nd.cz;
  const bool lf = nd.leaf != 0;
  q6[6 * k] = lf ? 0.0 : nd.qxx; q6[6 * k + 1] = lf ? 0.0 : nd.qyy; q6[6 * k + 2] = lf ? 0.0 : nd.qzz;
  q6[6 * k + 3] = lf ? 0.0 : nd.qxy; q6[6 * k + 4] = lf ? 0.0 : nd.qxz; q6[6 * k + 5] = lf ? 0.0 : nd.qyz;
}

inline unsigned grid_of(int64_t n) { return (unsigned)div_up(n, kBlock); }

}  // namespace

inline unsigned sys_grid(const SysArrays& sy) { return (unsigned)div_up(std::max(sy.nsys, 1), kBlock); }

void launch_fill_scalars(DevScalars* sc, int what, hipStream_t s) {
  hipLaunchKernelGGL(k_fill_scalars, dim3(1), dim3(kBlock), 0, s, sc, what);
}
void launch_fill_v2max(const SysArrays& sy, hipStream_t s) {
  hipLaunchKernelGGL(k_fill_v2max, dim3(sys_grid(sy)), dim3(kBlock), 0, s, sy);
}
void launch_set_dt(const SysArrays& sy, double dt, hipStream_t s) {
  hipLaunchKernelGGL(k_set_dt, dim3(sys_grid(sy)), dim3(kBlock), 0, s, sy, dt);
}
void launch_bbox(const StateArrays& st, const BoxBlock* blocks, int nblocks, const int32_t* block_off, double* part,
                 const SysArrays& sy, DevScalars* clear, hipStream_t s) {
  if (nblocks > 0) hipLaunchKernelGGL(k_bbox_partial, dim3(nblocks), dim3(kBlock), 0, s, st, blocks, part);
  hipLaunchKernelGGL(k_bbox_final, dim3((unsigned)std::max(sy.nsys, 1)), dim3(kWave), 0, s, part, block_off, sy,
                     clear);
}
void launch_keys(int64_t n, const StateArrays& st, const SysArrays& sy, uint64_t* key, uint32_t* idx,
                 DevScalars* scw, hipStream_t s) {
  if (n > 0) hipLaunchKernelGGL(k_keys, dim3(grid_of(n)), dim3(kBlock), 0, s, n, st, sy, key, idx, scw);
}
void launch_keys2(int64_t n, const StateArrays& st, const SysArrays& sy, uint64_t* key2, hipStream_t s) {
  if (n > 0) hipLaunchKernelGGL(k_keys2, dim3(grid_of(n)), dim3(kBlock), 0, s, n, st, sy, key2);
}
void launch_keys_export(int64_t n, const StateArrays& st, const SysArrays& sy, uint64_t* hi, uint64_t* lo,
                        hipStream_t s) {
  if (n > 0) hipLaunchKernelGGL(k_keys_export, dim3(grid_of(n)), dim3(kBlock), 0, s, n, st, sy, hi, lo);
}
void launch_fix_runs(int64_t n, const StateArrays& st, const SysArrays& sy, uint64_t* key, uint64_t* key2,
                     uint32_t* amag, int lo, hipStream_t s) {
  if (n > 1) hipLaunchKernelGGL(k_fix_runs, dim3(grid_of(n)), dim3(kBlock), 0, s, n, st, sy, key, key2, amag, lo);
}
void launch_rank_sort(int64_t n, const uint64_t* key, uint64_t* kout, const StateArrays& src, const StateArrays& dst,
                      const uint32_t* amag, uint32_t* amag_out, hipStream_t s) {
  if (n > 0)
    hipLaunchKernelGGL(k_rank_sort, dim3((unsigned)div_up(n, kWave)), dim3(kRankWaves * kWave), 0, s, (int32_t)n, key,
                       kout, src, dst, amag, amag_out);
}
void launch_set_ids(int64_t n, int32_t* id, int32_t id0, int32_t* sys, int32_t sys_no, hipStream_t s) {
  if (n > 0) hipLaunchKernelGGL(k_set_ids, dim3(grid_of(n)), dim3(kBlock), 0, s, n, id, id0, sys, sys_no);
}
void launch_out_index(int64_t cnt, const int32_t* id, int32_t base, uint32_t* inv, int32_t* bad, hipStream_t s) {
  if (cnt <= 0) return;
  hipLaunchKernelGGL(k_out_index, dim3(grid_of(cnt)), dim3(kBlock), 0, s, cnt, id, base, inv);
  hipLaunchKernelGGL(k_out_check, dim3(grid_of(cnt)), dim3(kBlock), 0, s, cnt, id, base, inv, bad);
}
void launch_out_gather(int64_t j0, int64_t len, int64_t cnt, const uint32_t* inv, const OutArrays& src, int m,
                       double* dst, hipStream_t s) {
  if (len > 0 && m > 0)
    hipLaunchKernelGGL(k_out_gather, dim3(grid_of(len)), dim3(kBlock), 0, s, j0, len, cnt, inv, src, m, dst);
}
void launch_iota(int64_t n, uint32_t* idx, hipStream_t s) {
  if (n > 0) hipLaunchKernelGGL(k_iota, dim3(grid_of(n)), dim3(kBlock), 0, s, n, idx);
}
void launch_gather_u64(int64_t n, const uint32_t* perm, const uint64_t* src, uint64_t* dst, hipStream_t s) {
  if (n > 0) hipLaunchKernelGGL(k_gather_u64, dim3(grid_of(n)), dim3(kBlock), 0, s, n, perm, src, dst);
}
void launch_gather_sys(int64_t n, const uint32_t* perm, const int32_t* sys, uint32_t* dst, hipStream_t s) {
  if (n > 0) hipLaunchKernelGGL(k_gather_sys, dim3(grid_of(n)), dim3(kBlock), 0, s, n, perm, sys, dst);
}
void launch_gather_u32(int64_t n, const uint32_t* perm, const uint32_t* src, uint32_t* dst, hipStream_t s) {
  if (n > 0)
    hipLaunchKernelGGL(k_gather_sys, dim3(grid_of(n)), dim3(kBlock), 0, s, n, perm,
                       reinterpret_cast<const int32_t*>(src), dst);
}
void launch_gather_state(int64_t n, const uint32_t* perm, const StateArrays& src, const StateArrays& dst,
                         hipStream_t s) {
  if (n > 0) hipLaunchKernelGGL(k_gather_state, dim3(grid_of(n)), dim3(kBlock), 0, s, n, perm, src, dst);
}
void launch_lcp_count(int64_t n, const uint64_t* key, const uint64_t* key2, const int32_t* sys, int32_t* lcp,
                      uint32_t* cnt_s, uint32_t* part, DevScalars* sc, hipStream_t s) {
  if (n <= 0) return;
  const int64_t rows = grid_of(n);
  hipLaunchKernelGGL(k_lcp_count, dim3((unsigned)rows), dim3(kBlock), 0, s, n, key, key2, sys, lcp, cnt_s, part);
  hipLaunchKernelGGL(k_lcp_scan, dim3(kPartW), dim3(kBlock), 0, s, part, rows, key2 ? 1 : 0, sc);
}
void launch_remove_map(int64_t n_new, int64_t cut, int64_t len, uint32_t* perm, hipStream_t s) {
  if (n_new > 0) hipLaunchKernelGGL(k_remove_map, dim3(grid_of(n_new)), dim3(kBlock), 0, s, n_new, cut, len, perm);
}
void launch_relabel(int64_t n, int32_t* sys, int32_t removed, hipStream_t s) {
  if (n > 0) hipLaunchKernelGGL(k_relabel, dim3(grid_of(n)), dim3(kBlock), 0, s, n, sys, removed);
}
void launch_gather_f64(int64_t n, const uint32_t* perm, const double* src, double* dst, hipStream_t s) {
  if (n > 0) hipLaunchKernelGGL(k_gather_f64, dim3(grid_of(n)), dim3(kBlock), 0, s, n, perm, src, dst);
}
void launch_sys_roots(const SysArrays& sy, const uint32_t* pre_off, const DevScalars* sc, hipStream_t s) {
  hipLaunchKernelGGL(k_sys_roots, dim3(sys_grid(sy)), dim3(kBlock), 0, s, sy, pre_off, sc);
}
void launch_emit(int64_t n, const int32_t* lcp, const uint32_t* pre_off, const uint32_t* part,
                 const StateArrays& st, const SysArrays& sy, const DevScalars* sc, RefNode* nodes, WalkHead* heads,
                 int32_t* level_list, uint32_t* end_list, uint32_t cap_nodes, uint32_t cap_int, hipStream_t s) {
  if (n > 0)
    hipLaunchKernelGGL(k_emit, dim3(grid_of(n)), dim3(kBlock), 0, s, n, lcp, pre_off, part, st, sy, sc, nodes, heads,
                       level_list, end_list, cap_nodes, cap_int);
}
void launch_set_run(DevScalars* sc, int32_t step, hipStream_t s) {
  hipLaunchKernelGGL(k_set_run, dim3(1), dim3(1), 0, s, sc, step);
}
void launch_check(DevScalars* sc, int64_t cap_records, int64_t cap_list, int dmax, hipStream_t s) {
  hipLaunchKernelGGL(k_check, dim3(1), dim3(kWave), 0, s, sc, cap_records, cap_list, dmax);
}
void launch_upward_tail(int d_lo, const int32_t* level_list, const uint32_t* end_list, RefNode* nodes,
                        WalkHead* heads, double theta, const int32_t* sys, const double* root, const DevScalars* sc,
                        hipStream_t s) {
  if (d_lo < kMaxLevels)
    hipLaunchKernelGGL(k_upward_tail, dim3(1), dim3(kBlock), 0, s, d_lo, level_list, end_list, nodes, heads,
                       1.0 / theta, sys, root, sc);
}
void launch_upward_level(unsigned grid, int d, const int32_t* level_list, const uint32_t* end_list, RefNode* nodes,
                         WalkHead* heads, double theta, const int32_t* sys, const double* root, const DevScalars* sc,
                         hipStream_t s) {
  hipLaunchKernelGGL(k_upward_level, dim3(grid), dim3(kBlock), 0, s, d, level_list, end_list, nodes, heads,
                     1.0 / theta, sys, root, sc);
}
void launch_upward(const int32_t* level_list, const uint32_t* end_list, int64_t beg, int64_t cnt, int d,
                   RefNode* nodes, WalkHead* heads, double theta, const int32_t* sys, const double* root,
                   hipStream_t s) {
  if (cnt > 0)
    hipLaunchKernelGGL(k_upward, dim3(grid_of(cnt)), dim3(kBlock), 0, s, level_list, end_list, beg, cnt, d, nodes,
                       heads, 1.0 / theta, sys, root);
}
void launch_upward_all(const int32_t* counts, const int32_t* level_list, const uint32_t* end_list, RefNode* nodes,
                       WalkHead* heads, double theta, const int32_t* sys, const double* root, hipStream_t s) {
  int64_t off = 0;
  for (int d = 0; d < kMaxDepthSlots; ++d) off += counts[d];
  for (int d = kMaxDepthSlots - 1; d >= 0; --d) {
    off -= counts[d];
    launch_upward(level_list, end_list, off, counts[d], d, nodes, heads, theta, sys, root, s);
  }
}
void launch_upward_units(const UnitArgs& a, RefNode* nodes, WalkHead* heads, double theta, const int32_t* sys,
                   const SysArrays& sy, hipStream_t s) {
  if (a.n <= 0) return;
  if (sy.nsys == 1) sys = nullptr;                         // one root
  hipLaunchKernelGGL(k_upward_unit, dim3((unsigned)a.units), dim3(kBlock), 0, s, a, nodes, heads, 1.0 / theta, sys,
                     sy.root);
  if (a.units > 1)
    hipLaunchKernelGGL(k_upward_over, dim3((unsigned)std::min(sy.nsys, kOverBlocks)), dim3(kOverBlock), 0, s, a, sy,
                       nodes, heads, 1.0 / theta, sys);
}
void launch_walk(const Group* groups, int64_t ngroups, const RefNode* nodes, const WalkHead* heads,
                 const StateArrays& st,
                 const SysArrays& sy, double theta, double* ax, double* ay, double* az, DevScalars* sc, bool kick,
                 bool count, hipStream_t s) {
  if (ngroups <= 0) return;
  const unsigned nb = (unsigned)(div_up(ngroups, 8) * 8);
#define NBX_RW(K, C) \
  hipLaunchKernelGGL((k_walk<K, C>), dim3(nb), dim3(kWave), 0, s, groups, ngroups, nodes, heads, st, sy, theta, \
                     ax, ay, az, sc)
  if (kick && count) NBX_RW(true, true);
  else if (kick) NBX_RW(true, false);
  else if (count) NBX_RW(false, true);
  else NBX_RW(false, false);
#undef NBX_RW
}
void launch_fill_u32(int64_t n, uint32_t* a, uint32_t v, hipStream_t s) {
  if (n > 0) hipLaunchKernelGGL(k_fill_u32, dim3(grid_of(n)), dim3(kBlock), 0, s, n, a, v);
}
void launch_kick_drift(int64_t n, const StateArrays& st, const double* ax, const double* ay, const double* az,
                       const SysArrays& sy, float* amag, hipStream_t s) {
  if (n > 0) hipLaunchKernelGGL(k_kick_drift, dim3(grid_of(n)), dim3(kBlock), 0, s, n, st, ax, ay, az, sy, amag);
}
void launch_maxv2(int64_t n, const StateArrays& st, const SysArrays& sy, hipStream_t s) {
  if (n > 0)
    hipLaunchKernelGGL(k_maxv2, dim3((unsigned)div_up(n, (int64_t)kBlock * kMaxv2Items)), dim3(kBlock), 0, s, n, st,
                       sy);
}
void launch_dt(const SysArrays& sy, double base, double* dts, int64_t step, DevScalars* sc, hipStream_t s) {
  hipLaunchKernelGGL(k_dt, dim3(sys_grid(sy)), dim3(kBlock), 0, s, sy, base, dts, step, sc);
}
void launch_export(int64_t total, const RefNode* nodes, const uint64_t* key, const uint64_t* key2,
                   const int32_t* id, const SysArrays& sy, int32_t* depth, int32_t* leaf, int32_t* body,
                   int32_t* cmask, double* geo4, double* mass, double* com3, double* q6, hipStream_t s) {
  if (total > 0)
    hipLaunchKernelGGL(k_export, dim3(grid_of(total)), dim3(kBlock), 0, s, total, nodes, key, key2, id, sy, depth,
                       leaf, body, cmask, geo4, mass, com3, q6);
}

}  // namespace nbx

// Physics-mode kernels on gfx950: a bucket-leaf Barnes-Hut walk with
// traceless quadrupoles, Plummer softening and a group acceptance test, plus
// an FP64 direct sum.
//
// Tree: the same depth-first preorder octree as reference mode (one body per
// leaf, skip pointers), read through a compact 64-byte PhysNode.  A node
// whose body count is at most `nleaf` that must be opened is treated as a
// bucket: its bodies go straight to the direct-sum list.
//
// Multipoles (FP64): m, centre of mass, Q_ij = sum m (3 r_i r_j - r^2 d_ij)
// about the centre of mass, propagated with the parallel-axis rule
//   Q = sum_c [Q_c + m_c (3 r_c r_c^T - |r_c|^2 I)],  r_c = com_c - com,
// and bmax, a bound on the distance from the centre of mass to any body: the
// smaller of the distance to the farthest corner of the bodies' bounding box
// and max_c (|r_c| + bmax_c).  A refit (bodies moved, same order and
// topology) recomputes all of these from the current positions.
//
// Walk: one wave = one group of at most 64 targets packed from the tree
// (consecutive sibling subtrees inside one node).  The wave walks the
// preorder tree with a decision shared by the whole group: a node is
// accepted when the distance from its centre of mass to the group's bounding
// box exceeds bmax/theta (and, with the relative criterion, when its
// octupole-order term is small against the group's previous |a|).  Lanes
// walk disjoint ranges of the preorder array
// and hand work to idle lanes (k_phys_walk).  Accepted cells and bucket
// bodies are appended, relative to the group centre, to per-wave LDS lists;
// a full list is evaluated by all the group's lanes at once (entries read as
// LDS broadcasts), in launches of few groups by further waves of the group.
// Each flush's sum is formed in the evaluation precision and added to FP64
// totals.
//
// Bound in large launches by FP32 issue: 90 % of a walk's VALU instructions
// evaluate lists (33 per cell with v_rsq_f32, 14 per body), at 3.1 cycles per
// instruction and SIMD where independent ones take 2.3 to 2.7.
//
// Acceleration on a target at distance vector d = com - x from a cell:
//   a = m d / r^3 - Q d / r^5 + (5/2) (d^T Q d) d / r^7,  r^2 = |d|^2 + eps^2
// (the gradient of phi = -m/r - (1/2) x^T Q x / r^5 with x = -d).
#include "common.hpp"
#include "layout.hpp"
#include "phys_kernels.hpp"
#include "prims.hpp"

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstdint>

namespace nbx {
namespace {

struct PhysAux {
  double m, bmax;
  double q[6];          // xx yy zz xy xz yz
  double lo[3], hi[3];  // bounding box of the node's bodies
  double pad[2];
};
static_assert(sizeof(PhysAux) == kPhysAuxBytes, "PhysAux layout");

inline unsigned grid_of(int64_t n, int b) { return (unsigned)div_up(n, b); }

// A walk group of c bodies starts at sorted body f: marked in two zeroed
// per-body arrays, compacted in body (Morton) order afterwards.
__device__ __forceinline__ void mark_group(int32_t f, int32_t c, int32_t* gcnt, uint32_t* gmark) {
  gcnt[f] = c;
  gmark[f] = 1u;
}

// Node layout from the sorted keys, as k_emit does for the reference tree
// but writing walk records: for body i, the internal nodes that start at it
// (first body only; the skip pointer comes from k_phys_pair, the moments from
// k_phys_upward) and its leaf, complete.  A leaf is never accepted as a cell
// (rc2 = +inf), so its quadrupole slots carry its FP64 mass for the upward
// pass.  A leaf that is a system's root is that system's walk group.
__global__ __launch_bounds__(kBlock) void k_phys_emit(int64_t n, const int32_t* __restrict__ lcp,
                                                      const uint32_t* __restrict__ pre_off,
                                                      const uint32_t* __restrict__ part, StateArrays st,
                                                      const DevScalars* __restrict__ sc, PhysNode* __restrict__ pn,
                                                      int32_t* __restrict__ level_list,
                                                      uint32_t* __restrict__ end_list,
                                                      int32_t* __restrict__ gcnt, uint32_t* __restrict__ gmark,
                                                      uint32_t cap_nodes, uint32_t cap_int) {
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
  const int ns = li > lp ? li - lp : 0;
  for (int t = 0; t < ns; ++t) {
    const uint32_t p = pre + t;
    if (p >= cap_nodes) break;
    pn[p].first = (int32_t)i;
  }
  if (pre + ns < cap_nodes) {
    const uint32_t p = pre + ns;
    PhysNode nd;
    nd.cx = st.x[i]; nd.cy = st.y[i]; nd.cz = st.z[i];
    const double m = st.m[i];
    nd.m = (float)m;
    nd.rc2 = INFINITY;
    set_leaf_mass(nd, m);
    nd.qxy = nd.qxz = nd.qyz = 0.f;
    nd.skip = (int32_t)(p + 1);
    nd.first = (int32_t)i;
    nd.count = 1;
    pn[p] = nd;
  }
  if (li < 0 && lp < 0) mark_group((int32_t)i, 1, gcnt, gmark);
}

// Skip pointer of the k-th internal node of the per-depth list.
__global__ __launch_bounds__(kBlock) void k_phys_pair(int64_t m, const int32_t* __restrict__ level_list,
                                                      const uint32_t* __restrict__ end_list,
                                                      PhysNode* __restrict__ pn) {
  const int64_t k = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (k >= m) return;
  pn[level_list[k]].skip = (int32_t)end_list[k];
}

// The same with the count on the device (fixed grid striding over it).
__global__ __launch_bounds__(kBlock) void k_phys_pair_dev(const int32_t* __restrict__ level_list,
                                                          const uint32_t* __restrict__ end_list,
                                                          PhysNode* __restrict__ pn,
                                                          const DevScalars* __restrict__ sc) {
  if (sc->abort_flags) return;
  const int64_t m = (int64_t)sc->level_off[kMaxDepthSlots - 1] + sc->level_count[kMaxDepthSlots - 1];
  for (int64_t k = (int64_t)blockIdx.x * kBlock + threadIdx.x; k < m; k += (int64_t)gridDim.x * kBlock)
    pn[level_list[k]].skip = (int32_t)end_list[k];
}

// Eight lanes work on one node of the upward pass, a lane per child: a node's
// children (192 bytes each) come in at once and their terms are formed side
// by side; a sum runs over the children in order in one lane, the terms passed
// through LDS.  One thread per node waits for its children one after another
// and keeps 5 waves per SIMD at most: the pass's launches over all depths took
// 850 us at 4,194,304 bodies, 255 us at 2^20 and 317 us at 96 systems of
// 1.49 M bodies; now 593, 183 and 238 us.  (Units of bodies as in units.hpp,
// two launches in all: 154 us at 16,384 bodies against 95, 183 against 103 at
// 65,536, 244 at the 96 systems.)
constexpr int kNodeLanes = 8;
constexpr int kNodeTerms = 6;      // sums over the children exchanged at once
typedef double NodeXch[kNodeTerms * kNodeLanes];

__device__ __forceinline__ void wave_order() {   // LDS traffic of one wave keeps its order; so must the compiler
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Sum q over the node's children in order, in lane q < Q; v[q] is this lane's
// (this child's) term.
template <int Q>
__device__ __forceinline__ double sum_children(double* xch, int c, const double (&v)[Q]) {
  static_assert(Q <= kNodeTerms, "exchange buffer");
  wave_order();
#pragma unroll
  for (int q = 0; q < Q; ++q) xch[q * kNodeLanes + c] = v[q];
  wave_order();
  double s = 0.0;
  const double* row = xch + (c < Q ? c : 0) * kNodeLanes;
#pragma unroll
  for (int j = 0; j < kNodeLanes; ++j) s = s + row[j];
  return s;
}

// Internal nodes of one depth from their children (FP64), and the walk
// groups this node packs: a node of more than G bodies packs its children of
// at most G bodies into groups, consecutive siblings together while the sum
// stays within G; a system root of at most G bodies is a group of its own.
// Every body lands in exactly one group and a group's bodies lie inside one
// node, so groups are compact in space where runs of G consecutive Morton
// keys are not (such a run can straddle two distant cells).
//
// Called by the eight lanes of a node together; c: the lane's child.
__device__ __forceinline__ void phys_upward_node(double* xch, int32_t id, bool root_level, int c,
                                                 PhysNode* __restrict__ pn, PhysAux* __restrict__ aux,
                                                 double inv_theta, int G, int32_t* __restrict__ gcnt,
                                                 uint32_t* __restrict__ gmark) {
  const int32_t end = pn[id].skip;
  const int lead = lane_id() - c;
  const int32_t first = pn[id].first;
  int32_t ci = -1;                                           // this lane's child
  {
    int32_t p = id + 1;
#pragma unroll
    for (int j = 0; j < kNodeLanes; ++j) {
      if (p < end) {
        if (j == c) ci = p;
        p = pn[p].skip;
      }
    }
  }
  // a body (a point) or a cell with its moments and box
  int32_t cn = 0;
  double px = 0, py = 0, pz = 0, cm = 0, bc = 0;
  double cq[6] = {0, 0, 0, 0, 0, 0};
  double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
  if (ci >= 0) {
    const PhysNode& ch = pn[ci];
    cn = ch.count;
    px = ch.cx; py = ch.cy; pz = ch.cz;
    if (cn == 1) {
      cm = leaf_mass(ch);
      lo[0] = hi[0] = px; lo[1] = hi[1] = py; lo[2] = hi[2] = pz;
    } else {
      const PhysAux& a = aux[ci];
      cm = a.m;
      bc = a.bmax;
      for (int t = 0; t < 6; ++t) cq[t] = a.q[t];
      for (int k = 0; k < 3; ++k) { lo[k] = a.lo[k]; hi[k] = a.hi[k]; }
    }
  }
  const double sums = sum_children<4>(xch, c, {cm, px * cm, py * cm, pz * cm});
  const double M = __shfl(sums, lead, kWave);
  // lanes 1 to 3: x, y, z (of the first child where there is no mass)
  const double x0 = __shfl(px, lead, kWave), y0 = __shfl(py, lead, kWave), z0 = __shfl(pz, lead, kWave);
  const double com = M > 0 ? sums / M : c == 1 ? x0 : c == 2 ? y0 : z0;
  const double cx = __shfl(com, lead + 1, kWave), cy = __shfl(com, lead + 2, kWave), cz = __shfl(com, lead + 3, kWave);
  // (no child: 0, whose square times no mass is 0 at any distance of the centre)
  const double rx = ci >= 0 ? px - cx : 0.0, ry = ci >= 0 ? py - cy : 0.0, rz = ci >= 0 ? pz - cz : 0.0;
  const double r2 = rx * rx + ry * ry + rz * rz;
  double bsum = ci >= 0 ? sqrt(r2) + bc : 0.0;
  const double quad =
      sum_children<6>(xch, c, {cq[0] + cm * (3 * rx * rx - r2), cq[1] + cm * (3 * ry * ry - r2),
                               cq[2] + cm * (3 * rz * rz - r2), cq[3] + cm * 3 * rx * ry, cq[4] + cm * 3 * rx * rz,
                               cq[5] + cm * 3 * ry * rz});
  int32_t count = cn;
#pragma unroll
  for (int o = 1; o < kNodeLanes; o <<= 1) {
    count += __shfl_xor(count, o, kWave);
    bsum = fmax(bsum, __shfl_xor(bsum, o, kWave));
    for (int k = 0; k < 3; ++k) {
      lo[k] = fmin(lo[k], __shfl_xor(lo[k], o, kWave));
      hi[k] = fmax(hi[k], __shfl_xor(hi[k], o, kWave));
    }
  }
  // bmax: the farthest corner of the bodies' box from the centre of mass,
  // or the children's bound if that is smaller.
  const double ex = fmax(cx - lo[0], hi[0] - cx), ey = fmax(cy - lo[1], hi[1] - cy), ez = fmax(cz - lo[2], hi[2] - cz);
  double bmax = sqrt(ex * ex + ey * ey + ez * ez);
  if (bsum < bmax) bmax = bsum;
  // Cells of very few bodies cost more as a multipole than as bodies.
  const double rc = bmax * inv_theta;
  const float rc2 = count < 4 ? INFINITY : (float)(rc * rc * (1.0 + 1e-6));
  // The record in one store and the moments in two, 8 bytes a lane.
  static_assert(offsetof(PhysNode, cx) == 0 && offsetof(PhysNode, m) == 24 && offsetof(PhysNode, rc2) == 28 &&
                    offsetof(PhysNode, qxx) == 32 && offsetof(PhysNode, qxy) == 40 && offsetof(PhysNode, qyz) == 48 &&
                    offsetof(PhysNode, skip) == 52 && offsetof(PhysNode, first) == 56 && offsetof(PhysAux, q) == 16 &&
                    offsetof(PhysAux, lo) == 64,
                "stored by lane");
  const float qf = (float)quad;
  const float qxx = __shfl(qf, lead, kWave), qyy = __shfl(qf, lead + 1, kWave), qxy = __shfl(qf, lead + 3, kWave),
              qxz = __shfl(qf, lead + 4, kWave), qyz = __shfl(qf, lead + 5, kWave);
  const uint32_t wlo = c == 0   ? __float_as_uint((float)M)
                       : c == 4 ? __float_as_uint(qxx)
                       : c == 5 ? __float_as_uint(qxy)
                       : c == 6 ? __float_as_uint(qyz)
                                : (uint32_t)first;
  const uint32_t whi = c == 0   ? __float_as_uint(rc2)
                       : c == 4 ? __float_as_uint(qyy)
                       : c == 5 ? __float_as_uint(qxz)
                       : c == 6 ? (uint32_t)end
                                : (uint32_t)count;
  const double word = __longlong_as_double((long long)((uint64_t)wlo | ((uint64_t)whi << 32)));
  const bool is_com = c >= 1 && c <= 3;
  reinterpret_cast<double*>(pn + id)[is_com ? c - 1 : c == 0 ? 3 : c] = is_com ? com : word;
  double* const ax = reinterpret_cast<double*>(aux + id);
  ax[c < 6 ? 2 + c : c - 6] = c < 6 ? quad : c == 6 ? M : bmax;
  if (c < 6) ax[8 + c] = c == 0 ? lo[0] : c == 1 ? lo[1] : c == 2 ? lo[2] : c == 3 ? hi[0] : c == 4 ? hi[1] : hi[2];
  // walk groups
  if (count > G) {
    int32_t run_first = 0, run = 0, f = first;
#pragma unroll
    for (int j = 0; j < kNodeLanes; ++j) {
      const int32_t cc = __shfl(cn, lead + j, kWave);
      const int32_t cf = f;                                  // children's bodies follow one another
      f += cc;
      if (c != 0 || cc == 0) continue;
      if (cc > G) {                                          // packs its own children
        if (run > 0) mark_group(run_first, run, gcnt, gmark);
        run = 0;
        continue;
      }
      if (run > 0 && run + cc > G) { mark_group(run_first, run, gcnt, gmark); run = 0; }
      if (run == 0) run_first = cf;
      run += cc;
    }
    if (run > 0) mark_group(run_first, run, gcnt, gmark);
  } else if (root_level && c == 0) {
    mark_group(first, count, gcnt, gmark);
  }
}

__global__ __launch_bounds__(kBlock)
void k_phys_upward(const int32_t* __restrict__ level_list, int64_t beg, int64_t cnt, bool root_level,
                   PhysNode* __restrict__ pn, PhysAux* __restrict__ aux, double inv_theta, int G,
                   int32_t* __restrict__ gcnt, uint32_t* __restrict__ gmark) {
  __shared__ NodeXch xch[kBlock / kNodeLanes];
  const int64_t k = ((int64_t)blockIdx.x * kBlock + threadIdx.x) / kNodeLanes;
  if (k >= cnt) return;
  phys_upward_node(xch[threadIdx.x / kNodeLanes], level_list[beg + k], root_level, threadIdx.x % kNodeLanes, pn, aux,
                   inv_theta, G, gcnt, gmark);
}

// Depths d_lo .. 41 of a build whose counts stay on the device in one
// workgroup, deepest first, a barrier between depths (see k_upward_tail).
__global__ __launch_bounds__(kBlock)
void k_phys_upward_tail(int d_lo, const int32_t* __restrict__ level_list, PhysNode* __restrict__ pn,
                        PhysAux* __restrict__ aux, double inv_theta, int G, int32_t* __restrict__ gcnt,
                        uint32_t* __restrict__ gmark, const DevScalars* __restrict__ sc) {
  __shared__ NodeXch xch[kBlock / kNodeLanes];
  if (sc->abort_flags) return;
  for (int d = kMaxLevels - 1; d >= d_lo; --d) {
    const int64_t beg = sc->level_off[d], cnt = sc->level_count[d];
    if (cnt == 0) continue;
    for (int64_t k = threadIdx.x / kNodeLanes; k < cnt; k += kBlock / kNodeLanes)
      phys_upward_node(xch[threadIdx.x / kNodeLanes], level_list[beg + k], d == 0, threadIdx.x % kNodeLanes, pn, aux,
                       inv_theta, G, gcnt, gmark);
    __syncthreads();
  }
}

// Depth d of a build whose counts stay on the device (k_check): fixed grid
// striding over the depth's extent in the node list.
__global__ __launch_bounds__(kBlock)
void k_phys_upward_level(int d, const int32_t* __restrict__ level_list, PhysNode* __restrict__ pn,
                         PhysAux* __restrict__ aux, double inv_theta, int G, int32_t* __restrict__ gcnt,
                         uint32_t* __restrict__ gmark, const DevScalars* __restrict__ sc) {
  __shared__ NodeXch xch[kBlock / kNodeLanes];
  if (sc->abort_flags) return;
  const int64_t beg = sc->level_off[d], cnt = sc->level_count[d];
  for (int64_t k = ((int64_t)blockIdx.x * kBlock + threadIdx.x) / kNodeLanes; k < cnt;
       k += (int64_t)gridDim.x * (kBlock / kNodeLanes))
    phys_upward_node(xch[threadIdx.x / kNodeLanes], level_list[beg + k], d == 0, threadIdx.x % kNodeLanes, pn, aux,
                     inv_theta, G, gcnt, gmark);
}

template <typename T>
struct alignas(4 * sizeof(T)) V4 {
  T x, y, z, w;
};
template <typename T>
struct alignas(2 * sizeof(T)) V2 {
  T x, y;
};

// Sum over the lanes that share a target slot (lanes slot + p * width).
template <typename T>
__device__ __forceinline__ void combine_parts(T& fx, T& fy, T& fz, T& fp, int width) {
  for (int off = width; off < kWave; off <<= 1) {
    fx += __shfl_xor(fx, off, kWave);
    fy += __shfl_xor(fy, off, kWave);
    fz += __shfl_xor(fz, off, kWave);
    fp += __shfl_xor(fp, off, kWave);
  }
}

template <typename T>
__device__ __forceinline__ T rsq(T x);
template <>
__device__ __forceinline__ float rsq<float>(float x) { return __frsqrt_rn(x); }
template <>
__device__ __forceinline__ double rsq<double>(double x) { return rsqrt(x); }

// Group walk with work donation.  Every lane walks a contiguous range of
// the preorder node array with skip pointers (accept or bucket: jump past the
// subtree; open: step to the first child).  Lane 0 starts with the whole
// tree; when a lane opens a node, it hands the rest of its range after that
// node's subtree, [skip, end), to a per-wave LDS stack from which idle lanes
// take work (last in, first out).  Handing work over is optional, so a full
// stack only means a lane keeps walking its range itself: the stack cannot
// overflow.  All decisions are made in lockstep by one wave and compacted in
// lane order, so the lists, and every sum, come out in the same order on
// every run.
template <typename T, int LIST>
struct CellList {
  V4<T> a[LIST];   // relative centre of mass, mass
  V4<T> b[LIST];   // qxx qyy qxy qxz
  V2<T> q[LIST];   // qyz qzz
};
template <typename T, int LIST>
struct BodyList {
  V4<T> p[LIST];   // relative position, mass
};

// What a lane needs of its target to evaluate list entries.
template <typename T>
struct WalkTarget {
  T x, y, z, e2;   // relative to the group's centre; softening squared
  int width, parts, part;
};

// The sum over the n entries of a list for the wave's targets, every product
// fused into the sum it feeds: a = m d / r^3 + 2.5 (d.Q.d) d / r^7 - Q d / r^5
// and phi = -m / r - 0.5 (d.Q.d) / r^5, d from the target to the cell.
template <bool POT, typename T, int LIST>
__device__ __forceinline__ void sum_cells(const CellList<T, LIST>& L, int n, const WalkTarget<T>& t, T& fx, T& fy,
                                          T& fz, T& fp) {
  auto term = [&](int k) {
    const V4<T> a = L.a[k];
    const V4<T> b = L.b[k];
    const V2<T> q = L.q[k];
    const T dx = a.x - t.x, dy = a.y - t.y, dz = a.z - t.z;
    const T r2 = fma(dz, dz, fma(dy, dy, fma(dx, dx, t.e2)));
    const T ri = rsq<T>(r2);
    const T ri2 = ri * ri;
    const T ri3 = ri2 * ri;
    const T ri5 = ri3 * ri2;
    const T qdx = fma(b.w, dz, fma(b.z, dy, b.x * dx));
    const T qdy = fma(q.x, dz, fma(b.y, dy, b.z * dx));
    const T qdz = fma(q.y, dz, fma(q.x, dy, b.w * dx));
    const T dqd = fma(dz, qdz, fma(dy, qdy, dx * qdx));
    const T u = dqd * ri5;
    const T s = fma((T)2.5 * ri2, u, a.w * ri3);
    fx = fma(-ri5, qdx, fma(s, dx, fx));
    fy = fma(-ri5, qdy, fma(s, dy, fy));
    fz = fma(-ri5, qdz, fma(s, dz, fz));
    if (POT) fp = fma((T)-0.5, u, fma(-a.w, ri, fp));
  };
  // A group of more than 32 targets has one lane per target, and every lane
  // takes every entry: the loop is wave-uniform (scalar control, one LDS
  // address for all lanes).
  if (t.parts == 1) {
#pragma unroll 2
    for (int k = 0; k < n; ++k) term(k);
  } else {
    for (int k = t.part; k < n; k += t.parts) term(k);
    combine_parts(fx, fy, fz, fp, t.width);
  }
}

template <bool POT, typename T, int LIST>
__device__ __forceinline__ void sum_bodies(const BodyList<T, LIST>& L, int n, const WalkTarget<T>& t, T& fx, T& fy,
                                           T& fz, T& fp) {
  auto term = [&](int k) {
    const V4<T> b = L.p[k];
    const T dx = b.x - t.x, dy = b.y - t.y, dz = b.z - t.z;
    const T r2 = fma(dz, dz, fma(dy, dy, fma(dx, dx, t.e2)));
    const T ri = rsq<T>(r2);
    const T mri = b.w * ri;
    const T mr3 = mri * (ri * ri);
    fx = fma(mr3, dx, fx);
    fy = fma(mr3, dy, fy);
    fz = fma(mr3, dz, fz);
    if (POT) fp -= mri;
  };
  if (t.parts == 1) {
#pragma unroll 2
    for (int k = 0; k < n; ++k) term(k);
  } else {
    for (int k = t.part; k < n; k += t.parts) term(k);
    combine_parts(fx, fy, fz, fp, t.width);
  }
}

// Counters in LDS that waves of a workgroup wait on.
__device__ __forceinline__ int lds_get(const int* p) {
  return __builtin_amdgcn_readfirstlane(__hip_atomic_load(p, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP));
}
__device__ __forceinline__ void lds_put(int* p, int v) {   // after all the wave's LDS accesses before it
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  if (lane_id() == 0) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// EVAL > 0: the workgroup has EVAL more waves.  The first wave walks and hands
// every full list over as a job; job j is summed by wave 1 + j % EVAL, and the
// sums are added to the totals (LDS) in the order of the jobs, so the result is
// that of one wave, bit for bit.  A buffer is filled again when the job that
// held it has been added.  Every wait ends: the walk waits for jobs handed over
// before, a job only for the ones before it, and the waves beyond the last job
// for the walk's end.
template <typename T, int LIST, bool KICK, bool POT, bool COUNT, int EVAL>
__global__ __launch_bounds__(kPhysBlock * (1 + EVAL)) void k_phys_walk(const Group* __restrict__ groups,
                                                          const PhysNode* __restrict__ pn, StateArrays st,
                                                          SysArrays sy, double eps, int nleaf,
                                                          double* __restrict__ ax, double* __restrict__ ay,
                                                          double* __restrict__ az, double* __restrict__ pot,
                                                          DevScalars* sc, const float* __restrict__ amag,
                                                          float rel2, float th2) {
  __shared__ int32_t stk_b[kPhysStack];  // donated ranges [stk_b, stk_e)
  __shared__ int32_t stk_e[kPhysStack];
  __shared__ int32_t bfirst[kWave];      // buckets of the current step: first body,
  __shared__ int32_t bstart[kWave];      //   offset in the step's flattened body list
  // (Four buffers of 5 + 2 KB leave a CU 5 workgroups, as their registers do;
  // FP64's three of 10 + 4 KB, 3.)
  constexpr int kBufs = !EVAL ? 1 : sizeof(T) == 4 ? 4 : 3, kSums = POT ? 4 : 3;
  constexpr int kJobs = 8;                            // at most 2 kBufs jobs are out
  static_assert(2 * kBufs <= kJobs && kBufs <= 8, "job ring");
  __shared__ CellList<T, LIST> cells[kBufs];
  __shared__ BodyList<T, LIST> bodies[kBufs];
  __shared__ int job_at[EVAL ? kJobs : 1];            // job j: entries, buffer, kind at j % kJobs
  __shared__ int buf_job[EVAL ? 2 * kBufs : 1];       // last job that held a buffer (cells, bodies)
  __shared__ int handed, added, last;                 // jobs handed over, added; how many there are in the end
  __shared__ double total[EVAL ? kSums : 1][kWave];

  const int lane = lane_id(), wave = EVAL ? __builtin_amdgcn_readfirstlane(threadIdx.x / kWave) : 0;
  // The group count comes from the device (the compaction that wrote it ran
  // earlier on this stream), so the host need not read it back first; the
  // grid (a multiple of 8) is sized from a bound.  Blocks are dealt to the 8
  // XCDs round-robin: XCD x walks the contiguous (spatially coherent) range
  // [x per, (x + 1) per) of the groups with its gridDim / 8 blocks, so its L2
  // holds the part of the tree those groups touch, whatever the grid size.
  const int64_t ngroups = sc->abort_flags ? 0 : (int64_t)sc->tree_groups;   // nothing after an aborted build
  const int64_t per = (ngroups + 7) / 8;
  const int64_t xbase = (int64_t)(blockIdx.x % 8) * per;
  for (int64_t j = blockIdx.x / 8; j < per; j += gridDim.x / 8) {
    const int64_t gi = xbase + j;
    if (gi >= ngroups) break;                              // the last range is short
    const Group g = groups[gi];
    // A group of at most 32 (16, ...) targets puts 2 (4, ...) lanes on each
    // target: lane = slot + part * width, and the parts evaluate interleaved
    // entries of every list, their sums combined after each flush.
    int width = kWave;
    while (width > 1 && (width >> 1) >= g.count) width >>= 1;
    const int parts = kWave / width;
    const int slot = lane & (width - 1), part = lane / width;
    const int64_t i = g.first + slot;
    const bool valid = slot < g.count && part == 0;        // the lane that owns the result
    const int64_t ii = slot < g.count ? i : g.first;
    const double px = st.x[ii], py = st.y[ii], pz = st.z[ii];
    const uint64_t ltmask = lanemask_lt();
    const int32_t root = sy.sroot[g.sys], tree_end = sy.send[g.sys];   // this system's tree

    // group bounding box
    double lo[3] = {px, py, pz}, hi[3] = {px, py, pz};
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const double a = __shfl_xor(lo[k], off, kWave), b = __shfl_xor(hi[k], off, kWave);
        lo[k] = a < lo[k] ? a : lo[k];
        hi[k] = b > hi[k] ? b : hi[k];
      }
    }
    const double gcx = 0.5 * (lo[0] + hi[0]), gcy = 0.5 * (lo[1] + hi[1]), gcz = 0.5 * (lo[2] + hi[2]);
    const float hx = (float)(0.5 * (hi[0] - lo[0])) * (1.0f + 1e-6f);
    const float hy = (float)(0.5 * (hi[1] - lo[1])) * (1.0f + 1e-6f);
    const float hz = (float)(0.5 * (hi[2] - lo[2])) * (1.0f + 1e-6f);
    const WalkTarget<T> tg{(T)(px - gcx), (T)(py - gcy), (T)(pz - gcz), (T)(eps * eps), width, parts, part};
    // Relative criterion (amag != null): a cell that passes the geometric test
    // is accepted only if its first neglected (octupole) term, ~ m bmax^3 / d^5,
    // is at most alpha times the smallest previous |a| of the group:
    // m^2 bmax^6 <= alpha^2 amin^2 d^10, with bmax^2 = rc2 * theta^2.
    float arel = 0.f;
    if (amag) {
      float am = amag[ii];
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) am = fminf(am, __shfl_xor(am, off, kWave));
      arel = rel2 * am * am;
    }

    if (EVAL) {
      if (wave == 0) {
        if (lane < 2 * kBufs) buf_job[lane] = -1;
        if (lane == 0) { handed = 0; added = 0; last = INT32_MAX; }
        for (int k = 0; k < kSums; ++k) total[k][lane] = 0.0;
      }
      __syncthreads();
      if (wave > 0) {
        for (int j = wave - 1;; j += EVAL) {
          bool none = false;
          while (lds_get(&handed) <= j) {
            none = lds_get(&last) <= j;
            if (none) break;
            __builtin_amdgcn_s_sleep(1);
          }
          if (none) break;
          const int job = __builtin_amdgcn_readfirstlane(job_at[j % kJobs]);
          const int buf = job >> 1 & 7, cnt = job >> 4;
          T fx = 0, fy = 0, fz = 0, fp = 0;
          if (job & 1) sum_bodies<POT>(bodies[buf], cnt, tg, fx, fy, fz, fp);
          else sum_cells<POT>(cells[buf], cnt, tg, fx, fy, fz, fp);
          while (lds_get(&added) != j) __builtin_amdgcn_s_sleep(1);
          total[0][lane] += (double)fx; total[1][lane] += (double)fy; total[2][lane] += (double)fz;
          if (POT) total[kSums - 1][lane] += (double)fp;
          lds_put(&added, j + 1);
        }
        __syncthreads();                                   // the group's end
        continue;
      }
    }

    double Ax = 0, Ay = 0, Az = 0, P = 0;
    uint32_t ncell_tot = 0, npart_tot = 0, niter = 0, nopen = 0;
    int nc = 0, np = 0, cbuf = 0, bbuf = 0, jobs = 0;

    auto hand_over = [&](int kind, int& buf, int cnt) {
      if (lane == 0) {
        job_at[jobs % kJobs] = kind | buf << 1 | cnt << 4;
        buf_job[kind * kBufs + buf] = jobs;
      }
      lds_put(&handed, ++jobs);
      buf = buf + 1 < kBufs ? buf + 1 : 0;
      wave_order();
      const int before = __builtin_amdgcn_readfirstlane(buf_job[kind * kBufs + buf]);
      while (lds_get(&added) <= before) __builtin_amdgcn_s_sleep(1);
    };
    auto flush_cells = [&]() {
      wave_order();
      if (EVAL) {
        hand_over(0, cbuf, nc);
      } else {
        T fx = 0, fy = 0, fz = 0, fp = 0;
        sum_cells<POT>(cells[0], nc, tg, fx, fy, fz, fp);
        Ax += (double)fx; Ay += (double)fy; Az += (double)fz;
        if (POT) P += (double)fp;
      }
      if (COUNT) ncell_tot += nc;
      wave_order();
      nc = 0;
    };
    auto flush_parts = [&]() {
      wave_order();
      if (EVAL) {
        hand_over(1, bbuf, np);
      } else {
        T fx = 0, fy = 0, fz = 0, fp = 0;
        sum_bodies<POT>(bodies[0], np, tg, fx, fy, fz, fp);
        Ax += (double)fx; Ay += (double)fy; Az += (double)fz;
        if (POT) P += (double)fp;
      }
      if (COUNT) npart_tot += np;
      wave_order();
      np = 0;
    };

    int32_t cur = lane == 0 ? root : tree_end;                  // this lane's range [cur, end)
    int32_t end = tree_end;
    int sp = 0;                                              // donated ranges on the stack
    for (;;) {
      // idle lanes take ranges from the top of the stack
      const bool idle = cur >= end;
      const uint64_t im = __ballot(idle);
      const int take = __popcll(im) < sp ? (int)__popcll(im) : sp;
      if (idle) {
        const int r = (int)__popcll(im & ltmask);
        if (r < take) { cur = stk_b[sp - 1 - r]; end = stk_e[sp - 1 - r]; }
      }
      sp -= take;
      const bool busy = cur < end;
      if (!__ballot(busy)) break;
      if (COUNT) ++niter;
      if (nc > LIST - kWave) flush_cells();

      bool acc = false, bucket = false, donate = false;
      int32_t cnt = 0, first = 0, nskip = 0;
      double ncx = 0, ncy = 0, ncz = 0;
      if (busy) {
        const PhysNode nd = pn[cur];
        ncx = nd.cx; ncy = nd.cy; ncz = nd.cz;
        const float rx = (float)(ncx - gcx), ry = (float)(ncy - gcy), rz = (float)(ncz - gcz);
        const float dx = fmaxf(fabsf(rx) - hx, 0.f), dy = fmaxf(fabsf(ry) - hy, 0.f), dz = fmaxf(fabsf(rz) - hz, 0.f);
        const float d2 = fmaf(dz, dz, fmaf(dx, dx, dy * dy));
        cnt = nd.count;
        first = nd.first;
        nskip = nd.skip > cur ? nd.skip : cur + 1;           // skip > cur by construction
        if (d2 > nd.rc2) {
          acc = true;
          if (amag) {
            const float b2 = nd.rc2 * th2;
            const float d4 = d2 * d2;
            acc = nd.m * nd.m * (b2 * b2 * b2) <= arel * (d4 * d4 * d2);
          }
        }
        if (!acc) {
          if (cnt <= nleaf) bucket = true;
          else donate = nskip < end;                         // open; the rest of the range can go
        }
      }
      // accepted cells -> cell list
      const uint64_t am = __ballot(acc);
      if (acc) {
        const int pos = nc + (int)__popcll(am & ltmask);
        const PhysNode& nd = pn[cur];
        CellList<T, LIST>& L = cells[EVAL ? cbuf : 0];
        L.a[pos] = V4<T>{(T)(ncx - gcx), (T)(ncy - gcy), (T)(ncz - gcz), (T)nd.m};
        L.b[pos] = V4<T>{(T)nd.qxx, (T)nd.qyy, (T)nd.qxy, (T)nd.qxz};
        L.q[pos] = V2<T>{(T)nd.qyz, (T)(-((double)nd.qxx + (double)nd.qyy))};
      }
      nc += (int)__popcll(am);
      // opened nodes hand [skip, end) to the stack while it has room
      const uint64_t dm = __ballot(donate);
      const int room = kPhysStack - sp;
      if (donate) {
        const int r = (int)__popcll(dm & ltmask);
        if (r < room) { stk_b[sp + r] = nskip; stk_e[sp + r] = end; end = nskip; }
      }
      sp += (int)__popcll(dm) < room ? (int)__popcll(dm) : room;
      if (busy) cur = (acc || bucket) ? nskip : cur + 1;
      if (COUNT) nopen += (uint32_t)__popcll(__ballot(busy && !acc && !bucket));

      // buckets -> body list, all lanes loading bodies in parallel
      const uint32_t cb_n = bucket ? (uint32_t)cnt : 0u;
      const uint32_t bincl = wave_incl_scan_u32(cb_n);
      const int nbody = __builtin_amdgcn_readlane((int)bincl, kWave - 1);   // wave-uniform
      const uint64_t bm = __ballot(bucket);
      const int nb = (int)__popcll(bm);
      if (bucket) {
        const int j = (int)__popcll(bm & ltmask);
        bfirst[j] = first;
        bstart[j] = (int)(bincl - cb_n);
      }
      wave_order();
      for (int base = 0; base < nbody; base += kWave) {
        if (np > LIST - kWave) flush_parts();
        const int t = base + lane;
        if (t < nbody) {
          int lo_j = 0, hi_j = nb - 1;                       // last bucket with bstart <= t
          while (lo_j < hi_j) {
            const int mid = (lo_j + hi_j + 1) >> 1;
            if (bstart[mid] <= t) lo_j = mid; else hi_j = mid - 1;
          }
          const int32_t b = bfirst[lo_j] + (t - bstart[lo_j]);
          bodies[EVAL ? bbuf : 0].p[np + lane] = V4<T>{(T)(st.x[b] - gcx), (T)(st.y[b] - gcy), (T)(st.z[b] - gcz), (T)st.m[b]};
        }
        np += nbody - base < kWave ? nbody - base : kWave;
      }
      wave_order();
    }
    if (nc) flush_cells();
    if (np) flush_parts();
    if (EVAL) {
      lds_put(&last, jobs);
      while (lds_get(&added) < jobs) __builtin_amdgcn_s_sleep(1);
      Ax = total[0][lane]; Ay = total[1][lane]; Az = total[2][lane];
      if (POT) P = total[kSums - 1][lane];
      __syncthreads();                                     // the group's end
    }

    double v2 = 0.0;
    if (valid) {
      ax[i] = Ax; ay[i] = Ay; az[i] = Az;
      if (POT) pot[i] = P + st.m[i] / eps;                   // drop the self pair, -m_i/eps
      if (KICK) {
        const double half = sy.dt[g.sys] * 0.5;
        const double vx = st.vx[i] + Ax * half;
        const double vy = st.vy[i] + Ay * half;
        const double vz = st.vz[i] + Az * half;
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
    if (COUNT && lane == 0) {
      const uint32_t nv = (uint32_t)g.count;
      atomicAdd(&sc->n_pc, (unsigned long long)ncell_tot * nv);
      atomicAdd(&sc->n_pp, (unsigned long long)npart_tot * nv);
      atomicAdd(&sc->n_open, (unsigned long long)nopen);
      atomicAdd(&sc->n_iter, (unsigned long long)niter);
    }
    wave_order();                                          // the next group reuses the LDS lists
  }
}

// FP64 direct sum.  One target per lane, 64 consecutive bodies per wave; the
// sources are wave-uniform, so they come in by scalar loads and cost no LDS,
// no barrier and no vector load.  Every system's sources are split over the
// waves of a workgroup, whose sums meet in LDS, and over blockIdx.y
// (k_direct_sum), so that a small system fills the chip too.  A pair issues 19
// FP64 instructions and v_rsq_f64, so the sum is bound by FP64 issue: two sums
// over 65,537 bodies (forces, then energies) with the download 6.8 ms, against
// 36.1 of one target per thread with sources staged in LDS, a correctly rounded
// square root and divide per pair and 257 workgroups.  v_rsq_f64 (5.2e-8 at
// most) is refined by one step of third order, y (1 + h/2 + 3/8 h^2) with
// h = 1 - r^2 y^2: 1.38e-16 at most, where the square root and divide give
// 1.66e-16 and a Newton step, one instruction less and 6.40 ms, 4.1e-15.
//
// Only bodies of the target's own system act on it: a wave whose targets lie
// in several systems takes them one after another.  The lanes' own bodies are
// among 64 sources only; the rest of the loop does not test for the self pair.
//
// A system's sources are cut into kDirectChunks parts by the system's size
// alone, each part is summed from zero, and the parts are added in a balanced
// tree: a wave its consecutive parts, a workgroup its waves, k_direct_sum the
// halves.  How many parts a wave takes follows from the size of the launch and
// changes no bit, so a system's sums are the same alone and in a batch.
constexpr int kDirectChunks = 32;
struct DirectSum { double x, y, z, p; };

// Sources [j, end).  SELF: some of them are targets of the wave (body i of
// this lane).  ZERO: eps is 0, so a pair at distance 0 has an infinite 1 / r.
template <bool SELF, bool ZERO>
__device__ __forceinline__ void direct_range(const StateArrays& st, int64_t j, int64_t end, int64_t i, double px,
                                             double py, double pz, double e2, DirectSum& a) {
#pragma clang fp contract(off)   // the same roundings with and without SELF (a wave's neighbours decide which)
  typedef const __attribute__((address_space(4))) double* cptr;   // scalar loads
  const cptr X = (cptr)st.x, Y = (cptr)st.y, Z = (cptr)st.z, M = (cptr)st.m;
#pragma unroll 4
  for (; j < end; ++j) {
    const double dx = X[j] - px, dy = Y[j] - py, dz = Z[j] - pz;
    const double m = M[j];
    const double r2 = fma(dz, dz, fma(dy, dy, fma(dx, dx, e2)));
    const double y = __builtin_amdgcn_rsq(r2);
    // (the minimum keeps inf * 0 out: an overflowing distance contributes 0)
    const double h = fma(-(fmin(r2, 1.7976931348623157e308) * y), y, 1.0);
    double ri = fma(y, h * fma(0.375, h, 0.5), y);
    if (ZERO && r2 == 0.0) ri = INFINITY;
    double mr = m * ri;
    double mr3 = mr * (ri * ri);
    if (SELF && j == i) { mr = 0.0; mr3 = 0.0; }
    a.x = fma(dx, mr3, a.x);
    a.y = fma(dy, mr3, a.y);
    a.z = fma(dz, mr3, a.z);
    a.p -= mr;
  }
}

__device__ __forceinline__ DirectSum operator+(const DirectSum& a, const DirectSum& b) {
  return DirectSum{a.x + b.x, a.y + b.y, a.z + b.z, a.p + b.p};
}

// Component q of waves [w, w + N) of a workgroup, added in a balanced tree.
template <int N>
__device__ __forceinline__ double sum_waves(const double (*part)[4][kWave], int w, int q) {
  if constexpr (N == 1) return part[w][q][lane_id()];
  else return sum_waves<N / 2>(part, w, q) + sum_waves<N / 2>(part, w + N / 2, q);
}

// The W waves of a workgroup have the same 64 targets and PER consecutive
// parts of the sources each; blockIdx.y: which of the W PER parts.
template <bool ZERO, int W, int PER>
__global__ __launch_bounds__(W* kWave) __attribute__((amdgpu_waves_per_eu(PER < 8 ? 8 : 7)))
void k_direct64(int64_t n, StateArrays st, SysArrays sy, double e2, double* __restrict__ ax, double* __restrict__ ay,
                double* __restrict__ az, double* __restrict__ pot) {
  static_assert(W >= 4 && (PER == 1 || PER == 2 || PER == 4 || PER == 8), "waves of the last sum, levels of the tree");
  __shared__ double part[W][4][kWave];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int64_t i0 = (int64_t)blockIdx.x * kWave;
  const int64_t i1 = i0 + kWave < n ? i0 + kWave : n;        // targets [i0, i1)
  const int64_t i = i0 + lane_id();
  const bool valid = i < n;
  const int64_t ii = valid ? i : n - 1;
  const double px = st.x[ii], py = st.y[ii], pz = st.z[ii];
  const int32_t me = st.sys[ii];
  const int32_t s0 = __builtin_amdgcn_readfirstlane(st.sys[i0]), s1 = __builtin_amdgcn_readfirstlane(st.sys[i1 - 1]);
  const int c0 = ((int)blockIdx.y * W + wave) * PER;         // parts [c0, c0 + PER)
  DirectSum total{0.0, 0.0, 0.0, 0.0};
  for (int32_t s = s0; s <= s1; ++s) {
    const int32_t lo = sy.soff[s], cnt = sy.soff[s + 1] - lo;   // (a context holds at most 2^25 bodies: cnt * 32 fits)
    if (me == s) {
      DirectSum l1{}, l2{}, l4{};                            // sums of 1, 2 and 4 parts that wait for their neighbours
#pragma unroll 1
      for (int k = 0; k < PER; ++k) {
        // (wave-uniform, and told so: with one part the compiler lost track and loaded the sources by lane)
        const int64_t b = __builtin_amdgcn_readfirstlane(lo + cnt * (c0 + k) / kDirectChunks),
                      e = __builtin_amdgcn_readfirstlane(lo + cnt * (c0 + k + 1) / kDirectChunks);
        const int64_t o0 = i0 < b ? b : i0 < e ? i0 : e, o1 = i1 < b ? b : i1 < e ? i1 : e;   // own targets in [b, e)
        DirectSum a{0.0, 0.0, 0.0, 0.0};
        direct_range<false, ZERO>(st, b, o0, i, px, py, pz, e2, a);
        direct_range<true, ZERO>(st, o0, o1, i, px, py, pz, e2, a);
        direct_range<false, ZERO>(st, o1, e, i, px, py, pz, e2, a);
        if (PER > 1 && !(k & 1)) { l1 = a; continue; }
        if (PER > 1) a = l1 + a;
        if (PER > 2 && !(k & 2)) { l2 = a; continue; }
        if (PER > 2) a = l2 + a;
        if (PER > 4 && !(k & 4)) { l4 = a; continue; }
        if (PER > 4) a = l4 + a;
        total = a;
      }
    }
  }
  part[wave][0][lane_id()] = total.x; part[wave][1][lane_id()] = total.y;
  part[wave][2][lane_id()] = total.z; part[wave][3][lane_id()] = total.p;
  __syncthreads();
  if (wave >= 4 || !valid) return;                           // a wave per component
  const double v = sum_waves<W>(part, 0, wave);
  if (gridDim.y > 1) {                                       // halves: x y z p, n each
    ax[((int64_t)blockIdx.y * 4 + wave) * n + i] = v;
  } else {
    double* const out = wave == 0 ? ax : wave == 1 ? ay : wave == 2 ? az : pot;
    if (out) out[i] = v;
  }
}

// The two halves' sums.
__global__ __launch_bounds__(kBlock) void k_direct_sum(int64_t n, const double* __restrict__ part,
                                                       double* __restrict__ ax, double* __restrict__ ay,
                                                       double* __restrict__ az, double* __restrict__ pot) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  double v[4];
  for (int k = 0; k < 4; ++k) v[k] = part[k * n + i] + part[(4 + k) * n + i];
  ax[i] = v[0]; ay[i] = v[1]; az[i] = v[2];
  if (pot) pot[i] = v[3];
}

// Energy and momentum per system, over the segmented blocks of the
// bounding-box reduction; each system's blocks are summed in block order.
__global__ __launch_bounds__(kBlock) void k_energy_partial(StateArrays st, const double* __restrict__ pot,
                                                           const BoxBlock* __restrict__ blocks,
                                                           double* __restrict__ part) {
  __shared__ double red[kBlock / kWave][5];
  const BoxBlock b = blocks[blockIdx.x];
  double v[5] = {0, 0, 0, 0, 0};
  for (int64_t i = b.begin + threadIdx.x; i < b.end; i += kBlock) {
    const double m = st.m[i], vx = st.vx[i], vy = st.vy[i], vz = st.vz[i];
    v[0] += 0.5 * m * (vx * vx + vy * vy + vz * vz);
    if (pot) v[1] += 0.5 * m * pot[i];
    v[2] += m * vx; v[3] += m * vy; v[4] += m * vz;
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1)
    for (int k = 0; k < 5; ++k) v[k] += __shfl_xor(v[k], off, kWave);
  if (lane_id() == 0)
    for (int k = 0; k < 5; ++k) red[threadIdx.x / kWave][k] = v[k];
  __syncthreads();
  if (threadIdx.x < 5) {
    double t = 0;
    for (int w = 0; w < kBlock / kWave; ++w) t += red[w][threadIdx.x];
    part[5 * blockIdx.x + threadIdx.x] = t;
  }
}

__global__ __launch_bounds__(kBlock) void k_energy_final(const double* __restrict__ part,
                                                         const int32_t* __restrict__ block_off, int nsys,
                                                         double* out) {
  const int s = blockIdx.x * kBlock + threadIdx.x;
  if (s >= nsys) return;
  double t[5] = {0, 0, 0, 0, 0};
  for (int b = block_off[s]; b < block_off[s + 1]; ++b)
    for (int k = 0; k < 5; ++k) t[k] += part[5 * b + k];
  for (int k = 0; k < 5; ++k) out[5 * s + k] = t[k];
}

// Evaluating waves of a split launch (phys_walk_split).  Two: 275 us (FP32,
// 16,384 bodies) where three take 205; five or seven: 208.
constexpr int kWalkEval = 3;

template <typename T, int LIST>
void walk_dispatch(unsigned nb, const Group* groups, const PhysNode* pn, const StateArrays& st, const SysArrays& sy,
                   double eps, int nleaf, double* ax, double* ay, double* az, double* pot, DevScalars* sc, bool kick,
                   bool count, bool eval_waves, const float* amag, float rel2, float th2, hipStream_t s) {
#define NBX_PW(K, P, C, E)                                                                                      \
  hipLaunchKernelGGL((k_phys_walk<T, LIST, K, P, C, E>), dim3(nb), dim3(kPhysBlock * (1 + (E))), 0, s, groups, \
                     pn, st, sy, eps, nleaf, ax, ay, az, pot, sc, amag, rel2, th2)
  constexpr int kSplit = LIST == 128 ? kWalkEval : 0;
  const bool p = pot != nullptr, split = kSplit > 0 && !count && eval_waves;
  if (kick) {
    if (count) NBX_PW(true, false, true, 0);
    else if (split) NBX_PW(true, false, false, kSplit);
    else NBX_PW(true, false, false, 0);
  } else if (p) {
    if (count) NBX_PW(false, true, true, 0);
    else if (split) NBX_PW(false, true, false, kSplit);
    else NBX_PW(false, true, false, 0);
  } else {
    if (count) NBX_PW(false, false, true, 0);
    else if (split) NBX_PW(false, false, false, kSplit);
    else NBX_PW(false, false, false, 0);
  }
#undef NBX_PW
}

template <typename T>
void walk_dispatch_list(int list, unsigned nb, const Group* groups, const PhysNode* pn, const StateArrays& st,
                        const SysArrays& sy, double eps, int nleaf, double* ax, double* ay, double* az, double* pot,
                        DevScalars* sc, bool kick, bool count, bool split, const float* amag, float rel2,
                        float th2, hipStream_t s) {
  switch (list) {
    case 96: walk_dispatch<T, 96>(nb, groups, pn, st, sy, eps, nleaf, ax, ay, az, pot, sc, kick, count, split,
                                    amag, rel2, th2, s); break;
    case 192: walk_dispatch<T, 192>(nb, groups, pn, st, sy, eps, nleaf, ax, ay, az, pot, sc, kick, count, split,
                                    amag, rel2, th2, s); break;
    case 256: walk_dispatch<T, 256>(nb, groups, pn, st, sy, eps, nleaf, ax, ay, az, pot, sc, kick, count, split,
                                    amag, rel2, th2, s); break;
    default: walk_dispatch<T, 128>(nb, groups, pn, st, sy, eps, nleaf, ax, ay, az, pot, sc, kick, count, split,
                                    amag, rel2, th2, s); break;
  }
}

}  // namespace

// Group table in body order from the marks (gmark holds the exclusive scan
// of the marks by now; gcnt != 0 marks a group start).
__global__ __launch_bounds__(kBlock) void k_group_compact(int64_t n, const int32_t* __restrict__ gcnt,
                                                          const uint32_t* __restrict__ gidx,
                                                          const int32_t* __restrict__ body_sys,
                                                          Group* __restrict__ groups) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const int32_t c = gcnt[i];
  if (c != 0) groups[gidx[i]] = Group{(int32_t)i, c, body_sys[i], 0};
}

void launch_phys_emit(int64_t n, const int32_t* lcp, const uint32_t* pre_off, const uint32_t* part,
                      const StateArrays& st, const DevScalars* sc, PhysNode* pn, int32_t* level_list,
                      uint32_t* end_list, int32_t* gcnt, uint32_t* gmark, uint32_t cap_nodes, uint32_t cap_int,
                      hipStream_t s) {
  if (n > 0)
    hipLaunchKernelGGL(k_phys_emit, dim3(grid_of(n, kBlock)), dim3(kBlock), 0, s, n, lcp, pre_off, part, st, sc, pn,
                       level_list, end_list, gcnt, gmark, cap_nodes, cap_int);
}

void launch_phys_pair(int64_t m, const int32_t* level_list, const uint32_t* end_list, PhysNode* pn, hipStream_t s) {
  if (m > 0)
    hipLaunchKernelGGL(k_phys_pair, dim3(grid_of(m, kBlock)), dim3(kBlock), 0, s, m, level_list, end_list, pn);
}

void launch_phys_pair_dev(unsigned grid, const int32_t* level_list, const uint32_t* end_list, PhysNode* pn,
                          const DevScalars* sc, hipStream_t s) {
  hipLaunchKernelGGL(k_phys_pair_dev, dim3(grid), dim3(kBlock), 0, s, level_list, end_list, pn, sc);
}

void launch_phys_upward_tail(int d_lo, const int32_t* level_list, PhysNode* pn, void* aux, double theta,
                             int group_size, int32_t* gcnt, uint32_t* gmark, const DevScalars* sc, hipStream_t s) {
  if (d_lo < kMaxLevels)
    hipLaunchKernelGGL(k_phys_upward_tail, dim3(1), dim3(kBlock), 0, s, d_lo, level_list, pn,
                       reinterpret_cast<PhysAux*>(aux), 1.0 / theta, group_size, gcnt, gmark, sc);
}

void launch_phys_upward_level(unsigned grid, int d, const int32_t* level_list, PhysNode* pn, void* aux, double theta,
                              int group_size, int32_t* gcnt, uint32_t* gmark, const DevScalars* sc, hipStream_t s) {
  hipLaunchKernelGGL(k_phys_upward_level, dim3(grid * kNodeLanes), dim3(kBlock), 0, s, d, level_list, pn,
                     reinterpret_cast<PhysAux*>(aux), 1.0 / theta, group_size, gcnt, gmark, sc);
}

void launch_phys_upward(const int32_t* level_list, int64_t beg, int64_t cnt, int depth, PhysNode* pn, void* aux,
                        double theta, int group_size, int32_t* gcnt, uint32_t* gmark, hipStream_t s) {
  if (cnt > 0)
    hipLaunchKernelGGL(k_phys_upward, dim3(grid_of(cnt, kBlock / kNodeLanes)), dim3(kBlock), 0, s, level_list, beg, cnt,
                       depth == 0, pn, reinterpret_cast<PhysAux*>(aux), 1.0 / theta, group_size, gcnt, gmark);
}

void launch_group_compact(int64_t n, const int32_t* gcnt, uint32_t* gmark, const int32_t* body_sys, Group* groups,
                          uint32_t* ngroups, uint32_t* scratch, hipStream_t s) {
  if (n <= 0) return;
  scan_u32(gmark, gmark, n, ngroups, scratch, s);
  hipLaunchKernelGGL(k_group_compact, dim3(grid_of(n, kBlock)), dim3(kBlock), 0, s, n, gcnt, gmark, body_sys, groups);
}

void launch_phys_walk(const Group* groups, int64_t grid_groups, const PhysNode* pn, const StateArrays& st,
                      const SysArrays& sy, double eps, int nleaf, double* ax, double* ay, double* az, double* pot,
                      DevScalars* sc, bool kick, bool count, bool fp64, bool split, const float* amag, double alpha,
                      double theta, int list, hipStream_t s) {
  if (grid_groups <= 0) return;
  const unsigned nb = (unsigned)(div_up(grid_groups, 8) * 8);
  const float rel2 = (float)(alpha * alpha), th2 = (float)(theta * theta);
  if (alpha <= 0.0) amag = nullptr;
  if (fp64)
    walk_dispatch_list<double>(list, nb, groups, pn, st, sy, eps, nleaf, ax, ay, az, pot, sc, kick, count, split, amag,
                               rel2, th2, s);
  else
    walk_dispatch_list<float>(list, nb, groups, pn, st, sy, eps, nleaf, ax, ay, az, pot, sc, kick, count, split, amag,
                              rel2, th2, s);
}

// Waves per workgroup and halves of the sources: 8 waves on each of the 1,024
// SIMDs from 65,536 bodies on, at least 64 sources a wave below.  Workgroups
// of 16 waves serve where 4 would leave SIMDs with fewer than 4 waves; above,
// 2 resident ones per CU would leave the last round nearly empty.  No more
// than two halves: their sums are 64 bytes per body.
static int direct_waves(int64_t n) { return n <= 32768 ? 16 : 4; }

int direct_splits(int64_t n) {
  const int64_t groups = div_up(std::max<int64_t>(n, 1), kWave);
  const int w = direct_waves(n);
  return groups * w < 8192 && groups >= 2 * w ? 2 : 1;
}

template <bool ZERO, int W, int SPLITS>
static void direct_go(int64_t n, const StateArrays& st, const SysArrays& sy, double e2, double* ax, double* ay,
                      double* az, double* pot, hipStream_t s) {
  hipLaunchKernelGGL((k_direct64<ZERO, W, kDirectChunks / (W * SPLITS)>), dim3(grid_of(n, kWave), SPLITS),
                     dim3(W * kWave), 0, s, n, st, sy, e2, ax, ay, az, pot);
}

void launch_direct64(int64_t n, const StateArrays& st, const SysArrays& sy, double eps, double* part, double* ax,
                     double* ay, double* az, double* pot, hipStream_t s) {
  if (n <= 0) return;
  const bool halves = direct_splits(n) == 2, wide = direct_waves(n) == 16;
  double* const ox = halves ? part : ax;
  const double e2 = eps * eps;
#define NBX_DS(Z)                                                                                         \
  (wide ? (halves ? &direct_go<Z, 16, 2> : &direct_go<Z, 16, 1>) : (halves ? &direct_go<Z, 4, 2> : &direct_go<Z, 4, 1>))
  auto* const go = e2 > 0.0 ? NBX_DS(false) : NBX_DS(true);
#undef NBX_DS
  go(n, st, sy, e2, ox, ay, az, pot, s);
  if (halves)
    hipLaunchKernelGGL(k_direct_sum, dim3(grid_of(n, kBlock)), dim3(kBlock), 0, s, n, part, ax, ay, az, pot);
}

void launch_energy(const StateArrays& st, const double* pot, const BoxBlock* blocks, int nblocks,
                   const int32_t* block_off, int nsys, double* part, double* out, hipStream_t s) {
  if (nblocks > 0) hipLaunchKernelGGL(k_energy_partial, dim3(nblocks), dim3(kBlock), 0, s, st, pot, blocks, part);
  hipLaunchKernelGGL(k_energy_final, dim3(grid_of(nsys, kBlock)), dim3(kBlock), 0, s, part, block_off, nsys, out);
}

}  // namespace nbx

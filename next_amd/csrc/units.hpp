// Upward pass over units of consecutive bodies: reference trees of small
// systems.
//
// A unit is a run of about `span` bodies whose ends lie where neighbouring
// bodies share the fewest digits (the smallest lcp in a window of span / 2
// around each multiple of span), so it covers whole cells but for the few
// large ones that contain a unit's end.  One workgroup takes a unit and works
// through its internal nodes deepest first, a barrier between depths: every
// child of a node that ends inside the unit is in the unit too.  The unit's
// nodes of one depth are one piece of the per-depth node list (sorted by
// preorder).  A node that ends beyond its unit is the unit's last of its depth
// and goes to a table; one workgroup does those afterwards, depth by depth.
//
// A depth costs latency, not work, so what a node waits for is kept in LDS:
// the unit's node list and skip pointers, loaded once, and each node's mass and
// centre.
//
// A launch per depth takes 5 to 6 us for every depth of up to some thousand
// nodes (a dependent chain of list entry, up to 8 children one after another,
// system and root, and 400 to 900 FP64 instructions), 10 to 20 depths a build.
// Measured, whole upward pass: 1,000 bodies 53 -> 34 us, 16,384 69 -> 59, 65,536
// 88 -> 67, 262,144 96 -> 81, 366,000 107 -> 84, 128 systems of 2,000 76 -> 68.  A CU
// holds two units (80 KB of LDS each at most), the chip 512: with more, a second
// round of units costs what a launch per depth saves (512 systems of 1,000, 666
// units: 114 against 96 us, 2^20 bodies 203 against 178), and the nodes that end
// beyond their units, one workgroup's work, grow with the units.
#pragma once

#include <algorithm>

#include "common.hpp"
#include "ref_kernels.hpp"

namespace nbx {

// First body of unit u (1 <= u < units): after the body with the smallest lcp
// in [u span - span / 4, u span + span / 4), the first of several.  Called by
// every thread of a kBlock-thread block; scratch: kBlock / kWave words.
__device__ __forceinline__ int64_t unit_start(int64_t u, int32_t span, const int32_t* __restrict__ lcp,
                                              unsigned long long* scratch) {
  const int64_t lo = u * span - span / 4;                    // u span + span / 4 <= n - 1: units * span <= n
  unsigned long long best = ~0ull;
  for (int32_t k = threadIdx.x; k < span / 2; k += kBlock) {
    const unsigned long long v = ((unsigned long long)(uint32_t)(lcp[lo + k] + 1) << 32) | (uint32_t)k;
    if (v < best) best = v;
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const unsigned long long o = __shfl_xor(best, off, kWave);
    if (o < best) best = o;
  }
  if (lane_id() == 0) scratch[threadIdx.x / kWave] = best;
  __syncthreads();
  for (int w = 0; w < kBlock / kWave; ++w) best = scratch[w] < best ? scratch[w] : best;
  __syncthreads();
  return lo + (int64_t)(uint32_t)best + 1;
}

// A unit as its nodes see it: node k (preorder) is slot k - first of the LDS
// arrays when lds is set.
struct UnitView {
  int32_t first;
  bool lds;
  uint16_t* skips;          // skip pointer, as a slot
  __device__ __forceinline__ int slot(int32_t k) const { return k - first; }
};

// LDS of upward_unit, its alignment included.
template <int NODES>
constexpr size_t unit_lds() {
  return kBlock / kWave * 8 + 5 * kMaxDepthSlots * 4 + 2 * 4 + NODES * 6 + 8 * 16;
}

// The body of a unit kernel (kBlock threads, one unit per block).
// load(view, k): called once for every node k of the unit, in parallel, when
// the unit fits LDS (a leaf's data; an internal node's are written by node).
// node(view, id, end, depth): one internal node.
// NODES: nodes of a unit whose lists LDS holds (a unit of up to 1.5 span bodies
// has about 1.5 nodes per body); with more (clumps that share many digits) the
// lists and records are read from memory.
template <int NODES, class Load, class Node>
__device__ __forceinline__ void upward_unit(const UnitArgs& a, Load load, Node node) {
  __shared__ unsigned long long red[kBlock / kWave];
  __shared__ int32_t seg[2][kMaxDepthSlots];       // this unit's part of each depth's list
  __shared__ uint32_t off[kMaxDepthSlots];         // nodes of smaller depth
  __shared__ int32_t at[kMaxDepthSlots];           // where each depth's part starts in `list`
  __shared__ int32_t over[kMaxDepthSlots];         // list entry of the node that ends beyond the unit
  __shared__ uint32_t range[2];
  __shared__ uint32_t list[NODES];            // slots of a node and of its end (NODES: beyond the unit)
  __shared__ uint16_t skips[NODES];
  if (a.sc->abort_flags) return;
  const int t = threadIdx.x;
  const int64_t u = blockIdx.x;
  const int64_t s0 = u == 0 ? 0 : unit_start(u, a.span, a.lcp, red);
  const int64_t s1 = u + 1 == a.units ? a.n : unit_start(u + 1, a.span, a.lcp, red);
  if (t < kMaxDepthSlots) {
    const uint32_t v = (uint32_t)a.sc->level_count[t];
    off[t] = wave_incl_scan_u32(v) - v;
    over[t] = -1;
  }
  __syncthreads();
  if (t < 2 * kMaxDepthSlots) {
    // first entry of depth d at or after the unit's first (last + 1) body's first node
    const int d = t % kMaxDepthSlots, side = t / kMaxDepthSlots;
    const int64_t s = side ? s1 : s0;
    const uint32_t cnt = (uint32_t)a.sc->level_count[d];
    const uint32_t p = s < a.n ? a.pre_off[s] : (uint32_t)a.sc->total_nodes;
    uint32_t lo = cnt, hi = cnt;
    if (s < a.n) {
      const int64_t blk = s / kBlock, nblk = (a.n + kBlock - 1) / kBlock;   // the blocks of k_lcp_count
      lo = a.part[(int64_t)d * nblk + blk];
      hi = blk + 1 < nblk ? a.part[(int64_t)d * nblk + blk + 1] : cnt;
    }
    while (lo < hi) {
      const uint32_t mid = lo + (hi - lo) / 2;
      if ((uint32_t)a.level_list[off[d] + mid] < p) lo = mid + 1;
      else hi = mid;
    }
    seg[side][d] = (int32_t)(off[d] + lo);
    if (d == 0) range[side] = p;
  }
  __syncthreads();
  const uint32_t p0 = range[0], p1 = range[1];
  const UnitView view{(int32_t)p0, p1 - p0 < (uint32_t)NODES, skips};
  if (view.lds) {
    if (t < kMaxDepthSlots) {
      const uint32_t v = (uint32_t)(seg[1][t] - seg[0][t]);
      at[t] = (int32_t)(wave_incl_scan_u32(v) - v);
    }
    for (uint32_t k = t; k < p1 - p0; k += kBlock) {
      skips[k] = (uint16_t)(k + 1);                          // a leaf's
      load(view, (int32_t)(p0 + k));
    }
    __syncthreads();
    // a wave per depth copies its part of the lists
    for (int d = t / kWave; d < kMaxLevels; d += kBlock / kWave)
      for (int32_t k = seg[0][d] + lane_id(); k < seg[1][d]; k += kWave) {
        const uint32_t end = a.end_list[k];
        list[at[d] + (k - seg[0][d])] =
            ((uint32_t)a.level_list[k] - p0) | ((end > p1 ? (uint32_t)NODES : end - p0) << 16);
        if (end > p1) over[d] = k;
      }
    __syncthreads();
    for (int d = kMaxLevels - 1; d >= 0; --d) {
      const int32_t cnt = seg[1][d] - seg[0][d];
      if (cnt == 0) continue;                                // (uniform)
      for (int32_t k = t; k < cnt; k += kBlock) {
        const uint32_t e = list[at[d] + k], id = e & 0xffffu, end = e >> 16;
        if (end == (uint32_t)NODES) continue;
        node(view, (int32_t)(p0 + id), (int32_t)(p0 + end), d);
        skips[id] = (uint16_t)end;
      }
      __syncthreads();
    }
  } else {
    for (int d = kMaxLevels - 1; d >= 0; --d) {
      const int32_t b = seg[0][d], e = seg[1][d];
      if (b == e) continue;
      for (int32_t k = b + t; k < e; k += kBlock) {
        const uint32_t end = a.end_list[k];
        if (end > p1) over[d] = k;
        else node(view, a.level_list[k], (int32_t)end, d);
      }
      __syncthreads();
    }
  }
  if (a.units == 1) return;
  if (t < kMaxDepthSlots) {
    const int32_t k = over[t];
    if (t < kMaxLevels) a.over[(int64_t)t * a.units + u] = k;
    const unsigned long long m = __ballot(k >= 0);
    if (t == 0 && m) atomicOr(&a.sc->over_depths, m);
  }
}

// The nodes that end beyond their units, depth by depth: a workgroup of
// kOverBlock threads takes one system after another (a system's nodes are its
// own).  A system of at most span / 2 bodies has none: where a unit ends inside
// a system, the window its end was chosen from holds that system's bodies only.
// At most kOverBlocks workgroups: one for each of 16,000 systems of 16 bodies
// took 27 us to find nothing.  The depth mask is cleared by the next build's
// first kernel.
constexpr int kOverBlock = 1024, kOverBlocks = 512;
template <class Node>
__device__ __forceinline__ void upward_over(const UnitArgs& a, const SysArrays& sy, Node node) {
  __shared__ int32_t list[kOverBlock];
  __shared__ int32_t count;
  if (a.sc->abort_flags) return;
  const unsigned long long depths = a.sc->over_depths;
  if (depths == 0) return;
  const int t = threadIdx.x;
  const UnitView view{0, false, nullptr};
  for (int32_t s = blockIdx.x; s < sy.nsys; s += gridDim.x) {
    if (sy.soff[s + 1] - sy.soff[s] <= a.span / 2) continue;   // (uniform)
    const int32_t root = sy.sroot[s], end = sy.send[s];
    // units that can hold the system's bodies
    const int32_t ub = (int32_t)std::max<int64_t>((int64_t)sy.soff[s] / a.span - 1, 0);
    const int32_t ue = (int32_t)std::min<int64_t>((int64_t)sy.soff[s + 1] / a.span + 2, a.units);
    for (unsigned long long m = depths; m;) {
      const int d = 63 - __clzll((long long)m);
      m &= ~(1ull << d);
      for (int32_t u0 = ub; u0 < ue; u0 += kOverBlock) {
        if (t == 0) count = 0;
        __syncthreads();
        const int32_t k = u0 + t < ue ? a.over[(int64_t)d * a.units + u0 + t] : -1;
        if (k >= 0) {
          const int32_t id = a.level_list[k];
          if (id >= root && id < end) list[atomicAdd(&count, 1)] = k;
        }
        __syncthreads();
        for (int32_t j = t; j < count; j += kOverBlock)
          node(view, a.level_list[list[j]], (int32_t)a.end_list[list[j]], d);
        __syncthreads();
      }
    }
  }
}

}  // namespace nbx

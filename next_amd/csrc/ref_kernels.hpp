// Launchers for the reference-mode (FP64, NEXT-exact) kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "common.hpp"

namespace nbx {

// Particle state, structure of arrays (particle.h:22-52) plus `id`, the
// upload-order index of the body held in each slot, and `sys`, its system.
struct StateArrays {
  double *x, *y, *z, *vx, *vy, *vz, *m;
  int32_t *type, *id, *sys;
};

constexpr int kBlock = 256;
constexpr int kBoxSpan = 2048;      // bodies per block of the bounding-box reduction
// Row of per-block partial counts written by the lcp kernel: internal nodes
// started per depth (columns 0..63), ended per depth (64..127), deepest leaf,
// equal-key pairs.  k_lcp_scan turns the per-depth columns into exclusive
// prefixes over the blocks.
constexpr int kPartEnds = kMaxDepthSlots;
constexpr int kPartMaxDepth = 2 * kMaxDepthSlots;  // column: deepest leaf
constexpr int kPartEqual = 2 * kMaxDepthSlots + 1; // column: equal-key pairs
constexpr int kPartW = 2 * kMaxDepthSlots + 2;
inline int64_t lcp_part_words(int64_t n) { return ((n + kBlock - 1) / kBlock) * kPartW; }

void launch_fill_scalars(DevScalars* sc, int what, hipStream_t s);  // what: 1 build counters, 4 err, 8 walk counters
// v2max (the largest |v|^2 per system, which the closing kicks raise) to 0;
// k_dt also resets it once it has read it.
void launch_fill_v2max(const SysArrays& sy, hipStream_t s);
void launch_set_dt(const SysArrays& sy, double dt, hipStream_t s);
// Roots of the systems from their bodies' bounding boxes; clear (may be
// null): the scalars a tree build counts into, reset as launch_fill_scalars
// with what = 1 | 4 would.
void launch_bbox(const StateArrays& st, const BoxBlock* blocks, int nblocks, const int32_t* block_off, double* part,
                 const SysArrays& sy, DevScalars* clear, hipStream_t s);
void launch_keys(int64_t n, const StateArrays& st, const SysArrays& sy, uint64_t* key, uint32_t* idx,
                 DevScalars* scw, hipStream_t s);
void launch_keys2(int64_t n, const StateArrays& st, const SysArrays& sy, uint64_t* key2, hipStream_t s);
// Runs of bodies of one system with equal first key words (in the order of
// the sort by the first word) sorted in place by the second word, stably;
// key2 written for those bodies (amag, may be null, moves with them).
void launch_fix_runs(int64_t n, const StateArrays& st, const SysArrays& sy, uint64_t* key, uint64_t* key2,
                     uint32_t* amag, int lo, hipStream_t s);
void launch_iota(int64_t n, uint32_t* idx, hipStream_t s);
void launch_gather_u64(int64_t n, const uint32_t* perm, const uint64_t* src, uint64_t* dst, hipStream_t s);
void launch_gather_sys(int64_t n, const uint32_t* perm, const int32_t* sys, uint32_t* dst, hipStream_t s);
// dst[i] = src[perm[i]] for 32-bit words.
void launch_gather_u32(int64_t n, const uint32_t* perm, const uint32_t* src, uint32_t* dst, hipStream_t s);
void launch_gather_state(int64_t n, const uint32_t* perm, const StateArrays& src, const StateArrays& dst,
                         hipStream_t s);
// lcp of the sorted keys, each body's node count (its started internal
// nodes and its leaf) in cnt_s, the per-block rows of per-depth counts
// (scanned over the blocks) in part, and in sc the internal nodes per depth,
// the deepest leaf and the equal-key pairs.
void launch_lcp_count(int64_t n, const uint64_t* key, const uint64_t* key2, const int32_t* sys, int32_t* lcp,
                      uint32_t* cnt_s, uint32_t* part, DevScalars* sc, hipStream_t s);
void launch_sys_roots(const SysArrays& sy, const uint32_t* pre_off, const DevScalars* sc, hipStream_t s);
void launch_remove_map(int64_t n_new, int64_t cut, int64_t len, uint32_t* perm, hipStream_t s);
void launch_relabel(int64_t n, int32_t* sys, int32_t removed, hipStream_t s);
void launch_gather_f64(int64_t n, const uint32_t* perm, const double* src, double* dst, hipStream_t s);
// Leaf records and walk heads from the sorted keys' lcp and the scan of
// cnt_s (pre_off), and every internal node's place in the per-depth node list
// and the list of skip targets (layout.hpp); writes records below cap_nodes
// and list entries below cap_int only (the buffers' capacities), so it can
// run before the host knows the node counts.  The internal nodes' records
// come from the upward pass.
void launch_emit(int64_t n, const int32_t* lcp, const uint32_t* pre_off, const uint32_t* part,
                 const StateArrays& st, const SysArrays& sy, const DevScalars* sc, RefNode* nodes, WalkHead* heads,
                 int32_t* level_list, uint32_t* end_list, uint32_t cap_nodes, uint32_t cap_int, hipStream_t s);
// Builds whose counts stay on the device (no host read-back; a step of them
// can be captured): k_check derives each depth's offset and raises the abort
// flag when the tree does not fit cap_records node records, cap_list
// node-list entries or depth levels 0..dmax; the per-depth upward kernels
// take their counts from the scalars with fixed grids, and every tree kernel
// does nothing once the flag is set.
void launch_check(DevScalars* sc, int64_t cap_records, int64_t cap_list, int dmax, hipStream_t s);
// Start of a captured run: abort flag cleared, dt log entries from `step` on.
void launch_set_run(DevScalars* sc, int32_t step, hipStream_t s);
// Internal node records and heads of depth d (the list entries [beg, beg +
// cnt)), from their children's records; sys and root: the bodies' systems
// and the systems' roots (4 doubles each).
void launch_upward_level(unsigned grid, int d, const int32_t* level_list, const uint32_t* end_list, RefNode* nodes,
                         WalkHead* heads, double theta, const int32_t* sys, const double* root, const DevScalars* sc,
                         hipStream_t s);
// Depths d_lo .. 41 (whatever the build holds there) in one workgroup.
void launch_upward_tail(int d_lo, const int32_t* level_list, const uint32_t* end_list, RefNode* nodes,
                        WalkHead* heads, double theta, const int32_t* sys, const double* root, const DevScalars* sc,
                        hipStream_t s);
void launch_upward(const int32_t* level_list, const uint32_t* end_list, int64_t beg, int64_t cnt, int d,
                   RefNode* nodes, WalkHead* heads, double theta, const int32_t* sys, const double* root,
                   hipStream_t s);
// Every depth of a build whose per-depth counts the host holds (counts[d],
// the node list in depth order), one launch per depth, deepest first.  (A
// narrow level costs the latency of its nodes' child chains, not the launch:
// running the narrow levels at either end of the tree in one workgroup each
// measured slower.)
void launch_upward_all(const int32_t* counts, const int32_t* level_list, const uint32_t* end_list, RefNode* nodes,
                       WalkHead* heads, double theta, const int32_t* sys, const double* root, hipStream_t s);
// The same for a build of at most kUnitsMax bodies in two launches whose sizes
// need no counts on the host (units.hpp).  What it reads of the layout: the
// lcp and node offsets of the bodies, the scanned per-block counts of
// k_lcp_count, the per-depth node list and its skip targets; over holds
// kMaxLevels entries per unit; sys: the bodies' systems (after
// launch_sys_roots).
struct UnitArgs {
  int64_t n;
  int32_t units, span;
  const int32_t* lcp;
  const uint32_t* pre_off;
  const uint32_t* part;
  const int32_t* level_list;
  const uint32_t* end_list;
  DevScalars* sc;
  int32_t* over;
};
constexpr int32_t kUnitSpan = 768;   // bodies per unit: about 1,150 nodes
constexpr int64_t kUnitsMax = 512 * kUnitSpan;   // two units on each of 256 CUs
// Units of n / units bodies, at most kUnitSpan, and up to half as many more where
// the boundaries move to the smallest lcp (units.hpp): 1,152 bodies, which have
// about 1,700 nodes.  (All of kUnitSpan but a longer last one left that with up
// to 2,100 nodes, too many for LDS.)
constexpr int32_t unit_count(int64_t n) { return n <= 1230 ? 1 : (int32_t)((n + kUnitSpan - 1) / kUnitSpan); }
constexpr int32_t unit_span(int64_t n) { return (int32_t)(n / unit_count(n)); }
void launch_upward_units(const UnitArgs& a, RefNode* nodes, WalkHead* heads, double theta, const int32_t* sys,
                         const SysArrays& sy, hipStream_t s);
void launch_fill_u32(int64_t n, uint32_t* a, uint32_t v, hipStream_t s);
// Keys and body arrays (amag may be null) in ascending order of the keys,
// equal keys in their previous order: sort and gather in one launch, for
// systems of at most kRankSortMax bodies (n^2 compares).
constexpr int kRankWaves = 16;
constexpr int64_t kRankSortMax = 16384;
// Up to here also in place of the nearly-sorted path (three launches and the
// gather, 45 us at any small size).
constexpr int64_t kRankAlways = 4096;
void launch_rank_sort(int64_t n, const uint64_t* key, uint64_t* kout, const StateArrays& src, const StateArrays& dst,
                      const uint32_t* amag, uint32_t* amag_out, hipStream_t s);
// Upload indices id0, id0 + 1, ... and system number of n slots.
void launch_set_ids(int64_t n, int32_t* id, int32_t id0, int32_t* sys, int32_t sys_no, hipStream_t s);
// inv[j] = the slot (of cnt) that holds upload index base + j; *bad (host
// memory, 0 before) is set unless the slots hold a permutation of [base, base
// + cnt).
void launch_out_index(int64_t cnt, const int32_t* id, int32_t base, uint32_t* inv, int32_t* bad, hipStream_t s);
// Values of upload indices [j0, j0 + len) of m arrays, one array after
// another, len values each, into dst (host memory the device can write).
constexpr int kOutArrays = 6;
struct OutArrays {
  const double* p[kOutArrays];
};
void launch_out_gather(int64_t j0, int64_t len, int64_t cnt, const uint32_t* inv, const OutArrays& src, int m,
                       double* dst, hipStream_t s);
// Bodies per walk group of a system of n bodies, 8 to 64 (a group narrower
// than 64 puts 64 / width lanes on each target).  It depends on the system
// alone, so a system's sums are the same alone and in a batch.  Narrow
// groups give a small system enough waves and short ones; wide groups share
// more of the traversal, which is what a batch of many systems needs, the more
// so the larger theta, and what a large system needs too.  Up to 20,480 bodies
// the lines lie where the narrower groups would make a batch of Plummer spheres
// slower than one union traversal per 64 targets was ("u"); above, at the
// fastest width.  64 bodies are one wave's work either way.
// Walk (us, Plummer spheres), width u / 8 / 16 / 32 / 64:
//   theta  n        alone                              batch
//   0.3    64        39 /  29 /  32 /  41 /  41      4,000:   103 /   250 /   174 /   140 /   110
//   0.3    500      268 /  57 /  93 / 138 / 215        512:   475 /   573 /   505 /   512 /   542
//   0.3    1,000    403 / 107 / 133 / 198 / 295        512: 1,399 / 1,319 / 1,211 / 1,295 / 1,434
//   0.3    16,384   941 / 226 / 302 / 447 / 584         64: 5,600 / 4,926 / 4,816 / 5,194 / 5,504
//   0.39   200,003 1,011 / 752 / 675 / 685 / 740
//   0.35   2^20    5,155 / 5,032 / 4,372 / 4,160 / 3,750 (uniform 3,478 / 3,575 / 3,044 / 3,025 / 3,134)
//   0.3    2^20    7,500 / 6,544 / 6,089 / 6,240 / 5,917 (uniform 4,953 / 4,457 / 4,162 / 4,438 / 4,851)
//   0.39   2^22, uniform: 11,130 / 13,919 / 10,922 / 9,841 / 9,751
//   0.4    2,000    358 /  70 /  91 / 137 / 224        512: 2,105 / 2,527 / 2,076 / 1,984 / 2,078
//   0.44   100,000  592 / 338 / 303 / 285 / 302         10: 2,650 / 3,073 / 2,441 / 2,196 / 1,911
//   0.5    1,000    246 /  57 /  70 / 103 / 152        512:   767 /   885 /   677 /   635 /   643
//   0.5    2,000    270 /  57 /  78 / 112 / 162        512: 1,522 / 2,115 / 1,619 / 1,408 / 1,388
//   0.5    16,384   343 /  84 / 108 / 173 / 195         64: 1,972 / 2,577 / 1,975 / 1,686 / 1,485
//   0.5    32,768   378 / 117 / 121 / 200 / 232         32: 2,035 / 2,700 / 2,063 / 1,744 / 1,501
//   0.5    65,536   441 / 218 / 165 / 185 / 248         16: 2,101 / 2,801 / 2,131 / 1,790 / 1,491
//   0.5    100,000  458 / 305 / 258 / 233 / 265         10: 2,067 / 2,752 / 2,084 / 1,763 / 1,417
//   0.5    200,003  631 / 583 / 449 / 432 / 417
//   0.55   1,000    217 /  54 /  65 /  89 / 137        512:   667 /   833 /   623 /   567 /   575
//   0.55   16,384   305 /  78 /  94 / 126 / 181         64: 1,683 / 2,388 / 1,779 / 1,466 / 1,203
//   0.7    16,384   206 /  74 /  79 /  94 / 135         64: 1,210 / 2,021 / 1,419 / 1,115 /   782
//   0.85   16,384   165 /  61 /  83 / 107 / 111         64:   940 / 1,779 / 1,216 /   926 /   639
//   1.0    1,000    115 /  40 /  51 /  57 /  77        512:   330 /   621 /   429 /   327 /   285
//   1.0    16,384   130 /  83 /  82 /  91 /  91         64:   757 / 1,583 / 1,066 /   779 /   539
// Batches of uniform spheres, which have less to share, cross earlier: a step
// of 64 of 16,384 bodies at theta 0.5 takes 1,783 us against 1,676, of 512 of
// 2,000 1,479 against 1,315; alone the wider groups that would mend it cost
// 35 to 65 us of a walk of 80 to 110.
inline int32_t walk_width(int64_t n, double theta) {
  if (n <= 64) return 64;
  if (theta <= 0.32 && n >= 896 && n <= 4096) return 8;
  if (theta < 0.35) return 16;
  if (n <= (theta < 0.4 ? 524288 : theta < 0.45 ? 98304 : theta <= 0.5 ? 20480 : theta <= 0.55 ? 1500 : 0)) return 16;
  return n <= 1500 || (n <= 196608 && theta >= 0.4 && theta <= 0.8) ? 32 : 64;
}
void launch_walk(const Group* groups, int64_t ngroups, const RefNode* nodes, const WalkHead* heads,
                 const StateArrays& st,
                 const SysArrays& sy, double theta, double* ax, double* ay, double* az, DevScalars* sc, bool kick,
                 bool count, hipStream_t s);
// amag (may be null): |a| per body in FP32.
void launch_kick_drift(int64_t n, const StateArrays& st, const double* ax, const double* ay, const double* az,
                       const SysArrays& sy, float* amag, hipStream_t s);
void launch_maxv2(int64_t n, const StateArrays& st, const SysArrays& sy, hipStream_t s);
// dts (may be null) receives system 0's dt at entry `step`, or, for step < 0,
// at the entry the device's step counter gives (which it advances).
void launch_dt(const SysArrays& sy, double base, double* dts, int64_t step, DevScalars* sc, hipStream_t s);
void launch_export(int64_t total, const RefNode* nodes, const uint64_t* key, const uint64_t* key2,
                   const int32_t* id, const SysArrays& sy, int32_t* depth, int32_t* leaf, int32_t* body,
                   int32_t* cmask, double* geo4, double* mass, double* com3, double* q6, hipStream_t s);
void launch_keys_export(int64_t n, const StateArrays& st, const SysArrays& sy, uint64_t* hi, uint64_t* lo,
                        hipStream_t s);

}  // namespace nbx

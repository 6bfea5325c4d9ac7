// Launchers for the physics-mode kernels (phys_kernels.hip): bucket-leaf
// group walk with traceless quadrupoles and Plummer softening, and the FP64
// direct sum used for force errors and energies.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "common.hpp"
#include "ref_kernels.hpp"

namespace nbx {

// Walk record of a node (64 bytes): FP64 centre of mass for the
// group-relative conversion, FP32 moments, and the traversal links.
struct alignas(64) PhysNode {
  double cx, cy, cz;
  float m;
  float rc2;                  // (bmax / theta)^2; +inf: never accepted as a cell
  float qxx, qyy, qxy, qxz, qyz;   // traceless: qzz = -(qxx + qyy)
  int32_t skip;
  int32_t first;              // first body (sorted index)
  int32_t count;              // bodies in the subtree
};
static_assert(sizeof(PhysNode) == 64, "PhysNode layout");

// A leaf is never accepted as a cell (rc2 = +inf), so its first two
// quadrupole slots hold its FP64 mass, which the upward pass reads.
__host__ __device__ inline void set_leaf_mass(PhysNode& nd, double m) { __builtin_memcpy(&nd.qxx, &m, 8); }
__host__ __device__ inline double leaf_mass(const PhysNode& nd) {
  double m;
  __builtin_memcpy(&m, &nd.qxx, 8);
  return m;
}

constexpr int kPhysBlock = 64;      // one wave = one group of targets (further waves: k_phys_walk)
// Per-wave LDS (7.9 KB with these sizes) bounds the walk's occupancy at
// about 5 waves per SIMD; a 256-entry stack and body list (11 KB) allowed 3.
// Entries of the per-wave LDS lists (accepted cells, bodies of accepted
// buckets) a walk collects before it evaluates them: a walk setting
// (nbx_set_walk_list), one of kPhysLists.
constexpr int kPhysListDefault = 128;
constexpr int kPhysLists[] = {96, 128, 192, 256};
constexpr int kPhysMaxLeaf = 64;    // bucket size limit (one body per lane)
constexpr int kPhysStack = 32;      // per-wave LDS stack of donated node ranges
constexpr int kPhysAuxBytes = 128;  // FP64 moments per node (mass, bmax, Q, box)

// Walk groups are marked per first body in gcnt (body count) and gmark
// (1), both zeroed beforehand, then compacted in body order.
// Node layout from the sorted keys (the arguments of launch_emit, capacities
// included): leaf records complete, internal nodes' first body, their places
// in the per-depth node list and the list of skip targets; a leaf that is a
// system root is a one-body group.
void launch_phys_emit(int64_t n, const int32_t* lcp, const uint32_t* pre_off, const uint32_t* part,
                      const StateArrays& st, const DevScalars* sc, PhysNode* pn, int32_t* level_list,
                      uint32_t* end_list, int32_t* gcnt, uint32_t* gmark, uint32_t cap_nodes, uint32_t cap_int,
                      hipStream_t s);
// Skip pointers of the m internal nodes from the two lists.
void launch_phys_pair(int64_t m, const int32_t* level_list, const uint32_t* end_list, PhysNode* pn, hipStream_t s);
// The same two passes for builds whose counts stay on the device (see
// launch_check): fixed grids, counts from the scalars.
void launch_phys_pair_dev(unsigned grid, const int32_t* level_list, const uint32_t* end_list, PhysNode* pn,
                          const DevScalars* sc, hipStream_t s);
void launch_phys_upward_level(unsigned grid, int d, const int32_t* level_list, PhysNode* pn, void* aux, double theta,
                              int group_size, int32_t* gcnt, uint32_t* gmark, const DevScalars* sc, hipStream_t s);
void launch_phys_upward_tail(int d_lo, const int32_t* level_list, PhysNode* pn, void* aux, double theta,
                             int group_size, int32_t* gcnt, uint32_t* gmark, const DevScalars* sc, hipStream_t s);
// Internal nodes of one depth from their children (FP64 accumulation), and
// the walk groups of at most group_size bodies each node packs (see
// k_phys_upward).  `aux`: kPhysAuxBytes per node of FP64 moments (mass,
// bmax, quadrupole, bounding box of the bodies), internal nodes only.
void launch_phys_upward(const int32_t* level_list, int64_t beg, int64_t cnt, int depth, PhysNode* pn, void* aux,
                        double theta, int group_size, int32_t* gcnt, uint32_t* gmark, hipStream_t s);
// The group table from the marks (gmark is overwritten by its scan);
// *ngroups (device) receives the count; scratch as for scan_u32 over n.
void launch_group_compact(int64_t n, const int32_t* gcnt, uint32_t* gmark, const int32_t* body_sys, Group* groups,
                          uint32_t* ngroups, uint32_t* scratch, hipStream_t s);
// Group walk over the group table: accelerations (and potentials if
// pot != null), optionally followed by the closing half kick.  fp64 selects
// the FP64 evaluation.  With amag (|a| of each body from the previous
// evaluation, FP32) and alpha > 0, a cell that passes the geometric test
// (bmax / theta) is accepted only if m bmax^3 <= alpha |a|min d^5, |a|min
// the smallest |a| of the group and d the distance to the group's box.  The
// kernel takes the group count from sc->tree_groups; grid_groups (> 0) only
// sizes the grid, and a grid below the count walks the rest in more rounds.
// split: three further waves per group (list size 128 and no counting only); the
// bits are the same either way.
void launch_phys_walk(const Group* groups, int64_t grid_groups, const PhysNode* pn, const StateArrays& st,
                      const SysArrays& sy, double eps, int nleaf, double* ax, double* ay, double* az, double* pot,
                      DevScalars* sc, bool kick, bool count, bool fp64, bool split, const float* amag, double alpha,
                      double theta, int list, hipStream_t s);
// Whether a walk over about `groups` groups takes further waves; mean: the size
// of a body's system, averaged over the bodies (the larger systems' groups are
// the long ones).  Few groups leave most SIMDs with one wave at most, and a
// wave's time is then its evaluation's latency (about 2/3) plus its walk's: as
// long as all workgroups are resident at once (LDS: 5 on a CU in FP32, 3 in FP64)
// the further waves pay unless a group's lists are hardly ever full.  Beyond that
// they pay only where a group's work is long: larger systems, the more so the
// smaller the groups (whose lanes share the lists already), down to 17.
// Walk (us, Plummer spheres, theta 0.5), one wave per group / 1 + 3:
//   systems x bodies, group size   groups      FP32            FP64
//      1 x 2,000     64               60    125 /   67     158 /   77
//      1 x 16,384    64              373    511 /  177     677 /  253
//     30 x 1,000     64              990     99 /   68     117 /  119
//   1000 x 64        64            1,000     26 /   30
//      8 x 4,096     32            1,496    173 /  145     212 /  194
//     30 x 1,000     32            1,800     89 /  117     108 /  164
//    200 x 200       64            2,000     46 /   75      52 /  107
//    30 of 1-5,000   64            2,157    245 /  178     381 /  326
//      4 x 16,384    32            2,936    435 /  277     542 /  423
//      8 x 4,096     16            2,944    112 /  169     179 /  247
//    100 x 1,000     64            3,300    117 /  171     226 /  273
//     32 x 4,096     64            3,392    261 /  235     506 /  456
//     64 x 2,000     64            3,840    190 /  202     369 /  381
//   4000 x 64        64            4,000     34 /   94
//      1 x 200,000   64            4,436    578 /  492   1,119 / 1,064  (theta 0.8: 282 / 285, 537 / 560)
//     32 x 4,096     32            5,984    285 /  350     457 /  571
//    30 of 1-33,000  64            6,605    940 /  639   1,612 / 1,360  (theta 0.7: 716 / 466, 1,163 / 924)
//      5 x 65,536    64            7,335    753 /  680   1,489 / 1,509  (theta 0.8: 392 / 418, 734 / 835)
//    300 x 1,000     64            9,900    252 /  427     461 /  726
// They also shorten the longest group: two clusters of 140,000 bodies (6,174
// groups) take a third of the time (0.31 to 0.47 times), which is why even ones go
// on to 8,192 groups, where they lose up to a fifth in FP64 and above theta 0.6
// (a uniform ball of 280,000 bodies, 6,102 groups, FP64: 0.99 at theta 0.35, 1.14 at
// 0.62).
inline bool phys_walk_split(int64_t groups, int64_t mean, int group_size, bool fp64) {
  if (mean < 128) return false;
  if (groups <= (fp64 ? 768 : 1280)) return true;
  const bool narrow = group_size <= 32;
  if (group_size <= 16 || mean < (narrow ? 3072 : 1536)) return false;
  return groups <= (mean < (narrow ? 8192 : 3072) ? 2304 : 8192);
}
// FP64 direct sum with Plummer softening over all pairs of each system (G = 1).
// part: room for direct_splits(n) * 4 * n partial sums when that is two parts
// (fewer than 131,072 bodies).
int direct_splits(int64_t n);
void launch_direct64(int64_t n, const StateArrays& st, const SysArrays& sy, double eps, double* part, double* ax,
                     double* ay, double* az, double* pot, hipStream_t s);
// Kinetic energy, potential energy (0.5 sum m phi) and momentum of each
// system, reduced in a fixed order over the bounding-box blocks:
// out (device, 5 per system) = {ekin, epot, px, py, pz}; part holds 5 doubles
// per block.
void launch_energy(const StateArrays& st, const double* pot, const BoxBlock* blocks, int nblocks,
                   const int32_t* block_off, int nsys, double* part, double* out, hipStream_t s);

}  // namespace nbx

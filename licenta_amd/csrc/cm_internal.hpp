// Internal declarations of libclothmi: launch helpers shared between the
// kernel translation units and the body orchestration.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <algorithm>
#include <string>

#include "../../include/clothmi.h"
#include "cm_math.hpp"

namespace cm {

void set_error(const std::string& msg);

#define CM_HIP(expr)                                                                   \
  do {                                                                                 \
    hipError_t e_ = (expr);                                                            \
    if (e_ != hipSuccess) {                                                            \
      ::cm::set_error(std::string(#expr) + ": " + hipGetErrorString(e_));              \
      return CM_ERR_HIP;                                                               \
    }                                                                                  \
  } while (0)

#define CM_LAUNCH_CHECK()                                                              \
  do {                                                                                 \
    hipError_t e_ = hipGetLastError();                                                 \
    if (e_ != hipSuccess) {                                                            \
      ::cm::set_error(std::string("kernel launch: ") + hipGetErrorString(e_));         \
      return CM_ERR_HIP;                                                               \
    }                                                                                  \
  } while (0)

constexpr int kBlock = 256;  // 4 wave64s
constexpr int kXcds = 8;     // MI355X: workgroup i runs on XCD i mod 8

// Logical block for hardware block b of n so that each XCD gets a contiguous range
// of logical blocks (and so of data) instead of every eighth one. A bijection on
// [0, n).
__device__ __forceinline__ int xcd_block(int b, int n) {
  const int q = n / kXcds, r = n % kXcds;  // XCD x holds q + (x < r) blocks
  const int x = b % kXcds, k = b / kXcds;
  return x * q + min(x, r) + k;
}
inline int nblocks(int64_t n, int block = kBlock) {
  int64_t b = (n + block - 1) / block;
  return (int)(b < 1 ? 1 : b);
}
inline size_t align_up(size_t v, size_t a = 256) { return (v + a - 1) / a * a; }

// ---- primitives (k_prims.hip) --------------------------------------------
size_t scan_temp_bytes(int n_max);
// zero a scan temp before its first use (scans leave it zeroed for the next one)
int scan_temp_clear(void* temp, int n_max, hipStream_t s);
// exclusive prefix sum of in[0, n) into out[0, n), n = d_n ? min(*d_n, n_max) : n_max;
// *d_total (if non-null) receives the sum. out may alias in.
int scan_exclusive(const int* in, int* out, int n_max, const int* d_n, int* d_total, void* temp,
                   hipStream_t s);
// Tiles of the passes over a device-side number of items: one tile of 64 * R consecutive
// items per wave, lane l taking items base + l + 64 * j, j < R. R grows with the count, so
// that a short list still gives every SIMD a wave and a long one has few tile sums:
//   kTileSmall  R = 1 up to 8,192 tiles, else 4 (R = 4 -> 1: 64^2 k_ccd_test 40 -> 13.5
//               us, k_cand_count 8 -> 5.6; draped 131x97 k_ccd_test 48 -> 17)
//   kTilePlan   R = as many as leave kPlanWaves tiles, 1 to 8: a tile gathers the long
//               searches of its chunks, so long lists want large ones (R = 8 -> 1 at 64^2:
//               59 -> 22 us; R up to 16: 486 -> 522 us draped 256^2)
enum TileRule : int { kTileSmall, kTilePlan };
constexpr int kSmallWaves = 8192, kPlanWaves = 3072, kPlanLanes = 8;
__host__ __device__ inline int tile_lanes(TileRule rule, int items) {
  if (rule == kTileSmall) return items <= 64 * kSmallWaves ? 1 : 4;
  const int r = (int)(((int64_t)items + 64 * kPlanWaves - 1) / (64 * kPlanWaves));
  return r < 1 ? 1 : r > kPlanLanes ? kPlanLanes : r;
}
// most tiles that up to item_cap items can make
inline int64_t tile_max(TileRule rule, int64_t item_cap) {
  const int64_t few = rule == kTileSmall ? kSmallWaves : kPlanWaves;
  const int64_t per = 64 * (rule == kTileSmall ? 4 : kPlanLanes);
  return std::max<int64_t>(std::min<int64_t>((item_cap + 63) / 64, few),
                           (item_cap + per - 1) / per);
}
// Exclusive scan of n per-tile sums. packed: each sum holds two counts below 2^16,
// scanned into pre[2i] (low) and pre[2i+1] (high); else pre[i]. The totals (below 2^31),
// clamped to cap0 / cap1, go to *d_tot0 / *d_tot1. temp: a scan temp
// (scan_temp_bytes(m) with m >= the number of tiles).
int scan_tiles(int n, const int* sums, int* pre, int packed, int64_t cap0, int64_t cap1,
               int* d_tot0, int* d_tot1, void* temp, hipStream_t s);
// the same over the tiles of min(*d_items, item_cap) items
int scan_tiles_dev(const int* d_items, TileRule rule, int64_t item_cap, const int* sums, int* pre,
                   int packed, int64_t cap0, int64_t cap1, int* d_tot0, int* d_tot1, void* temp,
                   hipStream_t s);
size_t radix_sort_temp_bytes(int n);
int radix_sort(uint64_t* keys, uint32_t* vals, int n, int key_bits, void* temp, hipStream_t s);
int radix_sort_clear(void* temp, int n, hipStream_t s);  // before the first sort on a temp
// Stable LSD sort of the first min(*d_n, n_max) 32-bit keys (key_bits <= 32) with
// their values, with a launch shape independent of the count (graph-capturable). The
// result ends in keys_alt / vals_alt when *in_alt is set (an odd number of passes),
// else in keys / vals. hist (radix_sort_dev_temp_bytes()) holds the digit counts of the
// low 8 bits by workgroup, hist[256 * block + digit] over dev_sort_range's keys: the
// kernel that writes the keys counts them.
constexpr int kSortItems = 8;                   // keys per thread per tile
constexpr int kSortTile = kBlock * kSortItems;  // 2048 keys
// 256 workgroups of a few tiles: 1.16 M records of 96 cloths 110 us for the list, as with
// 1,024 and a scan in each pass (128: 124, 512: 121), none to 280,000 records 37 -> 22 (64^2)
// and 52 -> 47 us (draped 256^2).
constexpr int kDevSortBlocks = 256;
struct DevSortRange {
  int n, t0, t1, blocks;  // keys, this workgroup's tiles, workgroups that have any
};
__device__ __forceinline__ DevSortRange dev_sort_range(int n) {
  const int ntiles = (n + kSortTile - 1) / kSortTile;
  const int per = max(1, (ntiles + kDevSortBlocks - 1) / kDevSortBlocks);
  const int t0 = min(ntiles, (int)blockIdx.x * per);
  return {n, t0, min(ntiles, t0 + per), (ntiles + per - 1) / per};
}
size_t radix_sort_dev_temp_bytes();
int radix_sort_dev(uint32_t* keys, uint32_t* vals, uint32_t* keys_alt, uint32_t* vals_alt,
                   int n_max, const int* d_n, int key_bits, int* hist, int* in_alt,
                   hipStream_t s);
int fill_i32(int* p, int v, int64_t n, hipStream_t s);
int fill_u32(uint32_t* p, uint32_t v, int64_t n, hipStream_t s);

// ---- LBVH (k_lbvh.hip) -----------------------------------------------------
// ints per traversal hand-over record (leaf, pairs, depth, node, cap, visits, stack)
constexpr int kTravRec = 72;
// trees of fewer leaves are walked through their quantised nodes (26-bit ids)
constexpr int kQuantLeaves = 1 << 26;
// ints per leaf for the traversal stack entries below its LDS part
constexpr int kTravSpill = 55;

struct LbvhBufs {
  int t = 0;
  float4 *amin = nullptr, *amax = nullptr;  // 2T-1 (internal nodes first)
  int *lefts = nullptr, *rights = nullptr, *parents = nullptr, *rmll = nullptr, *rmlr = nullptr;
  int *claim_cnt = nullptr, *claim_hi = nullptr;  // 2T-1: claimants, highest claimant
  int2* ranges = nullptr;                           // T-1 key ranges
  // refit: per node 1 = finished by its chunk, 0 = deferred (top_index = list slot)
  int *state = nullptr, *top_list = nullptr, *top_index = nullptr, *ntop = nullptr;
  float4 *tmin = nullptr, *tmax = nullptr;  // deferred-node scratch (large trees)
  int *trm = nullptr, *tdone = nullptr;
  bool group = true;        // few leaves may be walked by groups of lanes
  uint4* qnodes = nullptr;  // quantised record of each internal node, 2 uint4 (k_lbvh.hip)
  float4* nodes = nullptr;  // exact records of a caller's irregular tree, 4 float4 a node
  int* irr = nullptr;       // per cloth: from 2 on its tree is walked through its exact boxes
  int trav_chunk = 4;       // traversal: tiles per chunk dealt to one XCD (launch shape only)
  // traversal: visits a leaf makes in the first pass before a wave takes it over (0:
  // one pass); records of kTravRec ints for up to rcap such leaves; hctl[0] their
  // count, zero between substeps (the pair compaction clears it). The pair lists are
  // the same with any budget.
  int trav_budget = 0;
  int* trec = nullptr;
  int rcap = 0;
  int* hctl = nullptr;
  int* spill = nullptr;  // kTravSpill ints per leaf: deep traversal stack entries
  uint32_t* warn = nullptr;
  // batch of cloths (ncloth == 0: one cloth): cloth c owns triangle slots (and, after
  // the sort, leaves) [tstart[c], tstart[c + 1]); its Morton keys carry c above bit 30
  int ncloth = 0;
  const int* tstart = nullptr;      // ncloth + 1
  const int* slot_cloth = nullptr;  // T: cloth of each triangle slot / leaf
  int* croot = nullptr;             // ncloth: internal node spanning the cloth (-1: none)
  const int* ccap = nullptr;        // ncloth: per-leaf pair cap of the cloth
  uint32_t* cbox = nullptr;         // 6 * ncloth: centroid box, order-preserving encoding
};
size_t lbvh_build_temp_bytes(int t);
size_t carve_build(int t, void* d_temp, LbvhBufs* b);  // b == nullptr: size only
size_t lbvh_pairs_temp_bytes(int t, int cap);
int launch_tri_update(int n, int t, const float4* x, const float4* p, const int4* tri, float th,
                      int bits, int normalize, float4* amin, float4* amax, uint64_t* keys,
                      uint32_t* vals, float4* centroid_tmp, float4* box_tmp, hipStream_t s);
// batch: swept AABBs, per-cloth centroid boxes and keys (cloth << 30 | Morton30)
int launch_tri_update_batch(const LbvhBufs& b, const float4* x, const float4* p, const int4* tri,
                            float th, uint64_t* keys, uint32_t* vals, float4* centroid_tmp,
                            hipStream_t s);
// cleared: launch_gather_tris has cleared what the build starts from. tri_from (or null):
// copied to tri_to on the way.
int launch_build(const LbvhBufs& b, const uint64_t* keys, int midpoint, bool cleared,
                 const int4* tri_from, int4* tri_to, hipStream_t s);
int launch_refit(const LbvhBufs& b, hipStream_t s);
// the traversal's node records; from_caller: check the caller's tree first
int launch_pack_nodes(const LbvhBufs& b, bool from_caller, hipStream_t s);
// pairs: traversal into chunk (T * cap ints: the pairs' second leaves) + per-leaf counts,
// then compaction.
int launch_pairs(const LbvhBufs& b, int cap, int* chunk, int* counts, int* offsets,
                 int2* pairs, int* d_npairs, void* scan_temp, hipStream_t s);
// whether groups of lanes walk the tree (k_traverse_group), without tile chunks or a budget
bool walked_by_groups(const LbvhBufs& b, int cap);
// the traversal kernel alone on the current tree (it rewrites the same pair chunk)
int launch_traverse_only(const LbvhBufs& b, int cap, int* chunk, int* counts, int* offsets,
                         hipStream_t s);
int launch_gather_tris(const LbvhBufs& b, const uint32_t* perm, const int4* tri_in, int4* tri_out,
                       int fix_leaves, float4* tmp_min, float4* tmp_max, hipStream_t s);

// ---- narrow phase (k_narrow.hip) ------------------------------------------
// A contact record in vertex order, self-contained for the Jacobi kernel: the
// contact's four vertex ids (bits 29-30 of ids.x hold this record's role, bit 31 is
// set for a VF contact) and the contact weights.
struct alignas(16) RecPayload {
  int4 ids;
  float4 w;
};

struct NarrowBufs {
  int n = 0, t = 0;
  int64_t pair_cap = 0;       // capacity of pairs (T*cap)
  int64_t vf_cap = 0, ee_cap = 0;          // candidate capacities
  int64_t vf_out_cap = 0, ee_out_cap = 0;  // contact (CCD survivor) capacities
  const int2* pairs = nullptr;
  const int* d_npairs = nullptr;
  uint16_t* mask = nullptr;   // per pair
  int* tile_sum = nullptr;  // per tile of pairs / candidates: packed counts
  int* tile_pre = nullptr;  // per tile: exclusive prefixes of the two counts
  int4 *cand_vf = nullptr, *cand_ee = nullptr;
  int *d_ncand_vf = nullptr, *d_ncand_ee = nullptr;
  uint64_t* near_mask = nullptr;  // a bit per candidate (VF then EE): near
  uint8_t* hit_flag = nullptr;    // per near index: hit
  int* near_ids = nullptr;       // candidates passing the box-gap rejection, in order
  int* d_nnear = nullptr;
  // CCD passes, per candidate (VF then EE, vf_cap + ee_cap), written for near
  // candidates only: plan word, critical points, and the secant root of each of its
  // (up to three) intervals
  int* cplan = nullptr;
  float2* ccp = nullptr;
  float* croot = nullptr;  // 3 * (vf_cap + ee_cap)
  int* d_ntotal = nullptr;
  int4 *vf_v = nullptr, *ee_v = nullptr;      // compacted contacts
  float4 *vf_w = nullptr, *vf_tn = nullptr, *ee_w = nullptr, *ee_tn = nullptr;
  int *d_nvf = nullptr, *d_nee = nullptr;
  // per-vertex dynamic record CSR, in solver order (rank: solver position of a vertex,
  // null: its id); the payloads' vertex ids are solver positions too
  const int* rank = nullptr;
  int *dcount = nullptr, *dprefix = nullptr;  // n + 1 each
  uint32_t* drec = nullptr;  // 4 * (vf_out_cap + ee_out_cap)
  uint32_t* dtmp = nullptr;  // same size: staging for very long record lists
  // same size: record payloads in drec order; between the solver's last read and
  // k_rec_place it holds the CCD hits' weights, time and normal per near index
  RecPayload* rec = nullptr;
  int* dlong = nullptr;      // n: vertices whose record lists are ordered by a workgroup
  // sorted_csr: the CSR comes from one radix sort of the records by vertex id
  // (else from per-vertex counts and atomic placement). skey: record keys then
  // alternate keys (2 * 4 * (vf_out_cap + ee_out_cap)), sort_hist:
  // radix_sort_dev_temp_bytes()
  bool sorted_csr = false;
  uint32_t* skey = nullptr;
  int* sort_hist = nullptr;
  int* d_nrec = nullptr;     // records of the substep (sorted CSR)
  uint32_t* warn = nullptr;
  void* scan_temp = nullptr;
};
// dcd: one proximity test per candidate at x instead of the CCD (CM_F_DCD)
// the CCD plan pass alone over the current candidate lists (kernel timing)
int launch_ccd_plan_only(const NarrowBufs& nb, const float4* x, const float4* v, float th,
                         float dt, int dcd, hipStream_t s);
int launch_narrow(const NarrowBufs& nb, const int4* tri, const float4* x, const float4* p,
                  const float4* v, float th, float dt, int ee_on, int dcd, hipStream_t s);
int launch_dynamic_csr(const NarrowBufs& nb, hipStream_t s);

// ---- PBD (k_pbd.hip) -------------------------------------------------------
// Jacobi tiles: the solver numbers the vertices in an order of its own (order[k] =
// vertex at solver position k, rank = its inverse) in which a tile is a run of
// consecutive positions: a patch of at most tile_v vertices that holds at most
// kTileSlots constraint slots. A tile lists the constraints touching it once, distance
// and bend apart, in tile-local vertex numbers: its own vertices first, then its halo
// (the other vertices of its constraints), whose solver positions are listed.
constexpr int kTileSlots = 3072;
// patches of neighbouring vertices a tile is made of when tiles are few: contacts
// gather in a few regions, and a tile of several small patches from all over the
// cloth holds about as many as any other
constexpr int kSubPatch = 32;
struct TileBufs {
  int n = 0;  // 0: no tiles (a vertex has more slots than a tile holds)
  int n_mem = 0;  // the last of them: halo too large for the LDS
  int threads = 256;                 // of a workgroup (256 or 512)
  int max_local = 0, lds_slots = 0;  // LDS per workgroup: positions and slots
  int* order = nullptr;   // n vertices (null: solver numbering = vertex ids)
  int* rank = nullptr;
  int* prefix = nullptr;  // n + 1: constraint slots before each solver position
  int4* hdr = nullptr;    // 2 per tile: {v0, nv, halo0, nhalo}, {s0, ns, b0, nb}
  int* halo = nullptr;    // solver positions
  // distance entries {id0 | id1 << 16, slot0 | slot1 << 16, l0, kp}; bend entries
  // {id0 | id1 << 16, id2 | id3 << 16, slot0 | slot1 << 16, slot2 | slot3 << 16} with
  // {kp, phi0}; tile-local ids and slots, slot 0xffff = not a vertex of the tile
  uint4 *sent = nullptr, *bent = nullptr;
  float2* bpar = nullptr;
  int *scid = nullptr, *bcid = nullptr;  // constraint of each entry
  int nsent = 0, nbent = 0;
};

struct PbdBufs {
  // collision sphere, centre and radius: in memory, so that moving it leaves the captured
  // substep as it is
  const float4* sphere = nullptr;
  int n = 0, S = 0, B = 0, F = 0;
  float4 *x = nullptr, *p = nullptr, *v = nullptr;  // .w of x/p = inverse mass
  float4 *q0 = nullptr, *q1 = nullptr;  // the solver's iterates, in solver order
  const uint8_t* pinned = nullptr;
  const int2* sid = nullptr;
  const float2* s_l0kp = nullptr;
  const int4* bid = nullptr;
  const float2* b_kpphi0 = nullptr;
  const int* vprefix = nullptr;
  const uint32_t* vslot = nullptr;
  TileBufs tl;
  const int* lra_fixed = nullptr;
  const float* lra_l0 = nullptr;
  uint8_t* lra_flag = nullptr;
  float4* ground = nullptr;  // qc.xyz, flag
  const float* mass = nullptr;
  float* damp_partials = nullptr;  // per block sums
  float* damp_state = nullptr;     // omega, xcm, vcm
};
struct PbdParams {
  float dt, th, gh;
  f3 g;
  int iters;
  uint32_t flags, ref_compat;
  f3 wmin, wmax;
  float kg, kd, kf;
};
int launch_predict(const PbdBufs& b, const PbdParams& pp, hipStream_t s);
int launch_set_sphere(float4* sphere, float4 value, hipStream_t s);
int launch_solver(const PbdBufs& b, const PbdParams& pp, const NarrowBufs& nb, hipStream_t s);
// the Jacobi iterations alone, and their result to p
int launch_solve_only(const PbdBufs& b, const PbdParams& pp, const NarrowBufs& nb, int iters,
                      hipStream_t s);
int launch_solve_result(const PbdBufs& b, int iters, hipStream_t s);
int launch_integrate(const PbdBufs& b, const PbdParams& pp, hipStream_t s);
// kp of every tile entry from the per-constraint parameters
int launch_tile_stiffness(const PbdBufs& b, hipStream_t s);
// LDS that the tiled kernels take (host check at tile building)
size_t tile_lds_bytes(int max_local, int lds_slots, bool adjoint);
int tile_lds_allow(size_t bytes);
int launch_integrate_from(const PbdBufs& b, const PbdParams& pp, const float4* pfin,
                          hipStream_t s);
int launch_friction(const PbdBufs& b, const PbdParams& pp, const NarrowBufs& nb, hipStream_t s);
int launch_revert_toc(const PbdBufs& b, const NarrowBufs& nb, hipStream_t s);
int launch_vertex_normals(int n, const int* vt_prefix, const int4* vt_tri, const float4* pos,
                          float4* nrm, int carry, int unit, hipStream_t s);
// the solver stage with every iterate kept, in solver order: pk[k * n, (k + 1) * n) =
// positions entering iteration k, pk[iters * n ...) the result
int launch_solver_rec(const PbdBufs& b, const PbdParams& pp, const NarrowBufs& nb, float4* pk,
                      hipStream_t s);

// ---- adjoint (k_pbd.hip) ---------------------------------------------------
struct AdjBufs {
  float4 *lx = nullptr, *lv = nullptr;  // dL/dx, dL/dv (n)
  float4 *lp = nullptr, *la = nullptr;  // dL/dp of the iterates (n each, alternating; solver order)
  int* cnt = nullptr;  // Jacobi count per iteration and vertex (iters * n), solver order
  double *gks = nullptr, *gkb = nullptr;  // dL/dkp per distance / bend constraint
};
// The contact set of substep `slot`: the per-vertex records (dprefix[n] of them) are
// appended to arena; ctl[0] = records used, ctl[1] = overflow, ctl[2 + slot] = first.
int launch_tape_records(int n, const int* dprefix, const RecPayload* rec, RecPayload* arena,
                        int64_t cap, int* ctl, int slot, hipStream_t s);
// One substep backwards: (lx, lv) = dL/d(x, v) after the substep in, before it out;
// dL/dkp added to gks / gkb. pk: the substep's iterates (launch_solver_rec);
// dprefix / rec: its contact records (null: none).
int launch_adj_substep(const PbdBufs& b, const PbdParams& pp, const AdjBufs& ab, const float4* pk,
                       const int* dprefix, const RecPayload* rec, hipStream_t s);

}  // namespace cm

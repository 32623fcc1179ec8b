// Morton/LBVH stages of the substep as gfx950 kernels.
//
//  k_tri_update   <- DeformableUtils::_UpdateTrianglesContinuous
//                    (LicentaV2/LicentaV2/Physics/CudaDeformableUtils.cu:120-151)
//  k_build        <- CudaBVH::_GenerateBVH2 / FindRange / FindSplit
//                    (Collision/CudaBVH.cu:163-242), Delta/sgn (Core/CudaUtils.cu:338-362)
//  k_refit_local,
//  k_refit_top    <- CudaBVH::ComputeTreeAABBs (Collision/CudaBVH.cu:128-149)
//  k_traverse     <- CudaBVH::_GetAABBCollisions (Collision/CudaBVH.cu:23-113)
//
// Layout: node AABBs are float4 min / float4 max arrays of 2T-1 entries, internal
// nodes [0, T-1) then leaves [T-1, 2T-1), as in the reference. Parent writes are
// made deterministic with claim records (count, highest claimant): parents[c] =
// highest claimant, which is what the reference's last writer in thread order
// produces. The refit pulls each node from its two children, so a node shared by
// several parents (midpoint split on tied codes) is still the union of its two
// children.
#include "cm_internal.hpp"

#include <algorithm>
#include <climits>

namespace cm {

namespace {

// ---- per-triangle swept AABB and Morton key --------------------------------
__device__ __forceinline__ void swept_aabb(const float4* __restrict__ x,
                                           const float4* __restrict__ p, int4 tr, float th,
                                           f3& smn, f3& smx) {
  const f3 p1 = xyz(p[tr.x]), p2 = xyz(p[tr.y]), p3 = xyz(p[tr.z]);
  const f3 q1 = xyz(x[tr.x]), q2 = xyz(x[tr.y]), q3 = xyz(x[tr.z]);
  const f3 mn = subs(min3(p1, p2, p3), th), mx = adds(max3(p1, p2, p3), th);
  const f3 pmn = subs(min3(q1, q2, q3), th), pmx = adds(max3(q1, q2, q3), th);
  smn = vmin(mn, pmn);
  smx = vmax(mx, pmx);
}

__global__ void __launch_bounds__(kBlock) k_tri_update(
    int t, const float4* __restrict__ x, const float4* __restrict__ p,
    const int4* __restrict__ tri, float th, int bits, float4* __restrict__ amin,
    float4* __restrict__ amax, uint64_t* __restrict__ keys, uint32_t* __restrict__ vals,
    float4* __restrict__ centroid, float4* __restrict__ box_partials) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  f3 c = mk3(0, 0, 0);
  bool valid = i < t;
  if (valid) {
    f3 smn, smx;
    swept_aabb(x, p, tri[i], th, smn, smx);
    amin[t - 1 + i] = f4(smn, 0.f);
    amax[t - 1 + i] = f4(smx, 0.f);
    c = add(smn, divs(sub(smx, smn), 2.f));
    if (vals) vals[i] = (uint32_t)i;
    if (centroid) {
      centroid[i] = f4(c, 0.f);
    } else if (bits == 30) {
      keys[i] = morton30(c, mk3(0, 0, 0), mk3(1, 1, 1));
    } else {
      keys[i] = morton63(c);
    }
  }
  if (box_partials) {  // block min/max of the centroids (exact)
    __shared__ float smin[3][kBlock], smax[3][kBlock];
    const float inf = __builtin_huge_valf();
    smin[0][threadIdx.x] = valid ? c.x : inf;
    smin[1][threadIdx.x] = valid ? c.y : inf;
    smin[2][threadIdx.x] = valid ? c.z : inf;
    smax[0][threadIdx.x] = valid ? c.x : -inf;
    smax[1][threadIdx.x] = valid ? c.y : -inf;
    smax[2][threadIdx.x] = valid ? c.z : -inf;
    __syncthreads();
    for (int s = kBlock / 2; s >= 1; s >>= 1) {
      if (threadIdx.x < s)
        for (int a = 0; a < 3; ++a) {
          smin[a][threadIdx.x] = fminf(smin[a][threadIdx.x], smin[a][threadIdx.x + s]);
          smax[a][threadIdx.x] = fmaxf(smax[a][threadIdx.x], smax[a][threadIdx.x + s]);
        }
      __syncthreads();
    }
    if (threadIdx.x == 0) {
      box_partials[2 * blockIdx.x] = make_float4(smin[0][0], smin[1][0], smin[2][0], 0.f);
      box_partials[2 * blockIdx.x + 1] = make_float4(smax[0][0], smax[1][0], smax[2][0], 0.f);
    }
  }
}

// The box of nb block boxes (min, max in turn), in every thread of the workgroup.
__device__ __forceinline__ void box_of(const float4* __restrict__ box, int nb, f3& lo, f3& hi) {
  __shared__ float smin[3][kBlock], smax[3][kBlock];
  const float inf = __builtin_huge_valf();
  float mn[3] = {inf, inf, inf}, mx[3] = {-inf, -inf, -inf};
  for (int b = threadIdx.x; b < nb; b += kBlock) {
    float4 a = box[2 * b], c = box[2 * b + 1];
    mn[0] = fminf(mn[0], a.x); mn[1] = fminf(mn[1], a.y); mn[2] = fminf(mn[2], a.z);
    mx[0] = fmaxf(mx[0], c.x); mx[1] = fmaxf(mx[1], c.y); mx[2] = fmaxf(mx[2], c.z);
  }
  for (int a = 0; a < 3; ++a) {
    smin[a][threadIdx.x] = mn[a];
    smax[a][threadIdx.x] = mx[a];
  }
  __syncthreads();
  for (int s = kBlock / 2; s >= 1; s >>= 1) {
    if (threadIdx.x < s)
      for (int a = 0; a < 3; ++a) {
        smin[a][threadIdx.x] = fminf(smin[a][threadIdx.x], smin[a][threadIdx.x + s]);
        smax[a][threadIdx.x] = fmaxf(smax[a][threadIdx.x], smax[a][threadIdx.x + s]);
      }
    __syncthreads();
  }
  lo = mk3(smin[0][0], smin[1][0], smin[2][0]);
  hi = mk3(smax[0][0], smax[1][0], smax[2][0]);
}

// single block: reduce the per-block boxes; result in box[2*nb], box[2*nb+1]
__global__ void __launch_bounds__(kBlock) k_box_reduce(float4* __restrict__ box, int nb) {
  f3 lo, hi;
  box_of(box, nb, lo, hi);
  if (threadIdx.x == 0) {
    box[2 * nb] = make_float4(lo.x, lo.y, lo.z, 0.f);
    box[2 * nb + 1] = make_float4(hi.x, hi.y, hi.z, 0.f);
  }
}

// kReduce: every workgroup reduces the block boxes itself, which up to kFewBoxes of them
// (16 KB from the L2) costs it less than k_box_reduce's launch of 3 to 4.5 us.
constexpr int kFewBoxes = 512;
template <bool kReduce>
__global__ void __launch_bounds__(kBlock) k_keys30(int t, const float4* __restrict__ centroid,
                                                   const float4* __restrict__ box, int nb,
                                                   uint64_t* __restrict__ keys) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  f3 lo, hi;
  if (kReduce) {
    box_of(box, nb, lo, hi);
  } else {
    lo = xyz(box[2 * nb]);
    hi = xyz(box[2 * nb + 1]);
  }
  if (i < t) keys[i] = morton30(xyz(centroid[i]), lo, hi);
}

// ---- per-cloth centroid boxes of a batch -------------------------------------------
// Floats are mapped to unsigned integers of the same order, so the box is a pair of
// integer atomic min/max per axis: exact, and independent of the order of arrival.
__device__ __forceinline__ uint32_t ford(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float funord(uint32_t e) {
  return __uint_as_float((e & 0x80000000u) ? (e & 0x7fffffffu) : ~e);
}

__global__ void __launch_bounds__(kBlock) k_cloth_box_init(int ncloth, uint32_t* __restrict__ cbox) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < 6 * ncloth) cbox[i] = (i % 6) < 3 ? 0xffffffffu : 0u;  // min xyz, max xyz
}

__device__ __forceinline__ uint32_t wave_min_u(uint32_t v) {
  for (int o = 32; o >= 1; o >>= 1) v = min(v, (uint32_t)__shfl_xor((int)v, o, 64));
  return v;
}
__device__ __forceinline__ uint32_t wave_max_u(uint32_t v) {
  for (int o = 32; o >= 1; o >>= 1) v = max(v, (uint32_t)__shfl_xor((int)v, o, 64));
  return v;
}

// Centroid box of each cloth.
// A wave takes kBoxRun chunks of 64 consecutive slots and keeps one cloth's box in its lanes
// until the cloth changes, then adds it to the cloth's with 6 atomics: they all go to a few
// cache lines and bound the pass (6 for each 64 slots, 6 for each slot of a chunk with two
// cloths: 108 us for 96 cloths of 938 k triangles, now 18). A chunk of more than kBoxCloths
// cloths, tiny ones, goes by one atomic a bound and slot.
constexpr int kBoxRun = 16, kBoxCloths = 4;
__global__ void __launch_bounds__(kBlock) k_cloth_box(int t, const float4* __restrict__ cen,
                                                      const int* __restrict__ slot_cloth,
                                                      uint32_t* __restrict__ cbox) {
  const int lane = threadIdx.x & 63;
  const int64_t base = ((int64_t)blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6)) * 64 * kBoxRun;
  int cur = -1;  // the cloth whose box e holds
  uint32_t e[6];
  auto flush = [&] {
    if (cur >= 0) {
#pragma unroll
      for (int a = 0; a < 6; ++a) e[a] = a < 3 ? wave_min_u(e[a]) : wave_max_u(e[a]);
      if (lane == 0)
        for (int a = 0; a < 6; ++a)
          if (a < 3) atomicMin(&cbox[6 * cur + a], e[a]); else atomicMax(&cbox[6 * cur + a], e[a]);
    }
#pragma unroll
    for (int a = 0; a < 6; ++a) e[a] = a < 3 ? 0xffffffffu : 0u;
  };
  for (int j = 0; j < kBoxRun && base + j * 64 < t; ++j) {
    const int64_t i = base + j * 64 + lane;
    const bool valid = i < t;
    const int c = valid ? slot_cloth[i] : -1;
    const f3 p = valid ? xyz(cen[i]) : mk3(0, 0, 0);
    const uint32_t o[3] = {ford(p.x), ford(p.y), ford(p.z)};
    uint64_t left = __ballot(valid);
    const int before = __shfl_up(c, 1, 64);
    if (__popcll(__ballot(valid && lane > 0 && c != before)) >= kBoxCloths) {
      if (valid)
        for (int a = 0; a < 3; ++a) {
          atomicMin(&cbox[6 * c + a], o[a]);
          atomicMax(&cbox[6 * c + 3 + a], o[a]);
        }
      continue;
    }
    while (left) {  // once for each cloth of the chunk
      const int cc = __shfl(c, __ffsll((long long)left) - 1, 64);
      if (cc != cur) {
        flush();
        cur = cc;
      }
      const bool mine = c == cc;
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        e[a] = min(e[a], mine ? o[a] : 0xffffffffu);
        e[3 + a] = max(e[3 + a], mine ? o[a] : 0u);
      }
      left &= ~__ballot(mine);
    }
  }
  flush();
}

__global__ void __launch_bounds__(kBlock) k_keys30_cloth(int t, const float4* __restrict__ cen,
                                                         const int* __restrict__ slot_cloth,
                                                         const uint32_t* __restrict__ cbox,
                                                         uint64_t* __restrict__ keys) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= t) return;
  const int c = slot_cloth[i];
  const uint32_t* bx = cbox + 6 * c;
  const f3 lo = mk3(funord(bx[0]), funord(bx[1]), funord(bx[2]));
  const f3 hi = mk3(funord(bx[3]), funord(bx[4]), funord(bx[5]));
  keys[i] = ((uint64_t)c << 30) | morton30(xyz(cen[i]), lo, hi);
}

// ---- Karras build -----------------------------------------------------------
// Core/CudaUtils.cu:338-351. In a batch, equal keys belong to one cloth and the
// index tie-break uses cloth-local indices, so each cloth's subtree is the tree its
// own keys would build.
__device__ __forceinline__ int delta(const uint64_t* __restrict__ k, int i, int j, int maxj,
                                     const int* __restrict__ tstart) {
  if (j < 0 || j > maxj) return -1;
  const uint64_t x = k[i] ^ k[j];
  if (x) return clz64(x);
  const int base = tstart ? tstart[(int)(k[i] >> 30)] : 0;
  return clz64((uint64_t)(i - base) ^ (uint64_t)(j - base)) + 64;
}
__device__ __forceinline__ int sgn(int a) { return signbit((float)a) ? -1 : 1; }

// What the build and the refit start from; thread i of at least max(2t - 1, ncloth).
struct BuildInit {
  int t;
  int *cnt, *hi, *ntop, *irr;
  int ncloth;
  int* croot;
};
__device__ __forceinline__ void build_init(const BuildInit& b, int i) {
  if (i < 2 * b.t - 1) {
    b.cnt[i] = 0;
    b.hi[i] = -1;
  }
  if (i < b.ncloth) b.croot[i] = -1;
  if (i < max(b.ncloth, 1)) b.irr[i] = 0;
  if (i == 0) *b.ntop = 0;  // deferred-node count of the refit
}
__global__ void __launch_bounds__(kBlock) k_build_init(BuildInit b) {
  build_init(b, blockIdx.x * kBlock + threadIdx.x);
}

__global__ void __launch_bounds__(kBlock) k_build(int t, const uint64_t* __restrict__ k,
                                                  int midpoint, int* __restrict__ lefts,
                                                  int* __restrict__ rights, int* __restrict__ cnt,
                                                  int* __restrict__ hi, int2* __restrict__ ranges,
                                                  uint32_t* __restrict__ warn,
                                                  const int* __restrict__ tstart,
                                                  int* __restrict__ croot) {
  const int id = blockIdx.x * kBlock + threadIdx.x;
  const int nin = t - 1;
  if (id >= nin) return;
  // range (Collision/CudaBVH.cu:190-212)
  const int d = sgn(delta(k, id, id + 1, nin, tstart) - delta(k, id, id - 1, nin, tstart));
  const int dmin = delta(k, id, id - d, nin, tstart);
  int lmax = 2;
  while (delta(k, id, id + lmax * d, nin, tstart) > dmin) lmax <<= 1;
  int l = 0;
  for (int s = lmax / 2; s >= 1; s /= 2)
    if (delta(k, id, id + (l + s) * d, nin, tstart) > dmin) l += s;
  const int j = id + l * d;
  const int first = min(id, j), last = max(id, j);
  ranges[id] = make_int2(first, last);
  if (tstart) {  // the node spanning exactly one cloth is that cloth's root
    const int c = (int)(k[first] >> 30);
    if (first == tstart[c] && last == tstart[c + 1] - 1) croot[c] = id;
  }
  // split (Collision/CudaBVH.cu:214-242)
  const uint64_t fc = k[first], lc = k[last];
  int split;
  if (midpoint && fc == lc) {
    split = (first + last) >> 1;
  } else {
    const int com = midpoint ? clz64(fc ^ lc) : delta(k, first, last, nin, tstart);
    split = first;
    int step = last - first;
    do {
      step = (step + 1) >> 1;
      const int ns = split + step;
      if (ns < last) {
        const int pref = midpoint ? clz64(fc ^ k[ns]) : delta(k, first, ns, nin, tstart);
        if (pref > com) split = ns;
      }
    } while (step > 1);
  }
  const int left = split == first ? nin + split : split;
  const int right = split + 1 == last ? nin + split + 1 : split + 1;
  lefts[id] = left;
  rights[id] = right;
  const int o1 = atomicAdd(&cnt[left], 1);
  atomicMax(&hi[left], id);
  const int o2 = atomicAdd(&cnt[right], 1);
  atomicMax(&hi[right], id);
  if (o1 > 0 || o2 > 0) atomicOr(warn, (uint32_t)CM_WARN_BROKEN_TREE);
}

__global__ void __launch_bounds__(kBlock) k_parents(int t, const int* __restrict__ cnt,
                                                    const int* __restrict__ hi,
                                                    int* __restrict__ parents,
                                                    const int4* __restrict__ tri_from,
                                                    int4* __restrict__ tri_to) {
  const int c = blockIdx.x * kBlock + threadIdx.x;
  if (tri_from && c < t) tri_to[c] = tri_from[c];
  if (c >= 2 * t - 1) return;
  if (cnt[c] > 0) parents[c] = hi[c];
}

// ---- bottom-up refit ------------------------------------------------------------
constexpr int kRefitCH = 1024;  // leaves (and node ids) per refit workgroup
constexpr int kTopCap = 2048;   // deferred nodes the top pass keeps in LDS
constexpr int kTopList = 8192;  // pending deferred nodes the top pass lists in LDS
constexpr int kIrregular = 2;   // irr from which on a tree is walked through its exact boxes

// Whether any thread changed something in this pass (1, 2, ...), for all threads, with the
// one barrier that a pass needs anyway: three flags in turn, the next one cleared while this
// one is set (f[0..2] start at 0). __syncthreads_or takes about 1,200 cycles on 1,024
// threads, and a refit makes 14 to 27 passes: 64^2 local pass 15.7 -> 12.6 us, top pass
// 14.4 -> 11.1, draped 131x97 19.5 -> 15.0 and 20.7 -> 16.4, 2 M leaves 168 -> 161 and
// 90 -> 82 (the rest of a pass is its chain of LDS reads).
__device__ __forceinline__ bool any_changed(int* f, int pass, bool changed) {
  if (changed) f[pass % 3] = 1;
  if (threadIdx.x == 0) f[(pass + 1) % 3] = 0;
  __syncthreads();
  return f[pass % 3] != 0;
}

// Refit, pass 1: one workgroup per chunk of 1024 consecutive leaves. Internal node
// q belongs to the chunk holding index q (a Karras node's index lies in its key
// range). Nodes whose range lies inside the chunk are finished here: in each
// synchronised pass a node whose children are leaves of the chunk or nodes finished
// in an earlier pass takes the union of its children (Collision/CudaBVH.cu:140-144),
// all in LDS. Every other node of the chunk (its range crosses the chunk, or a child
// is unfinished) is appended to the deferred list for k_refit_top. A node is the
// union of its two children however many parents claimed it.
__global__ void __launch_bounds__(kRefitCH) k_refit_local(
    int t, const int* __restrict__ lefts, const int* __restrict__ rights,
    const int2* __restrict__ ranges, float4* __restrict__ amin, float4* __restrict__ amax,
    int* __restrict__ rmll, int* __restrict__ rmlr, int* __restrict__ state, int* __restrict__ top_list, int* __restrict__ top_index,
    int* __restrict__ ntop, int* __restrict__ gdone) {
  __shared__ float4 lmin[kRefitCH], lmax[kRefitCH];  // leaf boxes of the chunk
  __shared__ float4 nmin[kRefitCH], nmax[kRefitCH];  // node boxes of the chunk
  __shared__ int nrm[kRefitCH];                      // max(rmll, rmlr) of each node
  __shared__ int ndone[kRefitCH];                    // pass that finished the node, 0 = not
  __shared__ int flag[3];
  const int nin = t - 1, base = blockIdx.x * kRefitCH, tid = threadIdx.x;
  if (base + tid < t) {
    lmin[tid] = amin[nin + base + tid];
    lmax[tid] = amax[nin + base + tid];
  }
  const int q = base + tid;
  int l = 0, r = 0;
  bool pending = false;
  if (q < nin) {
    const int2 rg = ranges[q];
    if (rg.x >= base && rg.y < base + kRefitCH) {
      l = lefts[q];
      r = rights[q];
      // children must be leaves or nodes of this chunk
      const int lo = l >= nin ? l - nin : l, ro = r >= nin ? r - nin : r;
      pending = lo >= base && lo < base + kRefitCH && ro >= base && ro < base + kRefitCH;
    }
  }
  ndone[tid] = 0;
  if (tid < 3) flag[tid] = 0;
  __syncthreads();
  bool fin = false;
  f3 lmn = mk3(0, 0, 0), lmx = lmn, rmn = lmn, rmx = lmn;
  int a = 0, b = 0;
  for (int pass = 1;; ++pass) {
    bool changed = false;
    if (pending) {
      const bool rl = l >= nin || (ndone[l - base] != 0 && ndone[l - base] < pass);
      const bool rr = r >= nin || (ndone[r - base] != 0 && ndone[r - base] < pass);
      if (rl && rr) {
        if (l >= nin) {
          lmn = xyz(lmin[l - nin - base]); lmx = xyz(lmax[l - nin - base]); a = l;
        } else {
          lmn = xyz(nmin[l - base]); lmx = xyz(nmax[l - base]); a = nrm[l - base];
        }
        if (r >= nin) {
          rmn = xyz(lmin[r - nin - base]); rmx = xyz(lmax[r - nin - base]); b = r;
        } else {
          rmn = xyz(nmin[r - base]); rmx = xyz(nmax[r - base]); b = nrm[r - base];
        }
        nmin[tid] = f4(vmin(lmn, rmn), 0.f);
        nmax[tid] = f4(vmax(lmx, rmx), 0.f);
        nrm[tid] = max(a, b);
        ndone[tid] = pass;
        pending = false;
        fin = true;
        changed = true;
      }
    }
    if (!any_changed(flag, pass, changed)) break;
  }
  if (q >= nin) return;
  if (fin) {
    amin[q] = nmin[tid];
    amax[q] = nmax[tid];
    rmll[q] = a;
    rmlr[q] = b;
    state[q] = 1;
  } else {
    state[q] = 0;
    const int j = atomicAdd(ntop, 1);
    top_list[j] = q;
    top_index[q] = j;
    gdone[j] = 0;  // pending for the later passes
  }
}

// child c of a deferred node: a leaf or a node finished by k_refit_local is final
// in global memory (kind 0); otherwise it is deferred node top_index[c] (kind 1)
__device__ __forceinline__ void top_child(int c, int nin, const int* __restrict__ state,
                                          const int* __restrict__ top_index,
                                          const float4* __restrict__ amin,
                                          const float4* __restrict__ amax,
                                          const int* __restrict__ rmll,
                                          const int* __restrict__ rmlr, bool& deferred,
                                          int& ref, f3& mn, f3& mx) {
  deferred = c < nin && state[c] == 0;
  if (deferred) {
    ref = top_index[c];
  } else {
    mn = xyz(amin[c]);
    mx = xyz(amax[c]);
    ref = c >= nin ? c : max(rmll[c], rmlr[c]);
  }
}

// a finished deferred node j (node qq): its box and rightmost leaf in the deferred
// scratch (for its parent) and in the tree
__device__ __forceinline__ void put_deferred(int j, int qq, int a, int b, f3 lmn, f3 lmx,
                                             f3 rmn, f3 rmx, float4* __restrict__ gmin,
                                             float4* __restrict__ gmax, int* __restrict__ grm,
                                             float4* __restrict__ amin, float4* __restrict__ amax,
                                             int* __restrict__ rmll, int* __restrict__ rmlr) {
  gmin[j] = f4(vmin(lmn, rmn), 0.f);
  gmax[j] = f4(vmax(lmx, rmx), 0.f);
  grm[j] = max(a, b);
  amin[qq] = gmin[j];
  amax[qq] = gmax[j];
  rmll[qq] = a;
  rmlr[qq] = b;
}

constexpr int kSuper = 64 * kRefitCH;  // leaves per workgroup of the middle pass
constexpr int kMidCap = 8192;          // deferred nodes one middle workgroup holds

// Refit, middle pass (large trees: more deferred nodes than the top pass holds in
// LDS): one workgroup per range of kSuper leaves finishes the deferred nodes whose
// key range lies inside it, with the synchronised passes of k_refit_local over the
// deferred scratch. A deferred child outside the range (possible only in a broken
// tree) leaves its parent to the top pass. Finished nodes are marked gdone = -pass;
// the top pass treats them as finished before its first pass.
__global__ void __launch_bounds__(1024) k_refit_mid(
    int t, const int* __restrict__ lefts, const int* __restrict__ rights,
    const int2* __restrict__ ranges, float4* __restrict__ amin, float4* __restrict__ amax,
    int* __restrict__ rmll, int* __restrict__ rmlr, const int* __restrict__ state, const int* __restrict__ top_list,
    const int* __restrict__ top_index, const int* __restrict__ ntop, float4* __restrict__ gmin,
    float4* __restrict__ gmax, int* __restrict__ grm, int* __restrict__ gdone) {
  __shared__ int own[kMidCap];
  __shared__ int nown, flag[3];
  const int nin = t - 1, tid = threadIdx.x;
  const int nt = *ntop;
  if (nt <= kTopCap) return;  // the top pass keeps a short list in LDS
  const int sbase = blockIdx.x * kSuper, send = sbase + kSuper;
  if (tid == 0) nown = 0;
  if (tid < 3) flag[tid] = 0;
  __syncthreads();
  for (int j = tid; j < nt; j += 1024) {
    const int2 rg = ranges[top_list[j]];
    if (rg.x >= sbase && rg.y < send) {
      const int k = atomicAdd(&nown, 1);
      if (k < kMidCap) own[k] = j;
    }
  }
  __syncthreads();
  const int no = nown;
  if (no > kMidCap) return;  // too many: all of them are left to the top pass
  auto inside = [&](int c) {
    const int2 rg = ranges[c];
    return rg.x >= sbase && rg.y < send;
  };
  for (int pass = 1;; ++pass) {
    bool changed = false;
    for (int k = tid; k < no; k += 1024) {
      const int j = own[k];
      if (gdone[j] != 0) continue;
      const int qq = top_list[j], ll = lefts[qq], rr = rights[qq];
      bool lt, rt;
      int a, b;
      f3 lmn, lmx, rmn, rmx;
      top_child(ll, nin, state, top_index, amin, amax, rmll, rmlr, lt, a, lmn, lmx);
      top_child(rr, nin, state, top_index, amin, amax, rmll, rmlr, rt, b, rmn, rmx);
      if (lt && !(inside(ll) && gdone[a] < 0 && -gdone[a] < pass)) continue;
      if (rt && !(inside(rr) && gdone[b] < 0 && -gdone[b] < pass)) continue;
      if (lt) { lmn = xyz(gmin[a]); lmx = xyz(gmax[a]); a = grm[a]; }
      if (rt) { rmn = xyz(gmin[b]); rmx = xyz(gmax[b]); b = grm[b]; }
      put_deferred(j, qq, a, b, lmn, lmx, rmn, rmx, gmin, gmax, grm, amin, amax, rmll,
                   rmlr);
      __threadfence_block();
      gdone[j] = -pass;
      changed = true;
    }
    if (!any_changed(flag, pass, changed)) break;
  }
}

// Refit, pass 2: one workgroup finishes the deferred nodes with the same
// synchronised passes. Up to kTopCap deferred nodes keep their boxes in LDS and
// their children in registers (two per thread); beyond that the boxes live in
// global scratch and node data is re-read each pass. Clears the list count.
__global__ void __launch_bounds__(1024) k_refit_top(
    int t, const int* __restrict__ lefts, const int* __restrict__ rights,
    float4* __restrict__ amin, float4* __restrict__ amax, int* __restrict__ rmll,
    int* __restrict__ rmlr, const int* __restrict__ state,
    const int* __restrict__ top_list, const int* __restrict__ top_index, int* __restrict__ ntop,
    float4* __restrict__ gmin, float4* __restrict__ gmax, int* __restrict__ grm,
    int* __restrict__ gdone, uint32_t* __restrict__ warn, int* __restrict__ irr, int ncloth) {
  __shared__ float4 smin[kTopCap], smax[kTopCap];
  __shared__ int srm[kTopCap], sdone[kTopCap];
  __shared__ int plist[kTopList];
  __shared__ int npend, flag[3];
  const int nin = t - 1, tid = threadIdx.x;
  const int nt = *ntop;
  bool left_over = false;
  if (tid < 3) flag[tid] = 0;  // a barrier follows on either way
  if (nt <= kTopCap) {
    constexpr int kPer = kTopCap / 1024;
    int q[kPer], l[kPer], r[kPer], la[kPer], ra[kPer];
    bool own[kPer], ltop[kPer], rtop[kPer];
    f3 lmn[kPer], lmx[kPer], rmn[kPer], rmx[kPer];
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int j = tid + k * 1024;
      own[k] = j < nt;
      if (own[k]) {
        q[k] = top_list[j];
        l[k] = lefts[q[k]];
        r[k] = rights[q[k]];
        top_child(l[k], nin, state, top_index, amin, amax, rmll, rmlr, ltop[k], la[k], lmn[k],
                  lmx[k]);
        top_child(r[k], nin, state, top_index, amin, amax, rmll, rmlr, rtop[k], ra[k], rmn[k],
                  rmx[k]);
        sdone[j] = 0;
      }
    }
    __syncthreads();
    for (int pass = 1;; ++pass) {
      bool changed = false;
#pragma unroll
      for (int k = 0; k < kPer; ++k) {
        const int j = tid + k * 1024;
        if (!own[k] || sdone[j] != 0) continue;
        const bool rl = !ltop[k] || (sdone[la[k]] != 0 && sdone[la[k]] < pass);
        const bool rr = !rtop[k] || (sdone[ra[k]] != 0 && sdone[ra[k]] < pass);
        if (!(rl && rr)) continue;
        if (ltop[k]) {
          const int c = la[k];
          lmn[k] = xyz(smin[c]); lmx[k] = xyz(smax[c]); la[k] = srm[c];
        }
        if (rtop[k]) {
          const int c = ra[k];
          rmn[k] = xyz(smin[c]); rmx[k] = xyz(smax[c]); ra[k] = srm[c];
        }
        smin[j] = f4(vmin(lmn[k], rmn[k]), 0.f);
        smax[j] = f4(vmax(lmx[k], rmx[k]), 0.f);
        srm[j] = max(la[k], ra[k]);
        sdone[j] = pass;
        changed = true;
      }
      if (!any_changed(flag, pass, changed)) break;
    }
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int j = tid + k * 1024;
      if (!own[k]) continue;
      if (sdone[j] == 0) {
        left_over = true;
        continue;
      }
      amin[q[k]] = smin[j];
      amax[q[k]] = smax[j];
      rmll[q[k]] = la[k];
      rmlr[q[k]] = ra[k];
    }
  } else {
    // gdone: 0 pending (set by k_refit_local), < 0 finished by k_refit_mid, > 0 the
    // pass of this kernel that finished it. The pending nodes are listed in LDS when
    // they fit, so the passes skip the finished ones.
    if (tid == 0) npend = 0;
    __syncthreads();
    for (int j = tid; j < nt; j += 1024)
      if (gdone[j] == 0) {
        const int k = atomicAdd(&npend, 1);
        if (k < kTopList) plist[k] = j;
      }
    __syncthreads();
    const int np = npend;
    const bool listed = np <= kTopList;
    const int nloop = listed ? np : nt;
    for (int pass = 1;; ++pass) {
      bool changed = false;
      for (int k = tid; k < nloop; k += 1024) {
        const int j = listed ? plist[k] : k;
        if (gdone[j] != 0) continue;
        const int qq = top_list[j], ll = lefts[qq], rr = rights[qq];
        bool lt, rt;
        int a, b;
        f3 lmn, lmx, rmn, rmx;
        top_child(ll, nin, state, top_index, amin, amax, rmll, rmlr, lt, a, lmn, lmx);
        top_child(rr, nin, state, top_index, amin, amax, rmll, rmlr, rt, b, rmn, rmx);
        if (lt && !(gdone[a] != 0 && gdone[a] < pass)) continue;
        if (rt && !(gdone[b] != 0 && gdone[b] < pass)) continue;
        if (lt) { lmn = xyz(gmin[a]); lmx = xyz(gmax[a]); a = grm[a]; }
        if (rt) { rmn = xyz(gmin[b]); rmx = xyz(gmax[b]); b = grm[b]; }
        put_deferred(j, qq, a, b, lmn, lmx, rmn, rmx, gmin, gmax, grm, amin, amax, rmll,
                     rmlr);
        __threadfence_block();
        gdone[j] = pass;
        changed = true;
      }
      if (!any_changed(flag, pass, changed)) break;
    }
    for (int k = tid; k < nloop; k += 1024)
      if (gdone[listed ? plist[k] : k] == 0) left_over = true;
  }
  if (__syncthreads_or(left_over)) {
    if (tid == 0) atomicOr(warn, (uint32_t)CM_WARN_REFIT_LIMIT);
    // an unfinished node's box need not hold its children's
    for (int c = tid; c < max(ncloth, 1); c += 1024) irr[c] = kIrregular;
  }
  if (tid == 0) *ntop = 0;
}

// ---- traversal ----------------------------------------------------------------
constexpr int kTravBlock = 128;  // 2 waves
constexpr int kStack = 63;       // usable entries, as the reference's int[64] with its -1 sentinel
// The first rows of a lane's stack live in LDS, 8 or 12 in the lane walks (WalkShape), 16 in
// k_traverse_redo; deeper ones, rare, go to the lane's global spill row of kSpill ints.
constexpr int kRedoStack = 16;
constexpr int kSpill = kStack - 8;
static_assert(kSpill == kTravSpill, "spill row");

// The tree as the traversal kernels take it
struct WalkTree {
  int t;
  const uint4* qnodes;  // null: the exact walk
  const float4* nodes;  // records of the exact walk of an irregular tree (k_pack_exact) or null
  const int *irr, *lefts, *rights, *rmll, *rmlr;  // irr: per cloth
  const float4 *amin, *amax;
  const int *slot_cloth, *croot, *ccap, *tstart;  // batch (null: one cloth)
};

// box b lies in box a (false when a bound is NaN)
__device__ __forceinline__ bool holds(f3 amn, f3 amx, f3 bmn, f3 bmx) {
  return amn.x <= bmn.x && amn.y <= bmn.y && amn.z <= bmn.z && amx.x >= bmx.x &&
         amx.y >= bmx.y && amx.z >= bmx.z;
}
// whether a leaf's own box can be quantised: one with a NaN bound overlaps every box by the
// exact test, and where no node holds its leaf (midpoint split on tied codes) the tree is
// regular all the same
__device__ __forceinline__ bool box_ordered(f3 mn, f3 mx) { return holds(mn, mx, mn, mx); }

// DFS of one leaf (Collision/CudaBVH.cu:23-113) from the root through the exact boxes:
// the second leaves of its pairs in the reference's order into out (at most cap); the
// stack is sstk[k][col]. Returns their number.
template <int kRow, int kLds, bool kPacked = false>
__device__ __forceinline__ int walk_exact(const WalkTree& T, int leaf, int root, f3 mn, f3 mx, int cap,
                          int* __restrict__ out, uint32_t& w, int (*sstk)[kRow], int col,
                          int* __restrict__ spill) {
  const int nin = T.t - 1, me = nin + leaf;
  const long long limit = 64ll * T.t + 4096;
  int node = root, top = 0, ncol = 0;
  for (long long visits = 0;;) {
    if (++visits > limit) {
      w |= CM_WARN_TRAVERSAL_LIMIT;
      break;
    }
    int l, r;
    bool ol, orr;
    if (kPacked) {
      const float4* n = T.nodes + 4 * (int64_t)node;
      const float4 ids = n[0], a = n[1], b = n[2], c = n[3];
      l = __float_as_int(ids.x);
      r = __float_as_int(ids.y);
      ol = (__float_as_int(ids.z) > me) & overlap(mn, mx, xyz(a), mk3(a.w, b.x, b.y));
      orr = (__float_as_int(ids.w) > me) & overlap(mn, mx, mk3(b.z, b.w, c.x), mk3(c.y, c.z, c.w));
    } else {
      l = T.lefts[node];
      r = T.rights[node];
      ol = (T.rmll[node] > me) & overlap(mn, mx, xyz(T.amin[l]), xyz(T.amax[l]));
      orr = (T.rmlr[node] > me) & overlap(mn, mx, xyz(T.amin[r]), xyz(T.amax[r]));
    }
    const bool el = ol & (l >= nin), er = orr & (r >= nin);
    // Past the cap the reference keeps walking but drops every further pair, so
    // stopping at the first dropped pair yields the same list.
    if (ncol + (int)el + (int)er > cap) {
      if (el && ncol < cap) out[ncol++] = l - nin;
      else if (er && ncol < cap) out[ncol++] = r - nin;
      w |= CM_WARN_PAIR_CAP;
      break;
    }
    if (el) out[ncol++] = l - nin;
    if (er) out[ncol++] = r - nin;
    const bool tl = ol & (l < nin), tr = orr & (r < nin);
    if (tl | tr) {
      node = tl ? l : r;
      if (tl & tr) {
        if (top >= kStack) {
          w |= CM_WARN_STACK_OVERFLOW;  // the push is dropped, as in the reference
        } else {
          if constexpr (kLds < kStack) {
            if (top < kLds) sstk[top][col] = r;
            else spill[top - kLds] = r;
          } else {
            sstk[top][col] = r;
          }
          ++top;
        }
      }
    } else {
      if (top == 0) break;
      --top;
      if constexpr (kLds < kStack) node = top < kLds ? sstk[top][col] : spill[top - kLds];
      else node = sstk[top][col];
    }
  }
  return ncol;
}

// ---- the walk through quantised nodes ----------------------------------------------
// The walk is bound by its instructions (nearly every branch is taken by some lane of a
// wave) and, where the nodes outgrow an L2, by the bytes of its gathers. A node's record
// is therefore 32 bytes, two loads:
//   .x  split (bits 0-25; the children are split and split + 1, as the build lays them),
//       bit 26 / 27: the left / right child is a leaf, bit 28: see .y
//   .y  the right child's rightmost leaf; the left one's is split (of a node with two
//       parents it can be another: then bit 28 is set and .y is the larger of the two)
//   then three words per child: its box in 16 bits a bound, (min x, min y),
//       (min z, 65535 - max x), (65535 - max y, 65535 - max z)
// Bounds are quantised by one monotone function over the root's box (in a batch the box of
// the cloth's root: cloths may lie far apart), the leaf's own box by the same one as
// (max x, max y), (max z, 65535 - min x), ..., so boxes that overlap have no word larger
// than the leaf's: three saturating 16-bit subtractions, an or and a compare. The test can
// pass boxes that do not overlap, so the leaves it finds are candidates: their exact boxes
// are tested after the walk (by 8 at a time, off its chain of loads), in order, and those
// that fail are dropped. The pairs and their order are walk_exact's: where a node's box
// holds its children's (irr small), a leaf whose exact box passes has ancestors that pass. A
// walk that reaches the stack limit or the visit limit is given up (kRedo) and done exactly,
// and so is the whole tree where the root's box is so large that leaves apart from each other
// fall together (coarse_frame).
// k_traverse with what finishes its long walks, exact records of 64 bytes and pairs
// stored as they are found -> now (walk_shape's rows): falling 256^2 614 -> 295 us, flat
// 54 -> 46, draped 319 -> 305, draped 131x97 217 -> 157, 64^2 134 -> 94, 2 M leaves
// 1,070 -> 850, crumpled 1024^2 1,740 -> 1,597 (there 65 vector and 30 scalar instructions
// a visit at 43% of the lanes bound it; refilling the lanes that finish early from a wave's
// queue of leaves was slower, 2,320, as is stepping two levels at a time: 650 instructions a
// step, or loading both children's records ahead).
constexpr uint32_t kSplitMask = (1u << 26) - 1, kLeftLeaf = 1u << 26, kRightLeaf = 1u << 27,
                   kOtherRight = 1u << 28;
struct Quant {
  f3 lo, scale;
};
__device__ __forceinline__ Quant quant_frame(float4 lo, float4 hi) {
  auto sc = [](float a, float b) { return b > a ? 65535.f / (b - a) : 0.f; };
  return {xyz(lo), mk3(sc(lo.x, hi.x), sc(lo.y, hi.y), sc(lo.z, hi.z))};
}
// monotone in v, whatever the frame (a frame without extent, or past the float range,
// gives one value for all)
__device__ __forceinline__ uint32_t q16(float v, float lo, float scale) {
  return (uint32_t)fminf(fmaxf((v - lo) * scale, 0.f), 65535.f);
}
// the three words of a box; of the leaf's own box with min and max exchanged
__device__ __forceinline__ uint3 q_box(Quant q, f3 mn, f3 mx) {
  return make_uint3(q16(mn.x, q.lo.x, q.scale.x) | (q16(mn.y, q.lo.y, q.scale.y) << 16),
                    q16(mn.z, q.lo.z, q.scale.z) | ((65535u - q16(mx.x, q.lo.x, q.scale.x)) << 16),
                    (65535u - q16(mx.y, q.lo.y, q.scale.y)) |
                        ((65535u - q16(mx.z, q.lo.z, q.scale.z)) << 16));
}
// per half: how far a is above b, 0 if it is not
__device__ __forceinline__ uint32_t above16(uint32_t a, uint32_t b) {
  typedef unsigned short us2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_sub_sat(__builtin_bit_cast(us2, a),
                                                                    __builtin_bit_cast(us2, b)));
}
__device__ __forceinline__ bool q_overlap(uint32_t a, uint32_t b, uint32_t c, uint3 q) {
  return (above16(a, q.x) | above16(b, q.y) | above16(c, q.z)) == 0;
}

struct QNode {
  int split;
  bool l, r, lleaf, rleaf;  // child passes, child is a leaf
};
__device__ __forceinline__ QNode q_visit(const uint4* __restrict__ qnodes, int node, int leaf,
                                         uint3 q) {
  const uint4* p = (const uint4*)((const char*)qnodes + ((uint32_t)node << 5));
  const uint4 a = p[0], b = p[1];
  QNode n;
  n.split = (int)(a.x & kSplitMask);
  const int rml = (a.x & kOtherRight) ? (int)a.y : n.split;
  n.l = (rml > leaf) & q_overlap(a.z, a.w, b.x, q);
  n.r = ((int)a.y > leaf) & q_overlap(b.y, b.z, b.w, q);
  n.lleaf = (a.x & kLeftLeaf) != 0;
  n.rleaf = (a.x & kRightLeaf) != 0;
  return n;
}

enum WalkEnd { kDone, kBudget, kRedo };
// State of a walk between two visits: the node to visit next (-1: none), the pending
// nodes (the last in tos, the one below it in row top - 1, the first in row 1), the
// candidates or pairs written, the visits made
struct WalkState {
  int node, top, tos, n, visits;
};

// One visit: the node's leaf children that pass join the candidates cand[n][col], st goes
// to the next node. The candidates are collected in LDS: a store to memory in the walk
// would have each visit wait for it, as loads and stores share one counter. Returns
// false when the stack limit is reached.
template <int kLds, int kRow>
__device__ __forceinline__ bool quant_step(const uint4* __restrict__ qnodes, int leaf, uint3 q,
                                           WalkState& st, int& n, int (*sstk)[kRow],
                                           int (*cand)[kRow], int col, int* __restrict__ spill) {
  bool fits = true;
  ++st.visits;
  const QNode v = q_visit(qnodes, st.node, leaf, q);
  if (v.l & v.lleaf) cand[n++][col] = v.split;
  if (v.r & v.rleaf) cand[n++][col] = v.split + 1;
  const bool tl = v.l & !v.lleaf, tr = v.r & !v.rleaf;
  if (tl & tr) {
    if (st.top < kLds) sstk[st.top][col] = st.tos;
    else if (st.top < kStack) spill[st.top - kLds] = st.tos;
    else fits = false;
    st.tos = v.split + 1;
    ++st.top;
  }
  st.node = tl ? v.split : v.split + 1;
  if (!(tl | tr)) {
    st.node = st.top > 0 ? st.tos : -1;
    st.top = max(st.top - 1, 0);
    st.tos = sstk[min(st.top, kLds - 1)][col];
    if (st.top >= kLds) st.tos = spill[st.top - kLds];
  }
  return fits;
}

// The exact boxes of the n candidates, kVerify at a time: the second leaves of those that
// pass go to out[m...), at most cap. Returns the pairs found, also past the cap.
template <int kVerify, int kRow>
__device__ __forceinline__ int verify(const WalkTree& T, f3 mn, f3 mx, int n, int m, int cap,
                                      int* __restrict__ out, int (*cand)[kRow], int col) {
  const int nin = T.t - 1;
  for (int k = 0; k < n; k += kVerify) {
    int c[kVerify];
    float4 a[kVerify], b[kVerify];
#pragma unroll
    for (int u = 0; u < kVerify; ++u) {
      c[u] = cand[min(k + u, n - 1)][col];
      a[u] = T.amin[nin + c[u]];
      b[u] = T.amax[nin + c[u]];
    }
#pragma unroll
    for (int u = 0; u < kVerify; ++u)
      if (k + u < n && overlap(mn, mx, xyz(a[u]), xyz(b[u]))) {
        if (m < cap) out[m] = c[u];
        ++m;
      }
  }
  return m;
}

__device__ __forceinline__ int visit_limit(int t) {
  return (int)min(64ll * t + 4096, (long long)INT_MAX - 1);
}

// Walks on from st until it ends or `budget` visits were made; the second leaves of its
// pairs go to out[0, st.n), at most cap. cand has ncand rows.
template <int kLds, int kVerify, int kRow>
__device__ __forceinline__ WalkEnd walk_quant(const WalkTree& T, int leaf, f3 mn, f3 mx, uint3 q,
                                              int cap, int* __restrict__ out, int budget,
                                              WalkState& st, uint32_t& w, int (*sstk)[kRow],
                                              int (*cand)[kRow], int ncand, int col,
                                              int* __restrict__ spill) {
  const int limit = visit_limit(T.t);
  const int bound = min(budget, limit);
  for (;;) {
    int n = 0;
    const int room = min(ncand - 2, cap - st.n);  // past the cap one more is looked for
    bool fits = true;
    while (st.node >= 0 && st.visits < bound && n <= room && fits)
      fits = quant_step<kLds>(T.qnodes, leaf, q, st, n, sstk, cand, col, spill);
    const int m = verify<kVerify>(T, mn, mx, n, st.n, cap, out, cand, col);
    st.n = min(m, cap);
    if (!fits) return kRedo;
    if (m > cap) {  // the reference drops every pair past the cap
      w |= CM_WARN_PAIR_CAP;
      return kDone;
    }
    if (st.node < 0) return kDone;
    if (st.visits >= bound) return st.visits >= limit ? kRedo : kBudget;
  }
}

// The first pass's budget is given in exact visits; quantised ones are cheaper, and 1.7
// for one give the shortest two passes (draped 256^2: 342 us at 200 visits, 331 at 340,
// 362 at 400; falling 256^2: 500, 353, 320; all with 16 rows of stack and 66 of candidates).
constexpr int quant_budget(int budget) { return budget + budget * 7 / 10; }

// A leaf whose walk outlasts the first pass's visit budget leaves its state in a
// record of kRec ints: leaf, pairs written, stack depth, next node, cap, visits, then
// the kStack stack entries. The second pass finishes it with a whole wave.
constexpr int kRec = kTravRec;
static_assert(kRec >= 6 + kStack, "record holds the stack");

template <int kLds, int kRow>
__device__ __forceinline__ void put_record(int* __restrict__ R, int leaf, int cap,
                                           const WalkState& st, int (*sstk)[kRow], int col,
                                           const int* __restrict__ spill) {
  R[0] = leaf;
  R[1] = st.n;
  R[2] = st.top;
  R[3] = st.node;
  R[4] = cap;
  R[5] = st.visits;
  for (int k = 1; k <= st.top; ++k)
    R[5 + k] = k == st.top ? st.tos : (k < kLds ? sstk[k][col] : spill[k - kLds]);
}

// Workgroups are dealt to the 8 XCDs in turn. Each XCD takes every eighth chunk of
// `xchunk` consecutive tiles (Morton-ordered leaves), so its L2 serves compact
// subtrees while the dense regions of the cloth, whose leaves visit many more
// nodes, are shared evenly between the XCDs. The grid is padded to whole rounds.
__device__ __forceinline__ int walk_tile(int xchunk) {
  const int j = blockIdx.x / kXcds, xcd = blockIdx.x % kXcds;
  return ((j / xchunk) * kXcds + xcd) * xchunk + j % xchunk;
}

// First pass: one lane per leaf, at most `budget` visits (no budget: budget <= 0 or
// no record buffer). A leaf still walking then takes a record slot, if one is left,
// and counts zero pairs here; past the slots it walks on to the end.
template <int kLds, int kVerify>
__global__ void __launch_bounds__(kTravBlock) k_traverse(WalkTree T, int cap, int ncand,
                                                         int* __restrict__ chunk,
                                                         int* __restrict__ counts,
                                                         uint32_t* __restrict__ warn,
                                                         int* __restrict__ tile_sum,
                                                         int xchunk, int budget,
                                                         int* __restrict__ rec, int rcap,
                                                         int* __restrict__ hctl,
                                                         int* __restrict__ spill) {
  // Row k of every lane's stack is one LDS row, so a wave's pushes and pops at equal
  // depths hit 64 consecutive banks.
  extern __shared__ int walk_lds[][kTravBlock];
  int(*sstk)[kTravBlock] = walk_lds, (*cand)[kTravBlock] = walk_lds + kLds;
  const int tile = walk_tile(xchunk);
  const int t = T.t;
  if (tile >= (t + kTravBlock - 1) / kTravBlock) return;
  if (T.nodes && *T.irr >= kIrregular) return;  // k_traverse_exact takes the tree
  const int leaf = tile * kTravBlock + threadIdx.x;
  const int stride = cap;  // every leaf's chunk holds the body's cap (a cloth's may be less)
  uint32_t w = 0;
  const int me = t - 1 + leaf;
  int root = 0, c = 0, ncol = 0;
  bool walk = leaf < t;
  if (walk && T.croot) {  // a batch: the root of the leaf's cloth, its cap
    c = T.slot_cloth[leaf];
    root = T.croot[c];
    cap = T.ccap[c];
    walk = root >= 0;  // a one-triangle cloth has no pairs
  }
  int* out = chunk + (int64_t)leaf * stride;
  int* sp = spill + (int64_t)leaf * kSpill;
  f3 mn = mk3(0, 0, 0), mx = mk3(0, 0, 0);
  uint3 q = make_uint3(0, 0, 0);
  WalkState st{root, 0, 0, 0, 0};
  WalkEnd end = kDone;
  if (walk) {
    mn = xyz(T.amin[me]);
    mx = xyz(T.amax[me]);
    end = kRedo;
    if (T.qnodes && T.irr[c] < kIrregular && box_ordered(mn, mx)) {
      q = q_box(quant_frame(T.amin[root], T.amax[root]), mx, mn);
      end = walk_quant<kLds, kVerify, kTravBlock>(T, leaf, mn, mx, q, cap, out,
                                   budget > 0 && rec ? budget : INT_MAX, st, w, sstk, cand, ncand,
                                   threadIdx.x, sp);
    }
  }
  // Leaves still walking claim record slots with one atomic per wave (thousands of
  // lanes on one counter would queue at its L2 channel).
  const int lane = threadIdx.x & 63;
  const uint64_t want = __ballot(end == kBudget);
  bool handed = false;
  if (want) {
    int base = 0;
    if (lane == 0) base = atomicAdd(hctl, __popcll(want));
    base = __shfl(base, 0, 64);
    if (end == kBudget) {
      const int slot = base + __popcll(want & ((1ull << lane) - 1));
      if (slot < rcap) {
        put_record<kLds>(rec + (int64_t)slot * kRec, leaf, cap, st, sstk, threadIdx.x, sp);
        handed = true;
      } else {
        end = walk_quant<kLds, kVerify, kTravBlock>(T, leaf, mn, mx, q, cap, out, INT_MAX, st, w,
                                                    sstk, cand, ncand, threadIdx.x, sp);
      }
    }
  }
  if (walk) ncol = handed ? 0 : st.n;
  if (end == kRedo) {
    w = 0;
    ncol = walk_exact<kTravBlock, kLds>(T, leaf, root, mn, mx, cap, out, w, sstk,
                                             threadIdx.x, sp);
  }
  if (leaf < t) counts[leaf] = ncol;
  // one warning atomic per wave: two thirds of the leaves of a draped cloth hit the cap
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) w |= __shfl_xor(w, o, 64);
  if (lane == 0 && w) atomicOr(warn, w);
  // pairs of the tile (its leaves' counts follow in the compaction)
  __shared__ int wsum[kTravBlock / 64];
  int v = ncol;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
  if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    int tot = 0;
    for (int k = 0; k < kTravBlock / 64; ++k) tot += wsum[k];
    tile_sum[tile] = tot;
  }
}

// ---- second pass: one wave finishes one handed-over leaf -------------------------
// The reference's DFS visits nodes in preorder and emits a node's left leaf child
// before its right one, so a pair's place in the leaf's list is the preorder place of
// the node that emits it. The wave expands up to 64 pending nodes at once, in any
// order, and tags every pair (a candidate whose exact box passes) with a 64-bit key
// that sorts in that preorder:
//   bits 63..58  rank of the pending subtree handed over (0 = the next node to visit,
//                then the stack entries from the top down: they are visited in that
//                order, each subtree before the next)
//   bits 57..8   the path below that subtree's root, one bit per level (0 = left)
//   bits  7..1   the depth of that path
//   bit   0      0 for the left leaf child, 1 for the right one
// Sorting (rank, path padded with zeros, depth, side) is preorder: a node comes before
// its descendants (same padded path, smaller depth) and a left subtree before the
// right one. Pending nodes are kept sorted by key (the smallest on top), so every pair
// below the top pending node's key is final. The wave stops once more than the
// remaining cap of pairs are final: the first `cap` are the leaf's list and one more
// means the reference dropped pairs (CM_WARN_PAIR_CAP). A leaf that overflows this
// pass's buffers or path bits, or could reach the stack limit (each pending node
// carries its stack depth) or the visit limit, is walked exactly by lane 0 alone.
constexpr int kPend = 512;     // pending nodes per leaf
constexpr int kHits = 256;     // pairs kept per leaf
constexpr int kPathBits = 50;
constexpr int kResumeBlocks = 4096;
constexpr int kResumeMaxCap = 96;  // kHits holds cap + 1 kept pairs and a round's 128 new ones
static_assert(kResumeMaxCap + 1 + 128 <= kHits, "hit buffer");

__device__ __forceinline__ int wave_excl_scan(int v, int lane, int& total) {
  int s = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(s, o, 64);
    if (lane >= o) s += y;
  }
  total = __shfl(s, 63, 64);
  return s - v;
}

__device__ __forceinline__ int wave_sum(int v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// More records than this and each is finished by one lane (k_traverse_lanes) instead
// of a whole wave: a wave per record pays off for the long tail of a few heavy
// leaves, while with many records the lanes' serial walks keep more of them going
// at once.
constexpr int kLaneModeMin = 16384;

__global__ void __launch_bounds__(64) k_traverse_resume(WalkTree T,
                                                        int* __restrict__ chunk, int stride,
                                                        int* __restrict__ counts,
                                                        uint32_t* __restrict__ warn,
                                                        int* __restrict__ tile_sum,
                                                        const int* __restrict__ rec, int rcap,
                                                        int* __restrict__ hctl) {
  __shared__ int pe[kPend];  // node | stack depth << 26
  __shared__ uint64_t pk[kPend];
  __shared__ uint64_t hk[kHits];
  __shared__ int hp[kHits];
  __shared__ int fstk[kStack][1];
  const int lane = threadIdx.x;
  const int nin = T.t - 1;
  const long long limit = 64ll * T.t + 4096;
  const int nres = min(hctl[0], rcap);
  if (nres > kLaneModeMin) return;  // k_traverse_lanes takes them
  uint32_t wacc = 0;
  for (int rid = blockIdx.x; rid < nres; rid += gridDim.x) {
    const int* R = rec + (int64_t)rid * kRec;
    const int leaf = R[0], ncol0 = R[1], top0 = R[2], cur = R[3], cap = R[4];
    const int root = T.croot ? T.croot[T.slot_cloth[leaf]] : 0;
    const long long visits0 = R[5];
    const f3 mn = xyz(T.amin[nin + leaf]), mx = xyz(T.amax[nin + leaf]);
    const uint3 q = q_box(quant_frame(T.amin[root], T.amax[root]), mx, mn);
    const int capr = cap - ncol0;  // pairs still to find (0: only whether one more exists)
    int* out = chunk + (int64_t)leaf * stride;
    // pending: the stack entries bottom-up, then the next node on top
    const int m = top0 + 1;
    for (int k = lane; k < m; k += 64) {
      pe[k] = (k < top0 ? R[6 + k] : cur) | (k << 26);  // visited at stack depth k
      pk[k] = (uint64_t)(top0 - k) << 58;
    }
    __syncthreads();
    int np = m, nh = 0;
    long long expanded = 0;
    bool fallback = cap > kResumeMaxCap;
    while (np > 0 && !fallback) {
      const int take = min(64, np);
      const int base = np - take;
      const bool act = lane < take;
      int node = 0, sd = 0;
      uint64_t key = 0;
      if (act) {
        const uint32_t e = (uint32_t)pe[np - 1 - lane];
        node = (int)(e & kSplitMask);
        sd = (int)(e >> 26);
        key = pk[np - 1 - lane];
      }
      __syncthreads();
      expanded += take;
      int nc = 0, ne = 0, ce[2] = {0, 0}, ep[2] = {0, 0};
      uint64_t ck[2] = {0, 0}, ek[2] = {0, 0};
      bool deep = false;
      if (act) {
        const QNode v = q_visit(T.qnodes, node, leaf, q);
        auto passes = [&](int c) {
          return overlap(mn, mx, xyz(T.amin[nin + c]), xyz(T.amax[nin + c]));
        };
        const bool el = (v.l & v.lleaf) && passes(v.split);
        const bool er = (v.r & v.rleaf) && passes(v.split + 1);
        if (el) {
          ek[ne] = key;
          ep[ne++] = v.split;
        }
        if (er) {
          ek[ne] = key | 1ull;
          ep[ne++] = v.split + 1;
        }
        const bool tl = v.l & !v.lleaf, tr = v.r & !v.rleaf;
        if (tl | tr) {
          const int d = (int)((key >> 1) & 127ull);
          const bool both = tl & tr;
          if (d + 1 > kPathBits || (both && sd >= kStack)) deep = true;
          const uint64_t kl = (key & ~0xffull) | ((uint64_t)(d + 1) << 1);
          const uint64_t kr = kl | (1ull << (57 - d));
          if (tl) {
            ce[nc] = v.split | ((both ? sd + 1 : sd) << 26);
            ck[nc++] = kl;
          }
          if (tr) {
            ce[nc] = (v.split + 1) | (sd << 26);
            ck[nc++] = kr;
          }
        }
      }
      int totc, tote;
      const int exc = wave_excl_scan(nc, lane, totc);
      const int exe = wave_excl_scan(ne, lane, tote);
      if (__any(deep) || base + totc > kPend || visits0 + expanded > limit) {
        fallback = true;
        break;
      }
      if (nh + tote > kHits) {
        // keep the capr + 1 smallest keys: a larger one can only move further back
        // once the pending subtrees add theirs, so it is never listed nor the stop
        int rk[kHits / 64];
        uint64_t kk[kHits / 64];
        int kp[kHits / 64];
#pragma unroll
        for (int u = 0; u < kHits / 64; ++u) {
          const int i = lane + 64 * u;
          rk[u] = kHits;
          if (i < nh) {
            kk[u] = hk[i];
            kp[u] = hp[i];
            int rank = 0;
            for (int j2 = 0; j2 < nh; ++j2) rank += hk[j2] < kk[u];
            rk[u] = rank;
          }
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < kHits / 64; ++u)
          if (rk[u] <= capr) {
            hk[rk[u]] = kk[u];
            hp[rk[u]] = kp[u];
          }
        nh = min(nh, capr + 1);
        __syncthreads();
      }
      for (int q = 0; q < nc; ++q) {
        const int at = base + totc - 1 - (exc + q);
        pe[at] = ce[q];
        pk[at] = ck[q];
      }
      for (int q = 0; q < ne; ++q) {
        hk[nh + exe + q] = ek[q];
        hp[nh + exe + q] = ep[q];
      }
      __syncthreads();
      np = base + totc;
      nh += tote;
      if (nh > capr) {
        const uint64_t bound = np > 0 ? pk[np - 1] : ~0ull;
        int below = 0;
        for (int i = lane; i < nh; i += 64) below += hk[i] < bound;
        if (wave_sum(below) > capr) break;
      }
    }
    int nout;
    uint32_t w = 0;
    if (fallback) {
      __syncthreads();
      nout = 0;
      if (lane == 0) {
        nout = walk_exact<1, kStack>(T, leaf, root, mn, mx, cap, out, w, fstk, 0, nullptr);
      }
    } else {
      // each pair's place is the number of smaller keys (keys are distinct)
      for (int i = lane; i < nh; i += 64) {
        const uint64_t ki = hk[i];
        int rank = 0;
        for (int j2 = 0; j2 < nh; ++j2) rank += hk[j2] < ki;
        if (rank < capr) out[ncol0 + rank] = hp[i];
      }
      __syncthreads();
      nout = ncol0 + min(nh, capr);
      if (nh > capr) w |= CM_WARN_PAIR_CAP;
    }
    if (lane == 0) {
      counts[leaf] = nout;
      atomicAdd(&tile_sum[leaf / kTravBlock], nout);
      wacc |= w;
    }
    __syncthreads();
  }
  // the workgroup's warnings in one atomic (the record count is cleared by the next
  // kernel on the stream, once every workgroup here has read it)
  if (lane == 0 && wacc) atomicOr(warn, wacc);
}

// Second pass when there are more than kLaneModeMin records: one lane per record
// walks on serially from the record's state (next node, stack, pairs written,
// visits), as the first pass would have without a budget.
template <int kLds, int kVerify>
__global__ void __launch_bounds__(kTravBlock) k_traverse_lanes(
    WalkTree T, int ncand, int* __restrict__ chunk, int stride, int* __restrict__ counts,
    uint32_t* __restrict__ warn, int* __restrict__ tile_sum, const int* __restrict__ rec, int rcap,
    const int* __restrict__ hctl, int* __restrict__ spill) {
  extern __shared__ int walk_lds[][kTravBlock];
  int(*sstk)[kTravBlock] = walk_lds, (*cand)[kTravBlock] = walk_lds + kLds;
  const int nres = min(hctl[0], rcap);
  if (nres <= kLaneModeMin) return;  // k_traverse_resume takes them
  const int nin = T.t - 1;
  uint32_t w = 0;
  for (int rid = blockIdx.x * kTravBlock + threadIdx.x; rid < nres;
       rid += gridDim.x * kTravBlock) {
    const int* R = rec + (int64_t)rid * kRec;
    const int leaf = R[0], top = R[2], cap = R[4];
    const int root = T.croot ? T.croot[T.slot_cloth[leaf]] : 0;
    int* sp = spill + (int64_t)leaf * kSpill;
    int* out = chunk + (int64_t)leaf * stride;
    for (int k = 1; k < top; ++k) {
      if (k < kLds) sstk[k][threadIdx.x] = R[5 + k];
      else sp[k - kLds] = R[5 + k];
    }
    const f3 mn = xyz(T.amin[nin + leaf]), mx = xyz(T.amax[nin + leaf]);
    WalkState st{R[3], top, top > 0 ? R[5 + top] : 0, R[1], R[5]};
    uint32_t wl = 0;
    int ncol;
    const uint3 q = q_box(quant_frame(T.amin[root], T.amax[root]), mx, mn);
    if (walk_quant<kLds, kVerify, kTravBlock>(T, leaf, mn, mx, q, cap, out, INT_MAX, st, wl, sstk,
                                              cand, ncand, threadIdx.x, sp) == kRedo) {
      wl = 0;
      ncol = walk_exact<kTravBlock, kLds>(T, leaf, root, mn, mx, cap, out, wl, sstk,
                                               threadIdx.x, sp);
    } else {
      ncol = st.n;
    }
    w |= wl;
    counts[leaf] = ncol;
    atomicAdd(&tile_sum[leaf / kTravBlock], ncol);
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) w |= __shfl_xor(w, o, 64);
  if ((threadIdx.x & 63) == 0 && w) atomicOr(warn, w);
}

// ---- a group of lanes per leaf ----------------------------------------------------
// On a tree of few leaves the first pass above leaves most of the chip idle behind its
// longest walk (64^2: 124 waves on 1,024 SIMDs, 200 dependent visits of about 0.4 us).
// Here kG lanes expand up to kG pending nodes of one leaf at once, with the keys and the
// order of k_traverse_resume (rank 0: the root is the one subtree). The leaves they meet
// join the hits by the quantised test alone and are tested exactly, kG at a time, when
// there are more than the cap of them and at the end. A leaf that overflows the buffers
// or the path bits, or could reach the stack limit or the visit limit (on a caller's tree
// of shared nodes: each path to a node is a visit), and any leaf of an irregular tree, is
// left to k_traverse_redo. Bound by the rounds' latency (about 1,550 cycles, a third of
// them the records' loads; 16 to 18 rounds at 64^2), on draped cloths by the instructions.
// k_traverse, with what finishes its long walks -> k_traverse_group: 60^2 72 -> 17 us, 64^2
// 94 -> 25, 96x83 119 -> 43, four of 64^2 67 -> 44, falling 128^2 174 -> 68, fit 128^2
// 64 -> 58, draped 131x97 157 -> 128. Where few boxes overlap the lanes of a group idle and
// it is the slower one: flat 128^2 33 -> 54, a crumpled ball of 128^2 139 -> 173.
constexpr int kGroup = 16;  // 8: 22, 34, 41 us for 60^2, 64^2 and 96x83, 143 draped 131x97
constexpr int kGroupPend = 128, kGroupHits = 112;
constexpr int kGroupMaxCap = kGroupHits - 1 - 2 * kGroup;
// Up to this many leaves. Beyond it a falling cloth gains little (256^2 295 -> 271 us), and a
// draped one, whose leaves meet several times the cap, loses (305 -> 655).
constexpr int kGroupLeaves = 1 << 15;

template <int kG>
__device__ __forceinline__ int group_sum(int v) {
#pragma unroll
  for (int o = kG / 2; o >= 1; o >>= 1) v += __shfl_xor(v, o, kG);
  return v;
}

template <int kG>
__global__ void __launch_bounds__(64) k_traverse_group(WalkTree T, int cap,
                                                       int* __restrict__ chunk,
                                                       int* __restrict__ counts,
                                                       uint32_t* __restrict__ warn) {
  constexpr int kPer = 64 / kG;  // leaves per wave
  __shared__ uint64_t spk[kPer][kGroupPend], shk[kPer][kGroupHits];
  __shared__ int spe[kPer][kGroupPend], shp[kPer][kGroupHits];  // pe: node | stack depth << 26
  const int lane = threadIdx.x, g = lane % kG, sub = lane / kG;
  uint64_t *pk = spk[sub], *hk = shk[sub];
  int *pe = spe[sub], *hp = shp[sub];
  const uint64_t mine = ((1ull << kG) - 1ull) << (sub * kG);
  const uint64_t below_me = mine & ((1ull << lane) - 1ull);
  // the group's kG bits of a ballot; earlier: the group's earlier lanes in two such fields
  auto field = [&](uint64_t b) { return (uint32_t)(b >> (sub * kG)) & ((1u << kG) - 1u); };
  const uint32_t earlier = ((1u << g) - 1u) * (1u | 1u << kG);
  // consecutive leaves to one XCD in chunks, as in k_traverse
  constexpr int kRun = 4 * kTravBlock / kPer;
  const int j = blockIdx.x / kXcds, xcd = blockIdx.x % kXcds;
  const int leaf = (((j / kRun) * kXcds + xcd) * kRun + j % kRun) * kPer + sub;
  const int t = T.t, nin = t - 1, stride = cap;
  // the lanes of a wave share the buffers: their accesses stay in program order
  auto order = [] { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); };
  int root = 0, c = 0;
  bool act = leaf < t, again = false;
  if (act && T.croot) {  // a batch: the root of the leaf's cloth, its cap
    c = T.slot_cloth[leaf];
    root = T.croot[c];
    cap = T.ccap[c];
    act = root >= 0;  // a one-triangle cloth has no pairs
  }
  f3 mn = mk3(0, 0, 0), mx = mk3(0, 0, 0);
  uint3 q = make_uint3(0, 0, 0);
  int np = 0, nh = 0, nv = 0;  // pending, hits, hits tested (the first nv)
  const int limit = visit_limit(t);
  int seen = 0;
  if (act) {
    const int irr = T.irr[c];
    mn = xyz(T.amin[nin + leaf]);
    mx = xyz(T.amax[nin + leaf]);
    q = q_box(quant_frame(T.amin[root], T.amax[root]), mx, mn);
    if (g == 0) {
      pe[0] = root;
      pk[0] = 0;
    }
    np = 1;
    again = irr >= kIrregular || !box_ordered(mn, mx);
    act = !again;
  }
  // tests hits nv to nh exactly and closes the gaps
  auto test_hits = [&] {
    for (int k0 = nv; k0 < nh; k0 += kG) {
      const int k = k0 + g;
      int c = 0;
      uint64_t key = 0;
      bool keep = false;
      if (k < nh) {
        c = hp[k];
        key = hk[k];
        keep = overlap(mn, mx, xyz(T.amin[nin + c]), xyz(T.amax[nin + c]));
      }
      const uint64_t m = __ballot(keep);
      if (keep) {
        const int at = nv + __popcll(m & below_me);
        hp[at] = c;
        hk[at] = key;
      }
      nv += __popcll(m & mine);
      order();
    }
    nh = nv;
  };
  while (act) {
    order();
    const int take = min(kG, np), base = np - take;
    seen += take;
    bool tl = false, tr = false, hl = false, hr = false, deep = false;
    int split = 0, sd = 0;
    uint64_t key = 0, kl = 0;
    if (g < take) {
      const uint32_t e = (uint32_t)pe[np - 1 - g];
      key = pk[np - 1 - g];
      const QNode v = q_visit(T.qnodes, (int)(e & kSplitMask), leaf, q);
      split = v.split;
      sd = (int)(e >> 26);
      hl = v.l & v.lleaf;
      hr = v.r & v.rleaf;
      tl = v.l & !v.lleaf;
      tr = v.r & !v.rleaf;
      const int d = (int)((key >> 1) & 127ull);
      deep = (tl | tr) & ((d + 1 > kPathBits) | (tl & tr & (sd >= kStack)));
      kl = (key & ~0xffull) | ((uint64_t)(d + 1) << 1);
    }
    // children and hits of the group's earlier lanes
    const uint32_t c2 = field(__ballot(tl)) | field(__ballot(tr)) << kG;
    const uint32_t h2 = field(__ballot(hl)) | field(__ballot(hr)) << kG;
    const int totc = __popc(c2), tote = __popc(h2);
    if (field(__ballot(deep)) || base + totc > kGroupPend || seen > limit) {
      again = true;
      break;
    }
    order();
    const int ca = base + totc - 1 - __popc(c2 & earlier), ha = nh + __popc(h2 & earlier);
    if (tl) {
      pe[ca] = split | (((tl & tr) ? sd + 1 : sd) << 26);
      pk[ca] = kl;
    }
    if (tr) {
      pe[ca - tl] = (split + 1) | (sd << 26);
      pk[ca - tl] = kl | (1ull << (57 - (int)((key >> 1) & 127ull)));
    }
    if (hl) {
      hp[ha] = split;
      hk[ha] = key;
    }
    if (hr) {
      hp[ha + hl] = split + 1;
      hk[ha + hl] = key | 1ull;
    }
    np = base + totc;
    nh += tote;
    order();
    if (nh > cap) test_hits();
    if (nh > cap) {
      // more than the cap of pairs are final: their keys are below every pending node's
      const uint64_t bound = np > 0 ? pk[np - 1] : ~0ull;
      int below = 0;
      for (int k = g; k < nh; k += kG) below += hk[k] < bound;
      if (group_sum<kG>(below) > cap) break;
      if (nh + 2 * kG > kGroupHits) {
        // keep the cap + 1 smallest keys: a larger one can only move further back
        constexpr int kMine = (kGroupHits + kG - 1) / kG;
        uint64_t kk[kMine];
        int kp[kMine], rk[kMine];
#pragma unroll
        for (int u = 0; u < kMine; ++u) {
          const int k = g + kG * u;
          rk[u] = kGroupHits;
          if (k < nh) {
            kk[u] = hk[k];
            kp[u] = hp[k];
            int rank = 0;
            for (int k2 = 0; k2 < nh; ++k2) rank += hk[k2] < kk[u];
            rk[u] = rank;
          }
        }
        order();
#pragma unroll
        for (int u = 0; u < kMine; ++u)
          if (rk[u] <= cap) {
            hk[rk[u]] = kk[u];
            hp[rk[u]] = kp[u];
          }
        nh = nv = min(nh, cap + 1);
        order();
      }
    }
    act = np > 0;
  }
  order();
  bool over = false;
  if (leaf < t && !again) {
    test_hits();
    // each pair's place is the number of smaller keys (keys are distinct)
    int* out = chunk + (int64_t)leaf * stride;
    for (int k = g; k < nh; k += kG) {
      const uint64_t key = hk[k];
      int rank = 0;
      for (int k2 = 0; k2 < nh; ++k2) rank += hk[k2] < key;
      if (rank < cap) out[rank] = hp[k];
    }
    over = nh > cap;
  }
  if (leaf < t && g == 0) counts[leaf] = again ? -1 : min(nh, cap);
  if (__any(over) && lane == 0) atomicOr(warn, (uint32_t)CM_WARN_PAIR_CAP);
}

// The leaves the groups left (count -1), walked exactly by one lane each, and the tiles'
// sums (added up here: an atomic a leaf to the tiles' two cache lines took 40 us at 64^2).
__global__ void __launch_bounds__(kTravBlock) k_traverse_redo(WalkTree T, int cap,
                                                              int* __restrict__ chunk,
                                                              int* __restrict__ counts,
                                                              uint32_t* __restrict__ warn,
                                                              int* __restrict__ tile_sum,
                                                              int* __restrict__ spill) {
  __shared__ int sstk[kRedoStack][kTravBlock];
  __shared__ int wsum[kTravBlock / 64];
  const int leaf = blockIdx.x * kTravBlock + threadIdx.x;
  int n = leaf < T.t ? counts[leaf] : 0;
  if (n < 0) {
    const int me = T.t - 1 + leaf, c = T.croot ? T.slot_cloth[leaf] : 0;
    uint32_t w = 0;
    n = walk_exact<kTravBlock, kRedoStack>(T, leaf, T.croot ? T.croot[c] : 0, xyz(T.amin[me]),
                                          xyz(T.amax[me]), T.croot ? T.ccap[c] : cap,
                                          chunk + (int64_t)leaf * cap, w, sstk, threadIdx.x,
                                          spill + (int64_t)leaf * kSpill);
    counts[leaf] = n;
    if (w) atomicOr(warn, w);
  }
  n = wave_sum(n);
  if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = n;
  __syncthreads();
  if (threadIdx.x == 0) tile_sum[blockIdx.x] = wsum[0] + wsum[1];
}

// A caller's irregular tree of many leaves through its exact records: one lane per leaf, and
// no more LDS than the stack's, so that eight waves a SIMD hide the gathers.
__global__ void __launch_bounds__(kTravBlock) k_traverse_exact(WalkTree T, int cap, int xchunk,
                                                               int* __restrict__ chunk,
                                                               int* __restrict__ counts,
                                                               uint32_t* __restrict__ warn,
                                                               int* __restrict__ tile_sum,
                                                               int* __restrict__ spill) {
  __shared__ int sstk[kRedoStack][kTravBlock];
  __shared__ int wsum[kTravBlock / 64];
  const int tile = walk_tile(xchunk), leaf = tile * kTravBlock + threadIdx.x;
  if (tile >= (T.t + kTravBlock - 1) / kTravBlock || *T.irr < kIrregular) return;
  int n = 0;
  uint32_t w = 0;
  if (leaf < T.t) {
    const int me = T.t - 1 + leaf;
    n = walk_exact<kTravBlock, kRedoStack, true>(T, leaf, 0, xyz(T.amin[me]), xyz(T.amax[me]), cap,
                                                 chunk + (int64_t)leaf * cap, w, sstk, threadIdx.x,
                                                 spill + (int64_t)leaf * kSpill);
    counts[leaf] = n;
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) w |= __shfl_xor(w, o, 64);
  n = wave_sum(n);
  if ((threadIdx.x & 63) == 0) {
    wsum[threadIdx.x >> 6] = n;
    if (w) atomicOr(warn, w);
  }
  __syncthreads();
  if (threadIdx.x == 0) tile_sum[tile] = wsum[0] + wsum[1];
}

__global__ void k_clear_records(int* __restrict__ hctl) {
  if (threadIdx.x == 0) hctl[0] = 0;
}

// Whether leaf i and another leaf of its cloth, drawn by a hash, fall together in the frame
// though they are apart by half the leaf's extent. One vertex far away, or a piece that falls
// without end, makes the root's box so large that the cloth is a few cells, and a walk then
// passes a share of all nodes: with a vertex 1e5 m off 1,770 us at 150^2 (45 through the
// exact boxes), 6,200 at 256^2 (56), growing with the square of the leaves. A fourth of the
// leaves draw, so the pairs found are a fourth of the leaves that a walk meets in vain: from
// kIrregular on the tree is left to the exact walk.
constexpr int kDraw = 4;
__device__ __forceinline__ bool coarse_frame(const WalkTree& T, int i, int c, Quant q) {
  const int nin = T.t - 1, first = T.croot ? T.tstart[c] : 0;
  const uint32_t n = (uint32_t)((T.croot ? T.tstart[c + 1] : T.t) - first);
  uint32_t h = (uint32_t)i * 0x9e3779b1u;
  h = (h ^ (h >> 15)) * 0x85ebca77u;
  const int j = first + (int)__umulhi(h ^ (h >> 13), n);
  const f3 amn = xyz(T.amin[nin + i]), amx = xyz(T.amax[nin + i]);
  const f3 bmn = xyz(T.amin[nin + j]), bmx = xyz(T.amax[nin + j]);
  const f3 e = sub(amx, amn);
  const float half = 0.5f * fmaxf(e.x, fmaxf(e.y, e.z));
  const float gap = fmaxf(fmaxf(fmaxf(bmn.x - amx.x, amn.x - bmx.x),
                                fmaxf(bmn.y - amx.y, amn.y - bmx.y)),
                          fmaxf(bmn.z - amx.z, amn.z - bmx.z));
  const uint3 o = q_box(q, bmn, bmx);
  return gap > half && q_overlap(o.x, o.y, o.z, q_box(q, amx, amn));
}

// The quantised node records, and whether they can be walked: every node's box has to
// hold its children's, and the frame be fine enough. kCaller (unit-level pair query, the
// caller's own tree): also its children have to lie side by side as the build lays them,
// its rightmost leaves must not shrink upwards, and no leaf below its left child may lie
// beyond a right child that is a leaf itself: the record's one rightmost leaf would let that
// right leaf pass for leaves at and past it (the build's right leaf is the last of its
// parent's range).
template <bool kCaller>
__global__ void __launch_bounds__(kBlock) k_pack_nodes(WalkTree T, uint4* __restrict__ qnodes,
                                                       int* __restrict__ irr) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  const int nin = T.t - 1;
  if (i >= nin) return;
  // a tree that others have found irregular needs no records
  if (kCaller &&
      __hip_atomic_load(irr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= kIrregular)
    return;
  const int l = T.lefts[i], r = T.rights[i], a = T.rmll[i], b = T.rmlr[i];
  const f3 mn = xyz(T.amin[i]), mx = xyz(T.amax[i]);
  // in a batch, a node that is walked and the leaf of its number belong to one cloth
  const int c = T.croot ? T.slot_cloth[i] : 0, root = T.croot ? max(T.croot[c], 0) : 0;
  const Quant q = quant_frame(T.amin[root], T.amax[root]);
  // before the children's boxes, whose loads wait for their numbers
  const bool coarse = i % kDraw == 0 && coarse_frame(T, i, c, q);
  const f3 lmn = xyz(T.amin[l]), lmx = xyz(T.amax[l]), rmn = xyz(T.amin[r]), rmx = xyz(T.amax[r]);
  const bool ll = l >= nin, rl = r >= nin;
  const int sp = ll ? l - nin : l;
  bool ok = holds(mn, mx, lmn, lmx) && holds(mn, mx, rmn, rmx);
  if (kCaller && ok)
    ok = sp + 1 == (rl ? r - nin : r) && (ll ? a == l : a >= max(T.rmll[l], T.rmlr[l])) &&
         (rl ? b == r && a <= b : b >= max(T.rmll[r], T.rmlr[r]));
  int found = !ok ? kIrregular : coarse ? 1 : 0;
  if (!T.croot) {  // one cloth: one lane adds for the wave
    const uint64_t any = __ballot(found), bad = __ballot(found == kIrregular);
    const bool adds = (threadIdx.x & 63) == __ffsll((long long)any) - 1;
    found = adds ? (bad ? kIrregular : __popcll(any)) : 0;
  }
  if (found && __hip_atomic_load(&irr[c], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < kIrregular)
    atomicAdd(&irr[c], found);
  const uint3 bl = q_box(q, lmn, lmx), br = q_box(q, rmn, rmx);
  const bool other = a != nin + sp;
  qnodes[2 * (int64_t)i] =
      make_uint4((uint32_t)sp | (ll ? kLeftLeaf : 0u) | (rl ? kRightLeaf : 0u) |
                     (other ? kOtherRight : 0u),
                 (uint32_t)((other ? max(a, b) : b) - nin), bl.x, bl.y);
  qnodes[2 * (int64_t)i + 1] = make_uint4(bl.z, br.x, br.y, br.z);
}

// 64-byte records of an irregular tree for the exact walk: children, rightmost leaves, both
// boxes. A caller's nodes may be numbered in any order, and four words and four boxes from as
// many places a visit then cost several times the record's one (500 k renumbered leaves 2,296
// us, with the records 535; 2 M 10,735 and 1,883). Up to kGroupLeaves leaves the caches hold
// the tree (30,000: 132 us, 137 by records), and a body's nodes lie as the build numbers them.
__global__ void __launch_bounds__(kBlock) k_pack_exact(WalkTree T, float4* __restrict__ nodes) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= T.t - 1 || *T.irr < kIrregular) return;
  const int l = T.lefts[i], r = T.rights[i];
  const f3 lmn = xyz(T.amin[l]), lmx = xyz(T.amax[l]), rmn = xyz(T.amin[r]), rmx = xyz(T.amax[r]);
  float4* o = nodes + 4 * (int64_t)i;
  o[0] = make_float4(__int_as_float(l), __int_as_float(r), __int_as_float(T.rmll[i]),
                     __int_as_float(T.rmlr[i]));
  o[1] = make_float4(lmn.x, lmn.y, lmn.z, lmx.x);
  o[2] = make_float4(lmx.y, lmx.z, rmn.x, rmn.y);
  o[3] = make_float4(rmn.z, rmx.x, rmx.y, rmx.z);
}

// One workgroup per traversal tile of kTravBlock leaves: the first wave scans the
// leaves' counts, then the workgroup writes the tile's pairs in order, kBlock
// consecutive output slots at a time (each thread finds its slot's leaf by binary
// search over the tile's prefixes), so reads and writes are contiguous runs.
// A tile's pairs are shared by gridDim.y workgroups, so that a few tiles fill the chip, and
// a thread looks up kAhead pairs at once: the searches and the loads after them are chains
// of latencies. kScan: the workgroup adds up the sums of the tiles before its own, and the
// last one writes the total (at most pair_cap), in place of a scan's launch of 5 us.
// k_compact_pairs with that scan, one workgroup a tile and one pair a thread at a time ->
// now: 64^2 17 -> 4.9 us, draped 131x97 31 -> 5.8, draped 256^2 39 -> 19; without it, 96
// cloths 66 -> 44, 2 M leaves 147 -> 105, crumpled 1024^2 125 -> 97.
constexpr int kAhead = 4;
constexpr int kScanMax = 1024;  // tiles; every workgroup reads the sums of all before its own
template <bool kScan>
__global__ void __launch_bounds__(kBlock) k_compact_pairs(int t, int stride,
                                                          const int* __restrict__ chunk,
                                                          const int* __restrict__ counts,
                                                          const int* __restrict__ tile_pre,
                                                          int2* __restrict__ pairs,
                                                          int* __restrict__ hctl,
                                                          int64_t pair_cap,
                                                          int* __restrict__ d_npairs) {
  static_assert(kTravBlock == 128, "two leaves per lane of the first wave");
  // the traversal's hand-over record count, read by its second pass, starts the next
  // substep at zero
  if (hctl && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) hctl[0] = 0;
  __shared__ int pre[kTravBlock + 1];
  __shared__ int wsum[kBlock / 64];
  const int tile = blockIdx.x, tid = threadIdx.x;
  const int l0 = tile * kTravBlock;
  if (kScan) {
    int v = 0;
    for (int k = tid; k < tile; k += kBlock) v += tile_pre[k];
    v = wave_sum(v);
    if ((tid & 63) == 0) wsum[tid >> 6] = v;
  }
  if (tid < 64) {
    const int i0 = l0 + 2 * tid, i1 = i0 + 1;
    const int c0 = i0 < t ? counts[i0] : 0, c1 = i1 < t ? counts[i1] : 0;
    int s = c0 + c1;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(s, o, 64);
      if (tid >= o) s += y;
    }
    const int ex = s - (c0 + c1);
    pre[2 * tid] = ex;
    pre[2 * tid + 1] = ex + c0;
    if (tid == 63) pre[kTravBlock] = s;
  }
  __syncthreads();
  const int total = pre[kTravBlock];
  int out0 = 0;
  if (kScan) {
#pragma unroll
    for (int w = 0; w < kBlock / 64; ++w) out0 += wsum[w];
    if (tile == (int)gridDim.x - 1 && blockIdx.y == 0 && tid == 0)
      *d_npairs = (int)min((int64_t)out0 + total, pair_cap);
  } else {
    out0 = tile_pre[tile];
  }
  const int step = kBlock * gridDim.y;
  for (int k0 = blockIdx.y * kBlock + tid; k0 < total; k0 += kAhead * step) {
    // the last leaf whose prefix is <= k holds slot k
    int lo[kAhead], c[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) lo[u] = 0;
#pragma unroll
    for (int h = kTravBlock / 2; h >= 1; h >>= 1)
#pragma unroll
      for (int u = 0; u < kAhead; ++u)
        if (pre[lo[u] + h] <= k0 + u * step) lo[u] += h;
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const int k = min(k0 + u * step, total - 1);
      c[u] = k0 + u * step < total ? chunk[(int64_t)(l0 + lo[u]) * stride + (k - pre[lo[u]])] : 0;
    }
#pragma unroll
    for (int u = 0; u < kAhead; ++u)
      if (k0 + u * step < total) pairs[out0 + k0 + u * step] = make_int2(l0 + lo[u], c[u]);
  }
}

// Also clears what the build starts from (a launch of its own otherwise).
__global__ void __launch_bounds__(kBlock) k_gather_tris(BuildInit init,
                                                        const uint32_t* __restrict__ perm,
                                                        const int4* __restrict__ tin,
                                                        int4* __restrict__ tout, int fix,
                                                        const float4* __restrict__ amin,
                                                        const float4* __restrict__ amax,
                                                        float4* __restrict__ tmin,
                                                        float4* __restrict__ tmax) {
  const int i = blockIdx.x * kBlock + threadIdx.x, t = init.t;
  build_init(init, i);
  if (i >= t) return;
  const uint32_t s = perm[i];
  tout[i] = tin[s];
  if (fix) {
    tmin[i] = amin[t - 1 + s];
    tmax[i] = amax[t - 1 + s];
  }
}
__global__ void __launch_bounds__(kBlock) k_put_leaves(int t, const float4* __restrict__ tmin,
                                                       const float4* __restrict__ tmax,
                                                       float4* __restrict__ amin,
                                                       float4* __restrict__ amax) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= t) return;
  amin[t - 1 + i] = tmin[i];
  amax[t - 1 + i] = tmax[i];
}
}  // namespace

// ---- launchers --------------------------------------------------------------
int launch_tri_update(int n, int t, const float4* x, const float4* p, const int4* tri, float th,
                      int bits, int normalize, float4* amin, float4* amax, uint64_t* keys,
                      uint32_t* vals, float4* centroid_tmp, float4* box_tmp, hipStream_t s) {
  (void)n;
  if (t <= 0) return CM_OK;
  const int nb = nblocks(t);
  const bool norm = bits == 30 && normalize;
  hipLaunchKernelGGL(k_tri_update, dim3(nb), dim3(kBlock), 0, s, t, x, p, tri, th, bits, amin,
                     amax, keys, vals, norm ? centroid_tmp : nullptr, norm ? box_tmp : nullptr);
  if (norm) {
    if (nb > kFewBoxes)
      hipLaunchKernelGGL(k_box_reduce, dim3(1), dim3(kBlock), 0, s, box_tmp, nb);
    hipLaunchKernelGGL((nb > kFewBoxes ? k_keys30<false> : k_keys30<true>), dim3(nb), dim3(kBlock),
                       0, s, t, centroid_tmp, box_tmp, nb, keys);
  }
  CM_LAUNCH_CHECK();
  return CM_OK;
}

int launch_tri_update_batch(const LbvhBufs& b, const float4* x, const float4* p, const int4* tri,
                            float th, uint64_t* keys, uint32_t* vals, float4* centroid_tmp,
                            hipStream_t s) {
  const int t = b.t;
  if (t <= 0) return CM_OK;
  hipLaunchKernelGGL(k_cloth_box_init, dim3(nblocks(6 * b.ncloth)), dim3(kBlock), 0, s, b.ncloth,
                     b.cbox);
  hipLaunchKernelGGL(k_tri_update, dim3(nblocks(t)), dim3(kBlock), 0, s, t, x, p, tri, th, 30,
                     b.amin, b.amax, keys, vals, centroid_tmp, nullptr);
  hipLaunchKernelGGL(k_cloth_box, dim3(nblocks(t, kBlock * kBoxRun)), dim3(kBlock), 0, s, t, centroid_tmp,
                     b.slot_cloth, b.cbox);
  hipLaunchKernelGGL(k_keys30_cloth, dim3(nblocks(t)), dim3(kBlock), 0, s, t, centroid_tmp,
                     b.slot_cloth, b.cbox, keys);
  CM_LAUNCH_CHECK();
  return CM_OK;
}

static BuildInit build_init_args(const LbvhBufs& b) {
  return {b.t, b.claim_cnt, b.claim_hi, b.ntop, b.irr, b.ncloth, b.croot};
}
static int build_init_grid(const LbvhBufs& b) { return nblocks(std::max(2 * b.t - 1, b.ncloth)); }

int launch_build(const LbvhBufs& b, const uint64_t* keys, int midpoint, bool cleared,
                 const int4* tri_from, int4* tri_to, hipStream_t s) {
  const int t = b.t;
  if (t < 2) return CM_OK;
  if (!cleared)
    hipLaunchKernelGGL(k_build_init, dim3(build_init_grid(b)), dim3(kBlock), 0, s,
                       build_init_args(b));
  hipLaunchKernelGGL(k_build, dim3(nblocks(t - 1)), dim3(kBlock), 0, s, t, keys, midpoint, b.lefts,
                     b.rights, b.claim_cnt, b.claim_hi, b.ranges, b.warn,
                     b.ncloth ? b.tstart : nullptr, b.croot);
  hipLaunchKernelGGL(k_parents, dim3(nblocks(2 * t - 1)), dim3(kBlock), 0, s, t, b.claim_cnt,
                     b.claim_hi, b.parents, tri_from, tri_to);
  CM_LAUNCH_CHECK();
  return CM_OK;
}

int launch_refit(const LbvhBufs& b, hipStream_t s) {
  const int t = b.t;
  if (t < 2) return CM_OK;
  hipLaunchKernelGGL(k_refit_local, dim3((t + kRefitCH - 1) / kRefitCH), dim3(kRefitCH), 0, s, t,
                     b.lefts, b.rights, b.ranges, b.amin, b.amax, b.rmll, b.rmlr, b.state,
                     b.top_list, b.top_index, b.ntop, b.tdone);
  if (t > 2 * kSuper)  // smaller trees defer at most a few hundred nodes
    hipLaunchKernelGGL(k_refit_mid, dim3((t + kSuper - 1) / kSuper), dim3(1024), 0, s, t, b.lefts,
                       b.rights, b.ranges, b.amin, b.amax, b.rmll, b.rmlr, b.state,
                       b.top_list, b.top_index, b.ntop, b.tmin, b.tmax, b.trm, b.tdone);
  hipLaunchKernelGGL(k_refit_top, dim3(1), dim3(1024), 0, s, t, b.lefts, b.rights, b.amin, b.amax,
                     b.rmll, b.rmlr, b.state, b.top_list, b.top_index, b.ntop, b.tmin,
                     b.tmax, b.trm, b.tdone, b.warn, b.irr, b.ncloth);
  CM_LAUNCH_CHECK();
  return CM_OK;
}

// The lane walks' LDS: rows of the stack and of the candidates a lane collects before it
// tests them, and how many it tests at a time (registers). Each walk that stops to test holds
// up its wave, so as many candidate rows, up to 66, as leave the launch one round of
// workgroups: a CU's 160 KB, given out by 1,280 bytes, hold four workgroups of 12 and 66 rows
// (131,072 leaves) and ten of 12 and 17. Against 16 and 66 rows up to 262,144 leaves: 130 k
// leaves flat 72 -> 46 us, crumpled 110 -> 70, falling 369 -> 297, draped 308 -> 309; 216 k
// flat 107 -> 57; 258 k flat 117 -> 60, falling 735 -> 593; 156 k flat 77 -> 50 but draped
// 343 -> 400 (49 pairs a leaf, 50 rows). Trees of more rounds want the waves: 8 and 24 rows
// take 1,592 us for 2 M crumpled leaves and 327 for 96 cloths (16 and 16 rows 1,740 and 355,
// 12 and 24 by 8 1,614 and 324).
struct WalkShape {
  int stack, cand, verify;
};
static WalkShape walk_shape(int nt) {
  constexpr int kCus = 256, kLdsBytes = 160 << 10, kGrain = 1280, kRow = kTravBlock * 4;
  const int per_cu = (nt + kCus - 1) / kCus;
  if (per_cu > 10) return {8, 24, 4};
  const int rows = (kLdsBytes / per_cu / kGrain * kGrain - 16) / kRow;  // 16: the tile sums
  return {12, std::min(66, rows - 12), per_cu > 8 ? 4 : 8};
}

static WalkTree walk_tree(const LbvhBufs& b) {
  return {b.t,      b.t < kQuantLeaves ? b.qnodes : nullptr,
          b.nodes,  b.irr,
          b.lefts,  b.rights,
          b.rmll,   b.rmlr,
          b.amin,   b.amax,
          b.ncloth ? b.slot_cloth : nullptr,
          b.ncloth ? b.croot : nullptr,
          b.ccap,   b.tstart};
}

bool walked_by_groups(const LbvhBufs& b, int cap) {
  return b.group && b.t <= kGroupLeaves && cap <= kGroupMaxCap;
}

// the second pass needs a budget, record buffers and quantised nodes
static bool two_passes(const LbvhBufs& b) {
  return b.t < kQuantLeaves && b.trav_budget > 0 && b.trec && b.hctl && b.rcap > 0;
}

static int launch_traverse(const LbvhBufs& b, int cap, int* chunk, int* counts, int* offsets,
                           hipStream_t s) {
  const int t = b.t;
  const int nt = (t + kTravBlock - 1) / kTravBlock;
  const int xchunk = b.trav_chunk > 0 ? b.trav_chunk : 4;
  const int round = kXcds * xchunk;
  const bool two = two_passes(b);
  const WalkTree T = walk_tree(b);
  if (walked_by_groups(b, cap)) {
    const int per = 64 / kGroup, nb = (t + per - 1) / per, rnd = kXcds * 4 * kTravBlock / per;
    hipLaunchKernelGGL(k_traverse_group<kGroup>, dim3((nb + rnd - 1) / rnd * rnd), dim3(64), 0, s,
                       T, cap, chunk, counts, b.warn);
    hipLaunchKernelGGL(k_traverse_redo, dim3(nt), dim3(kTravBlock), 0, s, T, cap, chunk, counts,
                       b.warn, offsets, b.spill);
    CM_LAUNCH_CHECK();
    return CM_OK;
  }
  const WalkShape ws = walk_shape(nt);
  const size_t lds = sizeof(int) * kTravBlock * (ws.stack + ws.cand);
  hipLaunchKernelGGL((ws.stack == 8    ? k_traverse<8, 4>
                      : ws.verify == 4 ? k_traverse<12, 4>
                                       : k_traverse<12, 8>),
                     dim3((nt + round - 1) / round * round), dim3(kTravBlock), lds, s, T, cap,
                     ws.cand, chunk, counts, b.warn, offsets, xchunk,
                     two ? quant_budget(b.trav_budget) : 0, two ? b.trec : nullptr, b.rcap, b.hctl,
                     b.spill);
  if (b.nodes)
    hipLaunchKernelGGL(k_traverse_exact, dim3((nt + round - 1) / round * round), dim3(kTravBlock),
                       0, s, T, cap, xchunk, chunk, counts, b.warn, offsets, b.spill);
  if (two) {  // one of the two finishes the records, the other returns at once
    hipLaunchKernelGGL(k_traverse_resume, dim3(std::min(b.rcap, kResumeBlocks)), dim3(64), 0, s, T,
                       chunk, cap, counts, b.warn, offsets, b.trec, b.rcap, b.hctl);
    if (b.rcap > kLaneModeMin)
      hipLaunchKernelGGL((ws.stack == 8    ? k_traverse_lanes<8, 4>
                          : ws.verify == 4 ? k_traverse_lanes<12, 4>
                                           : k_traverse_lanes<12, 8>),
                         dim3(std::min((b.rcap + kTravBlock - 1) / kTravBlock, 8192)),
                         dim3(kTravBlock), lds, s, T, ws.cand, chunk, cap, counts, b.warn, offsets,
                         b.trec, b.rcap, b.hctl, b.spill);
  }
  CM_LAUNCH_CHECK();
  return CM_OK;
}

int launch_pairs(const LbvhBufs& b, int cap, int* chunk, int* counts, int* offsets, int2* pairs,
                 int* d_npairs, void* scan_temp, hipStream_t s) {
  const int t = b.t;
  if (t < 2) return fill_i32(d_npairs, 0, 1, s);
  // offsets[0, nt): pair count of each tile of kTravBlock leaves; offsets[nt, 2nt): the
  // tiles' exclusive prefixes (2 * nt <= t)
  const int nt = (t + kTravBlock - 1) / kTravBlock;
  int rc = launch_traverse(b, cap, chunk, counts, offsets, s);
  if (rc) return rc;
  const dim3 grid(nt, std::max(1, std::min(8, 2048 / nt)));
  int* hctl = two_passes(b) ? b.hctl : nullptr;
  if (nt <= kScanMax) {
    hipLaunchKernelGGL(k_compact_pairs<true>, grid, dim3(kBlock), 0, s, t, cap, chunk, counts,
                       offsets, pairs, hctl, (int64_t)t * cap, d_npairs);
  } else {
    rc = scan_tiles(nt, offsets, offsets + nt, 0, (int64_t)t * cap, 0, d_npairs, nullptr, scan_temp,
                    s);
    if (rc) return rc;
    hipLaunchKernelGGL(k_compact_pairs<false>, grid, dim3(kBlock), 0, s, t, cap, chunk, counts,
                       offsets + nt, pairs, hctl, (int64_t)t * cap, d_npairs);
  }
  CM_LAUNCH_CHECK();
  return CM_OK;
}

int launch_traverse_only(const LbvhBufs& b, int cap, int* chunk, int* counts, int* offsets,
                         hipStream_t s) {
  if (b.t < 2) return CM_OK;
  const int rc = launch_traverse(b, cap, chunk, counts, offsets, s);
  if (rc || !two_passes(b)) return rc;
  hipLaunchKernelGGL(k_clear_records, dim3(1), dim3(64), 0, s, b.hctl);
  CM_LAUNCH_CHECK();
  return CM_OK;
}

int launch_pack_nodes(const LbvhBufs& b, bool from_caller, hipStream_t s) {
  const int t = b.t;
  if (t < 2 || t >= kQuantLeaves) return CM_OK;
  hipLaunchKernelGGL(from_caller ? k_pack_nodes<true> : k_pack_nodes<false>, dim3(nblocks(t - 1)),
                     dim3(kBlock), 0, s, walk_tree(b), b.qnodes, b.irr);
  if (b.nodes)
    hipLaunchKernelGGL(k_pack_exact, dim3(nblocks(t - 1)), dim3(kBlock), 0, s, walk_tree(b),
                       b.nodes);
  CM_LAUNCH_CHECK();
  return CM_OK;
}

int launch_gather_tris(const LbvhBufs& b, const uint32_t* perm, const int4* tri_in, int4* tri_out,
                       int fix_leaves, float4* tmp_min, float4* tmp_max, hipStream_t s) {
  const int t = b.t;
  if (t <= 0) return CM_OK;
  hipLaunchKernelGGL(k_gather_tris, dim3(build_init_grid(b)), dim3(kBlock), 0, s,
                     build_init_args(b), perm, tri_in, tri_out, fix_leaves, b.amin, b.amax,
                     tmp_min, tmp_max);
  if (fix_leaves)
    hipLaunchKernelGGL(k_put_leaves, dim3(nblocks(t)), dim3(kBlock), 0, s, t, tmp_min, tmp_max,
                       b.amin, b.amax);
  CM_LAUNCH_CHECK();
  return CM_OK;
}

// Build/refit scratch carved from one buffer; with b == nullptr only the size.
size_t carve_build(int t, void* d_temp, LbvhBufs* b) {
  const size_t m = t > 0 ? 2 * (size_t)t - 1 : 0;
  const size_t tt = (size_t)(t > 0 ? t : 1);
  char* tp = (char*)d_temp;
  size_t off = 0;
  auto take = [&](auto** dst, size_t bytes) {
    if (b) *dst = (std::remove_reference_t<decltype(**dst)>*)(tp + off);
    off += align_up(bytes);
  };
  LbvhBufs dummy;
  LbvhBufs* o = b ? b : &dummy;
  take(&o->claim_cnt, sizeof(int) * m);
  take(&o->claim_hi, sizeof(int) * m);
  take(&o->state, sizeof(int) * tt);
  take(&o->top_list, sizeof(int) * tt);
  take(&o->top_index, sizeof(int) * tt);
  take(&o->ntop, sizeof(int));
  take(&o->irr, sizeof(int));
  take(&o->ranges, sizeof(int2) * tt);
  take(&o->qnodes, 2 * sizeof(uint4) * tt);
  take(&o->tmin, sizeof(float4) * tt);
  take(&o->tmax, sizeof(float4) * tt);
  take(&o->trm, sizeof(int) * tt);
  take(&o->tdone, sizeof(int) * tt);
  return off;
}

size_t lbvh_build_temp_bytes(int t) { return carve_build(t, nullptr, nullptr); }
// bytes of the exact walk's records for a caller's tree
static size_t exact_bytes(int t) {
  return t > kGroupLeaves && t < kQuantLeaves ? align_up(4 * sizeof(float4) * (size_t)t) : 0;
}
size_t lbvh_pairs_temp_bytes(int t, int cap) {
  return align_up(sizeof(int) * (size_t)t * cap) +
         2 * align_up(sizeof(int) * (size_t)t) + align_up(2 * sizeof(uint4) * (size_t)t) +
         exact_bytes(t) + align_up(sizeof(int) * kSpill * (size_t)t) + align_up(sizeof(int)) +
         scan_temp_bytes(t);
}

}  // namespace cm

// ---- unit-level C ABI ---------------------------------------------------------
using namespace cm;

extern "C" int cm_tri_update(int32_t n, int32_t t, const void* d_x, const void* d_p,
                             const void* d_tri, float thickness, int32_t morton_bits,
                             int32_t morton_normalize, void* d_aabb_min, void* d_aabb_max,
                             uint64_t* d_keys, void* stream) {
  if (t < 1 || n < 1 || !d_x || !d_p || !d_tri || !d_aabb_min || !d_aabb_max || !d_keys ||
      (morton_bits != 30 && morton_bits != 63)) {
    set_error("cm_tri_update: invalid argument");
    return CM_ERR_ARG;
  }
  hipStream_t s = (hipStream_t)stream;
  const bool norm = morton_bits == 30 && morton_normalize;
  float4* cen = nullptr;
  float4* box = nullptr;
  if (norm) {
    CM_HIP(hipMallocAsync((void**)&cen, sizeof(float4) * (size_t)t, s));
    CM_HIP(hipMallocAsync((void**)&box, sizeof(float4) * (2 * (size_t)nblocks(t) + 2), s));
  }
  int rc = launch_tri_update(n, t, (const float4*)d_x, (const float4*)d_p, (const int4*)d_tri,
                             thickness, morton_bits, morton_normalize, (float4*)d_aabb_min,
                             (float4*)d_aabb_max, d_keys, nullptr, cen, box, s);
  if (cen) hipFreeAsync(cen, s);
  if (box) hipFreeAsync(box, s);
  return rc;
}

extern "C" size_t cm_lbvh_sort_temp_bytes(int32_t t) { return radix_sort_temp_bytes(t); }

extern "C" int cm_lbvh_sort(int32_t t, int32_t key_bits, uint64_t* d_keys, uint32_t* d_vals,
                            void* d_temp, size_t temp_bytes, void* stream) {
  if (t < 0 || key_bits < 1 || key_bits > 64 || (t > 1 && (!d_keys || !d_vals || !d_temp))) {
    set_error("cm_lbvh_sort: invalid argument");
    return CM_ERR_ARG;
  }
  if (temp_bytes < radix_sort_temp_bytes(t)) {
    set_error("cm_lbvh_sort: temp buffer too small");
    return CM_ERR_ARG;
  }
  int rc = radix_sort_clear(d_temp, t, (hipStream_t)stream);
  if (rc) return rc;
  return radix_sort(d_keys, d_vals, t, key_bits, d_temp, (hipStream_t)stream);
}

extern "C" size_t cm_lbvh_build_temp_bytes(int32_t t) { return lbvh_build_temp_bytes(t); }


extern "C" int cm_lbvh_build(int32_t t, const uint64_t* d_keys, int32_t midpoint_split,
                             int32_t* d_lefts, int32_t* d_rights, int32_t* d_parents,
                             uint32_t* d_warn, void* d_temp, size_t temp_bytes, void* stream) {
  if (t < 2 || !d_keys || !d_lefts || !d_rights || !d_parents || !d_warn || !d_temp ||
      temp_bytes < lbvh_build_temp_bytes(t)) {
    set_error("cm_lbvh_build: invalid argument");
    return CM_ERR_ARG;
  }
  LbvhBufs b;
  b.t = t;
  b.lefts = d_lefts;
  b.rights = d_rights;
  b.parents = d_parents;
  b.warn = d_warn;
  carve_build(t, d_temp, &b);
  return launch_build(b, d_keys, midpoint_split, false, nullptr, nullptr, (hipStream_t)stream);
}

// d_temp must be the same buffer that the preceding cm_lbvh_build used (claim records).
extern "C" int cm_lbvh_refit(int32_t t, const int32_t* d_lefts, const int32_t* d_rights,
                             const int32_t* d_parents, void* d_aabb_min, void* d_aabb_max,
                             int32_t* d_rmll, int32_t* d_rmlr, uint32_t* d_warn, void* d_temp,
                             size_t temp_bytes, void* stream) {
  (void)d_parents;
  if (t < 2 || !d_lefts || !d_rights || !d_aabb_min || !d_aabb_max || !d_rmll || !d_rmlr ||
      !d_warn || !d_temp || temp_bytes < lbvh_build_temp_bytes(t)) {
    set_error("cm_lbvh_refit: invalid argument");
    return CM_ERR_ARG;
  }
  LbvhBufs b;
  b.t = t;
  b.lefts = (int*)d_lefts;
  b.rights = (int*)d_rights;
  b.amin = (float4*)d_aabb_min;
  b.amax = (float4*)d_aabb_max;
  b.rmll = d_rmll;
  b.rmlr = d_rmlr;
  b.warn = d_warn;
  carve_build(t, d_temp, &b);
  return launch_refit(b, (hipStream_t)stream);
}

extern "C" size_t cm_lbvh_pairs_temp_bytes(int32_t t, int32_t cap) {
  return lbvh_pairs_temp_bytes(t, cap);
}

extern "C" int cm_lbvh_pairs(int32_t t, const int32_t* d_lefts, const int32_t* d_rights,
                             const void* d_aabb_min, const void* d_aabb_max,
                             const int32_t* d_rmll, const int32_t* d_rmlr, int32_t cap,
                             int32_t* d_pairs, int32_t* d_n_pairs, uint32_t* d_warn,
                             void* d_temp, size_t temp_bytes, void* stream) {
  if (t < 2 || cap < 1 || !d_lefts || !d_rights || !d_aabb_min || !d_aabb_max || !d_rmll ||
      !d_rmlr || !d_pairs || !d_n_pairs || !d_warn || !d_temp ||
      temp_bytes < lbvh_pairs_temp_bytes(t, cap)) {
    set_error("cm_lbvh_pairs: invalid argument");
    return CM_ERR_ARG;
  }
  LbvhBufs b;
  b.t = t;
  b.lefts = (int*)d_lefts;
  b.rights = (int*)d_rights;
  b.amin = (float4*)d_aabb_min;
  b.amax = (float4*)d_aabb_max;
  b.rmll = (int*)d_rmll;
  b.rmlr = (int*)d_rmlr;
  b.warn = d_warn;
  char* tp = (char*)d_temp;
  int* chunk = (int*)tp;
  tp += align_up(sizeof(int) * (size_t)t * cap);
  int* counts = (int*)tp;
  tp += align_up(sizeof(int) * (size_t)t);
  int* offsets = (int*)tp;
  tp += align_up(sizeof(int) * (size_t)t);
  b.qnodes = (uint4*)tp;
  tp += align_up(2 * sizeof(uint4) * (size_t)t);
  if (exact_bytes(t)) b.nodes = (float4*)tp;
  tp += exact_bytes(t);
  b.spill = (int*)tp;
  tp += align_up(sizeof(int) * kSpill * (size_t)t);
  b.irr = (int*)tp;
  tp += align_up(sizeof(int));
  int rc = fill_i32(b.irr, 0, 1, (hipStream_t)stream);
  if (rc) return rc;
  rc = launch_pack_nodes(b, true, (hipStream_t)stream);
  if (rc) return rc;
  rc = scan_temp_clear(tp, t, (hipStream_t)stream);
  if (rc) return rc;
  return launch_pairs(b, cap, chunk, counts, offsets, (int2*)d_pairs, d_n_pairs, tp,
                      (hipStream_t)stream);
}

// Device-wide primitives of libclothmi, written for CDNA4 wave64:
//  * single-pass exclusive int32 scan over a device-side element count
//    (decoupled look-back, one launch, graph-capturable);
//  * stable LSD radix sort of (uint64 key, uint32 value) with 8-bit digits.
// They replace the CUB primitives the reference calls through
// LicentaV2/LicentaV2/Core/CubWrappers.cuh:24-183 (DeviceScan::ExclusiveSum,
// DeviceSelect::Flagged, DeviceRadixSort::SortPairs). Integer results are exact
// and independent of the launch shape.
#include "cm_internal.hpp"

namespace cm {

namespace {

__device__ __forceinline__ int lane_id() { return threadIdx.x & 63; }

__device__ __forceinline__ int wave_incl_scan(int v) {
  const int lane = lane_id();
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    int t = __shfl_up(v, o, 64);
    if (lane >= o) v += t;
  }
  return v;
}

__device__ __forceinline__ int wave_reduce(int v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Exclusive scan across a 256-thread block; lds needs 5 ints.
__device__ __forceinline__ int block_excl_scan(int v, int* lds, int& total) {
  const int lane = lane_id(), wid = threadIdx.x >> 6;
  int inc = wave_incl_scan(v);
  if (lane == 63) lds[wid] = inc;
  __syncthreads();
  if (threadIdx.x == 0) {
    int run = 0;
    for (int w = 0; w < kBlock / 64; ++w) {
      int t = lds[w];
      lds[w] = run;
      run += t;
    }
    lds[kBlock / 64] = run;
  }
  __syncthreads();
  int res = inc - v + lds[wid];
  total = lds[kBlock / 64];
  __syncthreads();
  return res;
}

// ---- single-pass exclusive scan -------------------------------------------------
// Tiles of kScanTile elements are taken in order from a ticket counter; each tile
// publishes its sum, looks back over its predecessors (one wave reads 64 tile
// states at a time) until it meets an inclusive prefix, then publishes its own
// inclusive prefix and writes its outputs. A tile state is one 64-bit word (flag
// in bits 62-63: 0 empty, 1 tile sum, 2 inclusive prefix; value in bits 0-31)
// written and read with device-scope relaxed atomics, so no cache-wide fences are
// needed. The last workgroup to finish clears the states and counters, leaving the
// temp ready for the next scan on the stream.
constexpr int kScanItems = 16;
constexpr int kScanTile = kBlock * kScanItems;  // 4096
constexpr int kScanMaxGrid = 256;
constexpr unsigned long long kFlagAgg = 1ull << 62, kFlagInc = 2ull << 62;

__device__ __forceinline__ unsigned long long ld_state(const unsigned long long* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_state(unsigned long long* p, unsigned long long v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__global__ void __launch_bounds__(kBlock) k_scan(const int* in, int* out, int n_max,
                                                 const int* __restrict__ d_n,
                                                 int* __restrict__ d_total, int* __restrict__ ctr,
                                                 unsigned long long* __restrict__ state) {
  __shared__ int lds[kBlock / 64 + 1];
  __shared__ int s_tile, s_prefix, s_last;
  const int n = max(0, d_n ? min(*d_n, n_max) : n_max);
  const int ntiles = (n + kScanTile - 1) / kScanTile;
  const int lane = lane_id();
  if (n == 0 && blockIdx.x == 0 && threadIdx.x == 0 && d_total) *d_total = 0;
  const bool vec = ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 15) == 0;
  for (;;) {
    if (threadIdx.x == 0) s_tile = atomicAdd(&ctr[0], 1);
    __syncthreads();
    const int tile = s_tile;
    if (tile >= ntiles) break;
    const int base = tile * kScanTile + threadIdx.x * kScanItems;
    int v[kScanItems];
    if (vec && base + kScanItems <= n) {
#pragma unroll
      for (int q = 0; q < kScanItems / 4; ++q) {
        const int4 t4 = reinterpret_cast<const int4*>(in + base)[q];
        v[4 * q] = t4.x; v[4 * q + 1] = t4.y; v[4 * q + 2] = t4.z; v[4 * q + 3] = t4.w;
      }
    } else {
#pragma unroll
      for (int k = 0; k < kScanItems; ++k) v[k] = base + k < n ? in[base + k] : 0;
    }
    int sum = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) sum += v[k];
    int total;
    const int ex = block_excl_scan(sum, lds, total);
    if (threadIdx.x < 64) {
      int prefix = 0;
      if (tile > 0) {
        if (lane == 0) st_state(&state[tile], kFlagAgg | (unsigned)total);
        int j = tile - 1;
        for (;;) {
          const int idx = j - lane;  // lane 0 is the nearest predecessor
          const unsigned long long st = idx >= 0 ? ld_state(&state[idx]) : kFlagInc;
          const unsigned flag = (unsigned)(st >> 62);
          const unsigned long long pm = __ballot(flag == 2u), zm = __ballot(flag == 0u);
          const int first = pm ? __ffsll((long long)pm) - 1 : 64;
          const unsigned long long need = first == 64 ? ~0ull : ((2ull << first) - 1ull);
          if (zm & need) continue;  // a predecessor up to the first prefix is still empty
          prefix += wave_reduce(lane <= first ? (int)(unsigned)st : 0);
          if (first < 64) break;
          j -= 64;
        }
      }
      if (lane == 0) {
        st_state(&state[tile], kFlagInc | (unsigned)(prefix + total));
        s_prefix = prefix;
      }
    }
    __syncthreads();
    int run = s_prefix + ex;
    if (vec && base + kScanItems <= n) {
#pragma unroll
      for (int q = 0; q < kScanItems / 4; ++q) {
        int4 o;
        o.x = run; run += v[4 * q];
        o.y = run; run += v[4 * q + 1];
        o.z = run; run += v[4 * q + 2];
        o.w = run; run += v[4 * q + 3];
        reinterpret_cast<int4*>(out + base)[q] = o;
      }
    } else {
#pragma unroll
      for (int k = 0; k < kScanItems; ++k)
        if (base + k < n) {
          out[base + k] = run;
          run += v[k];
        }
    }
    if (tile == ntiles - 1 && threadIdx.x == 0 && d_total) *d_total = s_prefix + total;
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    __threadfence();
    s_last = atomicAdd(&ctr[1], 1) == (int)gridDim.x - 1;
  }
  __syncthreads();
  if (s_last) {
    for (int i = threadIdx.x; i < ntiles; i += kBlock) st_state(&state[i], 0ull);
    if (threadIdx.x == 0) {
      ctr[0] = 0;
      ctr[1] = 0;
    }
  }
}

__global__ void k_fill_i32(int* __restrict__ p, int v, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

// ---- radix sort ------------------------------------------------------------
constexpr int kWaves = kBlock / 64;

// Lanes whose digit equals this lane's, among those in `valid`. A bit costs a shift, a
// compare, and an xor and an and for each half of the mask (before, with a select for each
// half: 2.1 M keys of 30 bits 231 us, now 172).
__device__ __forceinline__ uint64_t match_digit(uint32_t d, uint64_t valid) {
  uint64_t m = valid;
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    const int sx = (int)(d << (31 - b)) >> 31;  // the bit in every place
    m &= ~(__ballot(sx != 0) ^ (uint64_t)(int64_t)sx);
  }
  return m;
}

// Digit counts of each tile: hist[digit * nblk + tile] for the scan, or, with by_tile,
// hist[tile * 256 + digit] for scatter kernels that add up the tiles before theirs.
__global__ void __launch_bounds__(kBlock) k_radix_hist(const uint64_t* __restrict__ keys, int n,
                                                       int shift, int nblk, int by_tile,
                                                       int* __restrict__ hist) {
  __shared__ int h[256];
  h[threadIdx.x] = 0;
  __syncthreads();
  const int base = blockIdx.x * kSortTile;
#pragma unroll
  for (int k = 0; k < kSortItems; ++k) {
    int i = base + k * kBlock + threadIdx.x;
    if (i < n) atomicAdd(&h[(keys[i] >> shift) & 255u], 1);
  }
  __syncthreads();
  hist[by_tile ? blockIdx.x * 256 + threadIdx.x : threadIdx.x * nblk + blockIdx.x] =
      h[threadIdx.x];
}

// Up to this many tiles a scatter kernel adds up the tiles' digit counts itself, which costs
// it about 1 us where the scan is a launch of 5: 32,258 keys of 30 bits 73 -> 53 us, 130,050
// 79 -> 60. Every tile reads all counts, so many tiles are left to the scan: 500,000 keys
// 91 us by the scan, 93 or more by the tiles.
constexpr int kByTileMax = 64;

// Where thread d's digit begins for block blk of nblk, from hist[block * 256 + digit]: the
// digits below it and the blocks before this one.
__device__ __forceinline__ int digit_start(const int* __restrict__ hist, int blk, int nblk) {
  __shared__ int lds[kBlock / 64 + 1];
  int before = 0, total = 0;
  for (int b0 = 0; b0 < nblk; b0 += 16) {  // 16 loads at a time, also for the last few
    int v[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) v[j] = hist[min(b0 + j, nblk - 1) * 256 + threadIdx.x];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      before += b0 + j < blk ? v[j] : 0;
      total += b0 + j < nblk ? v[j] : 0;
    }
  }
  int all;
  return block_excl_scan(total, lds, all) + before;
}

// Stable scatter: wave w ranks the contiguous slice [w*64*ITEMS, (w+1)*64*ITEMS)
// of the tile in order, using 8 ballots per 64-key chunk to find equal digits.
// kByTile: offsets holds the tiles' digit counts, else where each (digit, tile) begins.
template <bool kByTile>
__global__ void __launch_bounds__(kBlock) k_radix_scatter(
    const uint64_t* __restrict__ kin, const uint32_t* __restrict__ vin,
    uint64_t* __restrict__ kout, uint32_t* __restrict__ vout, int n, int shift, int nblk,
    const int* __restrict__ offsets) {
  __shared__ int cnt[kWaves][256];
  __shared__ int wbase[kWaves][256];
  const int lane = lane_id(), wid = threadIdx.x >> 6;
  for (int d = threadIdx.x; d < kWaves * 256; d += kBlock) (&cnt[0][0])[d] = 0;
  __syncthreads();
  const int base = blockIdx.x * kSortTile + wid * 64 * kSortItems;
  uint64_t key[kSortItems];
  uint32_t val[kSortItems];
  int rank[kSortItems];
  const uint64_t lt = (1ull << lane) - 1ull;
  const int start = kByTile ? digit_start(offsets, blockIdx.x, nblk)
                            : offsets[threadIdx.x * nblk + blockIdx.x];
#pragma unroll
  for (int c = 0; c < kSortItems; ++c) {
    const int i = base + c * 64 + lane;
    const bool valid = i < n;
    key[c] = valid ? kin[i] : 0ull;
    val[c] = valid ? vin[i] : 0u;
    const uint32_t d = (uint32_t)(key[c] >> shift) & 255u;
    const uint64_t m = match_digit(d, __ballot(valid));
    int r = 0;
    if (valid) {
      const int before = __popcll(m & lt);
      const int old = cnt[wid][d];
      r = old + before;
      if (before == 0) cnt[wid][d] = old + __popcll(m);
    }
    rank[c] = r;
  }
  __syncthreads();
  {
    const int d = threadIdx.x;  // kBlock == 256 digits
    int run = start;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      wbase[w][d] = run;
      run += cnt[w][d];
    }
  }
  __syncthreads();
#pragma unroll
  for (int c = 0; c < kSortItems; ++c) {
    const int i = base + c * 64 + lane;
    if (i < n) {
      const uint32_t d = (uint32_t)(key[c] >> shift) & 255u;
      const int pos = wbase[wid][d] + rank[c];
      kout[pos] = key[c];
      vout[pos] = val[c];
    }
  }
}

// ---- radix sort in one workgroup ---------------------------------------------------
// Up to kBlockSort keys are sorted by one workgroup, the keys (their low 32 bits where no
// higher one is sorted by) and their 16-bit places in its LDS, in one launch for all
// passes. A thread holds its keys in registers from one pass's read to the next one's
// write. Bound by the ranking (about four vector instructions a bit for 64 keys) on one
// CU, so longer sorts go to the whole chip. 6,962 keys of 30 bits 69 -> 33 us, of 63 bits
// 136 -> 64; 8,192 keys 68 -> 37 (51 on the whole chip), 12,000 keys
// 72 -> 51 there and 54 here.
constexpr int kSortThreads = 1024, kSortWaves = kSortThreads / 64;
constexpr int kBlockItems = 8;  // most keys per thread
constexpr int kBlockSort = kBlockItems * kSortThreads;
constexpr int kSortHead = sizeof(int) * (kSortWaves * 256 + 4);

template <typename K>
__global__ void __launch_bounds__(kSortThreads) k_sort_block(uint64_t* keys, uint32_t* vals, int n,
                                                             int passes) {
  extern __shared__ char sort_lds[];
  int(*cnt)[256] = (int(*)[256])sort_lds;  // per wave and digit: count, then first place
  int* wtot = (int*)(cnt + kSortWaves);    // 4: digit totals of 64 digits
  K* skey = (K*)(wtot + 4);
  uint16_t* sidx = (uint16_t*)(skey + n);
  const int lane = lane_id(), wid = threadIdx.x >> 6;
  const uint64_t below = (1ull << lane) - 1ull;
  // wave w takes the n items in order from w * per
  const int items = (n + kSortThreads - 1) / kSortThreads;
  const int base = wid * 64 * items + lane;
  K key[kBlockItems];
  uint32_t at[kBlockItems];  // place in the caller's order (low half), rank in the wave (high)
#pragma unroll
  for (int c = 0; c < kBlockItems; ++c) {
    const int i = base + c * 64;
    key[c] = c < items && i < n ? (K)keys[i] : (K)0;
    at[c] = (uint32_t)i & 0xffffu;
  }
  for (int pass = 0; pass < passes; ++pass) {
    const int shift = 8 * pass;
    for (int d = lane; d < 256; d += 64) cnt[wid][d] = 0;
#pragma unroll
    for (int c = 0; c < kBlockItems; ++c) {
      if (c >= items) break;
      const bool valid = base + c * 64 < n;
      const uint32_t d = (uint32_t)(key[c] >> shift) & 255u;
      const uint64_t m = match_digit(d, __ballot(valid));
      const int before = __popcll(m & below);
      if (valid) {
        const int old = cnt[wid][d];
        if (before == 0) cnt[wid][d] = old + __popcll(m);
        at[c] |= (uint32_t)(old + before) << 16;
      }
    }
    __syncthreads();
    if (threadIdx.x < 256) {
      int run = 0;
#pragma unroll
      for (int w = 0; w < kSortWaves; ++w) {
        const int v = cnt[w][threadIdx.x];
        cnt[w][threadIdx.x] = run;
        run += v;
      }
      const int inc = wave_incl_scan(run);
      if (lane == 63) wtot[wid] = inc;
      cnt[0][threadIdx.x] = inc - run;  // wave 0's own base is 0: here the digit's base
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < kBlockItems; ++c) {
      if (c >= items) break;
      if (base + c * 64 < n) {
        const uint32_t d = (uint32_t)(key[c] >> shift) & 255u;
        int pos = cnt[0][d] + (int)(at[c] >> 16) + (wid ? cnt[wid][d] : 0);
#pragma unroll
        for (int w = 0; w < 3; ++w) pos += (int)(d >> 6) > w ? wtot[w] : 0;
        skey[pos] = key[c];
        sidx[pos] = (uint16_t)at[c];
      }
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < kBlockItems; ++c) {
      const int i = base + c * 64;
      if (c < items && i < n) {
        key[c] = skey[i];
        at[c] = sidx[i];
      }
    }
  }
  // whole keys and values from the caller's order; all are read before one is written
  uint64_t k64[kBlockItems];
  uint32_t v32[kBlockItems];
#pragma unroll
  for (int c = 0; c < kBlockItems; ++c)
    if (c < items && base + c * 64 < n) {
      k64[c] = keys[at[c]];
      v32[c] = vals[at[c]];
    }
  __syncthreads();
#pragma unroll
  for (int c = 0; c < kBlockItems; ++c)
    if (c < items && base + c * 64 < n) {
      keys[base + c * 64] = k64[c];
      vals[base + c * 64] = v32[c];
    }
}

// ---- radix sort of 32-bit keys with a device-side count --------------------------
// A fixed grid of kDevSortBlocks workgroups; workgroup b takes the run of tiles that
// dev_sort_range gives it, so one histogram per workgroup keeps the sort stable and the
// launch shape does not depend on n. A workgroup adds up the counts of the workgroups
// before it (digit_start), which a few workgroups do faster than a scan's launch takes.
__global__ void __launch_bounds__(kBlock) k_radix_hist_dev(const uint32_t* __restrict__ keys,
                                                           const int* __restrict__ d_n, int n_max,
                                                           int shift, int* __restrict__ hist) {
  __shared__ int h[256];
  const DevSortRange r = dev_sort_range(min(*d_n, n_max));
  if (r.t0 >= r.t1) return;
  h[threadIdx.x] = 0;
  __syncthreads();
  for (int tile = r.t0; tile < r.t1; ++tile) {
#pragma unroll
    for (int k = 0; k < kSortItems; ++k) {
      const int i = tile * kSortTile + k * kBlock + threadIdx.x;
      if (i < r.n) atomicAdd(&h[(keys[i] >> shift) & 255u], 1);
    }
  }
  __syncthreads();
  hist[blockIdx.x * 256 + threadIdx.x] = h[threadIdx.x];
}

// k_radix_scatter over the workgroup's run of tiles, each digit's running place carried
// from tile to tile (thread d owns digit d of carry, wbase and the count sums)
__global__ void __launch_bounds__(kBlock) k_radix_scatter_dev(
    const uint32_t* __restrict__ kin, const uint32_t* __restrict__ vin,
    uint32_t* __restrict__ kout, uint32_t* __restrict__ vout, const int* __restrict__ d_n,
    int n_max, int shift, const int* __restrict__ hist) {
  __shared__ int cnt[kWaves][256];
  __shared__ int wbase[kWaves][256];
  const DevSortRange r = dev_sort_range(min(*d_n, n_max));
  if (r.t0 >= r.t1) return;
  const int lane = lane_id(), wid = threadIdx.x >> 6;
  int carry = digit_start(hist, blockIdx.x, r.blocks);
  const uint64_t lt = (1ull << lane) - 1ull;
  uint32_t nkey[kSortItems], nval[kSortItems];  // the next tile's, loaded a tile ahead
  auto load = [&](int tile) {
#pragma unroll
    for (int c = 0; c < kSortItems; ++c) {
      const int i = min(tile * kSortTile + (wid * kSortItems + c) * 64 + lane, r.n - 1);
      nkey[c] = kin[i];
      nval[c] = vin[i];
    }
  };
  load(r.t0);
  for (int tile = r.t0; tile < r.t1; ++tile) {
    for (int d = threadIdx.x; d < kWaves * 256; d += kBlock) (&cnt[0][0])[d] = 0;
    const int base = tile * kSortTile + wid * 64 * kSortItems;
    uint32_t key[kSortItems], val[kSortItems];
    int rank[kSortItems];
#pragma unroll
    for (int c = 0; c < kSortItems; ++c) {
      key[c] = nkey[c];
      val[c] = nval[c];
    }
    if (tile + 1 < r.t1) load(tile + 1);
    __syncthreads();
#pragma unroll
    for (int c = 0; c < kSortItems; ++c) {
      const bool valid = base + c * 64 + lane < r.n;
      const uint32_t d = (key[c] >> shift) & 255u;
      const uint64_t m = match_digit(d, __ballot(valid));
      int q = 0;
      if (valid) {
        const int before = __popcll(m & lt);
        const int old = cnt[wid][d];
        q = old + before;
        if (before == 0) cnt[wid][d] = old + __popcll(m);
      }
      rank[c] = q;
    }
    __syncthreads();
    {
      const int d = threadIdx.x;  // kBlock == 256 digits
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        wbase[w][d] = carry;
        carry += cnt[w][d];
      }
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < kSortItems; ++c) {
      const int i = base + c * 64 + lane;
      if (i < r.n) {
        const uint32_t d = (key[c] >> shift) & 255u;
        const int pos = wbase[wid][d] + rank[c];
        kout[pos] = key[c];
        vout[pos] = val[c];
      }
    }
    __syncthreads();
  }
}

// ---- scan of per-tile sums ----------------------------------------------------------
// Kernels that produce counts in tiles of consecutive items also write each tile's sum;
// this scan turns the sums into tile prefixes, and the consuming kernel adds the
// exclusive scan within its tile. The counts are then read once instead of three
// times. A packed sum holds two counts below 2^16 (low and high half), scanned
// separately; the totals are clamped to the buffers they index. It is the
// single-pass look-back scan above carried over to a pair of counts: a thread adds
// both as one 64-bit sum (first count in the low word), and a tile state holds the
// two running counts in 31 bits each (every count and total is below 2^31).
__device__ __forceinline__ unsigned long long wave_incl_scan64(unsigned long long v) {
  const int lane = lane_id();
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned long long t = __shfl_up(v, o, 64);
    if (lane >= o) v += t;
  }
  return v;
}
__device__ __forceinline__ unsigned long long wave_reduce64(unsigned long long v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
__device__ __forceinline__ unsigned long long pair_of(int v, int packed) {
  return packed ? (unsigned long long)(v & 0xffff) | ((unsigned long long)((unsigned)v >> 16) << 32)
                : (unsigned long long)(unsigned)v;
}
// 64-bit pair sum <-> the 62 value bits of a tile state
__device__ __forceinline__ unsigned long long pack31(unsigned long long x) {
  return (x & 0x7fffffffull) | (((x >> 32) & 0x7fffffffull) << 31);
}
__device__ __forceinline__ unsigned long long unpack31(unsigned long long st) {
  return (st & 0x7fffffffull) | (((st >> 31) & 0x7fffffffull) << 32);
}

__global__ void __launch_bounds__(kBlock) k_scan_tiles(
    const int* __restrict__ d_items, TileRule rule, int64_t n_max, const int* sums, int* pre,
    int packed, int64_t cap0, int64_t cap1, int* __restrict__ d_tot0, int* __restrict__ d_tot1,
    int* __restrict__ ctr, unsigned long long* __restrict__ state) {
  __shared__ unsigned long long lds[kBlock / 64 + 1];
  __shared__ unsigned long long s_prefix;
  __shared__ int s_tile, s_last;
  int n = (int)n_max;  // tiles; with d_items, the tiles of at most n_max items
  if (d_items) {
    const int items = (int)min((int64_t)max(0, *d_items), n_max);
    const int per = 64 * tile_lanes(rule, items);
    n = items / per + (items % per != 0);
  }
  const int ntiles = (n + kScanTile - 1) / kScanTile;
  const int lane = lane_id(), wid = threadIdx.x >> 6;
  if (n == 0 && blockIdx.x == 0 && threadIdx.x == 0) {
    if (d_tot0) *d_tot0 = 0;
    if (packed && d_tot1) *d_tot1 = 0;
  }
  const bool vin = (reinterpret_cast<uintptr_t>(sums) & 15) == 0;
  const bool vout = (reinterpret_cast<uintptr_t>(pre) & 15) == 0;
  for (;;) {
    if (threadIdx.x == 0) s_tile = atomicAdd(&ctr[0], 1);
    __syncthreads();
    const int tile = s_tile;
    if (tile >= ntiles) break;
    const int base = tile * kScanTile + threadIdx.x * kScanItems;
    const bool full = base + kScanItems <= n;
    int v[kScanItems];
    if (vin && full) {
#pragma unroll
      for (int q = 0; q < kScanItems / 4; ++q) {
        const int4 t4 = reinterpret_cast<const int4*>(sums + base)[q];
        v[4 * q] = t4.x; v[4 * q + 1] = t4.y; v[4 * q + 2] = t4.z; v[4 * q + 3] = t4.w;
      }
    } else {
#pragma unroll
      for (int k = 0; k < kScanItems; ++k) v[k] = base + k < n ? sums[base + k] : 0;
    }
    unsigned long long sum = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) sum += pair_of(v[k], packed);
    // exclusive scan of the thread sums over the workgroup
    const unsigned long long inc = wave_incl_scan64(sum);
    if (lane == 63) lds[wid] = inc;
    __syncthreads();
    if (threadIdx.x == 0) {
      unsigned long long run = 0;
      for (int w = 0; w < kBlock / 64; ++w) {
        const unsigned long long t = lds[w];
        lds[w] = run;
        run += t;
      }
      lds[kBlock / 64] = run;
    }
    __syncthreads();
    const unsigned long long ex = inc - sum + lds[wid];
    const unsigned long long total = lds[kBlock / 64];
    if (threadIdx.x < 64) {
      unsigned long long prefix = 0;
      if (tile > 0) {
        if (lane == 0) st_state(&state[tile], kFlagAgg | pack31(total));
        int j = tile - 1;
        for (;;) {
          const int idx = j - lane;  // lane 0 is the nearest predecessor
          const unsigned long long st = idx >= 0 ? ld_state(&state[idx]) : kFlagInc;
          const unsigned flag = (unsigned)(st >> 62);
          const unsigned long long pm = __ballot(flag == 2u), zm = __ballot(flag == 0u);
          const int first = pm ? __ffsll((long long)pm) - 1 : 64;
          const unsigned long long need = first == 64 ? ~0ull : ((2ull << first) - 1ull);
          if (zm & need) continue;  // a predecessor up to the first prefix is still empty
          prefix += wave_reduce64(lane <= first ? unpack31(st) : 0ull);
          if (first < 64) break;
          j -= 64;
        }
      }
      if (lane == 0) {
        st_state(&state[tile], kFlagInc | pack31(prefix + total));
        s_prefix = prefix;
      }
    }
    __syncthreads();
    unsigned long long run = s_prefix + ex;
    if (vout && full) {
      if (packed) {
#pragma unroll
        for (int q = 0; q < kScanItems / 2; ++q) {
          int4 o;
          o.x = (int)(unsigned)run;
          o.y = (int)(run >> 32);
          run += pair_of(v[2 * q], 1);
          o.z = (int)(unsigned)run;
          o.w = (int)(run >> 32);
          run += pair_of(v[2 * q + 1], 1);
          reinterpret_cast<int4*>(pre + 2 * base)[q] = o;
        }
      } else {
#pragma unroll
        for (int q = 0; q < kScanItems / 4; ++q) {
          int4 o;
          o.x = (int)run; run += (unsigned)v[4 * q];
          o.y = (int)run; run += (unsigned)v[4 * q + 1];
          o.z = (int)run; run += (unsigned)v[4 * q + 2];
          o.w = (int)run; run += (unsigned)v[4 * q + 3];
          reinterpret_cast<int4*>(pre + base)[q] = o;
        }
      }
    } else {
#pragma unroll
      for (int k = 0; k < kScanItems; ++k)
        if (base + k < n) {
          if (packed) {
            pre[2 * (base + k)] = (int)(unsigned)run;
            pre[2 * (base + k) + 1] = (int)(run >> 32);
          } else {
            pre[base + k] = (int)(unsigned)run;
          }
          run += pair_of(v[k], packed);
        }
    }
    if (tile == ntiles - 1 && threadIdx.x == 0) {
      const unsigned long long all = s_prefix + total;
      if (d_tot0) *d_tot0 = (int)min<int64_t>((int64_t)(all & 0xffffffffull), cap0);
      if (packed && d_tot1) *d_tot1 = (int)min<int64_t>((int64_t)(all >> 32), cap1);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    __threadfence();
    s_last = atomicAdd(&ctr[1], 1) == (int)gridDim.x - 1;
  }
  __syncthreads();
  if (s_last) {
    for (int i = threadIdx.x; i < ntiles; i += kBlock) st_state(&state[i], 0ull);
    if (threadIdx.x == 0) {
      ctr[0] = 0;
      ctr[1] = 0;
    }
  }
}

}  // namespace

static int lookback_tiles(int64_t n_max) {
  return (int)std::max<int64_t>(1, (n_max + kScanTile - 1) / kScanTile);
}

size_t scan_temp_bytes(int n_max) {
  return 256 + align_up(sizeof(unsigned long long) * (size_t)lookback_tiles(n_max));
}

int scan_temp_clear(void* temp, int n_max, hipStream_t s) {
  return fill_i32((int*)temp, 0, (int64_t)(scan_temp_bytes(n_max) / sizeof(int)), s);
}

int scan_exclusive(const int* in, int* out, int n_max, const int* d_n, int* d_total, void* temp,
                   hipStream_t s) {
  int* ctr = (int*)temp;
  unsigned long long* state = (unsigned long long*)((char*)temp + 256);
  const int grid = std::min(lookback_tiles(n_max), kScanMaxGrid);
  hipLaunchKernelGGL(k_scan, dim3(grid), dim3(kBlock), 0, s, in, out, n_max, d_n, d_total, ctr,
                     state);
  CM_LAUNCH_CHECK();
  return CM_OK;
}

static int scan_tiles_grid(const int* d_items, TileRule rule, int64_t n_max, int64_t ntile,
                    const int* sums, int* pre, int packed, int64_t cap0, int64_t cap1,
                    int* d_tot0, int* d_tot1, void* temp, hipStream_t s) {
  int* ctr = (int*)temp;
  unsigned long long* state = (unsigned long long*)((char*)temp + 256);
  const int grid = std::min(lookback_tiles(ntile), kScanMaxGrid);
  hipLaunchKernelGGL(k_scan_tiles, dim3(grid), dim3(kBlock), 0, s, d_items, rule, n_max, sums, pre,
                     packed, cap0, cap1, d_tot0, d_tot1, ctr, state);
  CM_LAUNCH_CHECK();
  return CM_OK;
}

int scan_tiles(int n, const int* sums, int* pre, int packed, int64_t cap0, int64_t cap1,
               int* d_tot0, int* d_tot1, void* temp, hipStream_t s) {
  return scan_tiles_grid(nullptr, kTileSmall, n, n, sums, pre, packed, cap0, cap1, d_tot0, d_tot1,
                         temp, s);
}

int scan_tiles_dev(const int* d_items, TileRule rule, int64_t item_cap, const int* sums, int* pre,
                   int packed, int64_t cap0, int64_t cap1, int* d_tot0, int* d_tot1, void* temp,
                   hipStream_t s) {
  return scan_tiles_grid(d_items, rule, item_cap, tile_max(rule, item_cap), sums, pre, packed,
                         cap0, cap1, d_tot0, d_tot1, temp, s);
}

int fill_i32(int* p, int v, int64_t n, hipStream_t s) {
  if (n <= 0) return CM_OK;
  int grid = (int)std::min<int64_t>((n + kBlock - 1) / kBlock, 4096);
  hipLaunchKernelGGL(k_fill_i32, dim3(grid), dim3(kBlock), 0, s, p, v, n);
  CM_LAUNCH_CHECK();
  return CM_OK;
}
int fill_u32(uint32_t* p, uint32_t v, int64_t n, hipStream_t s) {
  return fill_i32((int*)p, (int)v, n, s);
}

static int sort_blocks(int n) { return (n + kSortTile - 1) / kSortTile; }

size_t radix_sort_temp_bytes(int n) {
  int nb = sort_blocks(n);
  return align_up(sizeof(uint64_t) * (size_t)n) + align_up(sizeof(uint32_t) * (size_t)n) +
         align_up(sizeof(int) * 256 * (size_t)nb) + scan_temp_bytes(256 * nb);
}

// The scan part of a sort temp must start zeroed (each scan leaves it zeroed).
int radix_sort_clear(void* temp, int n, hipStream_t s) {
  const int nb = sort_blocks(n);
  char* tp = (char*)temp + align_up(sizeof(uint64_t) * (size_t)n) +
             align_up(sizeof(uint32_t) * (size_t)n) + align_up(sizeof(int) * 256 * (size_t)nb);
  return scan_temp_clear(tp, 256 * nb, s);
}

size_t radix_sort_dev_temp_bytes() { return align_up(sizeof(int) * 256 * kDevSortBlocks); }

int radix_sort_dev(uint32_t* keys, uint32_t* vals, uint32_t* keys_alt, uint32_t* vals_alt,
                   int n_max, const int* d_n, int key_bits, int* hist, int* in_alt,
                   hipStream_t s) {
  const int passes = std::min(4, (key_bits + 7) / 8);
  uint32_t *ka = keys, *va = vals, *kb = keys_alt, *vb = vals_alt;
  for (int pass = 0; pass < passes; ++pass) {
    const int shift = 8 * pass;
    if (pass > 0)
      hipLaunchKernelGGL(k_radix_hist_dev, dim3(kDevSortBlocks), dim3(kBlock), 0, s, ka, d_n,
                         n_max, shift, hist);
    hipLaunchKernelGGL(k_radix_scatter_dev, dim3(kDevSortBlocks), dim3(kBlock), 0, s, ka, va, kb,
                       vb, d_n, n_max, shift, hist);
    CM_LAUNCH_CHECK();
    std::swap(ka, kb);
    std::swap(va, vb);
  }
  *in_alt = passes & 1;
  return CM_OK;
}

template <typename K>
static int sort_block(uint64_t* keys, uint32_t* vals, int n, int passes, hipStream_t s) {
  const size_t lds = kSortHead + (sizeof(K) + 2) * (size_t)n;
  // the most that any call needs, whatever this one does: other threads sort too
  CM_HIP(hipFuncSetAttribute((const void*)k_sort_block<K>,
                             hipFuncAttributeMaxDynamicSharedMemorySize,
                             (int)(kSortHead + (sizeof(K) + 2) * kBlockSort)));
  hipLaunchKernelGGL(k_sort_block<K>, dim3(1), dim3(kSortThreads), lds, s, keys, vals, n,
                     passes);
  CM_LAUNCH_CHECK();
  return CM_OK;
}

int radix_sort(uint64_t* keys, uint32_t* vals, int n, int key_bits, void* temp, hipStream_t s) {
  if (n <= 1) return CM_OK;
  const int nb = sort_blocks(n);
  char* tp = (char*)temp;
  uint64_t* kalt = (uint64_t*)tp;
  tp += align_up(sizeof(uint64_t) * (size_t)n);
  uint32_t* valt = (uint32_t*)tp;
  tp += align_up(sizeof(uint32_t) * (size_t)n);
  int* hist = (int*)tp;
  tp += align_up(sizeof(int) * 256 * (size_t)nb);
  void* stemp = tp;
  int passes = (key_bits + 7) / 8;
  if (passes & 1) ++passes;  // even number of passes: result ends in the input buffers
  if (n <= kBlockSort)
    return passes <= 4 ? sort_block<uint32_t>(keys, vals, n, passes, s)
                       : sort_block<uint64_t>(keys, vals, n, passes, s);
  uint64_t* ka = keys;
  uint32_t* va = vals;
  uint64_t* kb = kalt;
  uint32_t* vb = valt;
  for (int pass = 0; pass < passes; ++pass) {
    const int shift = 8 * pass;
    const bool by_tile = nb <= kByTileMax;
    hipLaunchKernelGGL(k_radix_hist, dim3(nb), dim3(kBlock), 0, s, ka, n, shift, nb, by_tile, hist);
    if (by_tile) {
      hipLaunchKernelGGL(k_radix_scatter<true>, dim3(nb), dim3(kBlock), 0, s, ka, va, kb, vb, n,
                         shift, nb, hist);
    } else {
      int rc = scan_exclusive(hist, hist, 256 * nb, nullptr, nullptr, stemp, s);
      if (rc) return rc;
      hipLaunchKernelGGL(k_radix_scatter<false>, dim3(nb), dim3(kBlock), 0, s, ka, va, kb, vb, n,
                         shift, nb, hist);
    }
    CM_LAUNCH_CHECK();
    std::swap(ka, kb);
    std::swap(va, vb);
  }
  return CM_OK;
}

}  // namespace cm

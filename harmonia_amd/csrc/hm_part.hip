// One-pass partition of a query batch for searches that return their results in input order, and its
// undoing.
//
// Measured, 2^24 queries: histogram 33 us, scan 17, scatter 72, un-scatter 92, where the two 8-bit passes
// took 58, 10, 132 and 159; 2^20 queries: 4.0, 4.7, 8.9 and 9.8 against 8.7, 8.5, 25 and 20.  The whole
// search went 699 -> 565 us at 2^24 on 2^26 keys and 82 -> 48 us at 2^20 on 2^20.  What bounds it: memory at
// the copy rate (the histogram reads 134 MB, the scatter moves 318 MB); the un-scatter's 2048 short runs per
// tile (nine or ten bits instead of eleven: 81 and 96 us for then 120, but the search reads more leaves
// twice, 455 and 423 us for 404; 1024 threads per tile: 124).  It gathered the found flags too, a second
// line per run: 120 us until a mark among the values took their place.
//
// Such a search may take its queries in any order that brings neighbours together, so the batch is split
// once by the top bits of the tree's key range into buckets of a few thousand queries (histogram, scan,
// scatter) and each block of the search sorts its share of a bucket further in LDS.  A second global pass
// (two 8-bit digits, stable) cost another histogram, scan, scatter and un-scatter.  The order inside a
// bucket is left open, so an LDS atomic gives each key its place in the tile.
//
// Undoing: the scatter recorded each query's place in its tile's staging (16 bits) and the offsets of the
// tile's runs, so a block gathers its tile's runs from the results, stages them in LDS and writes them in
// input order.
#include "hm_block.h"
#include "hm_internal.h"

namespace hm {
namespace {

constexpr int kThreads = 512;
constexpr int kItems = 16;
constexpr int kTile = kThreads * kItems;
constexpr int kDigits = 1 << kPartMaxBits;
constexpr int kDPer = kDigits / kThreads;  // digits per thread
static_assert(kDPer == 4, "a thread's digits are one 16-byte load");
static_assert(kTile <= 65536, "staging indices are 16-bit");

// As the radix sort: XCD x takes a contiguous eighth of the tiles, so partial cache lines at the ends of
// neighbouring tiles' runs meet in one L2.
__device__ __forceinline__ uint32_t tiles_of(size_t n) { return (uint32_t)((n + kTile - 1) / kTile); }
unsigned grid_for(size_t nb) { return (unsigned)((nb + 7) / 8 * 8); }

// counts[tile][digit], one block per tile.  VEC: keys 16-byte aligned.
template <bool VEC>
__global__ __launch_bounds__(kThreads) void part_hist_kernel(const uint64_t* __restrict__ keys, size_t n, int shift,
                                                             uint32_t nd, uint32_t* __restrict__ counts,
                                                             uint32_t* __restrict__ clash,
                                                             const uint32_t* __restrict__ dn) {
  __shared__ uint32_t h[kDigits];
  if (dn) n = *dn;
  const uint32_t tile = xcd_share(blockIdx.x, tiles_of(n));
  if (tile >= tiles_of(n)) return;  // block-uniform
  if (clash && tile == 0 && threadIdx.x == 0) *clash = 0;
  const uint32_t mask = nd - 1;
  for (uint32_t d = threadIdx.x; d < nd; d += kThreads) h[d] = 0;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const size_t base = (size_t)tile * kTile + (size_t)w * 64 * kItems;
  if (VEC && (size_t)(tile + 1) * kTile <= n) {  // block-uniform
    const ulonglong2* src = reinterpret_cast<const ulonglong2*>(keys + base);
    ulonglong2 kk[kItems / 2];
#pragma unroll
    for (int r = 0; r < kItems / 2; ++r) kk[r] = src[r * 64 + lane];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kItems / 2; ++r) {
      const uint32_t dx = (uint32_t)(kk[r].x >> shift) & mask, dy = (uint32_t)(kk[r].y >> shift) & mask;
      const uint32_t d0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)dx);
      if (__ballot(dx == d0 && dy == d0) == ~0ull) {  // sorted runs, a hot key: one add for the wave's 128 keys
        if (lane == 0) atomicAdd(&h[d0], 128u);
      } else {
        atomicAdd(&h[dx], 1u);
        atomicAdd(&h[dy], 1u);
      }
    }
  } else {
    const size_t last = n - 1;
    uint64_t kk[kItems];
#pragma unroll
    for (int r = 0; r < kItems; ++r) {
      const size_t i = base + (size_t)r * 64 + lane;
      kk[r] = keys[i < last ? i : last];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kItems; ++r)
      if (base + (size_t)r * 64 + lane < n) atomicAdd(&h[(uint32_t)(kk[r] >> shift) & mask], 1u);
  }
  __syncthreads();
  for (uint32_t d = threadIdx.x; d < nd; d += kThreads) counts[(size_t)tile * nd + d] = h[d];
}

// Per digit: exclusive scan of its counts along the tiles (of the *dn keys there are, if dn), in place; the
// digit's total to row nb.  A block takes 16 digits (64-byte pieces of the rows), 64 segments of tiles side by side.
constexpr int kScanThreads = 1024;
constexpr int kScanDigits = 16;
constexpr int kScanSegs = kScanThreads / kScanDigits;
constexpr int kScanBatch = 8;
__global__ __launch_bounds__(kScanThreads) void part_scan_kernel(uint32_t* __restrict__ counts, uint32_t nd,
                                                                 uint32_t nb, uint32_t limit,
                                                                 uint32_t* __restrict__ flags, uint32_t flag,
                                                                 const uint32_t* __restrict__ dn) {
  __shared__ uint32_t sums[kScanSegs][kScanDigits];
  const uint32_t live = dn ? tiles_of(*dn) : nb;
  const uint32_t j = threadIdx.x % kScanDigits, seg = threadIdx.x / kScanDigits;
  uint32_t* col = counts + blockIdx.x * kScanDigits + j;
  const uint32_t per = (live + kScanSegs - 1) / kScanSegs;
  const uint32_t t0 = seg * per < live ? seg * per : live, t1 = t0 + per < live ? t0 + per : live;
  uint32_t s = 0;
  for (uint32_t t = t0; t < t1; t += kScanBatch) {
    uint32_t v[kScanBatch];
#pragma unroll
    for (int u = 0; u < kScanBatch; ++u) v[u] = t + u < t1 ? col[(size_t)(t + u) * nd] : 0u;
#pragma unroll
    for (int u = 0; u < kScanBatch; ++u) s += v[u];
  }
  sums[seg][j] = s;
  __syncthreads();
  uint32_t run = 0, total = 0;
  for (uint32_t x = 0; x < kScanSegs; ++x) {
    const uint32_t v = sums[x][j];
    run += x < seg ? v : 0u;
    total += v;
  }
  for (uint32_t t = t0; t < t1; t += kScanBatch) {
    uint32_t v[kScanBatch];
#pragma unroll
    for (int u = 0; u < kScanBatch; ++u) v[u] = t + u < t1 ? col[(size_t)(t + u) * nd] : 0u;
#pragma unroll
    for (int u = 0; u < kScanBatch; ++u) {
      if (t + u < t1) col[(size_t)(t + u) * nd] = run;
      run += v[u];
    }
  }
  if (seg == 0) {
    col[(size_t)nb * nd] = total;
    if (flags && total > limit) atomicOr(flags, flag);  // a bucket that its block could not hold
  }
}

__device__ __forceinline__ void load_digits(const uint32_t* __restrict__ row, uint32_t d0, uint32_t nd,
                                            uint32_t (&v)[kDPer]) {
  const uint4 x = d0 < nd ? *reinterpret_cast<const uint4*>(row + d0) : make_uint4(0, 0, 0, 0);
  v[0] = x.x, v[1] = x.y, v[2] = x.z, v[3] = x.w;
}
// In: one value per digit; out: the exclusive scan over all digits.
__device__ __forceinline__ void scan_digits(uint32_t (&v)[kDPer], uint32_t* sh) {
  uint32_t s = 0, total;
#pragma unroll
  for (int j = 0; j < kDPer; ++j) s += v[j];
  uint32_t run = block_exclusive_scan<uint32_t, kThreads>(s, sh, total);
#pragma unroll
  for (int j = 0; j < kDPer; ++j) {
    const uint32_t x = v[j];
    v[j] = run;
    run += x;
  }
}

// LDS: 64 KiB of keys, 8 KiB of digits: two blocks per CU.
__global__ __launch_bounds__(kThreads) void part_scatter_kernel(const uint64_t* __restrict__ kin,
                                                                uint64_t* __restrict__ kout,
                                                                uint16_t* __restrict__ place, size_t n, int shift,
                                                                uint32_t nd, const uint32_t* __restrict__ offsets,
                                                                uint32_t nb, const uint32_t* __restrict__ dn) {
  __shared__ uint64_t skeys[kTile];
  __shared__ __align__(16) uint32_t dig[kDigits];  // counts, then tile offsets, then output minus tile offsets
  __shared__ uint32_t scan_sh[kThreads / 64 + 1];
  if (dn) n = *dn;
  const uint32_t tile = xcd_share(blockIdx.x, tiles_of(n));
  if (tile >= tiles_of(n)) return;  // block-uniform
  const uint32_t mask = nd - 1, d0 = threadIdx.x * kDPer;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const size_t tile0 = (size_t)tile * kTile, base = tile0 + (size_t)w * 64 * kItems;
  uint32_t g[kDPer], tot[kDPer];
  load_digits(offsets + (size_t)nb * nd, d0, nd, tot);
  load_digits(offsets + (size_t)tile * nd, d0, nd, g);
  uint64_t kk[kItems];
  const size_t last = n - 1;
#pragma unroll
  for (int r = 0; r < kItems; ++r) {
    const size_t i = base + (size_t)r * 64 + lane;
    kk[r] = kin[i < last ? i : last];
  }
  if (d0 < nd) *reinterpret_cast<uint4*>(dig + d0) = make_uint4(0, 0, 0, 0);
  scan_digits(tot, scan_sh);  // ends with a barrier
  uint32_t rank[kItems];
#pragma unroll
  for (int r = 0; r < kItems; ++r) {
    const bool valid = base + (size_t)r * 64 + lane < n;
    const uint32_t d = (uint32_t)(kk[r] >> shift) & mask;
    const uint32_t f = (uint32_t)__builtin_amdgcn_readfirstlane((int)d);
    if (__ballot(valid && d == f) == ~0ull) {  // one digit in the whole wave: one add
      uint32_t b = 0;
      if (lane == 0) b = atomicAdd(&dig[f], 64u);
      rank[r] = (uint32_t)__builtin_amdgcn_readfirstlane((int)b) + lane;
    } else {
      rank[r] = valid ? atomicAdd(&dig[d], 1u) : 0u;
    }
  }
  __syncthreads();
  uint32_t b[kDPer];
  load_digits(dig, d0, nd, b);
  scan_digits(b, scan_sh);  // ends with a barrier: every thread has read its counts
  if (d0 < nd) *reinterpret_cast<uint4*>(dig + d0) = make_uint4(b[0], b[1], b[2], b[3]);
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kItems; ++r) {
    const size_t i = base + (size_t)r * 64 + lane;
    if (i < n) {
      const uint32_t lp = dig[(uint32_t)(kk[r] >> shift) & mask] + rank[r];
      skeys[lp] = kk[r];
      place[i] = (uint16_t)lp;
    }
  }
  __syncthreads();
  if (d0 < nd)
    *reinterpret_cast<uint4*>(dig + d0) = make_uint4(tot[0] + g[0] - b[0], tot[1] + g[1] - b[1], tot[2] + g[2] - b[2],
                                                     tot[3] + g[3] - b[3]);
  __syncthreads();
  const uint32_t cnt = (uint32_t)(n - tile0 < (size_t)kTile ? n - tile0 : (size_t)kTile);
#pragma unroll 4
  for (uint32_t i = threadIdx.x; i < cnt; i += kThreads) {
    const uint64_t k = skeys[i];
    kout[dig[(uint32_t)(k >> shift) & mask] + i] = k;
  }
}

// (vin, fin) in partitioned order -> (vout, fout) in input order.  The digit of staging index i is the
// last one whose run starts at or before i: run starts are marked in LDS and a running maximum fills the
// gaps (a binary search of the 2048 starts per index took longer).  VEC: vout 16-byte, fout 4-byte aligned;
// each lane then writes 4 consecutive results.
template <bool VEC>
__global__ __launch_bounds__(kThreads) void part_unscatter_kernel(const uint64_t* __restrict__ vin,
                                                                  const uint8_t* __restrict__ fin,
                                                                  uint64_t* __restrict__ vout,
                                                                  uint8_t* __restrict__ fout,
                                                                  const uint16_t* __restrict__ place, size_t n,
                                                                  uint32_t nd, const uint32_t* __restrict__ offsets,
                                                                  uint32_t nb, Clash clash,
                                                                  const uint32_t* __restrict__ dn) {
  __shared__ __align__(16) uint64_t sv[kTile];       // first the digit of each index (16 bits)
  __shared__ __align__(16) uint32_t adj[kDigits];    // output minus tile offset; then the found flags
  __shared__ uint32_t scan_sh[kThreads / 64 + 1];
  static_assert(sizeof(adj) >= kTile, "the found flags fit");
  uint8_t* sf = reinterpret_cast<uint8_t*>(adj);
  uint16_t* dg = reinterpret_cast<uint16_t*>(sv);
  if (dn) n = *dn;
  const uint32_t live = tiles_of(n), tile = xcd_share(blockIdx.x, live);
  if (tile >= live) return;  // block-uniform
  const bool flags = *clash.any != 0;  // uniform
  const uint32_t d0 = threadIdx.x * kDPer;
  const size_t tile0 = (size_t)tile * kTile;
  const uint32_t cnt = (uint32_t)(n - tile0 < (size_t)kTile ? n - tile0 : (size_t)kTile);
  uint32_t g[kDPer], nx[kDPer], tot[kDPer], c[kDPer];
  load_digits(offsets + (size_t)nb * nd, d0, nd, tot);
  load_digits(offsets + (size_t)tile * nd, d0, nd, g);
  load_digits(offsets + (size_t)(tile + 1 < live ? tile + 1 : nb) * nd, d0, nd, nx);  // row nb: the totals
  uint2 pw[VEC ? kItems / 4 : 1];
  if constexpr (VEC) {
#pragma unroll
    for (int r = 0; r < kItems / 4; ++r) {
      const uint32_t j0 = (threadIdx.x + r * kThreads) * 4;
      pw[r] = j0 + 3 < cnt ? *reinterpret_cast<const uint2*>(place + tile0 + j0) : make_uint2(0u, 0u);
    }
  }
  uint4* dg4 = reinterpret_cast<uint4*>(dg);
#pragma unroll
  for (int k = 0; k < kItems / 8; ++k) dg4[threadIdx.x + k * kThreads] = make_uint4(0, 0, 0, 0);
#pragma unroll
  for (int j = 0; j < kDPer; ++j) c[j] = nx[j] - g[j];
  uint32_t has = 0;
#pragma unroll
  for (int j = 0; j < kDPer; ++j) has |= c[j] ? 1u << j : 0u;
  scan_digits(tot, scan_sh);
  scan_digits(c, scan_sh);  // ends with a barrier: the marks are cleared
  if (d0 < nd) {
#pragma unroll
    for (int j = 0; j < kDPer; ++j)
      if ((has >> j) & 1u) dg[c[j]] = (uint16_t)(d0 + j);
    *reinterpret_cast<uint4*>(adj + d0) = make_uint4(tot[0] + g[0] - c[0], tot[1] + g[1] - c[1], tot[2] + g[2] - c[2],
                                                     tot[3] + g[3] - c[3]);
  }
  __syncthreads();
  {
    // running maximum over 16 consecutive marks per thread, then over the threads
    uint4 q[2] = {dg4[2 * threadIdx.x], dg4[2 * threadIdx.x + 1]};
    uint32_t m[kItems];
    const uint32_t* qw = reinterpret_cast<const uint32_t*>(q);
    uint32_t run = 0;
#pragma unroll
    for (int k = 0; k < kItems; ++k) {
      const uint32_t x = (qw[k / 2] >> (16 * (k & 1))) & 0xFFFFu;
      run = x > run ? x : run;
      m[k] = run;
    }
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t inc = run;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t y = __shfl_up(inc, o, 64);
      if (lane >= o) inc = y > inc ? y : inc;
    }
    if (lane == 63) scan_sh[w] = inc;
    uint32_t before = __shfl_up(inc, 1, 64);
    if (lane == 0) before = 0;
    __syncthreads();
    for (int x = 0; x < w; ++x) before = scan_sh[x] > before ? scan_sh[x] : before;
    uint32_t o[kItems / 2];
#pragma unroll
    for (int k = 0; k < kItems / 2; ++k) {
      const uint32_t a = m[2 * k] > before ? m[2 * k] : before, b = m[2 * k + 1] > before ? m[2 * k + 1] : before;
      o[k] = a | b << 16;
    }
    dg4[2 * threadIdx.x] = make_uint4(o[0], o[1], o[2], o[3]);
    dg4[2 * threadIdx.x + 1] = make_uint4(o[4], o[5], o[6], o[7]);
  }
  __syncthreads();
  uint64_t v[kItems];
  uint32_t ff = 0;
#pragma unroll
  for (int r = 0; r < kItems; ++r) {
    const uint32_t i = threadIdx.x + r * kThreads;
    const uint32_t src = i < cnt ? adj[dg[i]] + i : 0u;
    v[r] = i < cnt ? vin[src] : 0ull;
    if (flags) {
      const bool mark = i < cnt && v[r] == kMissMark;
      ff |= (mark ? clash.part[src / kClashPart] && fin[src] : i < cnt) ? 1u << r : 0u;
    }
  }
  __syncthreads();  // marks and offsets are read: their memory takes the results
#pragma unroll
  for (int r = 0; r < kItems; ++r) {
    const uint32_t i = threadIdx.x + r * kThreads;
    if (i < cnt) {
      sv[i] = v[r];
      if (flags) sf[i] = (ff >> r) & 1u;
    }
  }
  __syncthreads();
  auto result = [&](uint32_t l, uint64_t& val) -> uint32_t {
    const uint64_t x = sv[l];
    const uint32_t found = flags ? (uint32_t)sf[l] : (x != kMissMark ? 1u : 0u);
    val = found ? x : 0ull;
    return found;
  };
  if constexpr (VEC) {
#pragma unroll
    for (int r = 0; r < kItems / 4; ++r) {
      const uint32_t j0 = (threadIdx.x + r * kThreads) * 4;
      if (j0 + 3 < cnt) {
        const uint32_t l0 = pw[r].x & 0xFFFFu, l1 = pw[r].x >> 16, l2 = pw[r].y & 0xFFFFu, l3 = pw[r].y >> 16;
        uint64_t a, b, c, d;
        const uint32_t f = result(l0, a) | result(l1, b) << 8 | result(l2, c) << 16 | result(l3, d) << 24;
        *reinterpret_cast<ulonglong2*>(vout + tile0 + j0) = make_ulonglong2(a, b);
        *reinterpret_cast<ulonglong2*>(vout + tile0 + j0 + 2) = make_ulonglong2(c, d);
        *reinterpret_cast<uint32_t*>(fout + tile0 + j0) = f;
      } else {
        for (uint32_t j = j0; j < cnt; ++j) {  // at most 3
          uint64_t a;
          fout[tile0 + j] = (uint8_t)result(place[tile0 + j], a);
          vout[tile0 + j] = a;
        }
      }
    }
  } else {
#pragma unroll
    for (int r = 0; r < kItems; ++r) {
      const uint32_t j = threadIdx.x + r * kThreads;
      if (j < cnt) {
        uint64_t a;
        fout[tile0 + j] = (uint8_t)result(place[tile0 + j], a);
        vout[tile0 + j] = a;
      }
    }
  }
}

// The same for (key, value) pairs: 128 KiB of pairs, one block of 1024 threads per CU.  Nothing is recorded.
// Does nothing once *flags has `skip`.
constexpr int kPairThreads = 1024;
constexpr int kPairItems = kTile / kPairThreads;
constexpr int kPairDPer = kDigits / kPairThreads;
__global__ __launch_bounds__(kPairThreads) void part_pairs_kernel(const uint64_t* __restrict__ kin,
                                                                  const uint64_t* __restrict__ vin,
                                                                  uint64_t* __restrict__ kout,
                                                                  uint64_t* __restrict__ vout, size_t n, int shift,
                                                                  uint32_t nd, const uint32_t* __restrict__ offsets,
                                                                  uint32_t nb, const uint32_t* __restrict__ flags,
                                                                  uint32_t skip) {
  __shared__ uint64_t skeys[kTile], svals[kTile];
  __shared__ __align__(16) uint32_t dig[kDigits];
  __shared__ uint32_t scan_sh[kPairThreads / 64 + 1];
  const uint32_t tile = xcd_share(blockIdx.x, nb);
  if (tile >= nb || (*flags & skip)) return;  // block-uniform
  const uint32_t mask = nd - 1, d0 = threadIdx.x * kPairDPer;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const size_t tile0 = (size_t)tile * kTile, base = tile0 + (size_t)w * 64 * kPairItems;
  uint32_t tot[kPairDPer], g[kPairDPer], all;
#pragma unroll
  for (int j = 0; j < kPairDPer; ++j) {
    tot[j] = d0 < nd ? offsets[(size_t)nb * nd + d0 + j] : 0u;
    g[j] = d0 < nd ? offsets[(size_t)tile * nd + d0 + j] : 0u;
  }
  uint64_t kk[kPairItems], vv[kPairItems];
#pragma unroll
  for (int r = 0; r < kPairItems; ++r) {
    const size_t i = base + (size_t)r * 64 + lane, c = i < n ? i : n - 1;
    kk[r] = kin[c];
    vv[r] = vin[c];
  }
  for (uint32_t d = threadIdx.x; d < nd; d += kPairThreads) dig[d] = 0;
  uint32_t dbase = block_exclusive_scan<uint32_t, kPairThreads>(tot[0] + tot[1], scan_sh, all);  // ends with a barrier
  uint32_t rank[kPairItems];
#pragma unroll
  for (int r = 0; r < kPairItems; ++r)
    rank[r] = base + (size_t)r * 64 + lane < n ? atomicAdd(&dig[(uint32_t)(kk[r] >> shift) & mask], 1u) : 0u;
  __syncthreads();
  const uint32_t c0 = d0 < nd ? dig[d0] : 0u, c1 = d0 < nd ? dig[d0 + 1] : 0u;
  const uint32_t b0 = block_exclusive_scan<uint32_t, kPairThreads>(c0 + c1, scan_sh, all), b1 = b0 + c0;
  if (d0 < nd) dig[d0] = b0, dig[d0 + 1] = b1;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kPairItems; ++r)
    if (base + (size_t)r * 64 + lane < n) {
      const uint32_t lp = dig[(uint32_t)(kk[r] >> shift) & mask] + rank[r];
      skeys[lp] = kk[r];
      svals[lp] = vv[r];
    }
  __syncthreads();
  if (d0 < nd) dig[d0] = dbase + g[0] - b0, dig[d0 + 1] = dbase + tot[0] + g[1] - b1;
  __syncthreads();
  const uint32_t cnt = (uint32_t)(n - tile0 < (size_t)kTile ? n - tile0 : (size_t)kTile);
#pragma unroll 4
  for (uint32_t i = threadIdx.x; i < cnt; i += kPairThreads) {
    const uint64_t k = skeys[i];
    const uint32_t p = dig[(uint32_t)(k >> shift) & mask] + i;
    kout[p] = k;
    vout[p] = svals[i];
  }
}
static_assert(kPairDPer == 2, "the offsets above are written for two digits per thread");

size_t offsets_bytes(size_t n, int bits) {
  const size_t nb = (n + kTile - 1) / kTile;
  return ((nb + 1) * ((size_t)4 << bits) + 255) / 256 * 256;
}

}  // namespace

int partition_bits(size_t n) {
  int b = kPartMinBits;
  while (b < kPartMaxBits && (n >> b) > (size_t)kPartBucket) ++b;
  return b;
}

size_t partition_bytes(size_t n) { return offsets_bytes(n, partition_bits(n)) + (n * 2 + 255) / 256 * 256; }

hipError_t partition_keys(const uint64_t* q, size_t n, int top, uint64_t* out, void* rec, const Clash& clash,
                          hipStream_t s, const uint32_t* dn) {
  if (n == 0) return hipSuccess;
  const int bits = partition_bits(n);
  if (top < bits || top > 64) return hipErrorInvalidValue;
  const uint32_t nd = 1u << bits, nb = (uint32_t)((n + kTile - 1) / kTile);
  const int shift = top - bits;
  uint32_t* offsets = reinterpret_cast<uint32_t*>(rec);
  uint16_t* place = reinterpret_cast<uint16_t*>(reinterpret_cast<char*>(rec) + offsets_bytes(n, bits));
  {
    ProfScope prof("psa_hist", s);
    if ((reinterpret_cast<uintptr_t>(q) & 15) == 0)
      hipLaunchKernelGGL(part_hist_kernel<true>, dim3(grid_for(nb)), dim3(kThreads), 0, s, q, n, shift, nd, offsets,
                         clash.any, dn);
    else
      hipLaunchKernelGGL(part_hist_kernel<false>, dim3(grid_for(nb)), dim3(kThreads), 0, s, q, n, shift, nd, offsets,
                         clash.any, dn);
  }
  {
    ProfScope prof("scan", s);
    hipLaunchKernelGGL(part_scan_kernel, dim3(nd / kScanDigits), dim3(kScanThreads), 0, s, offsets, nd, nb, 0u,
                       (uint32_t*)nullptr, 0u, dn);
  }
  ProfScope prof("psa_scatter", s);
  hipLaunchKernelGGL(part_scatter_kernel, dim3(grid_for(nb)), dim3(kThreads), 0, s, q, out, place, n, shift, nd,
                     (const uint32_t*)offsets, nb, dn);
  return hipGetLastError();
}

int pair_bits(size_t n) {
  int b = kPartMinBits;
  while (b <= kPartMaxBits && (n >> b) > (size_t)kPairBucket) ++b;
  return b <= kPartMaxBits ? b : 0;
}

size_t partition_pairs_bytes(size_t n) { return offsets_bytes(n, pair_bits(n)); }

hipError_t partition_pairs(const uint64_t* keys, const uint64_t* vals, size_t n, int top, uint64_t* kout,
                           uint64_t* vout, void* tmp, uint32_t* flags, uint32_t flag, const uint32_t** totals,
                           hipStream_t s) {
  const int bits = n ? pair_bits(n) : 0;
  if (!bits || top < 1 || top > 64) return hipErrorInvalidValue;
  const uint32_t nd = 1u << bits, nb = (uint32_t)((n + kTile - 1) / kTile);
  const int shift = top > bits ? top - bits : 0;  // fewer varying bits than digits: the digits above stay empty
  uint32_t* offsets = reinterpret_cast<uint32_t*>(tmp);
  ProfScope prof("build", s);
  if ((reinterpret_cast<uintptr_t>(keys) & 15) == 0)
    hipLaunchKernelGGL(part_hist_kernel<true>, dim3(grid_for(nb)), dim3(kThreads), 0, s, keys, n, shift, nd, offsets,
                       (uint32_t*)nullptr, (const uint32_t*)nullptr);
  else
    hipLaunchKernelGGL(part_hist_kernel<false>, dim3(grid_for(nb)), dim3(kThreads), 0, s, keys, n, shift, nd, offsets,
                       (uint32_t*)nullptr, (const uint32_t*)nullptr);
  hipLaunchKernelGGL(part_scan_kernel, dim3(nd / kScanDigits), dim3(kScanThreads), 0, s, offsets, nd, nb,
                     kBucketSortMax, flags, flag, (const uint32_t*)nullptr);
  hipLaunchKernelGGL(part_pairs_kernel, dim3(grid_for(nb)), dim3(kPairThreads), 0, s, keys, vals, kout, vout, n, shift,
                     nd, (const uint32_t*)offsets, nb, (const uint32_t*)flags, flag);
  *totals = offsets + (size_t)nb * nd;
  return hipGetLastError();
}

hipError_t unpartition_results(const uint64_t* vals, const uint8_t* found, size_t n, const void* rec,
                               const Clash& clash, uint64_t* out_vals, uint8_t* out_found, hipStream_t s,
                               const uint32_t* dn) {
  if (n == 0) return hipSuccess;
  const int bits = partition_bits(n);
  const uint32_t nd = 1u << bits, nb = (uint32_t)((n + kTile - 1) / kTile);
  const uint32_t* offsets = reinterpret_cast<const uint32_t*>(rec);
  const uint16_t* place = reinterpret_cast<const uint16_t*>(reinterpret_cast<const char*>(rec) + offsets_bytes(n, bits));
  ProfScope prof("unsort", s);
  if ((reinterpret_cast<uintptr_t>(out_vals) & 15) == 0 && (reinterpret_cast<uintptr_t>(out_found) & 3) == 0)
    hipLaunchKernelGGL(part_unscatter_kernel<true>, dim3(grid_for(nb)), dim3(kThreads), 0, s, vals, found, out_vals,
                       out_found, place, n, nd, offsets, nb, clash, dn);
  else
    hipLaunchKernelGGL(part_unscatter_kernel<false>, dim3(grid_for(nb)), dim3(kThreads), 0, s, vals, found, out_vals,
                       out_found, place, n, nd, offsets, nb, clash, dn);
  return hipGetLastError();
}

}  // namespace hm

// Leaf-chain range scan.
//
// Replaces range_prefix_sort_1thread_search_1_thread_scan_kernel (H/src/range.cu:101-227): descend
// to the leaf of `start`, then walk the leaves in key order (the leaf pool is contiguous in key
// order, leaf i -> i + 1, as the reference's BLeaf pool, H/src/range.cu:188-221), skipping padding.
// The reference emits at most Range_Size = 8 records per range (H/src/range.cu:32); here a range
// emits up to its own length, or every key of a closed interval [lo, hi] as
// find_range(start, end) does (H/regular_bpt/regular_bpt.cpp:320-338).
// A wave takes R ranges (calls in between give 8 lanes to each, group_kernel).  Their descents run together (R = 8:
// one 8-lane group per range; R = 1: the whole wave ranks a node in one step), then all 64 lanes walk the leaves:
// one 16-byte load per lane brings 8 leaves (1 KiB), lanes 0-3 of a leaf's 8 holding its keys and 4-7 its values,
// two ballots rank the qualifying keys, and one 16-byte store per lane writes the pairs, keys and values as
// contiguous runs.
//
// Large calls are bound by memory traffic: 2^20 ranges of 16..256 pairs on 2^26 keys (fanout 128) move
// 5.4 GB in 0.99-1.09 ms, the rate of a plain copy here (4.8-5.1 TB/s).  Walking each range with a group
// of 8 lanes took 1.28-1.31 ms: its loads and stores each touched eight short stretches of memory, which
// kept the address unit 92% busy.  Eight waves per SIMD, so that the grid of 8 blocks per CU is one whole
// round, matter most for short ranges (2^20 of 1..40 pairs: 269 us, 330 at seven, 301 with 8-lane groups).
// Nontemporal stores and an XCD-contiguous block order measured the same.  Small calls are bound by
// launches and the chain of dependent reads: 300 ranges 19.7 -> 7.9 us in one launch.
#include <algorithm>

#include "hm_device.h"

namespace hm {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
// Which kernel takes how many ranges; device times in us of a wave per range (R = 1), 8 lanes each and eight laid
// end to end (R = 8), trees of 2^20 to 2^25 keys, 1 to 8 keys to a leaf.
// R = 1 while waves are free: its descents have four dependent reads instead of eight.  4096 ranges of 1..3 pairs
// 10.5, 10.3, 11.2 (6 in the scan launches), of 16..256 13 to 41, 18 to 73, 22 to 123.  Above, for long ranges (by
// the capacity for them): 8192 of 16..256 25 to 68, 28 to 83, 34 to 140; 16384 47 to 123, 49 to 123, 51 to 165; of
// 1..40 38 to 64, 34 to 50, 36 to 58.
// R = 8 once there are enough of them that each of its loads is wanted: 24576 of 16..256 35 to 153, 38 to 160, 37 to
// 175, of 1..40 24 to 62, 18 to 35, 20 to 45; 65536 of 16..256 67 to 367, 67 to 376, 66 to 318, of 1..40 41 to 129, 29
// to 65, 28 to 71; 100000 of 16..256 98 to 526, 105 to 559, 104 to 477, of 1..40 54 to 195, 36 to 101, 34 to 102.
// Closed intervals may end anywhere before their capacity, which tells nothing then, and R = 8 would read many
// leaves for nothing: 4096 of 1..3 pairs 4 and 4 (R = 1, 8 lanes), of 1..40 5 to 7 and 5 to 14, of 16..256 7 to 32
// and 14 to 76; 8192 of 1..40 8 to 12 and 5 to 16; 24576 of 1..40 20 to 27 and 9 to 24.
constexpr uint32_t kOneMax = 4096, kOneMaxLong = 16384, kLongRange = 64, kGroupMax = 65536;
constexpr int kWalk = 4;   // loads (8 leaves each) in flight per step, R = 1
constexpr int kWalk8 = 3;  // the same, R = 8 (2 and 4 were slower, or even)

__device__ __forceinline__ uint32_t lane_u32(uint32_t v, int lane) {
  return (uint32_t)__builtin_amdgcn_readlane((int)v, lane);
}
__device__ __forceinline__ uint64_t lane_u64(uint64_t v, int lane) {
  return ((uint64_t)lane_u32((uint32_t)(v >> 32), lane) << 32) | lane_u32((uint32_t)v, lane);
}

// 16 bytes to an address that is only 8-byte aligned (outputs start at any pair).
__device__ __forceinline__ void store_pair(uint64_t* p, uint64_t x, uint64_t y) {
  typedef uint64_t u64x2 __attribute__((ext_vector_type(2), aligned(8)));
  u64x2 v = {x, y};
  *reinterpret_cast<u64x2*>(p) = v;
}

// Pairs of one range (every argument wave-uniform): up to L keys in [s, h] from `leaf` on, written at
// off + 0, 1, ...; returns how many there are (at most L).
__device__ __forceinline__ uint32_t walk_range(const TreeView& tv, uint32_t leaf, uint64_t s, uint64_t h, uint32_t L,
                                               uint64_t off, uint64_t* __restrict__ out_keys,
                                               uint64_t* __restrict__ out_vals, uint64_t capacity) {
  const int lane = threadIdx.x & 63;
  const int kl = (lane & ~7) | (lane & 3);  // the lane that holds this lane's two keys
  const uint64_t below = (1ull << kl) - 1ull;
  const bool is_key = (lane & 4) == 0;
  uint64_t* dst = is_key ? out_keys : out_vals;
  uint32_t got = 0;
  while (got < L) {  // wave-uniform
    // a leaf holds at most 8 keys and the first one may hold keys below s: no range needs more leaves
    const uint64_t need = (uint64_t)leaf + ((uint64_t)(L - got) + LEAF_KEYS - 1) / LEAF_KEYS + 1;
    const uint32_t stop = need < tv.n_leaves ? (uint32_t)need : tv.n_leaves;
    ulonglong2 x[kWalk];
#pragma unroll
    for (int u = 0; u < kWalk; ++u) {
      const uint32_t lf = leaf + 8 * u + (lane >> 3);
      x[u] = make_ulonglong2(KEY_MAX, KEY_MAX);
      if (lf < stop) x[u] = reinterpret_cast<const ulonglong2*>(tv.leaves + lf)[lane & 7];
    }
#pragma unroll
    for (int u = 0; u < kWalk; ++u) {
      if (got >= L || leaf + 8 * u >= stop) break;  // wave-uniform
      const bool t0 = is_key && x[u].x != KEY_MAX && x[u].x >= s && x[u].x <= h;
      const bool t1 = is_key && x[u].y != KEY_MAX && x[u].y >= s && x[u].y <= h;
      const bool past = is_key && ((x[u].x != KEY_MAX && x[u].x > h) || (x[u].y != KEY_MAX && x[u].y > h));
      const uint64_t m0 = __ballot(t0), m1 = __ballot(t1);
      const uint32_t rank = got + (uint32_t)__popcll(m0 & below) + (uint32_t)__popcll(m1 & below);
      const uint32_t b0 = (uint32_t)(m0 >> kl) & 1u, b1 = (uint32_t)(m1 >> kl) & 1u;
      const uint64_t o = off + rank;
      const bool w0 = b0 && rank < L && o < capacity;
      const bool w1 = b1 && rank + b0 < L && o + b0 < capacity;
      if (w0 && w1)
        store_pair(dst + o, x[u].x, x[u].y);
      else if (w0)
        dst[o] = x[u].x;
      else if (w1)
        dst[o + b0] = x[u].y;
      got += (uint32_t)(__popcll(m0) + __popcll(m1));
      if (__ballot(past)) return got < L ? got : L;
    }
    leaf = stop - leaf < 8 * kWalk ? stop : leaf + 8 * kWalk;  // leaves with free slots may leave some wanting
    if (leaf >= tv.n_leaves) break;
  }
  return got < L ? got : L;
}

// Pairs of a wave's eight ranges, range g held by lanes 8 g .. 8 g + 7 (s, L, off, the leaf of s; L = 0:
// none).  The leaves that the ranges still need are laid end to end and each load takes the next eight of
// them, whatever ranges they belong to, so short ranges fill the wave as well as long ones.  Returns the
// lane's range's count.
__device__ __forceinline__ uint32_t walk_ranges8(const TreeView& tv, uint32_t leaf, uint64_t s, uint32_t L,
                                                 uint64_t off, uint64_t* __restrict__ out_keys,
                                                 uint64_t* __restrict__ out_vals, uint64_t capacity) {
  // leaves of one range per round: nearly every range is done in one (leaves with free slots leave some)
  constexpr uint32_t most = 1u << 16;
  const int lane = threadIdx.x & 63;
  const int kl = (lane & ~7) | (lane & 3);  // the lane that holds this lane's two keys
  const uint64_t below = (1ull << kl) - 1ull;
  const bool is_key = (lane & 4) == 0;
  uint64_t* dst = is_key ? out_keys : out_vals;
  uint32_t got = 0;
  bool done = L == 0;
  while (true) {
    uint32_t need = 0;
    if (!done) {
      // a leaf holds at most 8 keys and the first one may hold keys below s
      const uint64_t want = ((uint64_t)(L - got) + LEAF_KEYS - 1) / LEAF_KEYS + 1;
      need = want < most ? (uint32_t)want : most;
      need = need < tv.n_leaves - leaf ? need : tv.n_leaves - leaf;
    }
    uint32_t P[8], T = 0, mine = 0;  // wave-uniform starts; the lane's own range's start
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      P[r] = T;
      if (r == (lane >> 3)) mine = T;
      T += lane_u32(need, 8 * r);
    }
    if (T == 0) break;
    for (uint32_t t0 = 0; t0 < T; t0 += 8 * kWalk8) {  // wave-uniform
      ulonglong2 x[kWalk8];
      int src[kWalk8];
      uint32_t first[kWalk8];  // start of the slot's range
#pragma unroll
      for (int u = 0; u < kWalk8; ++u) {
        const uint32_t t = t0 + 8 * u + (lane >> 3);
        int r = 0;
        first[u] = 0;
        x[u] = make_ulonglong2(KEY_MAX, KEY_MAX);
        if (t0 + 8 * u >= T) break;  // wave-uniform
#pragma unroll
        for (int k = 1; k < 8; ++k)
          if (P[k] <= t) r = k, first[u] = P[k];
        src[u] = 8 * r;
        const uint32_t lf = (uint32_t)__shfl((int)leaf, src[u]) + (t - first[u]);
        if (t < T) x[u] = reinterpret_cast<const ulonglong2*>(tv.leaves + lf)[lane & 7];
      }
#pragma unroll
      for (int u = 0; u < kWalk8; ++u) {
        const uint32_t tb = t0 + 8 * u;
        if (tb >= T) break;  // wave-uniform
        const uint64_t rs = __shfl(s, src[u]);
        const uint64_t ro = __shfl(off, src[u]);
        const uint32_t rL = __shfl(L, src[u]), rg = __shfl(got, src[u]);
        const bool t0k = is_key && x[u].x != KEY_MAX && x[u].x >= rs;
        const bool t1k = is_key && x[u].y != KEY_MAX && x[u].y >= rs;
        const uint64_t m0 = __ballot(t0k), m1 = __ballot(t1k);
        // rank among the range's keys: those counted before plus the ones below in this load
        const uint32_t f = first[u] > tb ? first[u] - tb : 0u;  // the range's first slot here, 0..7
        const uint64_t seg = below & (~0ull << (8 * f));
        const uint32_t rank = rg + (uint32_t)__popcll(m0 & seg) + (uint32_t)__popcll(m1 & seg);
        const uint32_t b0 = (uint32_t)(m0 >> kl) & 1u, b1 = (uint32_t)(m1 >> kl) & 1u;
        const uint64_t o = ro + rank;
        const bool w0 = b0 && rank < rL && o < capacity;
        const bool w1 = b1 && rank + b0 < rL && o + b0 < capacity;
        if (w0 && w1)
          store_pair(dst + o, x[u].x, x[u].y);
        else if (w0)
          dst[o] = x[u].x;
        else if (w1)
          dst[o + b0] = x[u].y;
        // the lane's own range: its slots [a, b) of this load
        const uint32_t a = mine > tb ? (mine - tb < 8 ? mine - tb : 8) : 0u;
        const uint32_t e = mine + need > tb ? (mine + need - tb < 8 ? mine + need - tb : 8) : 0u;
        const uint64_t own = e > a ? (~0ull >> (64 - 8 * (e - a))) << (8 * a) : 0ull;
        got += (uint32_t)__popcll(m0 & own) + (uint32_t)__popcll(m1 & own);
      }
    }
    leaf += need;
    done = done || got >= L || leaf >= tv.n_leaves;
  }
  return got < L ? got : L;
}

// SCAN (R = 1): out_offsets is written here, each wave adding up the lengths before its range, so a
// small call is one launch.
template <int F, int R, bool SCAN>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(8))) void range_kernel(TreeView tv, const uint64_t* __restrict__ start,
                                                         const uint64_t* __restrict__ hi,
                                                         const uint32_t* __restrict__ len, uint32_t cap_const,
                                                         uint32_t n, uint64_t* __restrict__ offsets,
                                                         uint64_t offset_stride, uint64_t* __restrict__ out_keys,
                                                         uint64_t* __restrict__ out_vals,
                                                         uint32_t* __restrict__ out_counts, uint64_t capacity) {
  static_assert(R == 1 || R == 8, "one range per wave or per 8-lane group");
  static_assert(!SCAN || R == 1, "");
  const int lane = threadIdx.x & 63;
  const uint32_t nw = gridDim.x * kWaves;
  for (uint32_t rb = (blockIdx.x * kWaves + (threadIdx.x >> 6)) * R; rb < n; rb += nw * R) {  // wave-uniform
    const uint32_t ri = rb + (R == 1 ? 0 : lane / (64 / R));
    const bool valid = ri < n;
    const uint64_t s = valid ? start[ri] : 0ull;
    const uint64_t h = (valid && hi) ? hi[ri] : KEY_MAX;
    const uint32_t L = valid ? (len ? len[ri] : cap_const) : 0u;
    uint64_t off = 0;
    if constexpr (SCAN) {
      uint64_t a = 0;
#pragma unroll 8
      for (uint32_t i = lane; i < ri; i += 64) a += len[i];
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) a += __shfl_xor(a, o);
      off = a;
      if (lane == 0) {
        offsets[ri] = off;
        if (ri == n - 1) offsets[n] = off + L;
      }
    } else {
      off = valid ? (offsets ? offsets[ri] : (uint64_t)ri * offset_stride) : 0ull;
    }
    const uint64_t sd = s == KEY_MAX ? KEY_MAX - 1 : s;
    uint32_t leaf;
    if constexpr (R == 1) {
      constexpr int G = F < 64 ? F : 64;
      uint32_t node = 0;
      for (int l = 0; l < tv.height; ++l)
        node = node_next_wide<F, G>(tv.inner + (size_t)node * node_slots(F), sd, lane % G, lane - lane % G);
      leaf = node - tv.n_inner;
    } else {
      leaf = descend<F, 8>(tv, 0, nullptr, sd, lane % 8, lane - lane % 8);
    }
    const uint32_t want = s > h || s == KEY_MAX ? 0u : L;
    uint32_t count;
    if constexpr (R == 1)
      count = walk_range(tv, lane_u32(leaf, 0), lane_u64(s, 0), lane_u64(h, 0), lane_u32(want, 0), lane_u64(off, 0),
                         out_keys, out_vals, capacity);
    else
      count = walk_ranges8(tv, leaf, s, want, off, out_keys, out_vals, capacity);
    if (valid && lane % (64 / R) == 0) out_counts[ri] = count;
  }
}

// 8 lanes per range or closed interval (HI), up to eight of its leaves on their way at a time (LDS-direct loads, a
// group's 8 lanes bring a whole leaf), consumed in order until the length is reached or one key lies past the end.
constexpr int kWalkInterval = 8;
template <int F, bool HI>
__global__ __launch_bounds__(kThreads) void group_kernel(TreeView tv, const uint64_t* __restrict__ start,
                                                         const uint64_t* __restrict__ hi,
                                                         const uint32_t* __restrict__ len, uint32_t cap_const,
                                                         uint32_t n, const uint64_t* __restrict__ offsets,
                                                         uint64_t offset_stride, uint64_t* __restrict__ out_keys,
                                                         uint64_t* __restrict__ out_vals,
                                                         uint32_t* __restrict__ out_counts, uint64_t capacity) {
  constexpr int G = 8;
  constexpr uint32_t gpb = kThreads / G;
  typedef __attribute__((address_space(1))) void global_void_t;
  typedef __attribute__((address_space(3))) void lds_void_t;
  // the wave's leaves of one step: step u holds its 8 groups' leaves, lane l's 16-byte piece at byte 16 l
  __shared__ __align__(16) uint64_t lbuf[kWaves][kWalkInterval][128];
  uint64_t* wb = &lbuf[threadIdx.x >> 6][0][0];
  const int lane = threadIdx.x & 63, gl = lane % G, gbase = lane - gl;
  const uint64_t lanes_below = (1ull << gl) - 1ull;
  for (uint32_t rb = blockIdx.x * gpb; rb < n; rb += gridDim.x * gpb) {  // uniform across the block
    const uint32_t ri = rb + threadIdx.x / G;
    const bool valid = ri < n;
    const uint64_t s = valid ? start[ri] : 0ull, h = !HI ? KEY_MAX : valid ? hi[ri] : 0ull;
    const uint32_t L = HI ? cap_const : valid ? len[ri] : 0u;
    const uint64_t off = HI ? (uint64_t)ri * offset_stride : valid ? offsets[ri] : 0ull;
    uint32_t leaf = descend<F, G>(tv, 0, nullptr, s == KEY_MAX ? KEY_MAX - 1 : s, gl, gbase);
    uint32_t got = 0;
    bool done = !valid || L == 0 || s > h || s == KEY_MAX;
    while (!done) {  // uniform inside the group
      uint64_t k[kWalkInterval], v[kWalkInterval];
      const uint64_t need = ((uint64_t)(L - got) + LEAF_KEYS - 1) / LEAF_KEYS + 1;  // got < L here
      const uint32_t step = need < (uint64_t)kWalkInterval ? (uint32_t)need : (uint32_t)kWalkInterval;
#pragma unroll
      for (int u = 0; u < kWalkInterval; ++u)
        if ((uint32_t)u < step) {  // group-uniform; the load writes LDS only
          const uint32_t lf = leaf + u < tv.n_leaves ? leaf + u : tv.n_leaves - 1;
          __builtin_amdgcn_global_load_lds(
              (const global_void_t*)(reinterpret_cast<const ulonglong2*>(tv.leaves + lf) + gl),
              (lds_void_t*)(wb + u * 128), 16, 0, 0);
        }
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's leaves are in LDS
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int u = 0; u < kWalkInterval; ++u) {
        const bool in = (uint32_t)u < step && leaf + u < tv.n_leaves;
        const uint64_t* lp = wb + u * 128 + gbase * 2;  // this group's leaf
        k[u] = in ? lp[gl] : KEY_MAX;
        v[u] = in ? lp[8 + gl] : 0ull;
      }
      __builtin_amdgcn_wave_barrier();  // the next step's loads overwrite the buffer after these reads
#pragma unroll
      for (int u = 0; u < kWalkInterval; ++u)
        if (!done && (uint32_t)u < step) {  // group-uniform
          const bool take = k[u] != KEY_MAX && k[u] >= s && k[u] <= h;
          const uint64_t m = (__ballot(take) >> gbase) & 0xFFull;
          const uint64_t beyond = (__ballot(k[u] != KEY_MAX && k[u] > h) >> gbase) & 0xFFull;
          const uint32_t rank = got + (uint32_t)__popcll(m & lanes_below);
          const uint64_t o = off + rank;
          if (take && rank < L && o < capacity) {
            out_keys[o] = k[u];
            out_vals[o] = v[u];
          }
          got += (uint32_t)__popcll(m);
          done = got >= L || beyond != 0 || leaf + u + 1 >= tv.n_leaves;
        }
      leaf += step;
    }
    if (valid && gl == 0) out_counts[ri] = got < L ? got : L;
  }
}

__global__ void offsets_tail_kernel(const uint32_t* len, uint64_t* offsets, uint32_t n) {
  if (threadIdx.x == 0 && blockIdx.x == 0) offsets[n] = n ? offsets[n - 1] + len[n - 1] : 0ull;
}

template <int F>
void launch_range_f(const TreeView& tv, const uint64_t* start, const uint64_t* hi, const uint32_t* len,
                    uint32_t cap_const, uint32_t n, uint64_t* offsets, bool scan, uint64_t offset_stride,
                    uint64_t* out_keys, uint64_t* out_vals, uint32_t* out_counts, uint64_t capacity, hipStream_t s) {
  const size_t cus = (size_t)launch_cfg().num_cus;
  const size_t max_nb = cus * 8;
  const uint32_t one = !hi && capacity / n >= kLongRange ? kOneMaxLong : kOneMax;
  if (n <= one) {
    const size_t nb = std::min<size_t>((n + kWaves - 1) / kWaves, max_nb);
    if (scan)
      hipLaunchKernelGGL((range_kernel<F, 1, true>), dim3((unsigned)nb), dim3(kThreads), 0, s, tv, start, hi, len,
                         cap_const, n, offsets, offset_stride, out_keys, out_vals, out_counts, capacity);
    else
      hipLaunchKernelGGL((range_kernel<F, 1, false>), dim3((unsigned)nb), dim3(kThreads), 0, s, tv, start, hi, len,
                         cap_const, n, offsets, offset_stride, out_keys, out_vals, out_counts, capacity);
  } else if (hi || n <= kGroupMax) {
    const size_t nb = std::min<size_t>((n + kWaves * 8 - 1) / (kWaves * 8), max_nb);
    if (hi)
      hipLaunchKernelGGL((group_kernel<F, true>), dim3((unsigned)nb), dim3(kThreads), 0, s, tv, start, hi, len, cap_const,
                         n, offsets, offset_stride, out_keys, out_vals, out_counts, capacity);
    else
      hipLaunchKernelGGL((group_kernel<F, false>), dim3((unsigned)nb), dim3(kThreads), 0, s, tv, start, hi, len,
                         cap_const, n, offsets, offset_stride, out_keys, out_vals, out_counts, capacity);
  } else {
    const size_t nb = std::min<size_t>((n + kWaves * 8 - 1) / (kWaves * 8), max_nb);
    hipLaunchKernelGGL((range_kernel<F, 8, false>), dim3((unsigned)nb), dim3(kThreads), 0, s, tv, start, hi, len,
                       cap_const, n, offsets, offset_stride, out_keys, out_vals, out_counts, capacity);
  }
}

}  // namespace

// scan: the offsets are computed here from the lengths (n <= kRangeScanMax), else they are there.
hipError_t launch_range(const TreeView& tv, const uint64_t* start, const uint64_t* hi, const uint32_t* len,
                        uint32_t cap_const, size_t n, uint64_t* offsets, bool scan, uint64_t offset_stride,
                        uint64_t* out_keys, uint64_t* out_vals, uint32_t* out_counts, uint64_t capacity,
                        hipStream_t s) {
  if (n == 0) return hipSuccess;
  if (scan && (n > kRangeScanMax || !len || !offsets)) return hipErrorInvalidValue;
  if (hi && (len || offsets)) return hipErrorInvalidValue;  // closed intervals: cap_const each, evenly spaced
  ProfScope prof("range", s);
  switch (tv.fanout) {
    case 32:
      launch_range_f<32>(tv, start, hi, len, cap_const, (uint32_t)n, offsets, scan, offset_stride, out_keys, out_vals,
                         out_counts, capacity, s);
      break;
    case 64:
      launch_range_f<64>(tv, start, hi, len, cap_const, (uint32_t)n, offsets, scan, offset_stride, out_keys, out_vals,
                         out_counts, capacity, s);
      break;
    case 128:
      launch_range_f<128>(tv, start, hi, len, cap_const, (uint32_t)n, offsets, scan, offset_stride, out_keys, out_vals,
                          out_counts, capacity, s);
      break;
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t range_offsets_tail(const uint32_t* len, uint64_t* offsets, size_t n, hipStream_t s) {
  hipLaunchKernelGGL(offsets_tail_kernel, dim3(1), dim3(64), 0, s, len, offsets, (uint32_t)n);
  return hipGetLastError();
}

}  // namespace hm

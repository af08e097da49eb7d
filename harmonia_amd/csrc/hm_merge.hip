// Stable merge sort of (key, staging index) for upsert batches, and the removal of all but the last write
// of each key.
//
// Chunks of 4096 keys are sorted in LDS, by a digit if their keys spread over it and by merges if not, then
// every pass merges pairs of runs.  Merges of two sorted runs go by tiles: a diagonal search splits the runs
// for each tile (merge path), the tile's keys go to LDS, and each thread finds its own diagonal there and
// merges eight keys in registers.  Equal keys of the left run go first, so the order of equal keys is the
// staging order.
//
// What bounds it: latency, not bytes (a pass over 2^20 keys moves 25 MB, 5 us at the copy rate).  A pass
// in which every key searched the other run in global memory (20 dependent reads) took 17 us, now 12;
// the chunks, sorted before by eight LSD radix passes in LDS (36 us for 2^20 keys, one block per CU, a block
// barrier every few hundred cycles), take 30 by merges and 18 by a digit.
#include <utility>

#include "hm_block.h"
#include "hm_internal.h"

namespace hm {
namespace {

constexpr int kPer = 8;             // keys per thread
constexpr int kChunkThreads = 512;  // 4096 keys per chunk
constexpr int kTileThreads = 256;   // 2048 keys per merge tile
constexpr uint32_t kTile = kTileThreads * kPer;
static_assert(kChunkThreads * kPer == (int)kSmallUpdate, "batches of one chunk take the small path");

// Element i sits at slot i + i / 8: threads that each touch eight consecutive elements hit all banks.
__device__ __forceinline__ uint32_t slot_of(uint32_t i) { return i + (i >> 3); }

template <int NT>
struct MergeLds {
  uint64_t k[NT * (kPer + 1)];
  uint32_t ix[NT * (kPer + 1)];
};

// Elements diag .. diag + 7 of the merge of the runs [a0, a0 + na) and [b0, b0 + nb) in LDS; past the end
// of both (KEY_MAX, ~0).
template <int NT>
__device__ __forceinline__ void merge_eight(const MergeLds<NT>& m, uint32_t a0, uint32_t na, uint32_t b0, uint32_t nb,
                                            uint32_t diag, uint64_t (&k)[kPer], uint32_t (&ix)[kPer]) {
  uint32_t lo = diag > nb ? diag - nb : 0u, hi = diag < na ? diag : na;
  while (lo < hi) {
    const uint32_t mid = (lo + hi) >> 1;
    if (m.k[slot_of(a0 + mid)] <= m.k[slot_of(b0 + diag - 1 - mid)])
      lo = mid + 1;
    else
      hi = mid;
  }
  uint32_t a = a0 + lo, b = b0 + diag - lo;
  const uint32_t ae = a0 + na, be = b0 + nb;
  uint64_t ka = a < ae ? m.k[slot_of(a)] : KEY_MAX, kb = b < be ? m.k[slot_of(b)] : KEY_MAX;
#pragma unroll
  for (int r = 0; r < kPer; ++r) {
    const bool left = a < ae && (b >= be || ka <= kb);
    const uint32_t src = left ? a : b;
    k[r] = left ? ka : kb;
    ix[r] = src < (left ? ae : be) ? m.ix[slot_of(src)] : 0xFFFFFFFFu;
    if (left) {
      ++a;
      ka = a < ae ? m.k[slot_of(a)] : KEY_MAX;
    } else if (b < be) {
      ++b;
      kb = b < be ? m.k[slot_of(b)] : KEY_MAX;
    }
  }
}

template <int NT>
__device__ __forceinline__ void put_eight(MergeLds<NT>& m, const uint64_t (&k)[kPer], const uint32_t (&ix)[kPer]) {
#pragma unroll
  for (int r = 0; r < kPer; ++r) {
    m.k[threadIdx.x * (kPer + 1) + r] = k[r];
    m.ix[threadIdx.x * (kPer + 1) + r] = ix[r];
  }
}

// A thread's eight keys: odd-even transposition, which moves no key past an equal one.
__device__ __forceinline__ void sort_eight(uint64_t (&k)[kPer], uint32_t (&ix)[kPer]) {
#pragma unroll
  for (int p = 0; p < kPer; ++p)
#pragma unroll
    for (int r = p & 1; r + 1 < kPer; r += 2)
      if (k[r] > k[r + 1]) {
        const uint64_t x = k[r];
        const uint32_t y = ix[r];
        k[r] = k[r + 1], ix[r] = ix[r + 1];
        k[r + 1] = x, ix[r + 1] = y;
      }
}

// n elements sorted by (key, element) into m without merges: by a digit of up to 11 bits, counted and placed
// in LDS, then each key's rank among the few that share its digit.  k[r] is the key of element r NT + thread;
// no key is padding.  False, for the whole block, if the keys crowd into few digits: then nothing is in m.
constexpr int kOrderBits = 11;
constexpr uint32_t kOrderDigits = 1u << kOrderBits;
constexpr uint32_t kOrderMost = 32;  // keys that share a digit; 4096 to 5120 evenly spread ones: 2 on average
template <int NT>
struct OrderLds {
  uint32_t cnt[kOrderDigits], sh[NT / 64 + 1], most;
};
template <int NT>
__device__ __forceinline__ bool order_by_digit(MergeLds<NT>& m, OrderLds<NT>& o, const uint64_t (&k)[kPer], uint32_t n,
                                               int shift, uint32_t mask) {
  constexpr uint32_t D = (kOrderDigits + NT - 1) / NT;  // digits per thread
  for (uint32_t d = threadIdx.x; d < kOrderDigits; d += NT) o.cnt[d] = 0;
  if (threadIdx.x == 0) o.most = 0;
  __syncthreads();
  uint32_t at[kPer];
#pragma unroll
  for (int r = 0; r < kPer; ++r)
    at[r] = r * NT + threadIdx.x < n ? atomicAdd(&o.cnt[(uint32_t)(k[r] >> shift) & mask], 1u) : 0u;
  __syncthreads();
  uint32_t c[D], s = 0, most = 0, total;
#pragma unroll
  for (uint32_t j = 0; j < D; ++j) {
    const uint32_t d = threadIdx.x * D + j;
    c[j] = d < kOrderDigits ? o.cnt[d] : 0u;
    s += c[j];
    most = c[j] > most ? c[j] : most;
  }
  if (most > kOrderMost) o.most = 1;
  uint32_t run = block_exclusive_scan<uint32_t, NT>(s, o.sh, total);  // ends with a barrier
  if (o.most) return false;
#pragma unroll
  for (uint32_t j = 0; j < D; ++j) {
    const uint32_t d = threadIdx.x * D + j;
    if (d < kOrderDigits) o.cnt[d] = run;
    run += c[j];
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kPer; ++r) {
    const uint32_t i = r * NT + threadIdx.x;
    if (i < n) {
      const uint32_t p = slot_of(o.cnt[(uint32_t)(k[r] >> shift) & mask] + at[r]);
      m.k[p] = k[r];
      m.ix[p] = i;
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kPer; ++r) {
    const uint32_t i = r * NT + threadIdx.x;
    if (i < n) {
      const uint32_t d = (uint32_t)(k[r] >> shift) & mask;
      const uint32_t b = o.cnt[d], e = d + 1 < kOrderDigits ? o.cnt[d + 1] : n;
      uint32_t rank = 0;
      for (uint32_t q = b; q < e; ++q) {
        const uint64_t x = m.k[slot_of(q)];
        rank += x < k[r] || (x == k[r] && m.ix[slot_of(q)] < i) ? 1u : 0u;
      }
      at[r] = slot_of(b + rank);
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kPer; ++r) {
    const uint32_t i = r * NT + threadIdx.x;
    if (i < n) {
      m.k[at[r]] = k[r];
      m.ix[at[r]] = i;
    }
  }
  __syncthreads();
  return true;
}

// Chunk c of 4096 staged keys sorted by (key, index); block 0 zeroes the epoch's 8 summary words.
__global__ __launch_bounds__(kChunkThreads) void chunk_sort_kernel(const uint64_t* __restrict__ pk, uint32_t n,
                                                                   uint64_t* __restrict__ ko,
                                                                   uint32_t* __restrict__ io,
                                                                   uint32_t* __restrict__ summary) {
  __shared__ MergeLds<kChunkThreads> m;
  __shared__ OrderLds<kChunkThreads> order;
  __shared__ uint64_t differ;
  constexpr uint32_t kChunk = kChunkThreads * kPer;
  if (blockIdx.x == 0 && threadIdx.x < 8) summary[threadIdx.x] = 0;
  const uint32_t c0 = blockIdx.x * kChunk, cnt = n - c0 < kChunk ? n - c0 : kChunk;
  uint64_t k[kPer];
#pragma unroll
  for (int r = 0; r < kPer; ++r) {
    const uint32_t i = r * kChunkThreads + threadIdx.x;
    k[r] = pk[c0 + (i < cnt ? i : 0u)];
  }
  // the digit: the 11 bits from the topmost one in which the chunk's keys differ
  const uint64_t k0 = pk[c0];
  uint64_t diff = 0;
#pragma unroll
  for (int r = 0; r < kPer; ++r) diff |= k[r] ^ k0;
#pragma unroll
  for (int s = 32; s > 0; s >>= 1) diff |= __shfl_xor(diff, s);
  if (threadIdx.x == 0) differ = 0;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) atomicOr(reinterpret_cast<unsigned long long*>(&differ), (unsigned long long)diff);
  __syncthreads();
  const int top = 64 - __builtin_clzll(differ | 1ull), shift = top > kOrderBits ? top - kOrderBits : 0;
  if (!order_by_digit(m, order, k, cnt, shift, (1u << (top - shift)) - 1u)) {
    const uint32_t t0 = threadIdx.x * kPer;
    uint32_t ix[kPer];
#pragma unroll
    for (int r = 0; r < kPer; ++r) {
      k[r] = t0 + r < cnt ? pk[c0 + t0 + r] : KEY_MAX;
      ix[r] = t0 + r;
    }
    sort_eight(k, ix);
    for (uint32_t w = kPer; w < kChunk; w <<= 1) {  // uniform across the block
      put_eight(m, k, ix);
      __syncthreads();
      const uint32_t base = t0 & ~(2 * w - 1);
      merge_eight(m, base, w, base + w, w, t0 - base, k, ix);
      __syncthreads();
    }
    put_eight(m, k, ix);
    __syncthreads();
  }
#pragma unroll
  for (int r = 0; r < kPer; ++r) {
    const uint32_t i = r * kChunkThreads + threadIdx.x;
    if (i < cnt) {
      ko[c0 + i] = m.k[slot_of(i)];
      io[c0 + i] = c0 + m.ix[slot_of(i)];
    }
  }
}

// Where diagonal `diag` splits the merge of A (na keys) and B (nb keys): how many come from A.  One wave,
// 64 probes per step (four steps for runs of 2^19).
__device__ __forceinline__ uint32_t wave_split(const uint64_t* __restrict__ A, uint32_t na,
                                               const uint64_t* __restrict__ B, uint32_t nb, uint32_t diag, int lane) {
  uint32_t lo = diag > nb ? diag - nb : 0u, hi = diag < na ? diag : na;
  while (lo < hi) {  // wave-uniform
    const uint32_t step = (hi - lo + 63) / 64;
    const uint32_t p = lo + (uint32_t)lane * step;
    const bool left = p < hi && A[p] <= B[diag - 1 - p];
    const uint32_t c = (uint32_t)__popcll(__ballot(left));  // the probes that hold are the first c
    if (c == 0) break;
    const uint32_t top = lo + c * step;
    lo = lo + (c - 1) * step + 1;
    hi = top < hi ? top : hi;
  }
  return lo;
}

// One pass over runs of length L: tile t writes elements [t kTile, (t + 1) kTile) of the merged pairs.
// LAST: also the tile's number of keys that differ from the next one, for the de-duplication.
template <bool LAST>
__global__ __launch_bounds__(kTileThreads) void merge_tile_kernel(const uint64_t* __restrict__ kin,
                                                                  const uint32_t* __restrict__ iin,
                                                                  uint64_t* __restrict__ kout,
                                                                  uint32_t* __restrict__ iout, uint32_t n, uint32_t L,
                                                                  uint32_t* __restrict__ tile_kept) {
  __shared__ MergeLds<kTileThreads> m;
  __shared__ uint32_t split[2], kept_w[kTileThreads / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const uint32_t t0 = blockIdx.x * kTile;
  const uint32_t base = t0 / (2 * L) * (2 * L);  // 2 L is a multiple of kTile: a tile lies in one pair
  const uint32_t mid = base + L < n ? base + L : n;
  const uint32_t end = mid + L < n ? mid + L : n;
  const uint32_t na = mid - base, nb = end - mid;
  const uint32_t d0 = t0 - base, d1 = d0 + kTile < na + nb ? d0 + kTile : na + nb;
  if (w < 2) {
    const uint32_t s = wave_split(kin + base, na, kin + mid, nb, w == 0 ? d0 : d1, lane);
    if (lane == 0) split[w] = s;
  }
  __syncthreads();
  const uint32_t a0 = split[0], a1 = split[1], b0 = d0 - a0, b1 = d1 - a1;
  const uint32_t ca = a1 - a0, cb = b1 - b0, cnt = d1 - d0;
  uint64_t k[kPer];
  uint32_t ix[kPer];
#pragma unroll
  for (int r = 0; r < kPer; ++r) {  // every load before the first LDS store
    const uint32_t i = r * kTileThreads + threadIdx.x;
    if (i < cnt) {
      const uint32_t src = i < ca ? base + a0 + i : mid + b0 + (i - ca);
      k[r] = kin[src];
      ix[r] = iin[src];
    }
  }
  // the key after the tile, for its last element
  uint64_t next = KEY_MAX;
  if (LAST && threadIdx.x == 0) {
    const uint64_t xa = a1 < na ? kin[base + a1] : KEY_MAX, xb = b1 < nb ? kin[mid + b1] : KEY_MAX;
    next = xa < xb ? xa : xb;
  }
#pragma unroll
  for (int r = 0; r < kPer; ++r) {
    const uint32_t i = r * kTileThreads + threadIdx.x;
    if (i < cnt) {
      m.k[slot_of(i)] = k[r];
      m.ix[slot_of(i)] = ix[r];
    }
  }
  __syncthreads();
  const uint32_t diag = threadIdx.x * kPer < cnt ? threadIdx.x * kPer : cnt;
  merge_eight(m, 0, ca, ca, cb, diag, k, ix);
  __syncthreads();
  put_eight(m, k, ix);
  __syncthreads();
  uint32_t kept = 0;
#pragma unroll
  for (int r = 0; r < kPer; ++r) {
    const uint32_t i = r * kTileThreads + threadIdx.x;
    if (i < cnt) {
      const uint64_t x = m.k[slot_of(i)];
      kout[t0 + i] = x;
      iout[t0 + i] = m.ix[slot_of(i)];
      if (LAST && i + 1 < cnt) kept += x != m.k[slot_of(i + 1)] ? 1u : 0u;
    }
  }
  if constexpr (LAST) {
    if (threadIdx.x == 0 && cnt) kept += m.k[slot_of(cnt - 1)] != next ? 1u : 0u;  // staged keys are below KEY_MAX
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) kept += __shfl_xor(kept, o);
    if (lane == 0) kept_w[w] = kept;
    __syncthreads();
    if (threadIdx.x == 0) tile_kept[blockIdx.x] = kept_w[0] + kept_w[1] + kept_w[2] + kept_w[3];
  }
}

// The same count for keys sorted elsewhere (the radix sort of the largest batches).
__global__ __launch_bounds__(kTileThreads) void count_kept_kernel(const uint64_t* __restrict__ sk, uint32_t n,
                                                                  uint32_t* __restrict__ tile_kept) {
  __shared__ uint32_t kept_w[kTileThreads / 64];
  uint32_t kept = 0;
#pragma unroll
  for (int r = 0; r < kPer; ++r) {
    const uint32_t i = blockIdx.x * kTile + r * kTileThreads + threadIdx.x;
    if (i < n) kept += i + 1 == n || sk[i] != sk[i + 1] ? 1u : 0u;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) kept += __shfl_xor(kept, o);
  if ((threadIdx.x & 63) == 0) kept_w[threadIdx.x >> 6] = kept;
  __syncthreads();
  if (threadIdx.x == 0) tile_kept[blockIdx.x] = kept_w[0] + kept_w[1] + kept_w[2] + kept_w[3];
}

// The last write of each key to (uk, uv), its value read at the staging index (si) or from the sorted
// values (si null); *dm = how many.  Each block adds up the tiles before its own (2048 words for 2^22 keys).
__global__ __launch_bounds__(kTileThreads) void compact_last_kernel(const uint64_t* __restrict__ sk,
                                                                    const uint32_t* __restrict__ si,
                                                                    const uint64_t* __restrict__ v, uint32_t n,
                                                                    const uint32_t* __restrict__ tile_kept,
                                                                    uint64_t* __restrict__ uk,
                                                                    uint64_t* __restrict__ uv,
                                                                    uint32_t* __restrict__ dm) {
  constexpr int kW = kTileThreads / 64;
  __shared__ uint32_t scan_sh[kW + 1];
  __shared__ uint32_t cnt[kPer * kW];  // kept keys per 64 consecutive ones, in order
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  uint64_t k[kPer], x[kPer];
  uint32_t at[kPer];
  bool last[kPer];
#pragma unroll
  for (int r = 0; r < kPer; ++r) {
    const uint32_t i = blockIdx.x * kTile + r * kTileThreads + threadIdx.x;
    k[r] = i < n ? sk[i] : KEY_MAX;
    last[r] = i < n && (i + 1 == n || sk[i + 1] != k[r]);
    at[r] = i < n ? (si ? si[i] : i) : 0u;
  }
#pragma unroll
  for (int r = 0; r < kPer; ++r) x[r] = v[at[r]];
  uint32_t part = 0, before;
  for (uint32_t t = threadIdx.x; t < blockIdx.x; t += kTileThreads) part += tile_kept[t];
#pragma unroll
  for (int r = 0; r < kPer; ++r) {
    const uint64_t b = __ballot(last[r]);
    at[r] = (uint32_t)__popcll(b & ((1ull << lane) - 1ull));
    if (lane == 0) cnt[r * kW + w] = (uint32_t)__popcll(b);
  }
  (void)block_exclusive_scan<uint32_t, kTileThreads>(part, scan_sh, before);  // its barriers cover cnt too
  uint32_t total = 0;
#pragma unroll
  for (int r = 0; r < kPer; ++r)
#pragma unroll
    for (int ww = 0; ww < kW; ++ww) {
      if (ww == w) at[r] += before + total;
      total += cnt[r * kW + ww];
    }
#pragma unroll
  for (int r = 0; r < kPer; ++r)
    if (last[r]) {
      uk[at[r]] = k[r];
      uv[at[r]] = x[r];
    }
  if (threadIdx.x == 0 && (blockIdx.x + 1) * (uint64_t)kTile >= n) *dm = before + total;
}

// ---- bulk build ---------------------------------------------------------------------------------
//
// A bucket of the build's pairs (at most kBucketSortMax), sorted in LDS like a chunk above, then written to
// its leaves: sorted pair g goes to slot g % fill of leaf g / fill.  The values are read from the bucket's own
// 40 KiB, which its block has just brought to L2.  4 million pairs: partition 45 us and this kernel 66 (132
// with nine merges in place of the digit), where eight radix passes, the validation, the leaf fill and the
// minima took 388; the build with one search of its keys went 656 -> 312 us.
constexpr int kBucketThreads = (int)kBucketSortMax / kPer;
__global__ __launch_bounds__(kBucketThreads) void bucket_sort_fill_kernel(
    const uint64_t* __restrict__ keys, const uint64_t* __restrict__ vals, size_t n, int shift,
    const uint32_t* __restrict__ totals, uint32_t fill, Leaf* __restrict__ leaves, uint64_t* __restrict__ mins,
    uint32_t* __restrict__ flags, uint32_t skip, uint64_t* __restrict__ edge) {
  __shared__ MergeLds<kBucketThreads> m;
  __shared__ OrderLds<kBucketThreads> order;
  __shared__ uint32_t part_w[kBucketThreads / 64], bad;
  if (*flags & skip) return;  // block-uniform: set before this launch
  const uint32_t cnt = totals[blockIdx.x];
  if (cnt == 0) return;
  uint32_t part = 0;  // the pairs before this bucket
  for (uint32_t b = threadIdx.x; b < blockIdx.x; b += kBucketThreads) part += totals[b];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) part += __shfl_xor(part, o);
  if ((threadIdx.x & 63) == 0) part_w[threadIdx.x >> 6] = part;
  if (threadIdx.x == 0) bad = 0;
  __syncthreads();
  uint32_t start = 0;
#pragma unroll
  for (int w = 0; w < kBucketThreads / 64; ++w) start += part_w[w];
  uint64_t k[kPer];
#pragma unroll
  for (int r = 0; r < kPer; ++r) {
    const uint32_t i = r * kBucketThreads + threadIdx.x;
    k[r] = keys[start + (i < cnt ? i : 0u)];
  }
  const int bits = shift < kOrderBits ? shift : kOrderBits;  // the digit: the bits below the bucket's
  if (!order_by_digit(m, order, k, cnt, shift - bits, (1u << bits) - 1u)) {
    const uint32_t t0 = threadIdx.x * kPer;
    uint32_t ix[kPer];
#pragma unroll
    for (int r = 0; r < kPer; ++r) {
      k[r] = t0 + r < cnt ? keys[start + t0 + r] : KEY_MAX;
      ix[r] = t0 + r;
    }
    sort_eight(k, ix);
    for (uint32_t w = kPer; w < cnt; w <<= 1) {  // uniform across the block
      put_eight(m, k, ix);
      __syncthreads();
      const uint32_t base = t0 & ~(2 * w - 1);
      const uint32_t na = base + w < kBucketSortMax ? w : kBucketSortMax - base;
      const uint32_t nb = base + na + w < kBucketSortMax ? w : kBucketSortMax - base - na;
      merge_eight(m, base, na, base + na, nb, t0 - base, k, ix);
      __syncthreads();
    }
    put_eight(m, k, ix);
    __syncthreads();
  }
#pragma unroll
  for (int r = 0; r < kPer; ++r) {
    const uint32_t i = r * kBucketThreads + threadIdx.x;
    if (i < cnt) {
      const uint64_t key = m.k[slot_of(i)];
      const uint32_t src = m.ix[slot_of(i)];
      const uint32_t g = start + i, leaf = g / fill, slot = g - leaf * fill;
      uint32_t f = key == KEY_MAX ? 1u : 0u;
      if (i + 1 < cnt && m.k[slot_of(i + 1)] == key) f |= 2u;  // equal keys share a bucket
      if (f) atomicOr(&bad, f);
      leaves[leaf].key[slot] = key;
      leaves[leaf].val[slot] = src < cnt ? vals[start + src] : 0ull;  // (a KEY_MAX key may stand for padding)
      if (slot == 0) mins[leaf] = key;
      if (slot + 1 == fill || g + 1 == n)
        for (uint32_t p = slot + 1; p < (uint32_t)LEAF_KEYS; ++p) {
          leaves[leaf].key[p] = KEY_MAX;
          leaves[leaf].val[p] = 0ull;
        }
      if (g == 0) edge[0] = key;
      if (g + 1 == n) edge[1] = key;
    }
  }
  __syncthreads();
  if (threadIdx.x == 0 && bad) atomicOr(flags, bad);
}

}  // namespace

hipError_t bucket_sort_fill(const uint64_t* keys, const uint64_t* vals, size_t n, int top, int bits,
                            const uint32_t* totals, int fill, Leaf* leaves, uint64_t* mins, uint32_t* flags,
                            uint32_t skip, uint64_t* edge, hipStream_t s) {
  ProfScope prof("build", s);
  hipLaunchKernelGGL(bucket_sort_fill_kernel, dim3(1u << bits), dim3(kBucketThreads), 0, s, keys, vals, n,
                     top > bits ? top - bits : 0, totals,
                     (uint32_t)fill, leaves, mins, flags, skip, edge);
  return hipGetLastError();
}

size_t dedupe_tmp_bytes(size_t n) { return ((n + kTile - 1) / kTile) * sizeof(uint32_t); }

hipError_t merge_sort_index(const uint64_t* pk, uint32_t n, uint64_t* k0, uint64_t* k1, uint32_t* i0, uint32_t* i1,
                            uint32_t* tile_kept, uint32_t* summary, hipStream_t s, const uint64_t** sorted_keys,
                            const uint32_t** sorted_index) {
  if (n <= kSmallUpdate || n > kMergeUpdate) return hipErrorInvalidValue;
  ProfScope prof("update", s);
  hipLaunchKernelGGL(chunk_sort_kernel, dim3((n + kSmallUpdate - 1) / kSmallUpdate), dim3(kChunkThreads), 0, s, pk, n,
                     k0, i0, summary);
  uint64_t *ka = k0, *kb = k1;
  uint32_t *ia = i0, *ib = i1;
  const dim3 grid((n + kTile - 1) / kTile);
  for (uint32_t L = kSmallUpdate; L < n; L *= 2) {
    if (2 * (uint64_t)L >= n)
      hipLaunchKernelGGL(merge_tile_kernel<true>, grid, dim3(kTileThreads), 0, s, ka, ia, kb, ib, n, L, tile_kept);
    else
      hipLaunchKernelGGL(merge_tile_kernel<false>, grid, dim3(kTileThreads), 0, s, ka, ia, kb, ib, n, L, tile_kept);
    std::swap(ka, kb);
    std::swap(ia, ib);
  }
  *sorted_keys = ka;
  *sorted_index = ia;
  return hipGetLastError();
}

hipError_t count_kept(const uint64_t* sorted_keys, size_t n, uint32_t* tile_kept, hipStream_t s) {
  if (!n) return hipErrorInvalidValue;
  ProfScope prof("update", s);
  hipLaunchKernelGGL(count_kept_kernel, dim3((unsigned)((n + kTile - 1) / kTile)), dim3(kTileThreads), 0, s,
                     sorted_keys, (uint32_t)n, tile_kept);
  return hipGetLastError();
}

hipError_t compact_last(const uint64_t* sorted_keys, const uint32_t* index, const uint64_t* vals, size_t n,
                        const uint32_t* tile_kept, uint64_t* uk, uint64_t* uv, uint32_t* dm, hipStream_t s) {
  if (!n) return hipErrorInvalidValue;
  ProfScope prof("update", s);
  hipLaunchKernelGGL(compact_last_kernel, dim3((unsigned)((n + kTile - 1) / kTile)), dim3(kTileThreads), 0, s,
                     sorted_keys, index, vals, (uint32_t)n, tile_kept, uk, uv, dm);
  return hipGetLastError();
}

}  // namespace hm

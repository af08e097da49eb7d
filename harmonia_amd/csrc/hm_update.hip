// Batched upsert on the device.
//
// The reference updates on the CPU: 56 threads upsert under per-leaf mutexes, splits are deferred
// to a serial pass, and the inner levels plus the prefix array are rebuilt breadth-first on the
// host (insert_parallel_Newupdate_batch / rebuild_without_leaf, H/src/bpt-ppi-update-batch.cpp:86-200,
// H/src/bpt-ppi-update.cpp:320-463).  Here a batch is sorted and de-duplicated (last write wins),
// each key is located in the tree, existing keys get their value overwritten in place, and new keys
// are merged into their leaf's free slots.  When some leaf would overflow, every leaf is re-laid
// out (overflowing leaves split evenly into ceil(total / fill) leaves) at offsets given by a device
// scan, and the caller rebuilds the inner levels and re-scans the prefix array on the device.
//
// The common serving case (a few thousand keys, no leaf overflows) stays O(batch) and is bound by its
// launches: the keys are placed in order by counting, de-duplicated and located in one launch, each
// leaf's keys form one run of the sorted batch, and one thread per run plans (overflow? how many new
// keys?) and then applies it.  An epoch of 4001 keys (2^24 stored) with the read of its keys: 115 us in
// 17 launches, now 59 us in six.
#include <algorithm>

#include "hm_device.h"

namespace hm {
namespace {

int grid_for(size_t work, int threads) {
  size_t g = (work + threads - 1) / threads;
  if (g < 1) g = 1;
  if (g > 65536) g = 65536;
  return (int)g;
}

// Register-array access with a run-time index, as unrolled selects: a dynamic index into a local
// array would put the whole leaf in scratch memory.
__device__ __forceinline__ uint64_t pick(const uint64_t (&a)[LEAF_KEYS], int i) {
  // masks rather than selects: the compiler folds a select chain back into one indexed load
  uint64_t r = 0;
#pragma unroll
  for (int s = 0; s < LEAF_KEYS; ++s) r |= a[s] & (0ull - (uint64_t)(i == s));
  return r;
}

__device__ __forceinline__ void put(uint64_t (&a)[LEAF_KEYS], int i, uint64_t v) {
#pragma unroll
  for (int s = 0; s < LEAF_KEYS; ++s) a[s] = i == s ? v : a[s];
}

// A leaf held in registers (a Leaf struct copy would live in scratch memory).
struct LeafRegs {
  uint64_t key[LEAF_KEYS];
  uint64_t val[LEAF_KEYS];
};

__device__ __forceinline__ LeafRegs load_leaf(const Leaf* p) {
  const ulonglong2* q = reinterpret_cast<const ulonglong2*>(p);
  LeafRegs r;
#pragma unroll
  for (int i = 0; i < LEAF_KEYS / 2; ++i) {
    const ulonglong2 a = q[i];
    r.key[2 * i] = a.x;
    r.key[2 * i + 1] = a.y;
  }
#pragma unroll
  for (int i = 0; i < LEAF_KEYS / 2; ++i) {
    const ulonglong2 b = q[LEAF_KEYS / 2 + i];
    r.val[2 * i] = b.x;
    r.val[2 * i + 1] = b.y;
  }
  return r;
}

__device__ __forceinline__ void store_leaf(Leaf* p, const LeafRegs& r) {
  ulonglong2* q = reinterpret_cast<ulonglong2*>(p);
#pragma unroll
  for (int i = 0; i < LEAF_KEYS / 2; ++i) q[i] = make_ulonglong2(r.key[2 * i], r.key[2 * i + 1]);
#pragma unroll
  for (int i = 0; i < LEAF_KEYS / 2; ++i) q[LEAF_KEYS / 2 + i] = make_ulonglong2(r.val[2 * i], r.val[2 * i + 1]);
}

__device__ __forceinline__ int leaf_count(const LeafRegs& l) {
  int c = 0;
#pragma unroll
  for (int i = 0; i < LEAF_KEYS; ++i) c += l.key[i] != KEY_MAX ? 1 : 0;
  return c;
}

__device__ __forceinline__ int leaf_count(const Leaf& l) {
  int c = 0;
#pragma unroll
  for (int i = 0; i < LEAF_KEYS; ++i) c += l.key[i] != KEY_MAX ? 1 : 0;
  return c;
}

// Stream the merge of a leaf's keys with its inserts (the batch keys from `start` on that are not
// found and map to this leaf; they are contiguous among the not-found keys because the batch is
// sorted) in key order, calling emit(i, key, value) for i = 0, 1, ...; returns the merged count.
template <typename Emit>
__device__ __forceinline__ int merge_leaf(const LeafRegs& l, uint32_t n_ins, uint32_t start, const uint64_t* __restrict__ bk,
                          const uint64_t* __restrict__ bv, const uint8_t* __restrict__ found, Emit emit) {
  const int cur = leaf_count(l);
  int a = 0, c = 0;
  uint32_t b = start, taken = 0;
  while (taken < n_ins && found[b]) ++b;  // skip existing keys interleaved with the inserts
  while (a < cur || taken < n_ins) {
    const uint64_t ka = pick(l.key, a);
    const bool take_leaf = taken >= n_ins || (a < cur && ka < bk[b]);
    if (take_leaf) {
      emit(c, ka, pick(l.val, a));
      ++a;
    } else {
      emit(c, bk[b], bv[b]);
      ++taken;
      ++b;
      while (taken < n_ins && found[b]) ++b;
    }
    ++c;
  }
  return c;
}

__device__ __forceinline__ bool run_head(const uint32_t* __restrict__ leaf, uint32_t i) {
  return i == 0 || leaf[i] != leaf[i - 1];
}

// Re-layout, the batch's runs: first[leaf] = the run's first entry, and there (two passes: the second looks
// its run up in first) the leaf's slots that the batch overwrites as a bit mask and the run's end.  A run's
// new keys are its entries less the mask's bits, so no thread walks a run and no two add to one word: 2^16
// keys appended after the largest took 40 ms in one thread of the plan, 18 in one of the merge and 0.7 in
// additions to one word; now all of it takes 25 us (an epoch: 50 ms, now 0.25).
__global__ void run_heads_kernel(const uint32_t* __restrict__ leaf, uint32_t m, uint32_t* __restrict__ first,
                                 uint32_t* __restrict__ mask) {
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < m; i += stride) {
    mask[i] = 0;
    if (run_head(leaf, i)) first[leaf[i]] = i;  // one writer per leaf
  }
}

__global__ void run_ends_kernel(const uint32_t* __restrict__ leaf, const uint32_t* __restrict__ slot,
                                const uint8_t* __restrict__ found, uint32_t m, const uint32_t* __restrict__ first,
                                uint32_t* __restrict__ mask, uint32_t* __restrict__ end) {
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < m; i += stride) {
    const uint32_t L = leaf[i];
    if (found[i]) atomicOr(&mask[first[L]], 1u << (slot[i] & 255u));
    if (i + 1 == m || leaf[i + 1] != L) end[first[L]] = i + 1;
  }
}

// New leaves per old leaf, and the new keys of the leaves that the batch touches (the locate step left the
// free slots beside the slot: no leaf is read).
__global__ void new_counts_kernel(const uint32_t* __restrict__ first, const uint32_t* __restrict__ mask,
                                  const uint32_t* __restrict__ end, const uint32_t* __restrict__ slot, size_t n_leaves,
                                  int fill, uint32_t* __restrict__ ins, uint32_t* __restrict__ cnt) {
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n_leaves; i += stride) {
    const uint32_t h = first[i];
    if (h == 0xFFFFFFFFu) {
      cnt[i] = 1u;
      continue;
    }
    const uint32_t a = end[h] - h - (uint32_t)__popc(mask[h]);
    const uint32_t total = (uint32_t)LEAF_KEYS - (slot[h] >> 8) + a;
    ins[i] = a;
    cnt[i] = total <= (uint32_t)LEAF_KEYS ? 1u : (total + fill - 1) / fill;
  }
}

// Re-layout, part 1: every leaf in [lo, hi) the batch does not touch moves unchanged to
// new_start[i].  Runs of untouched leaves shift by a constant, so this is a coalesced streaming copy
// in 16-byte pieces; the piece holding key[0] also records the leaf's minimum key for the inner
// rebuild (which then does not read a cache line per leaf again).
__global__ __launch_bounds__(256) void relayout_copy_kernel(const Leaf* __restrict__ old_leaves, size_t lo, size_t hi,
                                                            const uint32_t* __restrict__ first,
                                                            const uint32_t* __restrict__ new_start,
                                                            Leaf* __restrict__ new_leaves,
                                                            uint64_t* __restrict__ new_mins) {
  constexpr int kPieces = sizeof(Leaf) / 16;
  const ulonglong2* src = reinterpret_cast<const ulonglong2*>(old_leaves);
  ulonglong2* dst = reinterpret_cast<ulonglong2*>(new_leaves);
  const size_t end = hi * kPieces;
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t u = lo * kPieces + (size_t)blockIdx.x * blockDim.x + threadIdx.x; u < end; u += stride) {
    const size_t i = u / kPieces;
    if (first[i] == 0xFFFFFFFFu) {
      const ulonglong2 v = src[u];
      dst[(size_t)new_start[i] * kPieces + u % kPieces] = v;
      if (u % kPieces == 0) new_mins[new_start[i]] = v.x;
    }
  }
}

// Re-layout, part 2: one thread per batch entry.  A leaf that overflows is split evenly into
// ceil(total / fill) leaves at new_start[L]: part p holds the merged keys [p c / parts, (p + 1) c / parts),
// at most ceil(c / parts) <= fill <= 8 each.  The entry's place among the merged keys follows from its slot
// and from the new keys before it (entries since the run's head less those that overwrite a slot below its
// own).  It also moves the leaf's keys between its slot and the next entry's (the head those below its own),
// with the new value if it overwrites one.  Whoever places a part's last key pads the part.
__global__ __launch_bounds__(256) void relayout_touched_kernel(
    const Leaf* __restrict__ old_leaves, const uint32_t* __restrict__ ins, const uint32_t* __restrict__ first,
    const uint32_t* __restrict__ mask, const uint32_t* __restrict__ bleaf, const uint32_t* __restrict__ bslot,
    const uint64_t* __restrict__ bk, const uint64_t* __restrict__ bv, const uint8_t* __restrict__ found, uint32_t m,
    const uint32_t* __restrict__ new_start, int fill, Leaf* __restrict__ new_leaves, uint64_t* __restrict__ new_mins) {
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < m; i += stride) {
    const uint32_t L = bleaf[i], h = first[L], sl = bslot[i], s = sl & 255u;
    const uint32_t cur = (uint32_t)LEAF_KEYS - (sl >> 8);
    const uint32_t c = cur + ins[L];
    const uint32_t parts = c <= (uint32_t)LEAF_KEYS ? 1u : (c + (uint32_t)fill - 1u) / (uint32_t)fill;
    const bool upd = found[i] != 0;
    const uint32_t before = i - h - (uint32_t)__popc(mask[h] & ((1u << s) - 1u));
    const uint32_t j0 = i == h ? 0u : s;
    const uint32_t j1 = i + 1 < m && bleaf[i + 1] == L ? bslot[i + 1] & 255u : cur;
    Leaf* dst = new_leaves + new_start[L];
    uint64_t* dmin = new_mins + new_start[L];
    auto place = [&](uint32_t r, uint64_t k, uint64_t v) {
      uint32_t p = 0, lo = 0, hi = c;
      if (c > 65535u) {
        p = (uint32_t)(((uint64_t)(r + 1) * parts - 1) / c);
        lo = (uint32_t)((uint64_t)p * c / parts);
        hi = (uint32_t)((uint64_t)(p + 1) * c / parts);
      } else if (parts > 1) {  // the same in 32 bits: parts <= c
        p = ((r + 1) * parts - 1) / c;
        lo = p * c / parts;
        hi = (p + 1) * c / parts;
      }
      const uint32_t q = r - lo;
      dst[p].key[q] = k;
      dst[p].val[q] = v;
      if (q == 0) dmin[p] = k;  // every part gets at least one key
      if (r + 1 == hi)
        for (uint32_t x = q + 1; x < (uint32_t)LEAF_KEYS; ++x) {
          dst[p].key[x] = KEY_MAX;
          dst[p].val[x] = 0ull;
        }
    };
    if (!upd) place(s + before, bk[i], bv[i]);
    if (j0 >= j1) continue;
    const LeafRegs l = load_leaf(old_leaves + L);
#pragma unroll
    for (uint32_t j = 0; j < (uint32_t)LEAF_KEYS; ++j)
      if (j >= j0 && j < j1)
        place(j < s ? j : j + before + (upd ? 0u : 1u), l.key[j], upd && j == s ? bv[i] : l.val[j]);
  }
}

// Small batches (n <= kSmallUpdate), first kernel: every staged key's place in the order by (key, staging
// index), counted against all n keys held in LDS.  A block places 16 keys, 32 slices of the batch each, so
// 4096 keys take 256 blocks and 128 steps of two compares per thread.  One block sorting 4096 keys (LSD
// radix in LDS, eight passes) took 37.6 us on one CU with the others idle.
constexpr int kRankThreads = 512;
constexpr int kRankKeys = 16;
constexpr int kRankSlices = kRankThreads / kRankKeys;
__global__ __launch_bounds__(kRankThreads) void rank_keys_kernel(const uint64_t* __restrict__ pk, uint32_t n,
                                                                 uint64_t* __restrict__ sk, uint32_t* __restrict__ si,
                                                                 uint32_t* __restrict__ summary) {
  __shared__ ulonglong2 lk[kSmallUpdate / 2];
  __shared__ uint32_t place[kRankKeys];
  if (blockIdx.x == 0 && threadIdx.x < 8) summary[threadIdx.x] = 0;
  if (threadIdx.x < kRankKeys) place[threadIdx.x] = 0;
  const uint32_t pairs = (n + 1) / 2;
  for (uint32_t p = threadIdx.x; p < pairs; p += kRankThreads)
    lk[p] = make_ulonglong2(pk[2 * p], 2 * p + 1 < n ? pk[2 * p + 1] : KEY_MAX);
  __syncthreads();
  const uint32_t ki = blockIdx.x * kRankKeys + threadIdx.x % kRankKeys;
  // staged keys are below KEY_MAX, so an earlier equal key counts as smaller through key + 1
  const uint64_t key = ki < n ? pk[ki] : 0ull;
  uint32_t c = 0;
#pragma unroll 8
  for (uint32_t p = threadIdx.x / kRankKeys; p < pairs; p += kRankSlices) {
    const ulonglong2 v = lk[p];
    c += v.x < key + (2 * p < ki ? 1u : 0u) ? 1u : 0u;
    c += v.y < key + (2 * p + 1 < ki ? 1u : 0u) ? 1u : 0u;
  }
  c += __shfl_xor(c, 16);
  c += __shfl_xor(c, 32);
  if ((threadIdx.x & 63) < kRankKeys) atomicAdd(&place[threadIdx.x % kRankKeys], c);
  __syncthreads();
  if (threadIdx.x < kRankKeys && ki < n) {
    sk[place[threadIdx.x]] = key;
    si[place[threadIdx.x]] = ki;
  }
}

// Number of keys of a leaf's 8 (one per lane of an 8-lane group): its free slots.
__device__ __forceinline__ uint32_t group_room(uint64_t k, int gbase) {
  return (uint32_t)LEAF_KEYS - (uint32_t)__popcll((__ballot(k != KEY_MAX) >> gbase) & 0xFFull);
}

// Second kernel: the last write of each key kept (32 sorted entries per block, which counts the kept
// entries before its own: at most 32 KiB of keys, all in L2), and located, 8 lanes per key.
template <int F>
__global__ __launch_bounds__(256) void dedupe_locate_kernel(TreeView tv, const uint64_t* __restrict__ sk,
                                                            const uint32_t* __restrict__ si,
                                                            const uint64_t* __restrict__ pv, uint32_t n,
                                                            uint64_t* __restrict__ uk, uint64_t* __restrict__ uv,
                                                            uint32_t* __restrict__ leaf_out,
                                                            uint32_t* __restrict__ slot_out,
                                                            uint8_t* __restrict__ found_out, uint32_t* __restrict__ dm) {
  constexpr uint32_t kPer = 32;
  __shared__ uint32_t before_w[4];
  __shared__ uint32_t kept_s[kPer];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const uint32_t base = blockIdx.x * kPer;
  uint32_t c = 0;
  for (uint32_t p = threadIdx.x; p < base; p += 256) c += sk[p] != sk[p + 1] ? 1u : 0u;  // base < n
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o);
  if (lane == 0) before_w[w] = c;
  const int gl = lane & 7, gbase = lane - gl;
  const uint32_t g = threadIdx.x / 8, p = base + g;
  const uint64_t t = p < n ? sk[p] : 0ull;
  const bool kept = p < n && (p + 1 == n || sk[p + 1] != t);
  if (gl == 0) kept_s[g] = kept ? 1u : 0u;
  const uint32_t leaf = descend<F, 8>(tv, 0, nullptr, t, gl, gbase);
  const uint64_t k[1] = {tv.leaves[leaf].key[gl]};
  const int lt = group_count_lt<8, 1>(k, t, gbase);
  const bool eq = group_any_eq<8, 1>(k, t, gbase);
  const uint32_t room = group_room(k[0], gbase);
  __syncthreads();
  const uint32_t before = before_w[0] + before_w[1] + before_w[2] + before_w[3];
  const uint32_t km = (uint32_t)__ballot(lane < (int)kPer && kept_s[lane & (kPer - 1)] != 0u);
  if (kept && gl == 0) {
    const uint32_t o = before + (uint32_t)__popc(km & ((1u << g) - 1u));
    uk[o] = t;
    uv[o] = pv[si[p]];
    leaf_out[o] = leaf;
    slot_out[o] = (uint32_t)lt | room << 8;
    found_out[o] = eq ? 1 : 0;
  }
  if (threadIdx.x == 0 && base + kPer >= n) *dm = before + (uint32_t)__popc(km);
}

// Whether the run that starts at entry i overflows its leaf: at most 17 entries are read, for a leaf has at
// most 8 keys to overwrite and 8 free slots.
__device__ __forceinline__ bool run_overflows(const uint32_t* __restrict__ leaf, const uint32_t* __restrict__ slot,
                                              const uint8_t* __restrict__ found, uint32_t i, uint32_t m) {
  const uint32_t L = leaf[i], room = slot[i] >> 8;
  uint32_t ins = 0;
  for (uint32_t j = i; ins <= room && j < m && leaf[j] == L; ++j) ins += found[j] ? 0u : 1u;
  return ins > room;
}

// Plan an epoch, one thread per leaf the batch touches (its first batch entry: the batch is sorted, so a
// leaf's and a node's entries are contiguous).  Last-level node j holds leaves
// [j F, min((j + 1) F, n_leaves)): the bulk build and re-layouts fill every node but the last, and
// an in-node re-spread keeps each node's leaf count.  If a leaf of a node would overflow, the node goes
// on the re-spread list (nlist: node, first batch entry; count in summary[4]) when its leaves can hold all
// its keys, or else the epoch needs a full re-layout (summary[0] tells the other waves early: a hint).
// What a block has found (new keys, a node listed, a full node) travels in the one addition to summary[6..7]
// that also counts the block as finished: the block that finishes last has it all from the value returned,
// and no order among separate words matters (a barrier waits for no atomic whose result is unused).
// The locate step left each entry's leaf's free slots beside its slot, so the plan reads leaves only for
// nodes that overflow, and a thread walks one leaf's entries, not a node's: 2^20 entries took 61 us with
// one thread per node reading its leaves, now 12.  A node that overflows is planned by the wave that holds
// its first overflowing leaf, 64 entries at a step (2^16 new keys, most nodes of 2^16 overflowing: 109 us
// with one thread per node, now 11), and not at all once some node has asked for the re-layout (2^20 new
// keys of 2^22: 528 us on average over epochs of both kinds, now 47).  The block that
// finishes last writes the summary and the smallest and largest key to `host` (mapped pinned memory:
// words 0..4 and the two u64 at word 8), in place of two more launches.
constexpr uint32_t kPlanList = 1024;  // nodes that a block lists in LDS
// The word of that addition: new keys (fewer than 2^31 entries), then three counts of blocks, ten bits each.
constexpr int kPlanBlocks = 256;
constexpr int kPlanDone = 32, kPlanListed = 42, kPlanFull = 52;
static_assert(kPlanBlocks < 1024, "a count of blocks fits ten bits");
__global__ __launch_bounds__(1024) void plan_runs_kernel(const Leaf* __restrict__ leaves, uint32_t n_leaves, int F,
                                 const uint32_t* __restrict__ leaf, const uint32_t* __restrict__ slot,
                                 const uint8_t* __restrict__ found, const uint64_t* __restrict__ uk, size_t n_max,
                                 const uint32_t* __restrict__ dm, uint32_t* __restrict__ summary,
                                 uint32_t* __restrict__ nlist, uint32_t* __restrict__ host) {
  __shared__ uint32_t block_new, block_full, block_nodes, block_at;
  __shared__ uint32_t list[2 * kPlanList];
  __shared__ uint64_t all_found;
  if (threadIdx.x == 0) block_new = block_full = block_nodes = 0;
  __syncthreads();
  const uint32_t m = dm ? *dm : (uint32_t)n_max;
  const uint32_t stride = gridDim.x * blockDim.x;
  const uint32_t uF = (uint32_t)F;
  const uint32_t lane = threadIdx.x & 63;
  uint32_t my_new = 0;
  for (uint32_t w = blockIdx.x * blockDim.x + (threadIdx.x & ~63u); w < m; w += stride) {  // wave-uniform
    const uint32_t i = w + lane;
    uint32_t node = ~0u;  // no node: there are fewer than 2^32 leaves
    bool over = false, isnew = false;
    if (i < m) {
      node = leaf[i] / uF;
      isnew = !found[i];
      over = run_head(leaf, i) && run_overflows(leaf, slot, found, i, m);
    }
    my_new += isnew ? 1u : 0u;
    uint64_t todo = __ballot(over);
    if (todo && (__builtin_amdgcn_readfirstlane((int)__hip_atomic_load(&summary[0], __ATOMIC_RELAXED,
                                                                       __HIP_MEMORY_SCOPE_AGENT)) & 2))
      todo = 0;
    while (todo) {  // wave-uniform: the nodes of the wave's overflowing leaves, one after the other
      const uint32_t nd = (uint32_t)__builtin_amdgcn_readlane((int)node, __builtin_ctzll(todo));
      const uint64_t in0 = __ballot(node == nd);
      todo &= ~in0;
      uint32_t node_new = (uint32_t)__popcll(in0 & __ballot(isnew));
      uint32_t i0 = w + (uint32_t)__builtin_ctzll(in0);  // the node's first entry
      bool first = true;
      for (uint32_t b = w; b > 0 && i0 == b;) {  // back to it, unless an earlier leaf of the node overflows
        b -= 64;
        const uint32_t j = b + lane;
        const bool in = leaf[j] / uF == nd;
        first = !__any(in && run_head(leaf, j) && run_overflows(leaf, slot, found, j, m));
        const uint64_t inb = __ballot(in);
        if (!first || !inb) break;
        i0 = b + (uint32_t)__builtin_ctzll(inb);
        node_new += (uint32_t)__popcll(__ballot(in && !found[j]));
      }
      if (!first) continue;
      const uint32_t x0 = nd * uF, x1 = x0 + uF < n_leaves ? x0 + uF : n_leaves;
      const uint32_t cap = (x1 - x0) * (uint32_t)LEAF_KEYS;
      bool more = in0 >> 63;
      for (uint32_t b = w + 64; more && b < m && node_new <= cap; b += 64) {  // on to its last
        const uint32_t j = b + lane;
        const bool in = j < m && leaf[j] / uF == nd;
        node_new += (uint32_t)__popcll(__ballot(in && !found[j]));
        more = __all(in);
      }
      uint32_t total = 0;
      for (uint32_t x = x0 + lane; x < x1; x += 64) total += (uint32_t)leaf_count(leaves[x]);
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) total += (uint32_t)__shfl_xor((int)total, o);
      total += node_new;
      if (lane == 0) {
        if (total > cap) {
          if (!atomicExch(&block_full, 1u)) atomicOr(&summary[0], 2u);  // at once: the others need not go on
        } else {
          const uint32_t k = atomicAdd(&block_nodes, 1u);
          uint32_t* to = k < kPlanList ? list + 2 * k : nlist + 2 * atomicAdd(&summary[4], 1u);
          to[0] = nd;
          to[1] = i0;
        }
      }
    }
  }
  // new-key count: wave sum, then one LDS atomic per wave and one global atomic per block
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) my_new += __shfl_xor(my_new, o);
  if ((threadIdx.x & 63) == 0 && my_new) atomicAdd(&block_new, my_new);
  __syncthreads();
  // the block's nodes: one addition for their places (each takes about 10 ns, one after the other)
  const uint32_t nodes = block_nodes < kPlanList ? block_nodes : kPlanList;
  if (nodes > 0) {  // block-uniform
    if (threadIdx.x == 0) block_at = atomicAdd(&summary[4], nodes);
    __syncthreads();
    for (uint32_t x = threadIdx.x; x < 2 * nodes; x += blockDim.x) nlist[2 * block_at + x] = list[x];
  }
  __syncthreads();  // every wave has the results of its additions to summary[4], its list places
  if (threadIdx.x == 0) {
    // (A device-scope fence in every block would write the L2 back: 0.25 ms for 2^20 entries.)
    const uint64_t mine = (uint64_t)block_new | 1ull << kPlanDone | (nodes ? 1ull << kPlanListed : 0ull) |
                          (block_full ? 1ull << kPlanFull : 0ull);
    all_found = mine + atomicAdd(reinterpret_cast<unsigned long long*>(summary + 6), (unsigned long long)mine);
  }
  __syncthreads();
  const uint64_t all = all_found;
  if (((all >> kPlanDone) & 1023u) != gridDim.x) return;  // not the last block
  if (threadIdx.x < 5)
    host[threadIdx.x] = threadIdx.x == 0   ? (all >> kPlanFull ? 3u : (all >> kPlanListed) & 1023u ? 1u : 0u)
                        : threadIdx.x == 1 ? (uint32_t)all
                                           : __hip_atomic_load(&summary[threadIdx.x], __ATOMIC_RELAXED,
                                                               __HIP_MEMORY_SCOPE_AGENT);
  if (threadIdx.x == 64) {
    uint64_t* edge = reinterpret_cast<uint64_t*>(host + 8);
    edge[0] = m ? uk[0] : KEY_MAX;
    edge[1] = m ? uk[m - 1] : 0ull;
  }
}

// Mark the batch entries of the listed nodes (found |= 2) so the in-place merge leaves them to the
// node re-spread.  One block per listed node.
__global__ void mark_nodes_kernel(const uint32_t* __restrict__ nlist, uint32_t n_nodes, int F,
                                  const uint32_t* __restrict__ leaf, uint8_t* __restrict__ found,
                                  const uint32_t* __restrict__ dm) {
  const uint32_t m = *dm;
  for (uint32_t k = blockIdx.x; k < n_nodes; k += gridDim.x) {
    const uint32_t node = nlist[2 * k], i0 = nlist[2 * k + 1];
    for (uint32_t j = i0 + threadIdx.x;; j += blockDim.x) {
      if (j >= m || leaf[j] / (uint32_t)F != node) break;
      found[j] |= 2u;
    }
  }
}

// Re-spread one last-level node in place (one 64-lane block per listed node): its leaves' keys with
// the batch's values applied and its new keys merged in, spread evenly over the same leaves (leaf s
// gets merged keys [s K / c, (s + 1) K / c), at least one and at most 8 each), then the node's
// separators rewritten as the leaves' minima (key[s] = min of leaf s + 1) and its index granule
// (idx[g] = key[8 g + 7]; the last index slot, the node's prefix entry, is kept).  The node's
// smallest key does not change (new keys are >= the separator that leads to the node, which is that
// key), so the levels above stay valid.  Bounded cost: at most F leaves and one node per overflow.
template <int F>
__global__ __launch_bounds__(64) void node_respread_kernel(Leaf* __restrict__ leaves, uint64_t* __restrict__ nodes,
                                                           uint32_t n_leaves, const uint32_t* __restrict__ nlist,
                                                           uint32_t n_nodes, const uint32_t* __restrict__ leaf,
                                                           const uint32_t* __restrict__ slot,
                                                           const uint8_t* __restrict__ found,
                                                           const uint64_t* __restrict__ uk,
                                                           const uint64_t* __restrict__ uv,
                                                           const uint32_t* __restrict__ dm) {
  constexpr int CAP = LEAF_KEYS * F;
  constexpr int IS = idx_slots(F);
  constexpr int NS = node_slots(F);
  __shared__ uint64_t ek[CAP], ev[CAP];  // the node's keys in order (values updated), then merged
  __shared__ uint64_t nk[CAP], nv[CAP];  // its new keys in order
  __shared__ uint64_t mk[CAP], mv[CAP];
  __shared__ uint32_t off[F + 1];
  const int lane = threadIdx.x;
  const uint32_t m = *dm;
  for (uint32_t k = blockIdx.x; k < n_nodes; k += gridDim.x) {
    const uint32_t node = nlist[2 * k], i0 = nlist[2 * k + 1];
    const uint32_t x0 = node * (uint32_t)F;
    const uint32_t c = (x0 + F < n_leaves ? x0 + F : n_leaves) - x0;
    // leaf offsets in the node's key list: counts, then a wave scan (c <= F <= 128: two per lane)
    uint32_t c0 = 0, c1 = 0;
    if ((uint32_t)lane < c) c0 = (uint32_t)leaf_count(leaves[x0 + lane]);
    if ((uint32_t)lane + 64 < c) c1 = (uint32_t)leaf_count(leaves[x0 + 64 + lane]);
    const uint32_t s0 = wave_inclusive_scan(c0);
    const uint32_t t0 = (uint32_t)__shfl((int)s0, 63);
    const uint32_t s1 = wave_inclusive_scan(c1) + t0;
    if ((uint32_t)lane < c) off[lane] = s0 - c0;
    if ((uint32_t)lane + 64 < c) off[64 + lane] = s1 - c1;
    const uint32_t ke = (uint32_t)__shfl((int)s1, 63);  // existing keys
    if (lane == 0) off[c] = ke;
    __syncthreads();
    for (uint32_t u = lane; u < c * LEAF_KEYS; u += 64) {
      const uint32_t s = u / LEAF_KEYS, q = u % LEAF_KEYS;
      if (q < off[s + 1] - off[s]) {
        ek[off[s] + q] = leaves[x0 + s].key[q];
        ev[off[s] + q] = leaves[x0 + s].val[q];
      }
    }
    __syncthreads();
    // the batch entries of this node: values of existing keys, and the new keys compacted in order
    uint32_t kn = 0;
    for (uint32_t j0 = i0;; j0 += 64) {  // uniform: the node's entries are contiguous from i0
      const uint32_t j = j0 + lane;
      const bool in = j < m && leaf[j] / (uint32_t)F == node;
      const uint8_t f = in ? (found[j] & 1u) : 0u;
      if (in && f) ev[off[leaf[j] - x0] + (slot[j] & 255u)] = uv[j];
      const uint32_t isnew = in && !f ? 1u : 0u;
      const uint32_t inc = wave_inclusive_scan(isnew);
      if (isnew) {
        nk[kn + inc - 1] = uk[j];
        nv[kn + inc - 1] = uv[j];
      }
      kn += (uint32_t)__shfl((int)inc, 63);
      if (!__any(in) || j0 + 64 >= m) break;
    }
    __syncthreads();
    // merge: an element's place = its index + how many of the other list are smaller (keys distinct)
    const uint32_t K = ke + kn;
    for (uint32_t a = lane; a < ke; a += 64) {
      uint32_t lo = 0, hi = kn;
      while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (nk[mid] < ek[a]) lo = mid + 1; else hi = mid;
      }
      mk[a + lo] = ek[a];
      mv[a + lo] = ev[a];
    }
    for (uint32_t b = lane; b < kn; b += 64) {
      uint32_t lo = 0, hi = ke;
      while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (ek[mid] < nk[b]) lo = mid + 1; else hi = mid;
      }
      mk[b + lo] = nk[b];
      mv[b + lo] = nv[b];
    }
    __syncthreads();
    // leaves: leaf s = merged [s K / c, (s + 1) K / c), padded
    for (uint32_t u = lane; u < c * 2 * LEAF_KEYS; u += 64) {
      const uint32_t s = u / (2 * LEAF_KEYS), q = u % (2 * LEAF_KEYS);
      const uint32_t lo = s * K / c, hi = (s + 1) * K / c;
      const uint32_t p = lo + (q % LEAF_KEYS);
      Leaf* L = leaves + x0 + s;
      if (q < LEAF_KEYS)
        L->key[q] = p < hi ? mk[p] : KEY_MAX;
      else
        L->val[q - LEAF_KEYS] = p < hi ? mv[p] : 0ull;
    }
    // the node: separators, then the index slots below the last
    uint64_t* nd = nodes + (size_t)node * NS;
    for (uint32_t s = lane; s < (uint32_t)F; s += 64)
      nd[IS + s] = s + 1 < c ? mk[(s + 1) * K / c] : KEY_MAX;
    for (uint32_t g = lane; g + 1 < (uint32_t)IS; g += 64) {
      const uint32_t ks = 8 * g + 7;
      nd[g] = (g < (uint32_t)(F / 8) && ks + 1 < c) ? mk[(ks + 1) * K / c] : KEY_MAX;
    }
    __syncthreads();  // the LDS lists are reused by the next node
  }
}

__global__ void apply_runs_kernel(Leaf* __restrict__ leaves, const uint32_t* __restrict__ leaf,
                                  const uint32_t* __restrict__ slot, const uint8_t* __restrict__ found,
                                  const uint64_t* __restrict__ uk, const uint64_t* __restrict__ uv, size_t n_max,
                                  const uint32_t* __restrict__ dm) {
  const uint32_t m = dm ? *dm : (uint32_t)n_max;
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < m; i += stride) {
    if (!run_head(leaf, i) || (found[i] & 2u)) continue;  // marked: the node re-spread handles it
    const uint32_t L = leaf[i];
    uint32_t ins = 0;
    for (uint32_t j = i; j < m && leaf[j] == L; ++j) {
      if (found[j])
        leaves[L].val[slot[j] & 255u] = uv[j];
      else
        ++ins;
    }
    if (!ins) continue;
    const LeafRegs l = load_leaf(leaves + L);  // this thread's value writes above are visible to its own load
    LeafRegs o;
#pragma unroll
    for (int s = 0; s < LEAF_KEYS; ++s) {
      o.key[s] = KEY_MAX;
      o.val[s] = 0ull;
    }
    // the plan guarantees at most LEAF_KEYS merged keys
    merge_leaf(l, ins, i, uk, uv, found, [&](int idx, uint64_t k, uint64_t v) {
      put(o.key, idx, k);  // idx >= LEAF_KEYS matches no slot
      put(o.val, idx, v);
    });
    store_leaf(leaves + L, o);
  }
}

// Staging of an upsert batch: keys and values copied, and *flag (mapped pinned memory, may be null) set
// if a key is the reserved one.  One launch and no reduction: the flag is only ever written by a bad key.
// (Two copies, a memset, a validation that ended in 4096 atomics on one word and a copy of that word
// took 70 us for 2^20 pairs, 48 of them in the validation.)
constexpr int kStageUnroll = 4;
__global__ __launch_bounds__(256) void stage_pairs_kernel(const uint64_t* __restrict__ k, const uint64_t* __restrict__ v,
                                                          uint64_t* __restrict__ dk, uint64_t* __restrict__ dv,
                                                          size_t n, uint32_t* __restrict__ flag) {
  const size_t stride = (size_t)gridDim.x * 256;
  bool bad = false;
  for (size_t b = (size_t)blockIdx.x * 256 + threadIdx.x; b < n; b += kStageUnroll * stride) {
    uint64_t x[kStageUnroll], y[kStageUnroll];
#pragma unroll
    for (int u = 0; u < kStageUnroll; ++u) {
      const size_t i = b + u * stride;
      x[u] = i < n ? k[i] : 0ull;
      y[u] = i < n ? v[i] : 0ull;
    }
#pragma unroll
    for (int u = 0; u < kStageUnroll; ++u) {
      const size_t i = b + u * stride;
      if (i < n) {
        dk[i] = x[u];
        dv[i] = y[u];
        bad |= x[u] == KEY_MAX;
      }
    }
  }
  if (bad && flag) *flag = 1u;
}

}  // namespace

hipError_t stage_pairs(const uint64_t* k, const uint64_t* v, uint64_t* dk, uint64_t* dv, size_t n, uint32_t* flag,
                       hipStream_t s) {
  if (!n) return hipSuccess;
  ProfScope prof("update", s);
  size_t nb = (n + 256 * kStageUnroll - 1) / (256 * kStageUnroll);
  if (nb > 2048) nb = 2048;
  hipLaunchKernelGGL(stage_pairs_kernel, dim3((unsigned)nb), dim3(256), 0, s, k, v, dk, dv, n, flag);
  return hipGetLastError();
}

hipError_t small_sort_locate(const TreeView& tv, const uint64_t* pk, const uint64_t* pv, uint32_t n, uint64_t* sk,
                             uint32_t* si, uint64_t* uk, uint64_t* uv, uint32_t* leaf, uint32_t* slot, uint8_t* found,
                             uint32_t* summary, uint32_t* dm, hipStream_t s) {
  if (n == 0 || n > kSmallUpdate) return hipErrorInvalidValue;
  ProfScope prof("update", s);
  hipLaunchKernelGGL(rank_keys_kernel, dim3((n + kRankKeys - 1) / kRankKeys), dim3(kRankThreads), 0, s, pk, n, sk, si,
                     summary);
  const dim3 grid((n + 31) / 32);
  switch (tv.fanout) {
    case 32:
      hipLaunchKernelGGL(dedupe_locate_kernel<32>, grid, dim3(256), 0, s, tv, sk, si, pv, n, uk, uv, leaf, slot, found, dm);
      break;
    case 64:
      hipLaunchKernelGGL(dedupe_locate_kernel<64>, grid, dim3(256), 0, s, tv, sk, si, pv, n, uk, uv, leaf, slot, found, dm);
      break;
    case 128:
      hipLaunchKernelGGL(dedupe_locate_kernel<128>, grid, dim3(256), 0, s, tv, sk, si, pv, n, uk, uv, leaf, slot, found,
                         dm);
      break;
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t plan_runs(const Leaf* leaves, uint32_t n_leaves, int F, const uint32_t* leaf, const uint32_t* slot,
                     const uint8_t* found, const uint64_t* uk, size_t n, const uint32_t* dm, uint32_t* summary,
                     uint32_t* nlist, uint32_t* host, hipStream_t s) {
  if (!n) return hipSuccess;
  ProfScope prof("update", s);
  // Few blocks, each ends in an atomic on one word (~10 ns, one after the other): 2^20 entries take 22 us with
  // 1024 blocks of 256 threads, 16 with 512 of 512, 12 with 256 of 1024; 2^16 7.1 with 256 of 256, 5.4 with 64 of
  // 1024.  Small batches are spread (4001: 4.2 with 16 blocks for 4.6 with 4).
  const int threads = n >= (1u << 15) ? 1024 : 256;
  hipLaunchKernelGGL(plan_runs_kernel, dim3(std::min(grid_for(n, threads), kPlanBlocks)), dim3(threads), 0, s, leaves,
                     n_leaves, F, leaf, slot, found, uk, n, dm, summary, nlist, host);
  return hipGetLastError();
}

hipError_t mark_nodes(const uint32_t* nlist, uint32_t n_nodes, int F, const uint32_t* leaf, uint8_t* found,
                      const uint32_t* dm, hipStream_t s) {
  if (!n_nodes) return hipSuccess;
  ProfScope prof("update", s);
  const unsigned g = n_nodes < 4096 ? n_nodes : 4096;
  hipLaunchKernelGGL(mark_nodes_kernel, dim3(g), dim3(64), 0, s, nlist, n_nodes, F, leaf, found, dm);
  return hipGetLastError();
}

hipError_t node_respread(Leaf* leaves, uint64_t* last_level, uint32_t n_leaves, int F, const uint32_t* nlist,
                         uint32_t n_nodes, const uint32_t* leaf, const uint32_t* slot, const uint8_t* found,
                         const uint64_t* uk, const uint64_t* uv, const uint32_t* dm, hipStream_t s) {
  if (!n_nodes) return hipSuccess;
  ProfScope prof("update", s);
  const unsigned g = n_nodes < 4096 ? n_nodes : 4096;
  switch (F) {
    case 32:
      hipLaunchKernelGGL(node_respread_kernel<32>, dim3(g), dim3(64), 0, s, leaves, last_level, n_leaves, nlist,
                         n_nodes, leaf, slot, found, uk, uv, dm);
      break;
    case 64:
      hipLaunchKernelGGL(node_respread_kernel<64>, dim3(g), dim3(64), 0, s, leaves, last_level, n_leaves, nlist,
                         n_nodes, leaf, slot, found, uk, uv, dm);
      break;
    case 128:
      hipLaunchKernelGGL(node_respread_kernel<128>, dim3(g), dim3(64), 0, s, leaves, last_level, n_leaves, nlist,
                         n_nodes, leaf, slot, found, uk, uv, dm);
      break;
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t apply_runs(Leaf* leaves, const uint32_t* leaf, const uint32_t* slot, const uint8_t* found,
                      const uint64_t* uk, const uint64_t* uv, size_t n, const uint32_t* dm, hipStream_t s) {
  if (!n) return hipSuccess;
  ProfScope prof("update", s);
  hipLaunchKernelGGL(apply_runs_kernel, dim3(grid_for(n, 256)), dim3(256), 0, s, leaves, leaf, slot, found, uk, uv, n,
                     dm);
  return hipGetLastError();
}

hipError_t run_bounds(const uint32_t* leaf, const uint32_t* slot, const uint8_t* found, size_t m, uint32_t* first,
                      uint32_t* mask, uint32_t* end, hipStream_t s) {
  if (!m) return hipSuccess;
  ProfScope prof("update", s);
  const dim3 grid(grid_for(m, 256));
  hipLaunchKernelGGL(run_heads_kernel, grid, dim3(256), 0, s, leaf, (uint32_t)m, first, mask);
  hipLaunchKernelGGL(run_ends_kernel, grid, dim3(256), 0, s, leaf, slot, found, (uint32_t)m, first, mask, end);
  return hipGetLastError();
}

hipError_t new_leaf_counts(const uint32_t* first, const uint32_t* mask, const uint32_t* end, const uint32_t* slot,
                           size_t n_leaves, int fill, uint32_t* ins, uint32_t* cnt, hipStream_t s) {
  ProfScope prof("update", s);
  hipLaunchKernelGGL(new_counts_kernel, dim3(grid_for(n_leaves, 256)), dim3(256), 0, s, first, mask, end, slot,
                     n_leaves, fill, ins, cnt);
  return hipGetLastError();
}

hipError_t relayout_copy(const Leaf* old_leaves, size_t lo, size_t hi, const uint32_t* first, const uint32_t* new_start,
                         Leaf* new_leaves, uint64_t* new_mins, hipStream_t s) {
  if (hi <= lo) return hipSuccess;
  ProfScope prof("update", s);
  // a few blocks per CU: the copy streams at full rate and searches on other streams still get CUs
  const size_t pieces = (hi - lo) * (sizeof(Leaf) / 16);
  size_t nb = (pieces + 255) / 256;
  const size_t cap = (size_t)launch_cfg().num_cus * 4;
  if (nb > cap) nb = cap;
  hipLaunchKernelGGL(relayout_copy_kernel, dim3((unsigned)nb), dim3(256), 0, s, old_leaves, lo, hi, first, new_start,
                     new_leaves, new_mins);
  return hipGetLastError();
}

hipError_t relayout_touched(const Leaf* old_leaves, const uint32_t* ins, const uint32_t* first, const uint32_t* mask,
                            const uint32_t* bleaf, const uint32_t* bslot, const uint64_t* bkeys, const uint64_t* bvals,
                            const uint8_t* found, size_t m, const uint32_t* new_start, int fill, Leaf* new_leaves,
                            uint64_t* new_mins, hipStream_t s) {
  if (!m) return hipSuccess;
  ProfScope prof("update", s);
  hipLaunchKernelGGL(relayout_touched_kernel, dim3(grid_for(m, 256)), dim3(256), 0, s, old_leaves, ins, first, mask,
                     bleaf, bslot, bkeys, bvals, found, (uint32_t)m, new_start, fill, new_leaves, new_mins);
  return hipGetLastError();
}

}  // namespace hm

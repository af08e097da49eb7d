// Internal declarations shared by the HIP translation units of libharmonia_amd.
//
// Layout (all device memory, built on the device):
//   inner   : n_inner nodes in breadth-first order, node_slots(F) u64 each.
//             slots [0, IS)      index granule: idx[j] = key[8j+7] for j < F/8, else KEY_MAX
//             slots [IS, IS+F)   separators key[0..F-2] ascending, KEY_MAX padding; key[F-1] = KEY_MAX
//   prefix  : n_inner u32, prefix[g] = BFS index of the first child of node g
//             (= 1 + exclusive scan of child counts, H/regular_bpt/traversal.cpp:40,58).
//             BFS indices >= n_inner name leaves: leaf = index - n_inner.
//   leaves  : 128-byte records {key[8], val[8]}, keys ascending then KEY_MAX padding.
// On the device the last index slot, idx[IS-1] (KEY_MAX in the layout above: it would be
// key[F-1], or an unused slot), holds prefix[node] instead, so a descent step reads the next
// node's base with the index granule rather than as a separate load; rank computations treat that
// slot as KEY_MAX, and hm_tree_export restores KEY_MAX.
// Child choice is upper_bound (number of separators <= target), leaf match is exact equality
// (H/regular_bpt/prefix-sort.cu:147-173, 202-228; H/regular_bpt/regular_bpt.cpp:346-393).
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>
#include <cstddef>

namespace hm {

constexpr uint64_t KEY_MAX = ~0ull;
constexpr int LEAF_KEYS = 8;
constexpr int MAX_LEVELS = 16;

struct __attribute__((aligned(128))) Leaf {
  uint64_t key[8];
  uint64_t val[8];
};
static_assert(sizeof(Leaf) == 128, "leaf record must be 128 bytes");

__host__ __device__ constexpr int idx_slots(int F) { return F / 8 < 8 ? 8 : F / 8; }
__host__ __device__ constexpr int node_slots(int F) { return idx_slots(F) + F; }

// Everything a search kernel needs, passed by value.
struct TreeView {
  const uint64_t* inner;
  const uint32_t* prefix;
  const Leaf* leaves;
  uint32_t n_inner;
  uint32_t n_leaves;
  int32_t height;  // inner levels, >= 1
  int32_t fanout;
  uint32_t level_start[MAX_LEVELS + 1];
  // Host side: one past the highest bit in which the tree's keys differ (64 for fewer than two keys).
  // Every key agrees with the others above it, so a PSA window that ends there orders queries in the
  // key range as finely as its width allows.
  int32_t psa_top;
  uint64_t any_key;  // a key of the tree: its bits from psa_top on are every key's
};

// ---- launch helpers (host) -------------------------------------------------------------
struct LaunchCfg {
  int num_cus = 256;
  int max_lds = 160 * 1024;
};
const LaunchCfg& launch_cfg();

// Stage timing (HIP events on the launch stream); no-ops unless profiling is enabled.
struct ProfScope {
  ProfScope(const char* stage, hipStream_t s);
  ~ProfScope();
  int slot;
  hipStream_t stream;
};
// While one is alive, ProfScope records nothing on this thread (the allocation-free entry point:
// profiling events come from hipEventCreate).
struct ProfMute {
  ProfMute();
  ~ProfMute();
};

// ---- scan (hm_scan.hip) ----------------------------------------------------------------
// Exclusive scan of n u32 / u64 values; out may alias in.  tmp must hold scan_tmp_bytes(n).
size_t scan_tmp_bytes(size_t n);
hipError_t exclusive_scan_u32(const uint32_t* in, uint32_t* out, size_t n, uint32_t init, void* tmp,
                              hipStream_t s);
hipError_t exclusive_scan_u64(const uint64_t* in, uint64_t* out, size_t n, uint64_t init, void* tmp,
                              hipStream_t s);
// u32 input widened into a u64 exclusive scan (range offsets).
hipError_t exclusive_scan_u32_to_u64(const uint32_t* in, uint64_t* out, size_t n, void* tmp, hipStream_t s);

// ---- radix sort (hm_sort.hip) ----------------------------------------------------------
// Stable LSD radix sort of u64 keys with a payload over bits [begin_bit, end_bit).
// Ping-pong between (k0,v0) and (k1,v1); returns which buffer (0/1) holds the result in *which.
size_t radix_tmp_bytes(size_t n);
// payload = position 0..n-1 generated on the first pass (vals_in unused)
hipError_t radix_sort_pos(const uint64_t* keys_in, size_t n, int begin_bit, int end_bit, uint64_t* k0, uint32_t* v0,
                          uint64_t* k1, uint32_t* v1, void* tmp, hipStream_t s, int* which,
                          const uint32_t* dn = nullptr);
hipError_t radix_sort_u64pay(const uint64_t* keys_in, const uint64_t* vals_in, size_t n, int begin_bit, int end_bit,
                             uint64_t* k0, uint64_t* v0, uint64_t* k1, uint64_t* v1, void* tmp, hipStream_t s,
                             int* which);
// Keys-only stable LSD sort over bits [begin_bit, end_bit) that records how to undo it: per pass,
// the per-digit scanned (digit, tile) offsets with the digit totals, and each element's index in its
// tile's digit-ordered staging (16 bits).  `replay` must hold replay_bytes(n, end_bit - begin_bit).
size_t replay_bytes(size_t n, int bits);
hipError_t radix_sort_keys_replay(const uint64_t* keys_in, size_t n, int begin_bit, int end_bit, uint64_t* k0,
                                  uint64_t* k1, void* replay, hipStream_t s, int* which,
                                  const uint32_t* dn = nullptr);
// Route per-element results (vals, found) of the sorted order back to input order by running the
// recorded passes backwards: each pass gathers its tile's digit runs (coalesced) into LDS and writes
// the tile in its input order.  (v_tmp, f_tmp) hold n entries; (vals, found) are clobbered when
// there are three or more passes.
hipError_t unsort_results(uint64_t* vals, uint8_t* found, size_t n, int bits, const void* replay, uint64_t* v_tmp,
                          uint8_t* f_tmp, uint64_t* out_vals, uint8_t* out_found, hipStream_t s,
                          const uint32_t* dn = nullptr);

// ---- partition (hm_part.hip) -----------------------------------------------------------
// One pass that splits a batch by the key bits [top - b, top), b = partition_bits(n), into buckets of at
// most kPartBucket queries on average (more once b is kPartMaxBits), in no particular order inside a
// bucket, and records in rec (partition_bytes(n)) how to undo it.  n sizes the launches; dn (device) may
// hold a smaller count.
constexpr int kPartMinBits = 8, kPartMaxBits = 11, kPartBucket = 4096;
int partition_bits(size_t n);
size_t partition_bytes(size_t n);
// Results on their way back: the value kMissMark means not found, so the found flags need not travel.  Unless
// a key that was found has that very value: then *any (zeroed by the partition) and part[i / kClashPart] of its
// place i are set, and there the flags tell.
struct Clash {
  uint32_t* any = nullptr;
  uint8_t* part = nullptr;  // n / kClashPart + 2
};
constexpr uint32_t kClashPart = 2048;
constexpr uint64_t kMissMark = 0xB5D19F6E03C7A28Dull;  // any value: rarer among stored ones than 0
hipError_t partition_keys(const uint64_t* q, size_t n, int top, uint64_t* out, void* rec, const Clash& clash,
                          hipStream_t s, const uint32_t* dn);
hipError_t unpartition_results(const uint64_t* vals, const uint8_t* found, size_t n, const void* rec,
                               const Clash& clash, uint64_t* out_vals, uint8_t* out_found, hipStream_t s,
                               const uint32_t* dn);

// (key, value) pairs into buckets by the key bits [top - b, top), b = pair_bits(n) (0: too many pairs for
// buckets of kPairBucket on average).  *totals = the 2^b bucket sizes (device).  A bucket above kBucketSortMax
// sets `flag` in *flags, and the pairs are then not moved.  tmp: partition_pairs_bytes(n).
constexpr uint32_t kBucketSortMax = 5120;
constexpr int kPairBucket = 4608;  // 5120 is seven standard deviations above it for uniform keys
int pair_bits(size_t n);
size_t partition_pairs_bytes(size_t n);
hipError_t partition_pairs(const uint64_t* keys, const uint64_t* vals, size_t n, int top, uint64_t* kout,
                           uint64_t* vout, void* tmp, uint32_t* flags, uint32_t flag, const uint32_t** totals,
                           hipStream_t s);

// ---- build (hm_build.hip) --------------------------------------------------------------
// flags |= 1 if a key is KEY_MAX, |= 2 if keys are not strictly ascending; edge[0], edge[1] = the first and
// last key.
hipError_t validate_sorted(const uint64_t* keys, size_t n, uint32_t* d_flags, uint64_t* edge, hipStream_t s);
// ornor[0] |= the or of the keys, ornor[1] |= the or of their complements (to skip radix passes whose digit
// is constant).
hipError_t key_bit_summary(const uint64_t* keys, size_t n, uint64_t* ornor, hipStream_t s);
// mins[leaf] = the leaf's smallest key (KEY_MAX for the one leaf of an empty tree).
hipError_t fill_leaves(const uint64_t* keys, const uint64_t* vals, size_t n, int fill, Leaf* leaves, size_t n_leaves,
                       uint64_t* mins,
                       hipStream_t s);
// Leaf minimum keys (KEY_MAX for an empty leaf) -> child_min.
hipError_t leaf_min_keys(const Leaf* leaves, size_t n_leaves, uint64_t* child_min, hipStream_t s);
// One inner level: m nodes over m_child children whose minimum keys are child_min.
hipError_t build_level(const uint64_t* child_min, size_t m_child, int F, uint64_t* nodes, uint64_t* node_min,
                       uint32_t* nchild, size_t m, hipStream_t s);
// inner[node][IS-1] = prefix[node] for every node (after the prefix scan of a build or rebuild).
hipError_t fold_prefix(uint64_t* inner, const uint32_t* prefix, size_t n_inner, int F, hipStream_t s);

// ---- search (hm_search.hip) ------------------------------------------------------------
// Query segments: segment j holds n queries at src (device memory) whose results go to slots
// [dst, dst + n) of the output; the segments are sorted by dst and tile [0, total).  The list may live
// in mapped pinned host memory (the batcher writes it there before each graph replay).
// gran_first[g] = the first segment that reaches slot g * kSegGranule (a search block finds the
// segments of its chunk with one lookup).
struct QuerySeg {
  const uint64_t* src;
  uint64_t dst;
  uint64_t n;
};
struct QuerySegList {
  const QuerySeg* items;
  uint64_t n_items;
  uint64_t total;  // sum of n
  const uint32_t* gran_first;
};
// Queries per segment: the batcher cuts batches into pieces of at most this many.
constexpr uint64_t kSegPiece = 1u << 13;
constexpr int kSegGranuleLog2 = 12;

struct SearchLaunch {
  int group = 4;        // lanes per query
  int lds_levels = 2;   // levels staged in LDS
  int blocks_per_cu = 8;
  int queries_per_group = 2;  // independent descents interleaved per group
  bool sorted = false;        // queries are PSA-sorted: waves share node reads (group 1, or group 2 x 4)
  bool window = false;        // with sorted, OUT_DIRECT: the leaf-window kernel (dense batches)
  bool named = false;         // the caller named the shape, or one descent per query: no other kernel's place
  int window_blocks_per_cu = 2;
  // unsorted OUT_DIRECT searches with 1..8 lanes per query: read the queries from these segments
  // (blocks take whole segments) instead of the packed array
  const QuerySegList* segs = nullptr;
};
// Leaves a wave's LDS ring holds in the leaf-window search (64 B of keys each).
constexpr int kWindowLeaves = 256;
// Where a search writes result i of its (possibly PSA-sorted) query array:
enum SearchOut {
  OUT_DIRECT = 0,   // out_vals[i], out_found[i]
  OUT_SCATTER = 1,  // out_vals[pos[i]], out_found[pos[i]]
};
// n sizes the grid; with dn != nullptr the kernel reads the actual count (<= n) from device memory.
hipError_t launch_search(const TreeView& tv, const SearchLaunch& sl, const uint64_t* q, const uint32_t* pos,
                         uint64_t* out_vals, uint8_t* out_found, size_t n, SearchOut mode, hipStream_t s,
                         const uint32_t* dn = nullptr);
// Search of a partitioned batch (partition_keys over bits [top - bits, top)): result i of query q[i].  Keys that
// are not found get the value `miss`; with a clash record the flags are written only where it says so.
hipError_t launch_search_chunks(const TreeView& tv, const uint64_t* q, uint64_t* out_vals, uint8_t* out_found, size_t n,
                                int top, int bits, uint64_t miss, Clash clash, hipStream_t s, const uint32_t* dn);
// Bytes of LDS the top `levels` need.
size_t lds_bytes_for(const TreeView& tv, int levels);
// *p = v as a one-thread kernel (a graph-safe way to hand a count to the next replay).
hipError_t launch_set_u32(uint32_t* p, uint32_t v, hipStream_t s);
// dst[i] = src[i] for n u64 words as a kernel: either side may be device memory or mapped pinned
// host memory, so moving small buffers between host and device takes no DMA-engine copy.
hipError_t copy_words(uint64_t* dst, const uint64_t* src, size_t n, hipStream_t s);
hipError_t copy_u32s(uint32_t* dst, const uint32_t* src, size_t n, hipStream_t s);

// Comparator baselines (pointer-child trees): child[node * F + slot] = prefix[node] + slot, and a
// plain search kernel (one query per group) that follows child[] (kind 0: index + key granule,
// kind 1: granule-by-granule node scan) or, as the control, prefix[node] + slot (kind 2).
hipError_t build_child_array(const uint32_t* prefix, uint32_t n_inner, int F, uint32_t* child, hipStream_t s);
hipError_t launch_search_baseline(const TreeView& tv, const uint32_t* child, const uint64_t* q, uint64_t* out_vals,
                                  uint8_t* out_found, uint32_t n, int group, int kind, hipStream_t s);
// Locate sorted keys (update path): leaf, lower_bound slot (low byte) with the leaf's free slots (next byte)
// and found flag per key; n sizes the grid, dn (device) may hold the actual count.
hipError_t launch_locate(const TreeView& tv, int lds_levels, const uint64_t* keys, size_t n, uint32_t* leaf_out, uint32_t* slot_out,
                         uint8_t* found_out, hipStream_t s, const uint32_t* dn = nullptr);

// ---- range (hm_range.hip) --------------------------------------------------------------
// scan: the kernel computes offsets[0..n] from len itself (n <= kRangeScanMax), every wave adding up the
// lengths before its range: one launch instead of three (1027 ranges 9.5 us against 12.4 us with the scan
// launches).
constexpr size_t kRangeScanMax = 2048;
hipError_t launch_range(const TreeView& tv, const uint64_t* start, const uint64_t* hi, const uint32_t* len,
                        uint32_t cap_const, size_t n, uint64_t* offsets, bool scan, uint64_t offset_stride,
                        uint64_t* out_keys, uint64_t* out_vals, uint32_t* out_counts, uint64_t capacity, hipStream_t s);

// ---- update (hm_update.hip) ------------------------------------------------------------
// Copy a batch into the staging arrays; *flag (mapped pinned memory, may be null) = 1 if a key is KEY_MAX.
hipError_t stage_pairs(const uint64_t* k, const uint64_t* v, uint64_t* dk, uint64_t* dv, size_t n, uint32_t* flag,
                       hipStream_t s);
// Small batches (n <= kSmallUpdate): the staged pairs sorted by key (through sk, si), the last write of
// each key kept in (uk, uv), its count in *dm, and each kept key located as launch_locate does.  Zeroes
// the 8 words of summary.
constexpr uint32_t kSmallUpdate = 4096;
hipError_t small_sort_locate(const TreeView& tv, const uint64_t* pk, const uint64_t* pv, uint32_t n, uint64_t* sk,
                             uint32_t* si, uint64_t* uk, uint64_t* uv, uint32_t* leaf, uint32_t* slot, uint8_t* found,
                             uint32_t* summary, uint32_t* dm, hipStream_t s);
// Mid-size batches (kSmallUpdate < n <= kMergeUpdate, hm_merge.hip): the staged keys sorted with their
// staging indices, stable, through (k0, i0) and (k1, i1), as a merge sort: chunks of kSmallUpdate in LDS,
// then a pass per doubling.  tile_kept (dedupe_tmp_bytes) receives what compact_last needs; the 8 words of
// summary are zeroed.
constexpr uint32_t kMergeUpdate = 1u << 22;
size_t dedupe_tmp_bytes(size_t n);
hipError_t merge_sort_index(const uint64_t* pk, uint32_t n, uint64_t* k0, uint64_t* k1, uint32_t* i0, uint32_t* i1,
                            uint32_t* tile_kept, uint32_t* summary, hipStream_t s, const uint64_t** sorted_keys,
                            const uint32_t** sorted_index);
// tile_kept for keys sorted by other means.
hipError_t count_kept(const uint64_t* sorted_keys, size_t n, uint32_t* tile_kept, hipStream_t s);
// The last of each run of equal sorted keys to uk, its value vals[index[i]] (vals[i] without an index) to
// uv, the number of them to *dm.
hipError_t compact_last(const uint64_t* sorted_keys, const uint32_t* index, const uint64_t* vals, size_t n,
                        const uint32_t* tile_kept, uint64_t* uk, uint64_t* uv, uint32_t* dm, hipStream_t s);
// The buckets of partition_pairs (with its top) sorted, one block each, straight into the leaves (and mins);
// flags |= 1 if a key is KEY_MAX, |= 2 if two keys are equal; edge = the first and last key.  Nothing once
// *flags has `skip`.
hipError_t bucket_sort_fill(const uint64_t* keys, const uint64_t* vals, size_t n, int top, int bits, const uint32_t* totals,
                            int fill, Leaf* leaves, uint64_t* mins, uint32_t* flags, uint32_t skip, uint64_t* edge,
                            hipStream_t s);
// Over the m located unique keys (sorted, so each leaf's keys form one run and each last-level
// node's keys one range): counts the new keys and finds the leaves that would exceed 8 keys.  The node of
// such a leaf goes on the re-spread list (nlist: pairs of node index within the last level and first batch
// entry; summary[4] = their count) when its leaves can hold all its keys, else a full re-layout is needed.
// n sizes the grid; nlist holds 2 n entries; summary (8 words, zeroed) is the kernel's.  host (mapped pinned
// memory) receives in word 0 bit 0 if some leaf overflows and bit 1 if a re-layout is needed (the list is
// then incomplete), the new keys, summary[2..4] and, as two u64 at word 8, the smallest and largest of the
// *dm sorted unique keys (KEY_MAX, 0 if none).
hipError_t plan_runs(const Leaf* leaves, uint32_t n_leaves, int F, const uint32_t* leaf, const uint32_t* slot,
                     const uint8_t* found, const uint64_t* uk, size_t n, const uint32_t* dm, uint32_t* summary,
                     uint32_t* nlist, uint32_t* host, hipStream_t s);
// found[j] |= 2 for the batch entries of the listed nodes (the in-place merge then skips them).
hipError_t mark_nodes(const uint32_t* nlist, uint32_t n_nodes, int F, const uint32_t* leaf, uint8_t* found,
                      const uint32_t* dm, hipStream_t s);
// Re-spread each listed node in place: its keys, the batch's values and new keys merged, spread evenly
// over its own leaves, separators and index slots rewritten.  last_level = the first node of the last
// inner level.
hipError_t node_respread(Leaf* leaves, uint64_t* last_level, uint32_t n_leaves, int F, const uint32_t* nlist,
                         uint32_t n_nodes, const uint32_t* leaf, const uint32_t* slot, const uint8_t* found,
                         const uint64_t* uk, const uint64_t* uv, const uint32_t* dm, hipStream_t s);
// No leaf overflows: per run, overwrite the values of existing keys and merge the new keys in place.
hipError_t apply_runs(Leaf* leaves, const uint32_t* leaf, const uint32_t* slot, const uint8_t* found,
                      const uint64_t* uk, const uint64_t* uv, size_t n, const uint32_t* dm, hipStream_t s);
// The runs of the m located keys (sorted, so each leaf's form one): first[leaf] = its first entry h (first
// pre-filled with ~0), mask[h] = the leaf's slots that entries overwrite, end[h] = the entry after the last.
hipError_t run_bounds(const uint32_t* leaf, const uint32_t* slot, const uint8_t* found, size_t m, uint32_t* first,
                      uint32_t* mask, uint32_t* end, hipStream_t s);
// Out of place: new leaf count per old leaf (1 if it fits, else ceil(total / fill)), and the new keys (ins)
// of each leaf with a run.
hipError_t new_leaf_counts(const uint32_t* first, const uint32_t* mask, const uint32_t* end, const uint32_t* slot,
                           size_t n_leaves, int fill, uint32_t* ins, uint32_t* cnt, hipStream_t s);
// Re-layout into new_leaves (old leaves are only read); both parts also write each new leaf's
// minimum key to new_mins[new leaf].
//   relayout_copy: the old leaves in [lo, hi) that the batch does not touch, moved to new_start[i];
//   relayout_touched: the touched leaves -- batch values of existing keys applied, new keys merged,
//   overflowing leaves split evenly.
hipError_t relayout_copy(const Leaf* old_leaves, size_t lo, size_t hi, const uint32_t* first, const uint32_t* new_start,
                         Leaf* new_leaves, uint64_t* new_mins, hipStream_t s);
hipError_t relayout_touched(const Leaf* old_leaves, const uint32_t* ins, const uint32_t* first, const uint32_t* mask,
                            const uint32_t* bleaf, const uint32_t* bslot, const uint64_t* bkeys, const uint64_t* bvals,
                            const uint8_t* found, size_t m, const uint32_t* new_start, int fill, Leaf* new_leaves,
                            uint64_t* new_mins, hipStream_t s);

}  // namespace hm

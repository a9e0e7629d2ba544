// Host plan object shared by the planner (plan.cpp) and the run launchers
// (decode.hip, prefill.hip).  The plan is the work partition that
// BatchDecode/BatchPrefillWithPagedKVCacheWrapper.begin_forward builds in the
// reference (src/models/llama.py:86-147); the device copy of its work list
// lives in the caller's workspace.
#pragma once

#include <cstddef>
#include <cstdint>
#include <vector>

#include "common.h"

namespace pa {

enum PlanMode { kPlanNone = 0, kPlanDecode = 1, kPlanPrefill = 2 };

// One decode work item, processed by one head group of hg waves: pages
// [page_lo, page_hi) of sequence b for KV heads [h, h + hg), one wave per KV
// head and all its query heads.  slot < 0 means the item covers the whole
// sequence and writes the final output; otherwise wave i writes split
// partials to `slot + i` and the item takes part in merge group `merge`.
struct DecodeItem {
  int32_t b, h, page_lo, page_hi, slot, merge, pad0, pad1;
};

// Split-KV merge group: (sequence b, KV head h) owns the partial slots
// slot0 + k * stride, k in [0, nslots).
struct MergeItem {
  int32_t b, h, slot0, nslots, stride;
};

// One prefill work item: query tokens [q_lo, q_hi) of sequence b (relative to
// qo_indptr[b]) for one KV head and all its query heads.  slot 1 or 2 flags a
// paired tile (at most half a workgroup's rows), run for both KV heads of
// each head pair by the pair's even (1) or odd (2) head's workgroup; the
// planners alternate the two so that paired work lands on both XCDs of a
// pair.  slot -1: an ordinary tile.
struct PrefillItem {
  int32_t b, q_lo, q_hi, slot;
};

// One entry of a split prefill work list: piece k of the n that the KV tiles
// of query tokens [q_lo, q_hi) of sequence b are cut into (prefill_split_cost).
// n = 1: the whole tile, written to the output (`flag` as PrefillItem::slot);
// n > 1: split partials to slot `slot` of every KV head.
struct PrefillPiece {
  int32_t b, q_lo, q_hi, flag, k, n, slot, pad;
};

// A cut q-tile: its pieces hold slots [slot0, slot0 + n).
struct PrefillMerge {
  int32_t b, q_lo, q_hi, slot0, n, pad0, pad1, pad2;
};

// One item of a shared-item decode plan (decode_shared_kernel): sequence b,
// KV head h, its page pairs being chunks [chunk_lo, chunk_lo + n_chunks) of
// the workgroup's chunk sequence; the sequence's pages are kv_indices
// [ind_lo, ind_lo + npages), the last holding `last` tokens (the planned
// metadata, which the run's is, as with FlashInfer's plan and run: the
// kernel then reads no kv_indptr / kv_last_page_len before its first page
// ids).  Workgroup w's items are entries [w kSharedMaxItems, (w + 1)
// kSharedMaxItems) of the list, each carrying the workgroup's item count in
// wg_items (entries past it are padding), so the kernel's first load is its
// items themselves.
struct SharedItem {
  int32_t b, h, chunk_lo, n_chunks, ind_lo, npages, last, wg_items;
};

// Shared-item decode geometry the planner sizes its partition by: items per
// workgroup (the kernel's LDS table) and page pairs per chunk (one register
// stage).
constexpr int kSharedMaxItems = 8;
constexpr int kSharedStagePairs = 1;
// Sequences a device-planned shared-item decode ranks in every workgroup's
// prologue (B compares per sequence).
constexpr int kDevSharedMaxBatch = 512;

// Prefill geometry: 8 waves per workgroup (two per SIMD) share every K/V tile
// loaded into LDS, which halves the global-to-LDS traffic per MFMA against 4
// waves; each wave owns kPrefillRB blocks of 32 query rows.
constexpr int kPrefillWaves = 8;
constexpr int kPrefillRB = 1;
constexpr int kPrefillRows = kPrefillWaves * 32 * kPrefillRB;
// Device-planned prefill: sequences a plan may hold (the plan kernel's
// workgroup scans four per thread) and q-tiles it orders longest first
// (one rank each per thread; beyond this the tiles keep sequence order).
constexpr int kPrefillDevMaxBatch = 4096;
constexpr int kPrefillDevSortMax = 1024;
// Split-KV prefill: a step whose q-tiles x KV heads are fewer than the CUs
// cuts the KV tiles of its long q-tiles into pieces, one workgroup each, merged
// by a second launch.  The longest tile of t_max KV tiles gets P pieces (up to
// kPrefillSplitMaxPieces) of at most L = ceil(t_max / P) >=
// kPrefillSplitMinTiles, every other tile pieces of at most L, and all pieces
// run at once (at most `slots` of them per KV head, one workgroup per CU).  P
// is the one with the least estimated time, if that beats the whole tiles'.
//
// The estimate (half microseconds x slots, D = 128; at D = 64 all of it is
// about a third less): a KV tile takes 1.5 us on a mostly idle GPU and 2 us on a
// full one, and the partials and the merge launch 5 us plus 6 us on a full GPU.
// Measured on steps of 32/8 heads at D = 128, whole and cut: 1 x 8 workgroups
// of 16 KV tiles 30.7 and 12.5 us; 8 x 8 of 13 28.7 and 24.8 us, of 133 200
// and 85 us; 16 x 8 of 17 38.5 and 41.7 us (kept whole), of 24 45.7 and 44.7 us,
// of 141 212 and 157 us.  The same estimate serves the other types, where cutting
// gains about as much at the same tile counts: e4m3 pools 8 x 8 of 17 40.0 and 29.1
// us, 16 x 8 of 33 71.2 and 60.5 us; 32/4 heads at D = 64 16 x 4 of 17 24.4 and
// 19.6 us, 32 x 4 of 33 43.1 and 38.0 us, e4m3 55.2 and 41.6 us; 8/1 heads at D = 128
// e4m3 32 x 1 of 17 39.4 and 23.7 us.  Of 680 steps of all these heads and types, of
// 1 to 256 tiles over 64 to 23000 tokens, the rule made one slower by more than 0.3
// us (73 tiles of 8/1 heads over 95 tokens, fp16: 25.3 and 26.5 us).
constexpr int kPrefillSplitMaxPieces = 128;
constexpr int kPrefillSplitMinTiles = 3;
constexpr int kPrefillKvTile = 64;
inline __host__ __device__ int64_t prefill_split_cost(int len, int64_t pieces, int64_t slots) {
  return (3 * slots + pieces) * len + 10 * slots + 12 * pieces;
}
inline __host__ __device__ bool prefill_split_pays(int t_max, int len, int64_t cost,
                                                   int64_t slots) {
  return t_max - len >= 4 && cost < 3 * slots * t_max;
}

// Workspace of a prefill plan that may cut tiles, from the workspace start: the
// `tiles` whole tiles, the cut tiles' count, `entries` pieces and the merge list
// of at most `slots` pieces per KV head.
struct PrefillSplitLayout {
  size_t off_items, off_count, off_pieces, off_merges, end;
};

// Workspace layout: [0, kWsHeader) is reserved for the caller's device flags
// (the Python shim keeps the append error counter at offset 0).
constexpr size_t kWsHeader = 256;
constexpr size_t kWsAlign = 256;

inline size_t ws_align(size_t x) { return (x + kWsAlign - 1) & ~(kWsAlign - 1); }

inline PrefillSplitLayout prefill_split_layout(int64_t tiles, int64_t entries, int64_t slots) {
  PrefillSplitLayout l;
  l.off_items = kWsHeader;
  l.off_count = ws_align(l.off_items + sizeof(PrefillItem) * (size_t)tiles);
  l.off_pieces = l.off_count + kWsAlign;
  l.off_merges = ws_align(l.off_pieces + sizeof(PrefillPiece) * (size_t)entries);
  l.end = ws_align(l.off_merges + sizeof(PrefillMerge) * (size_t)(slots / 2 + 1));
  return l;
}

// A run's split partials: outputs of `rows` rows of d values, then from *off_lse
// their log-sum-exps.  Returns the bytes of both.
inline size_t partial_bytes(int64_t rows, int d, size_t* off_lse) {
  *off_lse = ws_align(sizeof(float) * (size_t)rows * d);
  return ws_align(*off_lse + sizeof(float) * (size_t)rows);
}

}  // namespace pa

struct pagedattn_plan {
  int mode = pa::kPlanNone;
  int batch_size = 0, hq = 0, hkv = 0, d = 0, page_size = 0;
  // n_items = head groups (decode) or work items (prefill)
  int n_items = 0, n_merge = 0, n_slots = 0, split_pages = 0;
  // decode, split: most pieces any (sequence, head group) was cut in
  int max_pieces = 0;
  // decode: log2 of the waves (KV heads) per head group
  int hg_shift = 0;
  // decode: the partition is made on the device at run time from kv_indptr
  // (n_items = number of shares); no work list in the workspace.
  // prefill: the q-tile list is built on the device at run time from
  // qo_indptr (n_items = its capacity)
  bool implicit = false;
  // decode, implicit: page-equivalents charged per (sequence, head group)
  // segment by the device-side split
  int item_cost = 0;
  // decode: whole (sequence, KV head) items shared by the waves of one
  // workgroup per CU (n_items = workgroups; no split partials, no merge)
  bool shared = false;
  // decode, shared: fixed chunk assignment (output bits independent of timing)
  bool deterministic = false;
  // decode, implicit and shared: the items were dealt into the workspace by
  // pagedattn_decode_plan_device_update (items_dev, the host plan's layout)
  // and the runs read them there instead of dealing in their prologue.
  // prefill, implicit: pagedattn_prefill_plan_device_update built the q-tile
  // list and the runs launch no plan kernel of their own
  bool dev_table = false;
  // prefill: query tokens per tile (rows = tokens * hq/hkv)
  int q_tile = 0;
  // prefill: tiles of at most half a workgroup's rows run as KV-head pairs
  // (device plans apply it at run time; host plans flag their items)
  bool prefill_pair = false;
  int64_t total_qo = 0;
  // > 0: the plan holds two work lists, one that cuts KV ranges and a whole one
  // that writes nothing but the outputs.  A run that brings this many bytes of
  // scratch for its split partials takes the cut list, any other the whole one,
  // so runs of one plan share no memory that they write and may overlap.
  // prefill: items_dev is the whole list, pieces_dev / merge_dev the cut one
  // with n_slots slots per KV head (device plans: the plan kernel writes both).
  // decode: items_dev / merge_dev are the cut list, whole_dev the shared items
  // of n_whole workgroups.
  size_t scratch_bytes = 0;
  size_t scratch_lse = 0;  // offset of the partial log-sum-exps in the scratch
  int n_pieces = 0;
  void* pieces_dev = nullptr;
  int32_t* n_merge_dev = nullptr;  // prefill: the cut tiles' count
  int n_whole = 0;
  void* whole_dev = nullptr;
  // device pointers into the workspace
  void* items_dev = nullptr;
  const int32_t* wave_ptr_dev = nullptr;  // decode: items of head group w
  void* merge_dev = nullptr;
  float* partial_o = nullptr;
  float* partial_lse = nullptr;
  void* workspace = nullptr;
  size_t workspace_bytes = 0;
  // host staging of the work lists (kept until the next plan so the async
  // copy never reads freed memory)
  std::vector<int32_t> host;
  // statistics for the Python shim / tests
  int64_t total_pages = 0;
  int max_pages = 0;
};

// Prefill planning on the host (BatchPrefillWithPagedKVCacheWrapper.plan,
// src/models/llama.py:86-116): the q-tile work list of
// pagedattn_prefill_plan, and the fixed shapes of a device plan
// (pagedattn_prefill_plan_device), whose list prefill.hip's plan kernel
// builds at run time.  Plain host C++ (no device code), so the planner
// can also be built and driven on a machine without a GPU, under the
// address and undefined-behaviour sanitizers.
#include <algorithm>
#include <climits>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "plan_internal.h"

namespace pa {

// Paired tiles (a q-tile of at most half a workgroup's rows, run for two KV
// heads by one workgroup) are planned by default; PAGEDATTN_PREFILL_PAIR=0
// plans every tile on its own.
static bool prefill_pairing() {
  const char* env = std::getenv("PAGEDATTN_PREFILL_PAIR");
  return !(env && std::atoi(env) == 0);
}

// Split-KV prefill (plan.h) is planned by default; PAGEDATTN_PREFILL_SPLIT=0
// keeps every q-tile whole.
static bool prefill_splitting() {
  const char* env = std::getenv("PAGEDATTN_PREFILL_SPLIT");
  return !(env && std::atoi(env) == 0);
}

// Pieces per KV head: one workgroup per CU.  (At D = 64 a CU holds two, but
// they share its matrix cores: cutting for 512 workgroups ran a 4 x 512-token
// TinyLlama step over 1000-token prefixes in 47 us, uncut 35 us.)
static int64_t prefill_split_slots(int hkv) {
  int cus = device_cu_count();
  if (cus <= 0) cus = 256;
  return std::max(1, cus / hkv);
}

// KV tiles per piece of the q-tiles with `tiles` KV tiles (the rule in
// plan.h; prefill_plan_kernel applies the same one), or 0 to keep them whole.
static int prefill_piece_tiles(const std::vector<int>& tiles, int64_t slots) {
  if (tiles.empty() || (int64_t)tiles.size() > slots) return 0;
  const int t_max = *std::max_element(tiles.begin(), tiles.end());
  int best = 0;
  int64_t best_cost = 0;
  for (int p = 2; p <= kPrefillSplitMaxPieces; ++p) {
    const int len = (t_max + p - 1) / p;
    if (len < kPrefillSplitMinTiles) break;
    int64_t n = 0;
    for (int t : tiles) n += t > 0 ? (t + len - 1) / len : 1;
    if (n > slots) break;  // more pieces only ever take more slots
    const int64_t cost = prefill_split_cost(len, n, slots);
    if (best == 0 || cost < best_cost) {
      best = len;
      best_cost = cost;
    }
  }
  return best > 0 && prefill_split_pays(t_max, best, best_cost, slots) ? best : 0;
}

// Rows of split partials of `slots` pieces per KV head.
static int64_t prefill_partial_rows(int64_t slots, int hkv) {
  return slots * hkv * kPrefillRows;
}

// Whether plans may cut tiles: the caller's workspace bounds the scratch that
// their runs ask for (the same bound for host and device plans, whose outputs
// then agree bit for bit).
static bool prefill_may_cut(int64_t slots, int hkv, int d, size_t workspace_bytes) {
  size_t off_lse;
  return prefill_splitting() && slots >= 2 &&
         kWsHeader + partial_bytes(prefill_partial_rows(slots, hkv), d, &off_lse) <=
             workspace_bytes;
}

// The cut list of a plan: n_pieces entries over `slots` slots per KV head.
static void set_split(pagedattn_plan* plan, const PrefillSplitLayout& lay, int64_t n_pieces,
                      int64_t slots) {
  char* ws = static_cast<char*>(plan->workspace);
  plan->n_pieces = (int)n_pieces;
  plan->n_slots = (int)slots;
  plan->pieces_dev = ws + lay.off_pieces;
  plan->merge_dev = ws + lay.off_merges;
  plan->n_merge_dev = reinterpret_cast<int32_t*>(ws + lay.off_count);
  plan->scratch_bytes = partial_bytes(prefill_partial_rows(slots, plan->hkv), plan->d,
                                      &plan->scratch_lse);
}

}  // namespace pa

using namespace pa;

extern "C" {

int pagedattn_prefill_plan(pagedattn_plan* plan, const int32_t* qo_indptr_host,
                           const int32_t* kv_indptr_host,
                           const int32_t* kv_last_page_len_host,
                           int32_t batch_size, int32_t num_qo_heads,
                           int32_t num_kv_heads, int32_t head_dim,
                           int32_t page_size, void* workspace,
                           size_t workspace_bytes, void* stream) {
  const char* who = "prefill_plan";
  if (!plan) return set_error(PAGEDATTN_ERR_INVALID, "%s: null plan", who);
  plan->mode = kPlanNone;
  plan->scratch_bytes = 0;
  if (batch_size < 0)
    return set_error(PAGEDATTN_ERR_INVALID, "%s: batch_size %d < 0", who,
                     batch_size);
  int rc = validate_heads(who, num_qo_heads, num_kv_heads, head_dim, page_size);
  if (rc) return rc;
  if (!workspace || ((uintptr_t)workspace & (kWsAlign - 1)))
    return set_error(PAGEDATTN_ERR_INVALID,
                     "%s: workspace must be a 256-byte aligned device buffer",
                     who);
  if (batch_size > 0 && !qo_indptr_host)
    return set_error(PAGEDATTN_ERR_INVALID, "%s: null qo_indptr", who);
  std::vector<int32_t> npages, kv_len;
  rc = validate_paged_metadata(who, kv_indptr_host, kv_last_page_len_host,
                               batch_size, page_size, &npages, &kv_len);
  if (rc) return rc;
  if (batch_size > 0 && qo_indptr_host[0] < 0)
    return set_error(PAGEDATTN_ERR_INVALID, "%s: qo_indptr[0] < 0", who);
  const int g = num_qo_heads / num_kv_heads;
  const int q_tile = kPrefillRows / g;
  const bool pair = prefill_pairing() && num_kv_heads % 2 == 0;
  // the q-tile count first: the work list must fit the workspace (and the
  // launch grid) before anything is built
  int64_t n_tiles = 0;
  for (int b = 0; b < batch_size; ++b) {
    const int64_t qo = (int64_t)qo_indptr_host[b + 1] - qo_indptr_host[b];
    if (qo < 0)
      return set_error(PAGEDATTN_ERR_INVALID,
                       "%s: qo_indptr is not monotone at %d", who, b);
    n_tiles += (qo + q_tile - 1) / q_tile;
  }
  if ((int64_t)sizeof(PrefillItem) * n_tiles > (int64_t)workspace_bytes ||
      n_tiles * num_kv_heads > INT32_MAX)
    return set_error(PAGEDATTN_ERR_WORKSPACE,
                     "%s: %lld q-tiles do not fit the %zu-byte workspace", who,
                     (long long)n_tiles, workspace_bytes);
  auto finish = [&](pagedattn_plan* pl) {
    pl->batch_size = batch_size;
    pl->hq = num_qo_heads;
    pl->hkv = num_kv_heads;
    pl->d = head_dim;
    pl->page_size = page_size;
    pl->q_tile = q_tile;
    pl->total_qo =
        batch_size > 0 ? (int64_t)qo_indptr_host[batch_size] - qo_indptr_host[0] : 0;
    pl->implicit = false;
    pl->shared = false;
    pl->dev_table = false;
    pl->mode = kPlanPrefill;
  };
  std::vector<PrefillItem> items;
  std::vector<int64_t> cost;
  items.reserve((size_t)n_tiles);
  cost.reserve((size_t)n_tiles);
  for (int b = 0; b < batch_size; ++b) {
    const int qo = qo_indptr_host[b + 1] - qo_indptr_host[b];  // >= 0, checked above
    for (int lo = 0; lo < qo; lo = qo - lo > q_tile ? lo + q_tile : qo) {
      const int hi = qo - lo > q_tile ? lo + q_tile : qo;
      // slot 1: a paired tile (kernels built without pairing -- e4m3 pools,
      // D = 64 -- run it like any other)
      const int flag = pair && (int64_t)(hi - lo) * g <= kPrefillRows / 2 ? 1 : -1;
      items.push_back(PrefillItem{b, lo, hi, flag});
      // kv tokens the tile's last row can see (causal)
      cost.push_back(std::max<int64_t>(
          0, std::min<int64_t>(kv_len[b], (int64_t)kv_len[b] - qo + hi)));
    }
  }
  // most expensive tiles first
  std::vector<int> order(items.size());
  for (size_t i = 0; i < order.size(); ++i) order[i] = (int)i;
  std::stable_sort(order.begin(), order.end(),
                   [&](int a, int c) { return cost[a] > cost[c]; });
  const int64_t slots = prefill_split_slots(num_kv_heads);
  int piece_tiles = 0;
  if (prefill_may_cut(slots, num_kv_heads, head_dim, workspace_bytes) &&
      (int64_t)items.size() <= slots) {
    std::vector<int> tiles;
    for (int64_t c : cost) tiles.push_back((int)((c + kPrefillKvTile - 1) / kPrefillKvTile));
    piece_tiles = prefill_piece_tiles(tiles, slots);
  }
  std::vector<PrefillPiece> pieces;
  std::vector<PrefillMerge> merges;
  if (piece_tiles > 0)
    for (int i : order) {
      const PrefillItem& it = items[i];
      const int t = (int)((cost[i] + kPrefillKvTile - 1) / kPrefillKvTile);
      const int n = std::max(1, (t + piece_tiles - 1) / piece_tiles);
      const int at = (int)pieces.size();
      for (int k = 0; k < n; ++k)
        pieces.push_back(PrefillPiece{it.b, it.q_lo, it.q_hi, -1, k, n, n > 1 ? at + k : -1, 0});
      if (n > 1) merges.push_back(PrefillMerge{it.b, it.q_lo, it.q_hi, at, n, 0, 0, 0});
    }
  const bool cut = !merges.empty();
  const PrefillSplitLayout lay = prefill_split_layout(n_tiles, (int64_t)pieces.size(), slots);
  const size_t host_bytes =
      cut ? lay.end - kWsHeader : sizeof(PrefillItem) * items.size();
  plan->host.assign((host_bytes + 3) / 4, 0);
  char* hb = reinterpret_cast<char*>(plan->host.data());
  if (cut) {
    const int32_t n_merge = (int32_t)merges.size();
    std::memcpy(hb + (lay.off_count - kWsHeader), &n_merge, sizeof(n_merge));
    std::memcpy(hb + (lay.off_pieces - kWsHeader), pieces.data(),
                sizeof(PrefillPiece) * pieces.size());
    std::memcpy(hb + (lay.off_merges - kWsHeader), merges.data(),
                sizeof(PrefillMerge) * merges.size());
  }
  auto* dst = reinterpret_cast<PrefillItem*>(hb);
  // paired tiles alternate between the even and the odd head of each pair in
  // list order, so the two XCDs that hold a head pair's workgroups share them
  int n_paired = 0;
  for (size_t i = 0; i < order.size(); ++i) {
    dst[i] = items[order[i]];
    if (dst[i].slot > 0) dst[i].slot = 1 + (n_paired++ & 1);
  }
  plan->workspace = workspace;
  plan->workspace_bytes = workspace_bytes;
  rc = upload_plan(plan, who, host_bytes, ws_align(kWsHeader + host_bytes),
                   stream);
  if (rc) return rc;
  plan->n_items = (int)items.size();
  plan->n_merge = (int)merges.size();
  plan->n_slots = 0;
  plan->items_dev = static_cast<char*>(workspace) + kWsHeader;
  finish(plan);
  if (cut) set_split(plan, lay, (int64_t)pieces.size(), (int64_t)pieces.size());
  return PAGEDATTN_OK;
}

int pagedattn_prefill_plan_device(pagedattn_plan* plan, int32_t batch_size,
                                  int32_t num_qo_heads, int32_t num_kv_heads,
                                  int32_t head_dim, int32_t page_size, int64_t max_qo_tokens,
                                  void* workspace, size_t workspace_bytes) {
  const char* who = "prefill_plan_device";
  if (!plan) return set_error(PAGEDATTN_ERR_INVALID, "%s: null plan", who);
  plan->mode = kPlanNone;
  plan->scratch_bytes = 0;
  if (batch_size < 0 || batch_size > kPrefillDevMaxBatch)
    return set_error(PAGEDATTN_ERR_UNSUPPORTED, "%s: batch_size %d outside [0, %d]", who,
                     batch_size, kPrefillDevMaxBatch);
  if (max_qo_tokens < 0)
    return set_error(PAGEDATTN_ERR_INVALID, "%s: max_qo_tokens %lld < 0", who,
                     (long long)max_qo_tokens);
  int rc = validate_heads(who, num_qo_heads, num_kv_heads, head_dim, page_size);
  if (rc) return rc;
  if (!workspace || ((uintptr_t)workspace & (kWsAlign - 1)))
    return set_error(PAGEDATTN_ERR_INVALID,
                     "%s: workspace must be a 256-byte aligned device buffer", who);
  const int g = num_qo_heads / num_kv_heads;
  const int q_tile = kPrefillRows / g;
  // every sequence may end in a partial tile
  const int64_t cap = (max_qo_tokens + q_tile - 1) / q_tile + batch_size;
  if ((int64_t)sizeof(PrefillItem) * cap > (int64_t)workspace_bytes - (int64_t)kWsHeader ||
      cap * num_kv_heads > INT32_MAX)
    return set_error(PAGEDATTN_ERR_WORKSPACE,
                     "%s: %lld q-tiles do not fit the %zu-byte workspace", who,
                     (long long)cap, workspace_bytes);
  plan->host.clear();
  plan->workspace = workspace;
  plan->workspace_bytes = workspace_bytes;
  plan->implicit = true;
  plan->shared = false;
  plan->dev_table = false;
  plan->prefill_pair = prefill_pairing() && num_kv_heads % 2 == 0;
  plan->batch_size = batch_size;
  plan->hq = num_qo_heads;
  plan->hkv = num_kv_heads;
  plan->d = head_dim;
  plan->page_size = page_size;
  plan->n_items = (int)cap;
  plan->n_merge = 0;
  plan->n_slots = 0;
  plan->q_tile = q_tile;
  plan->total_qo = max_qo_tokens;
  plan->items_dev = static_cast<char*>(workspace) + kWsHeader;
  // the plan kernel may cut tiles, on the host plan's rule (the tiles are known
  // to it only), where both lists fit
  const int64_t slots = prefill_split_slots(num_kv_heads);
  const int64_t entries = std::max(cap, slots);
  const PrefillSplitLayout lay = prefill_split_layout(cap, entries, slots);
  if (cap > 0 && prefill_may_cut(slots, num_kv_heads, head_dim, workspace_bytes) &&
      slots <= kPrefillDevSortMax && lay.end <= workspace_bytes &&
      entries * num_kv_heads <= INT32_MAX)
    set_split(plan, lay, entries, slots);
  plan->mode = kPlanPrefill;
  return PAGEDATTN_OK;
}

}  // extern "C"

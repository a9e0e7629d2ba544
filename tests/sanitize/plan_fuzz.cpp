// Drives the host planners of libpagedattn (pagedattn_decode_plan,
// pagedattn_decode_plan_device, pagedattn_prefill_plan, and the metadata
// validation they share) with randomized and malformed metadata, built with
// the address and undefined-behaviour sanitizers (Makefile next to this
// file).  The metadata is what the engine's callers build
// (src/engine/runtime/step_executor.py:98-165, 204-243) plus what a bad
// caller could pass: non-monotone or negative indptr, last_page_len outside
// [1, 16], lengths near INT32_MAX, bad head shapes, short or misaligned
// workspaces.  Every call must return a documented status with a message; a
// sanitizer report aborts the run.  The work-list upload is replaced by a copy
// into host memory (hipMemcpyAsync below), where the lists are then read back:
// every query token and page is covered once, and pieces, slots and merge
// entries agree and stay inside the workspace and the runs' scratch.
//
//   plan_fuzz <iterations> <seed>
#include <algorithm>
#include <cinttypes>
#include <climits>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <map>
#include <set>
#include <string>
#include <tuple>
#include <vector>

#include "pagedattn.h"
#include "plan_internal.h"

namespace {

// The workspace the planner was given: uploads must stay inside it.
char* g_ws = nullptr;
size_t g_ws_bytes = 0;
bool g_upload_inside = true;

}  // namespace

extern "C" hipError_t hipMemcpyAsync(void* dst, const void* src, size_t bytes, hipMemcpyKind,
                                     hipStream_t) {
  char* d = static_cast<char*>(dst);
  if (!g_ws || d < g_ws || bytes > g_ws_bytes || d + bytes > g_ws + g_ws_bytes) {
    g_upload_inside = false;
    return hipErrorInvalidValue;
  }
  std::memcpy(dst, src, bytes);
  return hipSuccess;
}

namespace {

std::mt19937_64 rng;

int64_t uni(int64_t lo, int64_t hi) {  // inclusive
  return std::uniform_int_distribution<int64_t>(lo, hi)(rng);
}
bool coin(double p) { return std::uniform_real_distribution<double>(0, 1)(rng) < p; }

struct Meta {
  std::vector<int32_t> indptr, last, qo;
  int32_t batch = 0;
  bool valid = true;  // the metadata satisfies every documented rule
};

// kv_indptr / kv_last_page_len (and qo_indptr) of `batch` sequences; with
// probability `bad` one rule is broken.
Meta make_meta(double bad) {
  Meta m;
  // a few sequences of much the same length: what leaves CUs idle
  const bool few = coin(0.3);
  m.batch = (int32_t)(coin(0.05) ? 0 : uni(1, few ? 6 : coin(0.1) ? 1200 : 64));
  const int max_pages = coin(0.2) ? 9000 : 80;
  const int few_pages = (int)uni(1, 3000);
  m.indptr.resize(m.batch + 1);
  m.last.resize(m.batch);
  m.qo.resize(m.batch + 1);
  m.indptr[0] = coin(0.3) ? (int32_t)uni(0, 5000) : 0;
  m.qo[0] = coin(0.3) ? (int32_t)uni(0, 5000) : 0;
  for (int b = 0; b < m.batch; ++b) {
    const int np = coin(0.05) ? 0 : few ? few_pages : (int)uni(1, max_pages);
    m.indptr[b + 1] = m.indptr[b] + np;
    m.last[b] = (int32_t)uni(1, 16);
    const int kv = np > 0 ? (np - 1) * 16 + m.last[b] : 0;
    m.qo[b + 1] = m.qo[b] + (int32_t)(kv > 0 ? uni(1, std::min(kv, 600)) : uni(0, 3));
  }
  if (m.batch > 0 && coin(bad)) {
    m.valid = false;
    const int b = (int)uni(0, m.batch - 1);
    switch (uni(0, 9)) {
      case 0: m.indptr[0] = -(int32_t)uni(1, INT_MAX); break;
      case 1: m.indptr[b + 1] = m.indptr[b] - (int32_t)uni(1, 100); break;  // not monotone
      case 2: m.last[b] = (int32_t)uni(17, INT_MAX); m.indptr[b + 1] = m.indptr[b] + 1; break;
      case 3: m.last[b] = -(int32_t)uni(0, INT_MAX); m.indptr[b + 1] = m.indptr[b] + 1; break;
      case 4:  // a sequence longer than INT32_MAX tokens
        m.indptr[b + 1] = m.indptr[b] + (int32_t)uni(134217728, INT_MAX / 2);
        for (int c = b + 1; c < m.batch; ++c) m.indptr[c + 1] = m.indptr[b + 1];
        break;
      case 5: m.indptr[m.batch] = INT_MAX; break;
      case 6: m.qo[b + 1] = m.qo[b] - (int32_t)uni(1, INT_MAX / 2); break;
      case 7: m.qo[b + 1] = INT_MIN + (int32_t)uni(0, 10); break;
      case 8: m.qo[0] = -(int32_t)uni(1, 1000); break;
      default:  // a huge chunk: qo near INT32_MAX
        m.qo[b + 1] = m.qo[b] + (int32_t)uni(INT_MAX / 4, INT_MAX / 2);
        for (int c = b + 1; c < m.batch; ++c) m.qo[c + 1] = m.qo[b + 1];
        break;
    }
  }
  return m;
}

const char* kEnv[] = {"PAGEDATTN_DECODE_SHARED", "PAGEDATTN_DECODE_DETERMINISTIC",
                      "PAGEDATTN_DECODE_HEAD_GROUP", "PAGEDATTN_DECODE_ITEM_COST",
                      "PAGEDATTN_DECODE_WAVES_PER_CU", "PAGEDATTN_DECODE_SHARED_SLACK_KB",
                      "PAGEDATTN_DECODE_SHARED_SLACK_PCT",
                      "PAGEDATTN_PREFILL_PAIR", "PAGEDATTN_PREFILL_SPLIT"};

void shuffle_env() {
  for (const char* e : kEnv) {
    if (coin(0.6)) {
      unsetenv(e);
      continue;
    }
    const long v = coin(0.2) ? (long)uni(-5, 2000) : (long)uni(0, 12);
    setenv(e, std::to_string(v).c_str(), 1);
  }
}

int failures = 0;

void check(const char* what, int rc, const Meta& m, bool args_valid, int64_t iter) {
  const char* msg = pagedattn_last_error();
  const bool known = rc >= PAGEDATTN_OK && rc <= PAGEDATTN_ERR_PLAN;
  bool ok = known && (rc == PAGEDATTN_OK || (msg && msg[0]));
  // valid metadata and arguments may only fail on the workspace size
  if (ok && m.valid && args_valid && rc != PAGEDATTN_OK && rc != PAGEDATTN_ERR_WORKSPACE)
    ok = false;
  if (!g_upload_inside) ok = false;
  if (!ok) {
    ++failures;
    std::fprintf(stderr, "iteration %" PRId64 ": %s returned %d (%s) on %s metadata, batch %d\n",
                 iter, what, rc, msg ? msg : "(null)", m.valid ? "valid" : "invalid", m.batch);
  }
}

int cut_prefill = 0, both_decode = 0;  // plans of two forms seen

// n entries of T at p, inside the workspace.
template <typename T>
bool inside(const void* p, int64_t n, std::vector<T>* out) {
  const char* c = static_cast<const char*>(p);
  if (n < 0 || c < g_ws + 256 || c + n * (int64_t)sizeof(T) > g_ws + g_ws_bytes) return false;
  out->resize(n);
  if (n) std::memcpy(out->data(), c, n * sizeof(T));
  return true;
}

int kv_len(const Meta& m, int b) {
  const int np = m.indptr[b + 1] - m.indptr[b];
  return np > 0 ? (np - 1) * 16 + m.last[b] : 0;
}

// What is wrong with a host prefill plan's lists, or null.
const char* prefill_lists(const pagedattn_plan* p, const Meta& m) {
  std::vector<pa::PrefillItem> items;
  if (!inside(p->items_dev, p->n_items, &items)) return "item list outside the workspace";
  std::set<std::tuple<int, int, int>> tiles;
  std::vector<int64_t> rows(m.batch, 0);
  for (auto& i : items) {
    if (i.b < 0 || i.b >= m.batch || i.q_lo < 0 || i.q_hi <= i.q_lo ||
        i.q_hi - i.q_lo > p->q_tile || i.q_hi > m.qo[i.b + 1] - m.qo[i.b])
      return "tile outside its sequence";
    if (!tiles.insert({i.b, i.q_lo, i.q_hi}).second) return "tile twice";
    rows[i.b] += i.q_hi - i.q_lo;
  }
  int64_t end = 0;  // disjoint: equal sums of equal tiles starting at distinct q_lo
  for (int b = 0; b < m.batch; ++b) {
    if (rows[b] != m.qo[b + 1] - m.qo[b]) return "query tokens not covered once";
    end += rows[b];
  }
  if (end != p->total_qo) return "query tokens";
  if (!p->scratch_bytes) return nullptr;
  ++cut_prefill;
  std::vector<pa::PrefillPiece> pieces;
  std::vector<pa::PrefillMerge> merges;
  std::vector<int32_t> count;
  if (!inside(p->pieces_dev, p->n_pieces, &pieces) || !inside(p->merge_dev, p->n_merge, &merges) ||
      !inside(p->n_merge_dev, 1, &count))
    return "cut lists outside the workspace";
  if (count[0] != p->n_merge || p->n_merge < 1) return "merge count";
  if (p->n_pieces > p->n_slots || (int64_t)p->n_pieces * p->hkv > 256) return "pieces past the CUs";
  const size_t n_rows = (size_t)p->n_slots * p->hkv * pa::kPrefillRows;
  if (p->scratch_lse < n_rows * p->d * 4 || p->scratch_bytes < p->scratch_lse + n_rows * 4 ||
      p->scratch_bytes > g_ws_bytes)
    return "scratch size";
  std::map<int, const pa::PrefillMerge*> by_slot;
  for (auto& g : merges) by_slot[g.slot0] = &g;
  size_t at = 0, cut = 0;
  while (at < pieces.size()) {
    const auto& f = pieces[at];
    if (!tiles.erase({f.b, f.q_lo, f.q_hi})) return "piece of no tile, or tile twice";
    if (f.n < 1 || at + f.n > pieces.size()) return "piece count";
    if (f.n > 1 && f.n > (kv_len(m, f.b) + 63) / 64) return "more pieces than KV tiles";
    for (int k = 0; k < f.n; ++k) {
      const auto& x = pieces[at + k];
      if (x.b != f.b || x.q_lo != f.q_lo || x.q_hi != f.q_hi || x.n != f.n || x.k != k)
        return "pieces of a tile";
      if (f.n == 1 ? x.slot != -1 : x.slot != (int)at + k || x.slot >= p->n_slots)
        return "piece slot";
    }
    if (f.n > 1) {
      ++cut;
      const auto g = by_slot.find((int)at);
      if (g == by_slot.end() || g->second->b != f.b || g->second->q_lo != f.q_lo ||
          g->second->q_hi != f.q_hi || g->second->n != f.n)
        return "merge entry";
    }
    at += f.n;
  }
  if (!tiles.empty()) return "tile without a piece";
  return cut == merges.size() ? nullptr : "merge entries";
}

// What is wrong with the lists of a host decode plan of both forms, or null.
const char* decode_lists(const pagedattn_plan* p, const Meta& m) {
  if (!p->scratch_bytes) return nullptr;
  ++both_decode;
  const int hg = 1 << p->hg_shift, g = p->hq / p->hkv;
  std::vector<pa::SharedItem> whole;
  std::vector<int32_t> wave_ptr;
  std::vector<pa::DecodeItem> items;
  std::vector<pa::MergeItem> merges;
  if (!inside(p->whole_dev, (int64_t)p->n_whole * pa::kSharedMaxItems, &whole) ||
      !inside(p->wave_ptr_dev, p->n_items + 1, &wave_ptr) || wave_ptr[0] != 0 ||
      !inside(p->items_dev, wave_ptr.back(), &items) ||
      !inside(p->merge_dev, p->n_merge, &merges))
    return "list outside the workspace";
  if (!std::is_sorted(wave_ptr.begin(), wave_ptr.end())) return "wave_ptr";
  std::set<std::pair<int, int>> heads;
  for (auto& s : whole) {
    if (s.b < 0) continue;
    if (s.b >= m.batch || s.h < 0 || s.h >= p->hkv || s.ind_lo != m.indptr[s.b] ||
        s.npages != m.indptr[s.b + 1] - m.indptr[s.b] ||
        (s.npages > 0 && s.last != m.last[s.b]) || !heads.insert({s.b, s.h}).second)
      return "shared item";
  }
  if (heads.size() != (size_t)m.batch * p->hkv) return "shared items missing";
  const size_t n_rows = (size_t)p->n_slots * g;
  if (p->scratch_lse < n_rows * p->d * 4 || p->scratch_bytes < p->scratch_lse + n_rows * 4 ||
      p->scratch_bytes > g_ws_bytes)
    return "scratch size";
  std::map<std::pair<int, int>, int> next;       // pages covered of (b, head group)
  std::map<std::pair<int, int>, std::vector<int>> slots;
  for (auto& i : items) {
    if (i.b < 0 || i.b >= m.batch || i.h < 0 || i.h + hg > p->hkv || i.h % hg) return "item";
    int& at = next[{i.b, i.h}];
    if (i.page_lo != at || i.page_hi < i.page_lo) return "pages not covered in order";
    at = i.page_hi;
    if ((i.slot >= 0) != (i.merge >= 0) || i.slot + hg > p->n_slots || i.merge >= p->n_merge)
      return "item slot";
    slots[{i.b, i.h}].push_back(i.slot);
  }
  int most = 0;
  std::set<int> used;
  for (int b = 0; b < m.batch; ++b)
    for (int h = 0; h < p->hkv; h += hg) {
      if (next[{b, h}] != m.indptr[b + 1] - m.indptr[b]) return "pages not covered";
      const auto& s = slots[{b, h}];
      most = std::max(most, (int)s.size());
      if (s.size() == 1 && s[0] != -1) return "slot of a whole item";
      if (s.size() > 1)
        for (size_t k = 0; k < s.size(); ++k)
          if (s[k] != s[0] + (int)k * hg || s[k] < 0) return "slots of a cut item";
    }
  if (most != p->max_pieces) return "most pieces";
  for (auto& x : merges) {
    const auto& s = slots[{x.b, x.h / hg * hg}];
    if (x.nslots != (int)s.size() || x.nslots < 2 || x.stride != hg || x.slot0 != s[0] + x.h % hg)
      return "merge entry";
    for (int k = 0; k < x.nslots; ++k)
      if (!used.insert(x.slot0 + k * x.stride).second) return "slot used twice";
  }
  return (int)used.size() == p->n_slots ? nullptr : "slots without a merge";
}

void check_lists(const char* what, const char* wrong, const Meta& m, int64_t iter) {
  if (!wrong) return;
  ++failures;
  std::fprintf(stderr, "iteration %" PRId64 ": %s: %s, batch %d\n", iter, what, wrong, m.batch);
}

}  // namespace

int main(int argc, char** argv) {
  const int64_t iters = argc > 1 ? std::atoll(argv[1]) : 2000;
  rng.seed(argc > 2 ? std::strtoull(argv[2], nullptr, 10) : 1);
  // a 256-byte aligned stand-in for the device workspace, as large as the
  // engine's (128 MiB): the work-list upload is the only access
  const size_t ws_bytes = (size_t)128 << 20;
  char* ws = static_cast<char*>(std::aligned_alloc(256, ws_bytes));
  if (!ws) return 2;
  const int hq_kv[][2] = {{32, 4}, {32, 8}, {64, 8}, {8, 8}, {16, 1}, {4, 2}};
  for (int64_t it = 0; it < iters; ++it) {
    shuffle_env();
    Meta m = make_meta(0.3);
    int hq = 32, hkv = 8, d = coin(0.5) ? 64 : 128, page = 16;
    const int pick = (int)uni(0, 5);
    hq = hq_kv[pick][0];
    hkv = hq_kv[pick][1];
    bool args_valid = true;
    if (coin(0.08)) {  // an unsupported or invalid shape
      args_valid = false;
      switch (uni(0, 4)) {
        case 0: d = (int)uni(-10, 300); break;
        case 1: hq = (int)uni(-4, 70); break;
        case 2: hkv = (int)uni(-4, 70); break;
        case 3: page = (int)uni(-4, 64); break;
        default: hq = 96; hkv = 3; break;  // group size 32
      }
      if (d == 64 || d == 128) args_valid = page == 16 && hq > 0 && hkv > 0 && hq % hkv == 0 &&
                                            hq / hkv <= 16 && ((hq / hkv) & (hq / hkv - 1)) == 0;
    }
    void* w = ws;
    size_t wb = coin(0.1) ? (size_t)uni(0, 4096) : coin(0.1) ? (size_t)uni(4096, 1 << 22) : ws_bytes;
    if (coin(0.03)) {
      w = ws + 8;  // misaligned
      args_valid = false;
    }
    if (coin(0.02)) {
      w = nullptr;
      args_valid = false;
    }
    const int32_t batch = coin(0.02) ? -(int32_t)uni(1, 5) : m.batch;
    if (batch < 0) args_valid = false;
    g_ws = ws;
    g_ws_bytes = wb;
    g_upload_inside = true;
    pagedattn_plan* plan = pagedattn_plan_create();
    switch (uni(0, 2)) {
      case 0: {
        static const int splits[] = {0, 0, -1, 8, 256, 3, 1000, INT_MAX, INT_MIN};
        const int split = splits[uni(0, 8)];
        const int rc = pagedattn_decode_plan(plan, m.indptr.data(), m.last.data(), batch, hq,
                                             hkv, d, page, split, w, wb, nullptr);
        check("decode_plan", rc, m, args_valid, it);
        if (rc == PAGEDATTN_OK) check_lists("decode_plan", decode_lists(plan, m), m, it);
        break;
      }
      case 1: {
        const int rc = pagedattn_decode_plan_device(plan, batch, hq, hkv, d, page, w, wb);
        Meta any = m;
        any.valid = true;  // the device plan reads no metadata on the host
        check("decode_plan_device", rc, any, args_valid, it);
        break;
      }
      default: {
        const int rc = pagedattn_prefill_plan(plan, m.qo.data(), m.indptr.data(), m.last.data(),
                                              batch, hq, hkv, d, page, w, wb, nullptr);
        check("prefill_plan", rc, m, args_valid, it);
        if (rc == PAGEDATTN_OK) check_lists("prefill_plan", prefill_lists(plan, m), m, it);
        break;
      }
    }
    pagedattn_plan_destroy(plan);
    if (failures > 0) break;  // stop at the first finding
  }
  std::free(ws);
  if (iters >= 2000 && !failures && (!cut_prefill || !both_decode)) {
    ++failures;
    std::fprintf(stderr, "no plan of two forms was made\n");
  }
  std::printf("plan_fuzz: %" PRId64 " iterations (%d cut prefill plans, %d decode plans of both "
              "forms), %d failures\n", iters, cut_prefill, both_decode, failures);
  return failures ? 1 : 0;
}

// load_plan.cpp -- host tables of a gather or a load, checked, ordered and packed
// for one upload. Part of libdaser_kv (host code, no HIP calls).
//
// A load of host tables is bound by the host until it moves some 300 MB: in
// numpy the checks, the sort by destination, the count of distinct records and
// the grouping cost 30-60 us for 16 pages and 3.5 ms for 32,768, and each table
// was an upload of its own (15 us of host time). Here one pass each over the
// tables, into one buffer.

#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <new>
#include <vector>

#include "daser_kv.h"

namespace {

int64_t round16(int64_t v) { return (v + 15) & ~(int64_t)15; }

// Numbers the distinct values of v in the order of their first appearance:
// open addressing over twice as many places, by the multipliers of Steele, Lea
// and Flood's SplitMix64.
class Distinct {
 public:
  explicit Distinct(int n) {
    int log = 4;
    while (((int64_t)1 << log) < 2 * (int64_t)n) ++log;
    shift_ = 64 - log;
    mask_ = ((uint64_t)1 << log) - 1;
    place_.assign((size_t)mask_ + 1, -1);
  }
  int id(int64_t v) {
    uint64_t h = (uint64_t)v * 0x9e3779b97f4a7c15ull;  // offsets step by several strides
    h = ((h ^ (h >> 29)) * 0xbf58476d1ce4e5b9ull) >> shift_;
    while (true) {
      const int32_t at = place_[h];
      if (at < 0) {
        place_[h] = (int32_t)values.size();
        values.push_back(v);
        return place_[h];
      }
      if (values[at] == v) return at;
      h = (h + 1) & mask_;
    }
  }
  std::vector<int64_t> values;

 private:
  int shift_;
  uint64_t mask_;
  std::vector<int32_t> place_;
};

// Entries in block order, of each block the last one listed.
void by_destination(const int64_t* ids, int n, int64_t num_blocks, std::vector<int32_t>* order) {
  order->clear();
  if (num_blocks <= 8 * (int64_t)n + 1024) {
    std::vector<int32_t> last((size_t)num_blocks, -1);
    for (int i = 0; i < n; ++i) last[(size_t)ids[i]] = i;
    for (int64_t b = 0; b < num_blocks; ++b)
      if (last[(size_t)b] >= 0) order->push_back(last[(size_t)b]);
    return;
  }
  std::vector<int32_t> all(n);
  for (int i = 0; i < n; ++i) all[i] = i;
  std::sort(all.begin(), all.end(), [&](int32_t x, int32_t y) {
    return ids[x] != ids[y] ? ids[x] < ids[y] : x < y;
  });
  for (int i = 0; i < n; ++i)
    if (i + 1 == n || ids[all[i]] != ids[all[i + 1]]) order->push_back(all[i]);
}

int check_record(int64_t off, int64_t rec_end, int64_t staging_bytes) {
  if (off < 0 || off > staging_bytes - rec_end) return DSR_PLAN_ERR_RECORD;
  return DSR_OK;
}

}  // namespace

extern "C" {

int dsr_plan_shared(const int64_t* slot_offsets, int n) {
  if (!slot_offsets || n < 0) return DSR_ERR_ARG;
  if (n < 2) return 0;
  try {
    Distinct d(n);
    for (int i = 0; i < n; ++i) {
      d.id(slot_offsets[i]);
      if (2 * (int64_t)d.values.size() > n) return 0;
    }
    return 1;
  } catch (const std::bad_alloc&) {
    return DSR_ERR_TOO_LARGE;
  }
}

int dsr_plan_load(const int64_t* page_ids, const int64_t* slot_offsets, const int64_t* rope_idx,
                  int n, int64_t num_blocks, int64_t rec_end, int64_t staging_bytes, int n_tables,
                  int fanout, void* out, int64_t out_bytes, dsr_plan* plan) {
  if (n < 0 || !plan || (n > 0 && (!page_ids || !slot_offsets || !out)) || num_blocks < 0 ||
      rec_end < 0)
    return DSR_ERR_ARG;
  memset(plan, 0, sizeof(*plan));
  if (out_bytes < DSR_PLAN_BYTES(n)) return DSR_ERR_TOO_LARGE;
  if (rope_idx)
    for (int i = 0; i < n; ++i)
      if (rope_idx[i] < -1 || rope_idx[i] >= n_tables) return DSR_PLAN_ERR_ROPE;
  for (int i = 0; i < n; ++i)
    if (page_ids[i] < 0 || page_ids[i] >= num_blocks) return DSR_PLAN_ERR_BLOCK;
  try {
    std::vector<int32_t> order;
    by_destination(page_ids, n, num_blocks, &order);
    const int m = (int)order.size();
    bool odd = false;
    for (int i = 0; i < m; ++i) {
      const int64_t off = slot_offsets[order[i]];
      if (const int rc = check_record(off, rec_end, staging_bytes)) return rc;
      odd |= (off & 15) != 0;
    }
    if (odd) return DSR_PLAN_ERR_ALIGN;
    uint8_t* const base = static_cast<uint8_t*>(out);
    plan->n_pages = m;
    if (!fanout) {
      plan->off_ids = round16(8 * (int64_t)m);
      plan->off_rope = plan->off_ids + round16(4 * (int64_t)m);
      plan->bytes = plan->off_rope + (rope_idx ? round16(4 * (int64_t)m) : 0);
      int64_t* const offs = reinterpret_cast<int64_t*>(base);
      int32_t* const ids = reinterpret_cast<int32_t*>(base + plan->off_ids);
      int32_t* const rope = reinterpret_cast<int32_t*>(base + plan->off_rope);
      for (int i = 0; i < m; ++i) {
        offs[i] = slot_offsets[order[i]];
        ids[i] = (int32_t)page_ids[order[i]];
        if (rope_idx) rope[i] = (int32_t)rope_idx[order[i]];
      }
      return DSR_OK;
    }
    // by source: the sources by offset, each one's destinations in block order
    Distinct d(m);
    std::vector<int32_t> src(m);
    for (int i = 0; i < m; ++i) src[i] = d.id(slot_offsets[order[i]]);
    const int ns = (int)d.values.size();
    std::vector<int32_t> at(ns), rank(ns), fill(ns + 1, 0);
    for (int s = 0; s < ns; ++s) at[s] = s;
    std::sort(at.begin(), at.end(),
              [&](int32_t x, int32_t y) { return d.values[x] < d.values[y]; });
    for (int r = 0; r < ns; ++r) rank[at[r]] = r;
    for (int i = 0; i < m; ++i) ++fill[rank[src[i]] + 1];
    for (int r = 0; r < ns; ++r) fill[r + 1] += fill[r];
    plan->n_src = ns;
    plan->off_start = round16(8 * (int64_t)ns);
    plan->off_ids = plan->off_start + round16(4 * ((int64_t)ns + 1));
    plan->off_rope = plan->off_ids + round16(4 * (int64_t)m);
    plan->bytes = plan->off_rope + (rope_idx ? round16(4 * (int64_t)m) : 0);
    int64_t* const srcs = reinterpret_cast<int64_t*>(base);
    int32_t* const start = reinterpret_cast<int32_t*>(base + plan->off_start);
    int32_t* const ids = reinterpret_cast<int32_t*>(base + plan->off_ids);
    int32_t* const rope = reinterpret_cast<int32_t*>(base + plan->off_rope);
    for (int r = 0; r < ns; ++r) srcs[r] = d.values[at[r]];
    for (int r = 0; r <= ns; ++r) start[r] = fill[r];
    for (int i = 0; i < m; ++i) {
      const int32_t to = fill[rank[src[i]]]++;
      ids[to] = (int32_t)page_ids[order[i]];
      if (rope_idx) rope[to] = (int32_t)rope_idx[order[i]];
    }
    return DSR_OK;
  } catch (const std::bad_alloc&) {
    return DSR_ERR_TOO_LARGE;
  }
}

int dsr_plan_gather(const int64_t* page_ids, const int64_t* slot_offsets, int n,
                    int64_t num_blocks, int64_t rec_end, int64_t rec_span, int64_t staging_bytes,
                    void* out, int64_t out_bytes, dsr_plan* plan) {
  if (n < 0 || !plan || (n > 0 && (!page_ids || !slot_offsets || !out)) || num_blocks < 0 ||
      rec_end < 0 || rec_span < 0)
    return DSR_ERR_ARG;
  memset(plan, 0, sizeof(*plan));
  if (out_bytes < DSR_PLAN_BYTES(n)) return DSR_ERR_TOO_LARGE;
  for (int i = 0; i < n; ++i)
    if (page_ids[i] < 0 || page_ids[i] >= num_blocks) return DSR_PLAN_ERR_BLOCK;
  bool odd = false, rising = true, apart = true;
  for (int i = 0; i < n; ++i) {
    if (const int rc = check_record(slot_offsets[i], rec_end, staging_bytes)) return rc;
    odd |= (slot_offsets[i] & 15) != 0;
    if (i) {
      rising &= slot_offsets[i] >= slot_offsets[i - 1];
      apart &= slot_offsets[i] - slot_offsets[i - 1] >= rec_span;
    }
  }
  if (odd) return DSR_PLAN_ERR_ALIGN;
  if (!rising) {
    try {
      std::vector<int64_t> s(slot_offsets, slot_offsets + n);
      std::sort(s.begin(), s.end());
      apart = true;
      for (int i = 1; i < n; ++i) apart &= s[i] - s[i - 1] >= rec_span;
    } catch (const std::bad_alloc&) {
      return DSR_ERR_TOO_LARGE;
    }
  }
  if (!apart) return DSR_PLAN_ERR_OVERLAP;
  plan->n_pages = n;
  plan->off_ids = plan->off_rope = round16(8 * (int64_t)n);
  plan->bytes = plan->off_ids + round16(4 * (int64_t)n);
  if (n) memcpy(out, slot_offsets, 8 * (size_t)n);
  int32_t* const ids = reinterpret_cast<int32_t*>(static_cast<uint8_t*>(out) + plan->off_ids);
  for (int i = 0; i < n; ++i) ids[i] = (int32_t)page_ids[i];
  return DSR_OK;
}

int dsr_plan_slots(const int64_t* slots, const int64_t* rows, const int64_t* rope_idx, int n,
                   int64_t num_blocks, int block_size, int64_t row_bytes, int64_t row_end,
                   int64_t staging_bytes, int n_tables, int mode, void* out, int64_t out_bytes,
                   dsr_slot_plan* plan) {
  if (n < 0 || !plan || (n > 0 && (!slots || !rows || !out)) || num_blocks < 0 ||
      block_size <= 0 || row_bytes <= 0 || row_end < 0 || (mode != 0 && mode != 1) ||
      num_blocks > INT64_MAX / block_size)
    return DSR_ERR_ARG;
  memset(plan, 0, sizeof(*plan));
  if (out_bytes < DSR_SLOT_PLAN_BYTES(n)) return DSR_ERR_TOO_LARGE;
  const int64_t num_slots = num_blocks * block_size;
  bool odd = false;
  for (int i = 0; i < n; ++i) {
    if (rope_idx && (rope_idx[i] < -1 || rope_idx[i] >= n_tables)) return DSR_PLAN_ERR_ROPE;
    if (slots[i] < 0) continue;
    if (slots[i] >= num_slots) return DSR_PLAN_ERR_SLOT;
    if (mode == 1 && check_record(rows[i], row_end, staging_bytes)) return DSR_PLAN_ERR_ROW;
    odd |= (rows[i] & 15) != 0;
  }
  if (mode == 1 && odd) return DSR_PLAN_ERR_ROWALIGN;
  try {
    std::vector<int32_t> order;
    order.reserve(n);
    bool rising = true;  // then no row repeats
    int64_t before = -1;
    for (int i = 0; i < n && mode == 1; ++i) {
      if (slots[i] < 0) continue;
      rising &= rows[i] > before;
      before = rows[i];
    }
    if (mode == 1 && rising) {
      for (int i = 0; i < n; ++i)
        if (slots[i] >= 0) order.push_back(i);
    } else if (mode == 1) {
      Distinct d(n);
      std::vector<int32_t> last;
      for (int i = 0; i < n; ++i) {
        if (slots[i] < 0) continue;
        const int r = d.id(rows[i]);
        if (r == (int)last.size()) last.push_back(i);
        else last[r] = i;
      }
      order = last;
      std::sort(order.begin(), order.end());
    } else if (num_slots <= 8 * (int64_t)n + 1024) {
      std::vector<int32_t> last((size_t)num_slots, -1);
      for (int i = 0; i < n; ++i)
        if (slots[i] >= 0) last[(size_t)slots[i]] = i;
      for (int64_t s = 0; s < num_slots; ++s)
        if (last[(size_t)s] >= 0) order.push_back(last[(size_t)s]);
    } else {
      std::vector<int32_t> all;
      all.reserve(n);
      for (int i = 0; i < n; ++i)
        if (slots[i] >= 0) all.push_back(i);
      std::sort(all.begin(), all.end(), [&](int32_t x, int32_t y) {
        return slots[x] != slots[y] ? slots[x] < slots[y] : x < y;
      });
      for (size_t i = 0; i < all.size(); ++i)
        if (i + 1 == all.size() || slots[all[i]] != slots[all[i + 1]]) order.push_back(all[i]);
    }
    const int m = (int)order.size();
    if (mode == 0) {  // a load: the rows that are read, not those of entries left out
      odd = false;
      for (int i = 0; i < m; ++i) {
        if (check_record(rows[order[i]], row_end, staging_bytes)) return DSR_PLAN_ERR_ROW;
        odd |= (rows[order[i]] & 15) != 0;
      }
      if (odd) return DSR_PLAN_ERR_ROWALIGN;
    }
    // whole blocks: their first entry's index in `order`
    std::vector<int32_t> first;
    std::vector<uint8_t> paged((size_t)m, 0);
    if (mode == 0) {
      for (int i = 0; i + block_size <= m;) {
        const int a = order[i];
        if (slots[a] % block_size) {
          ++i;
          continue;
        }
        int k = 1;
        for (; k < block_size; ++k) {
          const int b = order[i + k], p = order[i + k - 1];
          if (slots[b] != slots[p] + 1 || rows[b] != rows[p] + row_bytes ||
              (rope_idx && rope_idx[b] != rope_idx[p]))
            break;
        }
        if (k == block_size) {
          first.push_back(i);
          memset(&paged[i], 1, (size_t)block_size);
        }
        i += k;  // the entries passed start no block
      }
    }
    const int np = (int)first.size(), nt = m - np * block_size;
    uint8_t* const base = static_cast<uint8_t*>(out);
    plan->n_pages = np;
    plan->n_tokens = nt;
    plan->off_ids = 0;
    plan->off_offsets = round16(8 * (int64_t)np);
    plan->off_page_rope = plan->off_offsets + round16(8 * (int64_t)np);
    plan->off_slots = plan->off_page_rope + (rope_idx ? round16(8 * (int64_t)np) : 0);
    plan->off_rows = plan->off_slots + round16(8 * (int64_t)nt);
    plan->off_rope = plan->off_rows + round16(8 * (int64_t)nt);
    plan->bytes = plan->off_rope + (rope_idx ? round16(4 * (int64_t)nt) : 0) - plan->off_slots;
    int64_t* const ids = reinterpret_cast<int64_t*>(base);
    int64_t* const offs = reinterpret_cast<int64_t*>(base + plan->off_offsets);
    int64_t* const prope = reinterpret_cast<int64_t*>(base + plan->off_page_rope);
    for (int j = 0; j < np; ++j) {
      const int a = order[first[j]];
      ids[j] = slots[a] / block_size;
      offs[j] = rows[a];
      if (rope_idx) prope[j] = rope_idx[a];
    }
    int64_t* const ts = reinterpret_cast<int64_t*>(base + plan->off_slots);
    int64_t* const tr = reinterpret_cast<int64_t*>(base + plan->off_rows);
    int32_t* const tx = reinterpret_cast<int32_t*>(base + plan->off_rope);
    int t = 0;
    for (int i = 0; i < m; ++i) {
      if (paged[(size_t)i]) continue;
      ts[t] = slots[order[i]];
      tr[t] = rows[order[i]];
      if (rope_idx) tx[t] = (int32_t)rope_idx[order[i]];
      ++t;
    }
    return DSR_OK;
  } catch (const std::bad_alloc&) {
    return DSR_ERR_TOO_LARGE;
  }
}

}  // extern "C"

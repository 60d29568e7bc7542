// Work list of a prefill launch: which (row tile, key range) each workgroup
// takes. Plain host C++, built once per attention plan from the sequence
// lengths that the plan's owner has on the host; the CPU tests compile it with
// g++.
//
// A row tile sees all keys up to its last row, so a chunk of few rows on a long
// prefix is a handful of long items: taken whole they leave most of the 256 CUs
// idle (one 512-row chunk at position 15000, 32 q / 8 kv heads: 64 workgroups,
// 375 us), and a chunk of many rows ends in a partly empty round (4096 rows at
// position 28672, 56 q / 8 kv heads: 912 workgroups on 256 CUs, 3.56 rounds).
// An item can therefore be cut along its keys into pieces that leave
// unnormalised partial results, which prefill_merge_kernel combines: 375 -> 124
// us and 3.16 -> 3.01 ms for those two (whole op, same box); 263 rows at
// position 3840, 14 q / 2 kv heads, head_dim 64: 130 -> 29 us.
#pragma once

#include <algorithm>
#include <cstdint>
#include <functional>
#include <vector>

namespace gk {

// Query rows (row, head pairs) of a prefill workgroup and keys of a step.
constexpr int prefill_tile_qrows(int head_dim) { return head_dim > 128 ? 128 : 256; }
constexpr int prefill_step_keys(int head_dim) { return head_dim == 128 ? 64 : 32; }

struct PrefillSeq {
  int32_t first_row, rows, prefix;
};

// One workgroup's work for one kv head: query rows first_row .. + rows - 1 at
// positions pos .., steps of prefill_step_keys keys from key0 on. slot < 0: the
// whole item, output rows written directly; else the partial slot it fills.
struct PrefillItem {
  int32_t first_row, rows, pos, key0, steps, slot, pad[2];
};
constexpr int kPrefillItemWords = 8;
// A split item: its pieces filled slots slot .. slot + parts - 1.
struct PrefillMerge {
  int32_t first_row, rows, slot, parts;
};
constexpr int kPrefillMergeWords = 4;

struct PrefillWorkList {
  std::vector<PrefillItem> items;    // longest first
  std::vector<PrefillMerge> merges;
  int32_t slots = 0;                 // partial slots of one kv head
};

// Room for the words of any list of `tiles` row tiles: each worker's boundary
// leaves an extra piece at most, in the two ways of cutting three a worker.
inline int64_t prefill_row_tiles(int64_t rows, int group, int head_dim) {
  const int tile_rows = prefill_tile_qrows(head_dim) / group;
  return (rows + tile_rows - 1) / tile_rows;
}
inline int64_t prefill_words_bound(int64_t tiles, int kv_heads, int cus) {
  const int64_t slots = std::max(1, cus / kv_heads);
  return kPrefillItemWords * (tiles + 3 * slots + 1) + kPrefillMergeWords * std::min(tiles, 3 * slots + 1);
}

// What the choice weighs, in steps of the head dimension's kernel. Measured
// with every CU busy (256 workgroups, 1 to 64 steps each): a step takes 0.57 us
// at head_dim 64 (32 keys; two workgroups of a CU take 1.13, so one CU counts
// as one worker), 1.6-1.75 at 128 (64 keys) and 1.3 at 256 (32 keys); a
// workgroup's start and end 5-7 us. What a cut costs is fitted to 26000 drawn
// batches (up to 4096 rows on up to 20000 keys, windows, softcap), each launched
// cut and uncut: the smallest charges with which no batch that is then cut runs
// more than 2% longer for it (head_dim 64 and 128) or 0.2% (256, where pieces of
// different key ranges also find less of each other's K/V in the L2: steps of a
// cut list take 1.2 times as long); of 10765 other batches cut with them 2 ran
// longer by more than 2% (7%, 3%). With smaller charges (8, 3 and 4 a launch,
// 0.02 a partial) 2.7% of the batches ran up to 1.23 times as long: two chunks
// of 410 and 343 rows, 16 q / 8 kv heads, head_dim 256, 23.6 us uncut, 29.2 cut;
// 549 rows, 32 / 8, head_dim 128, 21.4 and 25.6. Over all of them cutting makes
// head_dim 64 1.94 times as fast, 128 1.72, 256 1.57.
struct PrefillCost {
  double piece;     // a workgroup's start and end
  double step;      // a step of a cut list
  double merge;     // the merge launch
  double partial;   // writing and reading one partial slot, spread over the GPU
  double merged;    // one split item of one kv head in the merge
  int least;        // shortest piece worth cutting
};
inline PrefillCost prefill_cost(int head_dim) {
  if (head_dim == 64) return {10.0, 1.0, 6.0, 0.04, 0.0, 8};
  if (head_dim == 128) return {4.0, 1.0, 4.0, 0.03, 0.0, 4};
  return {4.0, 1.2, 5.0, 0.03, 0.06, 8};
}

// Time at which `slots` workers, each taking the next piece when it falls free,
// finish pieces of the given lengths (longest first).
inline double prefill_makespan(const std::vector<PrefillItem>& items, int slots, double piece) {
  if ((int)items.size() <= slots) return items.empty() ? 0.0 : items.front().steps + piece;
  std::vector<double> busy(slots, 0.0);  // min-heap of the workers' times
  double last = 0.0;
  for (const auto& it : items) {
    std::pop_heap(busy.begin(), busy.end(), std::greater<double>());
    busy.back() += it.steps + piece;
    last = std::max(last, busy.back());
    std::push_heap(busy.begin(), busy.end(), std::greater<double>());
  }
  return last;
}

// A list's time by these costs (of an uncut list: its makespan).
inline double prefill_list_time(const PrefillWorkList& list, int slots, int kv_heads, const PrefillCost& cost) {
  const double busy = prefill_makespan(list.items, slots, cost.piece);
  if (list.merges.empty()) return busy;
  return cost.step * (busy - cost.piece) + cost.piece + cost.merge +
         kv_heads * (cost.partial * list.slots + cost.merged * list.merges.size());
}

inline void prefill_longest_first(std::vector<PrefillItem>& items) {
  // Pieces of one key range together: they read the same K/V.
  std::sort(items.begin(), items.end(), [](const PrefillItem& a, const PrefillItem& b) {
    if (a.steps != b.steps) return a.steps > b.steps;
    if (a.key0 != b.key0) return a.key0 > b.key0;
    return a.first_row < b.first_row;
  });
}

// Replaces `whole` with the pieces that end at the given step counts (the last
// one its length); one end leaves it whole.
inline void prefill_cut(PrefillWorkList& out, const PrefillItem& whole, const std::vector<int>& ends, int keys) {
  if (ends.size() == 1) {
    out.items.push_back(whole);
    return;
  }
  out.merges.push_back({whole.first_row, whole.rows, out.slots, (int32_t)ends.size()});
  int begin = 0;
  for (int end : ends) {
    PrefillItem p = whole;
    p.key0 += begin * keys;
    p.steps = end - begin;
    p.slot = out.slots++;
    out.items.push_back(p);
    begin = end;
  }
}

// Every row tile whole: a row's keys are taken in one order whatever else the
// list holds, so its output depends on its own sequence alone.
inline PrefillWorkList prefill_whole_list(const PrefillSeq* seqs, int count, int group, int head_dim, int window) {
  const int keys = prefill_step_keys(head_dim), tile_rows = prefill_tile_qrows(head_dim) / group;
  PrefillWorkList whole;
  for (int s = 0; s < count; ++s)
    for (int r0 = 0; r0 < seqs[s].rows; r0 += tile_rows) {
      const int nr = std::min(tile_rows, seqs[s].rows - r0), pos = seqs[s].prefix + r0;
      const int left = window > 0 ? std::max(0, pos - window + 1) : 0, key0 = left / keys * keys;
      const int steps = (pos + nr - key0 + keys - 1) / keys;
      whole.items.push_back({seqs[s].first_row + r0, nr, pos, key0, steps, -1, {0, 0}});
    }
  prefill_longest_first(whole.items);
  return whole;
}

inline PrefillWorkList prefill_work_list(const PrefillSeq* seqs, int count, int group, int kv_heads, int head_dim,
                                         int window, int cus) {
  const int keys = prefill_step_keys(head_dim);
  PrefillWorkList whole = prefill_whole_list(seqs, count, group, head_dim, window);
  int64_t total = 0;
  for (const auto& it : whole.items) total += it.steps;
  // Every kv head has the same list, and the grid gives each an equal share of
  // the GPU: balance one head's list over its share.
  const PrefillCost cost = prefill_cost(head_dim);
  const int n = (int)whole.items.size(), slots = std::max(1, cus / kv_heads);
  // Many items a worker: the last round is a small part (and the plan stays cheap).
  if (n == 0 || n > 12 * slots) return whole;
  const double uncut = prefill_makespan(whole.items, slots, cost.piece);
  const double even = (double)total / slots;
  if (uncut <= 1.04 * (even + cost.piece) + cost.merge) return whole;

  PrefillWorkList best;
  double best_time = uncut;
  const auto consider = [&](PrefillWorkList&& list) {
    if (list.merges.empty()) return;
    prefill_longest_first(list.items);
    const double time = prefill_list_time(list, slots, kv_heads, cost);
    if (time < best_time) {
      best_time = time;
      best = std::move(list);
    }
  };
  std::vector<int> ends;
  // Every item in equal pieces of at most `most` steps, the fewest steps with
  // which one round of workgroups holds all pieces.
  if (n <= slots) {
    int lo = std::max<int>(cost.least, (int)even), hi = std::max(lo, whole.items.front().steps);
    const auto pieces = [&](int most) {
      int64_t sum = 0;
      for (const auto& it : whole.items) sum += (it.steps + most - 1) / most;
      return sum;
    };
    while (lo < hi) {
      const int mid = (lo + hi) / 2;
      if (pieces(mid) <= slots) hi = mid;
      else lo = mid + 1;
    }
    PrefillWorkList list;
    for (const auto& it : whole.items) {
      const int k = (it.steps + lo - 1) / lo;
      ends.clear();
      for (int j = 1; j <= k; ++j) ends.push_back((int)((int64_t)it.steps * j / k));
      prefill_cut(list, it, ends, keys);
    }
    consider(std::move(list));
  }
  // The items laid end to end and cut into one equal share a worker: at most
  // one extra piece each, whatever the lengths.
  {
    const double share = (total + cost.piece * (n + slots)) / slots + 1.0;
    PrefillWorkList list;
    double room = share;
    for (const auto& it : whole.items) {
      ends.clear();
      int done = 0;
      while (done < it.steps) {
        int take = std::min(it.steps - done, (int)(room - cost.piece));
        if (take < std::min(cost.least, it.steps - done)) {
          room = share;
          take = std::min(it.steps - done, std::max(cost.least, (int)(room - cost.piece)));
        }
        if (it.steps - done - take < cost.least) take = it.steps - done;
        done += take;
        room -= take + cost.piece;
        ends.push_back(done);
      }
      prefill_cut(list, it, ends, keys);
    }
    consider(std::move(list));
  }
  return best.items.empty() ? whole : best;
}

}  // namespace gk

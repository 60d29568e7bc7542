// CPU checks of gaudirt_amd/csrc/prefill_schedule.hpp: for many sets of
// sequences, head geometries and windows the work list covers every step of
// every row tile exactly once, its partial slots are distinct and grouped as
// the merge records say, items come longest first, and the estimated time of
// the list never exceeds that of the uncut items; and batches that measured
// faster cut are cut, ones that measured faster whole stay whole. Prints OK on
// success.
#include <cstdio>
#include <map>
#include <random>
#include <vector>

#include "prefill_schedule.hpp"

namespace {

int failures = 0;
void expect(bool ok, const char* what, int trial) {
  if (!ok && failures++ < 10) std::printf("trial %d: %s\n", trial, what);
}

void check(const std::vector<gk::PrefillSeq>& seqs, int group, int kv_heads, int d, int window, int trial) {
  const auto list = gk::prefill_work_list(seqs.data(), (int)seqs.size(), group, kv_heads, d, window, 256);
  const int keys = gk::prefill_step_keys(d), tile_rows = gk::prefill_tile_qrows(d) / group;
  // Every tile's steps, by the tile's first row.
  std::map<int, std::vector<gk::PrefillItem>> pieces;
  for (const auto& it : list.items) pieces[it.first_row].push_back(it);
  std::vector<int> slot_used(list.slots, 0);
  size_t tiles = 0, split = 0;
  for (const auto& s : seqs)
    for (int r0 = 0; r0 < s.rows; r0 += tile_rows) {
      ++tiles;
      auto found = pieces.find(s.first_row + r0);
      expect(found != pieces.end(), "a row tile is missing", trial);
      if (found == pieces.end()) continue;
      auto& p = found->second;
      std::sort(p.begin(), p.end(), [](const auto& a, const auto& b) { return a.key0 < b.key0; });
      const int pos = s.prefix + r0, nr = std::min(tile_rows, s.rows - r0);
      const int left = window > 0 ? std::max(0, pos - window + 1) : 0;
      int at = left / keys * keys;
      for (const auto& it : p) {
        expect(it.key0 == at && it.steps > 0 && it.rows == nr && it.pos == pos, "a piece is out of place", trial);
        expect((it.slot >= 0) == (p.size() > 1), "partial slots and pieces disagree", trial);
        if (it.slot >= 0) {
          expect(it.slot < list.slots, "a slot out of range", trial);
          if (it.slot < list.slots) ++slot_used[it.slot];
        }
        at += it.steps * keys;
      }
      expect(at >= pos + nr && at - keys < pos + nr, "the pieces do not end with the last visible key", trial);
      if (p.size() > 1) ++split;
    }
  expect(pieces.size() == tiles, "items of rows that no tile has", trial);
  expect(split == list.merges.size(), "merge records and split items disagree", trial);
  for (const auto& m : list.merges) {
    const auto& p = pieces[m.first_row];
    expect((int)p.size() == m.parts && !p.empty() && p.front().rows == m.rows, "a merge record does not fit", trial);
    for (size_t i = 0; i < p.size(); ++i) expect(p[i].slot == m.slot + (int)i, "a merge's slots are not its pieces'", trial);
  }
  for (int u : slot_used) expect(u == 1, "a slot is filled by no piece or several", trial);
  for (size_t i = 1; i < list.items.size(); ++i)
    expect(list.items[i - 1].steps >= list.items[i].steps, "items are not longest first", trial);
  // At most one extra piece per worker and item, which bounds the workspace.
  const int slots = std::max(1, 256 / kv_heads);
  expect(list.slots <= 3 * slots + 1, "more partial slots than the workers can leave", trial);
  int64_t row_tiles = 0;
  for (const auto& s : seqs) row_tiles += gk::prefill_row_tiles(s.rows, group, d);
  expect((int64_t)tiles == row_tiles, "the count of row tiles is wrong", trial);
  expect((int64_t)(gk::kPrefillItemWords * list.items.size() + gk::kPrefillMergeWords * list.merges.size()) <=
             gk::prefill_words_bound(row_tiles, kv_heads, 256),
         "the list needs more words than the bound", trial);
  const auto whole = gk::prefill_whole_list(seqs.data(), (int)seqs.size(), group, d, window);
  expect(whole.merges.empty() && whole.items.size() == tiles, "an uncut list is cut", trial);
  const auto cost = gk::prefill_cost(d);
  expect(gk::prefill_list_time(list, slots, kv_heads, cost) <= gk::prefill_list_time(whole, slots, kv_heads, cost),
         "the list takes longer than the uncut items", trial);
}

// Batches measured both ways on a 256-CU GPU.
void check_choice(const std::vector<gk::PrefillSeq>& seqs, int group, int kv_heads, int d, bool cut, int trial) {
  const auto list = gk::prefill_work_list(seqs.data(), (int)seqs.size(), group, kv_heads, d, -1, 256);
  expect(list.merges.empty() != cut, cut ? "a batch that is faster cut stays whole" : "a batch that is faster whole is cut",
         trial);
}

}  // namespace

int main() {
  std::mt19937 rng(7);
  const int dims[] = {64, 128, 256}, groups[] = {1, 2, 3, 4, 7, 8, 16, 128}, heads[] = {1, 2, 3, 4, 8, 12, 16, 64, 256};
  auto upto = [&](int n) { return (int)(rng() % (unsigned)(n + 1)); };
  for (int trial = 0; trial < 4000; ++trial) {
    std::vector<gk::PrefillSeq> seqs;
    int row = upto(3);
    const int n = 1 + upto(trial % 5 ? 7 : 60);
    for (int s = 0; s < n; ++s) {
      const int rows = 1 + upto(trial % 3 ? 600 : 40), prefix = upto(3) ? upto(20000) : 0;
      seqs.push_back({row, rows, prefix});
      row += rows + upto(2);
    }
    const int window = upto(2) ? -1 : 1 + upto(5000);
    check(seqs, groups[upto(7)], heads[upto(8)], dims[upto(2)], window, trial);
  }
  // The ends of the range: one row and one key; a single very long sequence.
  for (int d : dims)
    for (int g : groups) {
      check({{0, 1, 0}}, g, 1, d, -1, -1);
      check({{0, 1, 1 << 24}}, g, 8, d, -1, -2);
      check({{5, 8192, 100000}}, g, 256, d, -1, -3);
      check({{0, 64, 1 << 20}}, g, 2, d, 1, -4);
    }
  // One chunk of few rows on a long prefix, cut: 375 -> 124 us, 130 -> 29 us, 86 -> 17 us, 85 -> 57 us.
  check_choice({{0, 512, 15000}}, 4, 8, 128, true, -10);
  check_choice({{0, 263, 3840}}, 7, 2, 64, true, -11);
  check_choice({{0, 8, 5222}}, 4, 8, 128, true, -12);
  check_choice({{0, 424, 1683}, {424, 424, 1261}}, 2, 8, 256, true, -13);
  // Whole 23.6 us against 29.2 cut, 23.4 / 28.0, 21.4 / 25.6, 24.8 / 29.6, and tiles that fill the GPU anyway.
  check_choice({{0, 410, 78}, {410, 343, 103}}, 2, 8, 256, false, -14);
  check_choice({{0, 247, 120}, {247, 204, 284}, {451, 212, 164}}, 2, 8, 256, false, -15);
  check_choice({{0, 549, 0}}, 4, 8, 128, false, -16);
  check_choice({{0, 305, 362}, {305, 240, 173}}, 2, 16, 128, false, -17);
  check_choice({{0, 4096, 2048}}, 4, 8, 128, false, -18);
  // No sequence: an empty list.
  if (!gk::prefill_work_list(nullptr, 0, 1, 1, 64, -1, 256).items.empty()) ++failures;
  if (failures) return 1;
  std::printf("OK\n");
  return 0;
}

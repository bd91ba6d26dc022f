// score_tables.cpp -- host-side work split of the generalized scoring kernel
// (score.hip): which targets each wave scores, and one table entry per
// 16-token tile (the last tile of a target holds its remaining 1..16 tokens;
// an empty target gets one empty tile).  A target costs its tiles + 1; targets
// go to waves longest first, each onto the least-loaded wave (LPT), as in
// scan_tables.cpp, with absolute target indices; more than 2^24 targets fall
// back to contiguous cost-balanced ranges.
#include <algorithm>
#include <queue>

#include "internal.hpp"

namespace msim {

namespace {
constexpr int64_t kMaxLocal = int64_t(1) << 24;  // target index bits of a tile entry
}  // namespace

void build_score_tables(const int64_t* off, const int64_t* targets, int64_t n, int64_t waves,
                        std::vector<int64_t>& info, std::vector<uint64_t>& tiles) {
  info.clear();
  tiles.clear();
  waves = std::max<int64_t>(1, std::min(waves, std::max<int64_t>(1, n)));
  auto doc_of = [&](int64_t t) { return targets ? targets[t] : t; };
  auto cost_of = [&](int64_t t) {
    const int64_t d = doc_of(t);
    return std::max<int64_t>(1, (off[d + 1] - off[d] + 15) / 16) + 1;
  };
  // Tiles of target t (index `local` relative to the wave's base).
  auto emit_target = [&](int64_t t, int64_t local) {
    const int64_t d = doc_of(t);
    const int64_t s = off[d], e = off[d + 1];
    if (s == e) {
      tiles.push_back(score_tile_entry(0, 1, true, true, local));
      return;
    }
    for (int64_t x = s; x < e; x += 16)
      tiles.push_back(score_tile_entry(x, std::min<int64_t>(16, e - x), x + 16 >= e, false, local));
  };
  auto close_wave = [&](int64_t base, int64_t count, int64_t tab0) {
    const int64_t ntiles = (int64_t)tiles.size() - tab0;
    tiles.push_back(score_tile_entry(0, 1, false, false, 0));
    const int64_t row[kScoreInfoWords] = {base, count, ntiles, tab0};
    info.insert(info.end(), row, row + kScoreInfoWords);
  };
  if (n < kMaxLocal) {
    std::vector<int64_t> order((size_t)n);
    for (int64_t t = 0; t < n; ++t) order[(size_t)t] = t;
    std::stable_sort(order.begin(), order.end(), [&](int64_t a, int64_t b) { return cost_of(a) > cost_of(b); });
    using Load = std::pair<int64_t, int64_t>;  // (cost so far, wave)
    std::priority_queue<Load, std::vector<Load>, std::greater<Load>> heap;
    for (int64_t w = 0; w < waves; ++w) heap.push({0, w});
    std::vector<std::vector<int64_t>> mine((size_t)waves);
    for (int64_t t : order) {
      Load l = heap.top();
      heap.pop();
      mine[(size_t)l.second].push_back(t);
      heap.push({l.first + cost_of(t), l.second});
    }
    for (auto& ts : mine) {
      std::sort(ts.begin(), ts.end());
      const int64_t tab0 = (int64_t)tiles.size();
      for (int64_t t : ts) emit_target(t, t);
      close_wave(0, (int64_t)ts.size(), tab0);
    }
  } else {
    std::vector<int64_t> cost(n + 1, 0);
    for (int64_t t = 0; t < n; ++t) cost[t + 1] = cost[t] + cost_of(t);
    int64_t t0 = 0;
    for (int64_t w = 1; w <= waves && t0 < n; ++w) {
      int64_t t1 = w == waves ? n : std::lower_bound(cost.begin(), cost.end(), (cost[n] * w) / waves) - cost.begin();
      t1 = std::min(t1, n);
      while (t0 < t1) {
        const int64_t e = std::min(t1, t0 + kMaxLocal - 1);
        const int64_t tab0 = (int64_t)tiles.size();
        for (int64_t t = t0; t < e; ++t) emit_target(t, t - t0);
        close_wave(t0, e - t0, tab0);
        t0 = e;
      }
    }
  }
  while ((info.size() / kScoreInfoWords) % kScanWavesPerGroup != 0 || info.empty()) {
    const int64_t tab0 = (int64_t)tiles.size();
    close_wave(n, 0, tab0);
  }
}

// Flat arrays throughout: it runs inside a corpus's first search, where a
// vector per list (and one of its records) took 80 us for 300 documents on 256
// lists, twice build_score_tables' time.
int64_t build_score_units(const int64_t* off, int64_t n, int64_t workgroups, int64_t min_tiles,
                          std::vector<int64_t>& info, std::vector<uint64_t>& tiles) {
  workgroups = std::max<int64_t>(1, std::min(workgroups, std::max<int64_t>(1, n)));
  auto tiles_of = [&](int64_t d) { return std::max<int64_t>(1, (off[d + 1] - off[d] + 15) / 16); };
  // Longest first, equal ones by index: one key each (a tile start has 34 bits,
  // so a document has fewer than 2^34 tiles).
  constexpr int kDocBits = 24;
  constexpr uint64_t kMostTiles = uint64_t(1) << 34, kDocMask = (uint64_t(1) << kDocBits) - 1;
  std::vector<uint64_t> order((size_t)n);
  int64_t total = 0;
  for (int64_t d = 0; d < n; ++d) {
    total += tiles_of(d);
    order[(size_t)d] = ((kMostTiles - (uint64_t)tiles_of(d)) << kDocBits) | (uint64_t)d;
  }
  std::sort(order.begin(), order.end());
  // A heap of (cost so far, list) keys, the least at the root.
  std::vector<uint64_t> heap((size_t)workgroups);
  for (int64_t w = 0; w < workgroups; ++w) heap[(size_t)w] = (uint64_t)w;
  std::vector<int64_t> list_of((size_t)n), first((size_t)workgroups + 1, 0);  // of the i-th longest; a list's first below
  for (int64_t i = 0; i < n; ++i) {
    const uint64_t list = heap[0] & kDocMask;
    list_of[(size_t)i] = (int64_t)list;
    ++first[(size_t)list + 1];
    const uint64_t key = heap[0] + ((kMostTiles - (order[(size_t)i] >> kDocBits) + 1) << kDocBits);
    size_t x = 0, child = 1;
    for (; child < heap.size(); x = child, child = 2 * x + 1) {
      if (child + 1 < heap.size() && heap[child + 1] < heap[child]) ++child;
      if (heap[child] >= key) break;
      heap[x] = heap[child];
    }
    heap[x] = key;
  }
  for (int64_t w = 0; w < workgroups; ++w) first[(size_t)w + 1] += first[(size_t)w];
  std::vector<int64_t> docs((size_t)n), at(first.begin(), first.end() - 1);  // list by list, each longest first
  for (int64_t i = 0; i < n; ++i) docs[(size_t)at[(size_t)list_of[(size_t)i]]++] = (int64_t)(order[(size_t)i] & kDocMask);

  tiles.resize((size_t)(total + 1));
  uint64_t* const table = tiles.data();
  table[0] = score_tile_entry(0, 1, false, true, 0);  // padding: what a wave loads past its list's end
  int64_t end = 1;
  std::vector<int64_t> records;  // kScoreInfoWords each, list by list
  records.reserve((size_t)(kScoreInfoWords * std::min(n, total / std::max<int64_t>(1, min_tiles) + workgroups)));
  std::vector<int64_t> ends((size_t)workgroups);  // records up to a list's end
  int64_t most = 1;
  for (int64_t w = 0; w < workgroups; ++w) {
    int64_t tab0 = end, count = 0;
    auto close = [&]() {
      const int64_t row[kScoreInfoWords] = {0, count, end - tab0, tab0};
      records.insert(records.end(), row, row + kScoreInfoWords);
      tab0 = end;
      count = 0;
    };
    for (int64_t i = first[(size_t)w]; i < first[(size_t)w + 1]; ++i) {
      const int64_t d = docs[(size_t)i], s = off[d], e = off[d + 1], last = tiles_of(d) - 1;
      for (int64_t x = 0; x < last; ++x) table[end + x] = score_tile_entry(s + 16 * x, 16, false, false, d);
      end += last;
      table[end++] = s == e ? score_tile_entry(0, 1, true, true, d)
                            : score_tile_entry(s + 16 * last, e - s - 16 * last, true, false, d);
      ++count;
      if (end - tab0 >= min_tiles) close();
    }
    if (count > 0) close();
    ends[(size_t)w] = (int64_t)records.size() / kScoreInfoWords;
    most = std::max(most, ends[(size_t)w] - (w > 0 ? ends[(size_t)w - 1] : 0));
  }
  info.assign((size_t)(workgroups * most * kScoreInfoWords), 0);
  for (int64_t w = 0; w < workgroups; ++w) {
    const int64_t from = w > 0 ? ends[(size_t)w - 1] : 0;
    std::copy(records.begin() + from * kScoreInfoWords, records.begin() + ends[(size_t)w] * kScoreInfoWords,
              info.begin() + w * most * kScoreInfoWords);
  }
  return most;
}

}  // namespace msim

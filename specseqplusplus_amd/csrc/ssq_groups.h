// Which clouds of a batched Rips call are built and reduced together, and on how many streams.  Host
// arithmetic on the clouds' sizes alone (ripsco_reduce runs the plan).
#pragma once
#include <algorithm>
#include <cstdint>
#include <utility>
#include <vector>

namespace ssq {

// Cells of one group: a bound well inside the engine's int32 cell ids, and small enough that
// the per-row tables of two consecutive groups' sizes fit beside each other as buffers grow.
constexpr int64_t kGroupCells = (int64_t)1 << 30;
// groups of a call that would leave streams without one (plan_groups)
constexpr int64_t kSplitCells = (int64_t)1 << 23;
constexpr int kSplitGroups = 6, kSplitStreams = 3;
// device bytes each engine keeps for its huge-column bit sets (k_add_huge regions)
constexpr int64_t kHugeRegionBytes = (int64_t)256 << 24;

// Device bytes of one group, by the buffers of the builder and of the engine, with the slack of
// their geometric growth (1.5x for the engine's buffers, 1.25x for the builder's).
inline double group_bytes(int64_t nv, int64_t ne, int64_t nt, int64_t n2, int64_t ew, int64_t tie_guess) {
  const double rows = 2.0 * ne + 3.0 * nt;
  const double engine = 4.0 * rows * 2.0                // pool: rows, then the arena (holds the staging)
                        + 42.0 * (double)(nv + ne + nt) // per-row tables: piv, leftone, flags, pivmeta
                        + 40.0 * (double)(nv + ne);     // per-column state and lists
  const double builder = 4.0 * (double)nt               // tie remap
                         + 4.0 * (double)n2             // rank matrices
                         + 10.0 * (double)ew            // Q bitsets and prefix counts
                         + 120.0 * (double)ne + 80.0 * (double)nv  // edge keys, runs, lists, lengths
                         + 32.0 * (double)tie_guess;
  return 1.5 * engine + 1.25 * builder + 64.0 * 1048576.0;
}

struct CloudSize {
  int64_t n, edges, tris;
};
struct GroupPlan {
  std::vector<int> order;                   // the clouds by decreasing triangle count
  std::vector<std::pair<int, int>> groups;  // [begin, end) in order
  int workers = 1;                          // streams that take groups
};

// Groups: clouds by decreasing triangle count, consecutive ones while the group's estimated
// bytes fit the budget and its cells stay below a limit.  The groups run on the streams side
// by side.  A group's rounds each last as long as the longest chase in them, which one
// workgroup runs, and clouds that share a group add up those times: 40 clouds of 64-2048
// points take 130 ms in one group, their longest alone 55 ms.  So where streams would be left
// without a group, the clouds are split further, into about kSplitGroups groups of at least
// kSplitCells cells (a group's launches and synchronisations are about 1 ms, the work on 8 million
// cells 2 ms or more).  A process with streams of its own has more than its four hardware queues, and
// a short group then waits behind another's long chase: a call takes kSplitStreams streams, or as
// many as it had groups before the split, whatever is more.
// Four hardware queues, ms in one group (or as many as kGroupCells asks for) / split on 3 streams /
// split on 4:
//   40 clouds of 64-2048 points  130 / 84 / 90-105     3 of 2000        119 / 88 / 87
//   6 of 1000                     30 / 20 / 29         12 of 300-600    7.1 / 5.5 / 5.5
//   60 of 64-1000                 32 / 24 / 24-28      200 of 100-400  13.2 / 12.2 / 12.0
//   100 of 64-2048 (3 groups)    185 / 172 / 174       31 of 500-900   26.0 / 27.8 / 28.6
// The last loses: its clouds are alike, and its seven groups fill three streams unevenly.  Half as many
// groups suit it better (23.7), but not 40 of 64-2048 (104).
// Sixteen queues, groups of 9 GB: 100 clouds of 64-2048 points make 14 groups, 128-164 ms on 14
// streams, 198-221 on 3.
inline GroupPlan plan_groups(const std::vector<CloudSize>& clouds, int64_t mem_budget, int nstreams) {
  GroupPlan p;
  const int count = (int)clouds.size();
  p.order.resize((size_t)count);
  for (int c = 0; c < count; c++) p.order[(size_t)c] = c;
  std::stable_sort(p.order.begin(), p.order.end(),
                   [&](int x, int y) { return clouds[(size_t)x].tris > clouds[(size_t)y].tris; });
  const auto make_groups = [&](int64_t cells) {
    p.groups.clear();
    for (int i0 = 0; i0 < count;) {
      int i1 = i0;
      int64_t nv = 0, ne = 0, nt = 0, n2 = 0, ew = 0;
      while (i1 < count) {
        const CloudSize& c = clouds[(size_t)p.order[(size_t)i1]];
        const int64_t W = (c.n + 63) / 64;
        const double bytes = group_bytes(nv + c.n, ne + c.edges, nt + c.tris, n2 + c.n * c.n, ew + c.edges * W,
                                         (nt + c.tris) / 16);
        const bool fits = nv + c.n + ne + c.edges + nt + c.tris <= cells && bytes <= (double)mem_budget;
        if (!fits && i1 > i0) break;
        nv += c.n;
        ne += c.edges;
        nt += c.tris;
        n2 += c.n * c.n;
        ew += c.edges * W;
        i1++;
        if (!fits) break;  // one cloud alone: try it anyway
      }
      p.groups.emplace_back(i0, i1);
      i0 = i1;
    }
  };
  make_groups(kGroupCells);
  const int whole = (int)p.groups.size();
  p.workers = nstreams;
  if (whole < nstreams) {
    int64_t cells = 0;
    for (const CloudSize& c : clouds) cells += c.n + c.edges + c.tris;
    make_groups(std::min(kGroupCells, std::max(kSplitCells, cells / kSplitGroups)));
    p.workers = std::min(nstreams, std::max(whole, kSplitStreams));
  }
  p.workers = std::min(p.workers, (int)p.groups.size());
  return p;
}

}  // namespace ssq

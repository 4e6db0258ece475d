// edge_plan.h -- the samples of edge checks in launches: levels, windows and
// the launches' edge and rank ranges.  Plain integer arithmetic, used by the
// host runtime, the kernels and (compiled for the host) the tests.
#pragma once

#include <algorithm>
#include <vector>

#if defined(__HIPCC__)
#define GPRM_EDGE_HD __host__ __device__ inline
#else
#define GPRM_EDGE_HD inline
#endif

namespace gprm {

// Samples of an edge in launch windows.  The testnum samples of an edge
// belong to levels: level 0 holds at most 16 evenly spaced ones, each next
// level fills up a spacing four times finer, the last level the rest:
// edge_levels(T) levels with spacings m_l, the multiples of m_l that are not
// multiples of m_(l-1).  A window covers levels [l0, l1) of every edge, in
// ascending sample order: adjacent items are adjacent samples, whose links
// stay close together, which is what the pair masks live on; and the first
// window's spread samples find most blocked edges.  The 6-DOF roadmap
// (longest edge 209 samples) takes two windows, of 15 and about 105 samples
// per edge.
constexpr int kLevelAll = 64;  // l1 of a window that takes every remaining sample
GPRM_EDGE_HD int edge_levels(int T) {
  if (T <= 16) return 1;
  if (T <= 256) return 2;
  int n = 3;
  for (long long lim = 512; T > lim; lim *= 4) ++n;
  return n;
}
// Samples of the window: the multiples of a that are not multiples of b (b =
// 0: every multiple of a).  count: how many.
GPRM_EDGE_HD void edge_window(int T, int l0, int l1, int* a, int* b, int* count) {
  const int n = edge_levels(T);
  *a = 1;
  *b = 0;
  *count = 0;
  if (T <= 0 || l0 >= n) return;
  int fine = 1;  // m_(n-2), and from it the coarser spacings
  if (n > 1) {
    const long long cnt = 16LL << (2 * (n - 2));
    fine = (int)((T + cnt - 1) / cnt);
  }
  if (l1 < n) *a = fine << (2 * (n - 1 - l1));
  if (l0 > 0) *b = fine << (2 * (n - 1 - l0));
  *count = (int)(((long long)T + *a - 1) / *a) - (*b ? (int)(((long long)T + *b - 1) / *b) : 0);
}
// Sample r (ascending) of that window.
GPRM_EDGE_HD int edge_window_sample(int a, int b, int r) {
  if (b == 0) return r * a;
  const int k = b / a - 1;
  return a * (r + r / k + 1);
}
// Most samples an edge of at most maxT samples has in the window.
inline int edge_window_most(int maxT, int l1) {
  long long lim = l1 == 1 ? 16 : 256;
  for (int l = 3; l <= l1 && lim < maxT; ++l) lim = l == 3 ? 512 : lim * 4;
  return (int)(lim < maxT ? lim : maxT);
}
// Item slots of an edge with count samples in a window: runs of more than
// kRunShort samples start at and are padded to multiples of 16 (a row of
// lanes), so that a row's items are one edge's.
constexpr int kRunShort = 8;
GPRM_EDGE_HD long long edge_run_slots(int count) {
  return count > kRunShort ? (count + 15LL) / 16 * 16 : count;
}
// A compaction block takes at most edge_slice ranks of each of its edges,
// further blocks the next slices, because a run is written by 16 lanes: one
// edge's million samples by one block's row took milliseconds, several times
// their checks.  A slice is a multiple of 16, so that only an edge's last one
// is padded.  There are at most kSliceBlocks blocks, or 16 slices where the
// edges alone are many blocks: those of edges that are blocked or short find
// nothing to do, but 16,384 of them cost about 15 us.
constexpr int kSliceLeast = 1024;
constexpr long long kSliceBlocks = 2048;
inline int edge_slice(int ranks, long long xblocks) {
  const long long most = std::max(kSliceBlocks / std::max(xblocks, 1LL), 16LL);
  const long long s = std::max<long long>(kSliceLeast, (ranks + most - 1) / most);
  return ((int)std::min<long long>(s, std::max(ranks, 1)) + 15) & ~15;
}
inline int edge_slices(int ranks, long long xblocks) {
  const int s = edge_slice(ranks, xblocks);
  return ranks > s ? (int)(((long long)ranks + s - 1) / s) : 1;
}
// What the blocks of n edges with at most `ranks` ranks each pad their packed
// short runs by, at most.
inline long long edge_block_pads(long long n, int ranks, int block) {
  const long long x = (n + block - 1) / block;
  return 16 * x * edge_slices(ranks, x);
}
// Item capacity for n edges of at most `ranks` ranks each in blocks of
// `block` edges.
inline long long edge_items_cap(long long n, int ranks, int block) {
  return n * edge_run_slots(ranks) + edge_block_pads(n, ranks, block);
}

// One launch of an edge call: of the window [l0, l1) of edges [e0, e1), the
// ranks [r0, r1), at most cap items (whole groups of 64, also the frames'
// plane stride).
struct EdgeLaunch {
  int e0, e1, l0, l1, r0, r1, cap;
};

// The launches of a window over N edges of at most maxT samples, total in all
// (-1: unknown), for compaction blocks of `block` edges: at most about budget
// items each.  Where a single edge's samples are more, its ranks are cut; an
// edge may have up to 2^31 samples, and one launch for all of them would need
// 48 bytes of frames per joint and sample.
inline void edge_plan_window(long long budget, int block, int N, int l0, int l1, int maxT, long long total,
                             std::vector<EdgeLaunch>* plan) {
  const int most = edge_window_most(maxT, l1);
  const auto groups = [](long long items) { return (int)((items + 63) / 64 * 64); };
  long long cap = edge_items_cap(N, most, block);
  if (total >= 0)  // every run padded by at most 15
    cap = std::min(cap, total + 15LL * N + edge_block_pads(N, most, block));
  if (cap <= budget) {
    plan->push_back({0, N, l0, l1, 0, most, groups(cap)});
    return;
  }
  // (the blocks' padding is at most 1/64 of an edge of several slices, and 16)
  const int ranks = (int)std::min<long long>(most, std::max(16LL, (budget - 64) * 64 / 65 / 16 * 16));
  const int per =
      (int)std::max(1LL, (budget - 64) / (edge_run_slots(ranks) + 1 + (ranks > kSliceLeast ? ranks / 64 + 1 : 0)));
  for (int e0 = 0, e1; e0 < N; e0 = e1) {
    e1 = N - e0 < per ? N : e0 + per;
    for (long long r0 = 0; r0 < most; r0 += ranks) {
      const int r1 = (int)std::min<long long>(most, r0 + ranks);
      plan->push_back({e0, e1, l0, l1, (int)r0, r1, groups(edge_items_cap(e1 - e0, r1 - (int)r0, block))});
    }
  }
}

}  // namespace gprm

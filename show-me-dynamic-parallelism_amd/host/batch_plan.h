// Host-only: which workgroups of a small-graph batch's launch solve which graph.
//
// A graph that one workgroup would hold up the batch with, or cannot hold at
// all, is solved by a team of workgroups that meet at a barrier after every
// round.  A barrier waits a bounded time (about a second), so it must only
// ever wait for a round of its own graph: teams are disjoint sets of
// consecutive workgroups, every member of a team works through the same list
// of graphs in the same order, and no workgroup belongs to two.  (Clusters
// placed one by one on the least loaded workgroups overlapped in part, and a
// workgroup then waited for the whole solve of another graph: 20 paths of
// 490000 vertices at one vertex a round, 3 to 5 us each, left some waiting for
// two seconds.)
//
// Graphs are taken by falling arcs.  Each opens a team of the size it is worth
// while workgroups are left; after that it joins the list of a team that is
// large enough, the one that would end first.
#pragma once
#include <stdint.h>

#include <algorithm>
#include <cmath>
#include <numeric>
#include <vector>

namespace smdp {

// Clusters (teams that keep the distances in LDS) are worth their exchanges
// from 4 workgroups on (or where the vertices need more than one), up to one
// per kClusterArcs arcs; a graph that one workgroup holds is left to it below
// kClusterMin arcs.  Single graphs, k workgroups, us: 32768 x 16 (1: 286, 2:
// 373, 4: 286, 8: 311), 32768 x 32 (390, 564, 349, 327), 65536 x 8 (2: 431, 4:
// 335, 8: 347, 16: 447), 65536 x 32 (2: 1000, 4: 561, 8: 462, 16: 515).
constexpr int64_t kClusterArcs = int64_t(1) << 18;
constexpr int64_t kClusterMin = int64_t(1) << 20;
constexpr int64_t kClusterRound = 64;  // a cluster's workgroups own multiples of so many vertices
// Solves in memory: a graph of at most so many arcs is left to one workgroup (30
// graphs of 8000 arcs 0.13 ms, on teams of 8 0.21; of 32000 arcs 0.39 both).
constexpr int64_t kGroupMin = int64_t(1) << 14;
constexpr double kMemoryCost = 8.0;    // an arc of a solve in memory against one in LDS, for the load of a team

struct BatchLimits {
  int32_t lds_verts;    // vertices whose distances one workgroup's LDS holds
  int32_t max_cluster;  // workgroups of a cluster at most; 1: no clusters
  int32_t max_group;    // workgroups that solve a graph in memory together at most
  int32_t resident;     // workgroups that are resident at once
  int32_t workgroups;   // workgroups of the launch at most
  double share;         // arcs of a workgroup's fair share of the batch
};

struct BatchPlan {
  struct Item {
    int32_t graph;
    int32_t team;
    bool cluster;  // distances in LDS; otherwise in memory
  };
  std::vector<int32_t> base;    // per team, and one more: its first workgroup
  std::vector<Item> items;      // graphs solved by teams, each team's in this order
  std::vector<int32_t> single;  // graphs solved by one workgroup each, by falling arcs
  std::vector<uint8_t> lds;     // per graph: one workgroup solves it in LDS
  int32_t team_size(int32_t t) const { return base[(size_t)t + 1] - base[(size_t)t]; }
  int32_t workgroups() const { return base.back(); }
};

// Vertices that a workgroup of a cluster of k owns of a graph of n.
inline int64_t cluster_block(int64_t n, int64_t k) {
  return ((n + k - 1) / k + kClusterRound - 1) / kClusterRound * kClusterRound;
}

// fit[i]: graph i's weights and arcs suit a solve in LDS.
inline BatchPlan plan_batch(const std::vector<int32_t>& nv, const std::vector<int64_t>& m,
                            const std::vector<uint8_t>& fit, const BatchLimits& lim) {
  const int32_t ng = (int32_t)nv.size();
  BatchPlan p;
  p.base.push_back(0);
  p.lds.assign((size_t)ng, 0);
  std::vector<double> load;  // per team, in arcs of a solve in LDS
  std::vector<int32_t> order((size_t)ng);
  std::iota(order.begin(), order.end(), 0);
  std::stable_sort(order.begin(), order.end(), [&](int32_t x, int32_t y) { return m[(size_t)x] > m[(size_t)y]; });
  const double share = std::max(1.0, lim.share);
  // Solves in memory take whole shares of the launch where graphs are few, and
  // else only what is above the graphs' mean: shares rounded up then asked for
  // more workgroups than there are.  Graphs of 500 to 100000 vertices, ms, mean
  // rounded up / shares rounded down / up: 40 graphs 6.6 / 2.2 / 2.2, 100 3.9 /
  // 2.8 / 7.2, 150 4.3 / 4.2 / 8.7, 255 5.0 / 7.0 / 10.9.
  const bool few = 2 * (int64_t)ng < lim.workgroups;
  const double of_mean = share * lim.workgroups / std::max(1, std::min(ng, lim.workgroups));
  // Puts a graph on a new team of `want` workgroups, of the `least` that are
  // left, or on an existing team of at least that size.
  auto place = [&](int32_t gi, int64_t want, int64_t least, bool cluster) {
    const int64_t left = lim.resident - p.workgroups();
    auto cost = [&](int64_t size) {
      return (cluster ? 1.0 : kMemoryCost) * (double)m[(size_t)gi] / (double)size + (double)kClusterArcs;
    };
    int32_t team = -1;
    if (left >= least) {
      team = (int32_t)load.size();
      p.base.push_back((int32_t)(p.workgroups() + std::min(left, want)));
      load.push_back(0.0);
    } else {
      for (int32_t t = 0; t < (int32_t)load.size(); ++t) {
        const int32_t size = p.team_size(t);
        if (size < least || size > (cluster ? lim.max_cluster : lim.max_group)) continue;
        if (team < 0 || load[(size_t)t] + cost(size) < load[(size_t)team] + cost(p.team_size(team))) team = t;
      }
    }
    if (team < 0) return false;
    load[(size_t)team] += cost(p.team_size(team));
    p.items.push_back({gi, team, cluster});
    return true;
  };
  for (int32_t gi : order) {
    const int64_t n = nv[(size_t)gi], arcs = m[(size_t)gi];
    const int64_t shares = (int64_t)std::ceil((double)arcs / share);
    if (fit[(size_t)gi] && n <= (int64_t)lim.lds_verts * lim.max_cluster) {
      const int64_t least = std::max<int64_t>(1, (n + lim.lds_verts - 1) / lim.lds_verts);
      int64_t k = least;
      if (least > 1 || arcs >= kClusterMin)
        k = std::max(least, std::min<int64_t>({(int64_t)lim.max_cluster, shares, std::max<int64_t>(4, arcs / kClusterArcs)}));
      // (rounding may leave the last workgroups without vertices)
      if (n > 0) k = std::max(least, (n + cluster_block(n, k) - 1) / cluster_block(n, k));
      if (k >= 2 && place(gi, k, std::max<int64_t>(2, least), true)) continue;
      if (n <= lim.lds_verts) {
        p.lds[(size_t)gi] = 1;
        p.single.push_back(gi);
        continue;
      }
    }
    const int64_t k = std::min<int64_t>(lim.max_group, (int64_t)(few ? (double)arcs / share : std::ceil((double)arcs / of_mean)));
    if (k >= 2 && arcs > kGroupMin && place(gi, k, 2, false)) continue;
    p.single.push_back(gi);
  }
  return p;
}

}  // namespace smdp

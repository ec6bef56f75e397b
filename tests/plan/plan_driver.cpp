// Prints the work plan of a batch: reads "resident share max_cluster graphs"
// and then "vertices arcs fits" per graph; prints the teams' first workgroups,
// one line "item graph team cluster" per graph of a team, one line "single
// graph lds" per other graph.
#include <stdio.h>

#include "batch_plan.h"

int main() {
  int resident, cluster, ng;
  double share;
  if (scanf("%d %lf %d %d", &resident, &share, &cluster, &ng) != 4) return 1;
  std::vector<int32_t> nv(ng);
  std::vector<int64_t> m(ng);
  std::vector<uint8_t> fit(ng);
  for (int i = 0; i < ng; ++i) {
    long long arcs;
    int f;
    if (scanf("%d %lld %d", &nv[i], &arcs, &f) != 3) return 1;
    m[i] = arcs;
    fit[i] = (uint8_t)f;
  }
  const smdp::BatchPlan p = smdp::plan_batch(nv, m, fit, smdp::BatchLimits{32768, cluster, 16, resident, resident, share});
  printf("base");
  for (int32_t b : p.base) printf(" %d", b);
  printf("\n");
  for (const auto& it : p.items) printf("item %d %d %d\n", it.graph, it.team, it.cluster ? 1 : 0);
  for (int32_t g : p.single) printf("single %d %d\n", g, p.lds[g]);
  return 0;
}

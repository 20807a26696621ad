// Test harness of the grouping of batched Rips calls (specseqplusplus_amd/csrc/ssq_groups.h): sizes
// in, each cloud's group and the number of streams out.  Host only.
#include "../../specseqplusplus_amd/csrc/ssq_groups.h"

extern "C" int ssq_harness_groups(int count, const int64_t* n, const int64_t* edges, const int64_t* tris,
                                  int64_t mem_budget, int nstreams, int32_t* group_of, double* bytes, int32_t* workers) {
  std::vector<ssq::CloudSize> c((size_t)count);
  for (int i = 0; i < count; i++) {
    c[(size_t)i] = {n[i], edges[i], tris[i]};
    const int64_t w = (n[i] + 63) / 64;
    bytes[i] = ssq::group_bytes(n[i], edges[i], tris[i], n[i] * n[i], edges[i] * w, tris[i] / 16);
  }
  const ssq::GroupPlan p = ssq::plan_groups(c, mem_budget, nstreams);
  for (int i = 0; i < count; i++) group_of[i] = -1;
  for (size_t g = 0; g < p.groups.size(); g++)
    for (int i = p.groups[g].first; i < p.groups[g].second; i++) {
      int32_t& at = group_of[p.order[(size_t)i]];
      if (at >= 0) return 1;  // a cloud in two groups
      at = (int32_t)g;
    }
  *workers = p.workers;
  return 0;
}

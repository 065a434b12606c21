// The plan of an ILU(0) sweep under a bound on its merged rows' entries.
#include "../../sysu_cfd_parallel_amd/csrc/device/ilu_plan.hpp"

// out: groups, slots, rows below depth 0, hash of the row order
extern "C" int probe_plan(int n, const int* rowptr, const int* col, const int* diag, int upper, int levels,
                          long most_entries, long* out) {
  std::vector<int> order(n);
  for (int i = 0; i < n; ++i) order[i] = i;
  const s355::IluPlan p = s355::ilu_plan(n, rowptr, col, diag, upper != 0, order, {0, n}, levels, s355::kMergeRows,
                                         most_entries);
  long h = 0;
  for (int i : p.rows) h = h * 31 + i;
  for (size_t k = 0; k < p.col.size(); ++k) h = h * 31 + p.col[k] + 7L * p.src[k];
  out[0] = static_cast<long>(p.group.size()) - 1;
  out[1] = static_cast<long>(p.col.size());
  out[2] = static_cast<long>(p.later.size());
  out[3] = h;
  return 0;
}

// Runs an ILU(0) sweep by its plan on the host, in FP64, one group after the
// other and every row of a group from what stood before the group.
#include <cmath>
#include <utility>
#include <vector>

#include "../../sysu_cfd_parallel_amd/csrc/device/ilu_plan.hpp"

using s355::IluPlan;
using s355::IluSub;

// out: groups, slots, terms, widest padded row, rows below depth 0, order violations
extern "C" int probe_sweep(int n, const int* rowptr, const int* col, const int* diag, int upper, int ncase,
                           const int* cases, int levels, int rows, const int* order, const double* lu, const double* r,
                           double* z, long* out) {
  const IluPlan p = s355::ilu_plan(n, rowptr, col, diag, upper != 0, std::vector<int>(order, order + n),
                                   std::vector<int>(cases, cases + ncase + 1), levels, rows);
  std::vector<double> c(p.col.size(), 0.0), own(n, 1.0);
  auto at = [&](int q, int u) { return static_cast<size_t>(p.slot(q, u)); };
  auto scale = [&](int q) {
    if (!upper) return;
    const double d = lu[diag[p.rows[q]]];
    for (int u = 0; u < p.len[q]; ++u) c[at(q, u)] /= d;
    own[q] = 1.0 / d;
  };
  for (int q = 0; q < n; ++q) {
    for (int u = 0; u < p.len[q]; ++u) c[at(q, u)] = p.src[at(q, u)] >= 0 ? -lu[p.src[at(q, u)]] : 0.0;
    if (p.depth[q] == 0) scale(q);
  }
  for (size_t k = 0; k < p.later.size(); ++k) {
    for (int x = p.sptr[k]; x < p.sptr[k + 1]; ++x)
      for (int y = p.uptr[x]; y < p.uptr[x + 1]; ++y)
        c[p.r[y]] -= lu[p.p[x]] * (p.q[y] < 0 ? own[-1 - p.q[y]] : c[p.q[y]]);
    scale(p.later[k]);
  }
  std::vector<double> buf(2 * static_cast<size_t>(n), NAN);
  for (int i = 0; i < n; ++i) buf[p.pos[i]] = r[i];
  long bad = 0, widest = 0, terms = 0;
  for (size_t g = 0; g + 1 < p.group.size(); ++g) {
    std::vector<std::pair<int, double>> res;
    for (int s = p.group[g]; s < p.group[g + 1]; ++s) {
      const IluSub& sub = p.subs[s];
      widest = sub.width > widest ? sub.width : widest;
      if (s > p.group[g] && sub.cls <= p.subs[s - 1].cls) ++bad;
      const int lanes = s355::kTermLanes[sub.cls];
      if (sub.cls + 1 < s355::kTermClasses ? sub.width != s355::kTermWidth[sub.cls]
                                           : sub.width % (lanes * s355::kTermBatch))
        ++bad;
      const bool even = sub.cls < 4 || sub.cls == 6 || sub.width % lanes == 0;
      for (int k = 0; k < sub.nrows; ++k) {
        const int q = sub.p0 + k;
        if (p.slot0[q] != sub.off + k * lanes || p.lanes[q] != lanes || p.stride[q] != sub.nrows * lanes ||
            p.len[q] > sub.width || !even)
          ++bad;
        double v = own[q] * buf[q];
        for (int u = 0; u < sub.width; ++u) {
          const int b = p.col[at(q, u)];
          if (b < 0 || b >= 2 * n || std::isnan(buf[b])) ++bad;
          if (u < p.len[q]) v += c[at(q, u)] * buf[b];
        }
        terms += p.len[q];
        res.emplace_back(q, v);
      }
    }
    for (const auto& x : res) buf[n + x.first] = x.second;
  }
  for (int i = 0; i < n; ++i) z[i] = buf[n + p.pos[i]];
  const long o[] = {static_cast<long>(p.group.size()) - 1, static_cast<long>(p.col.size()), terms, widest,
                    static_cast<long>(p.later.size()), bad};
  for (int k = 0; k < 6; ++k) out[k] = o[k];
  return 0;
}

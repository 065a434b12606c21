#include "ilu_plan.hpp"

#include <sys/mman.h>

#include <algorithm>
#include <memory>
#include <new>
#include <stdexcept>

#include "../mesh/parallel.hpp"

namespace s355 {
namespace {

constexpr long kMost = 0x7fffffffL;
constexpr size_t kHuge = size_t(1) << 21;

}  // namespace

void IntArray::resize(size_t m) {
  const size_t bytes = std::max<size_t>(m, 1) * sizeof(int);
  const bool huge = bytes >= 2 * kHuge;
  int* q = static_cast<int*>(huge ? std::aligned_alloc(kHuge, (bytes + kHuge - 1) / kHuge * kHuge) : std::malloc(bytes));
  if (!q) throw std::bad_alloc();
  if (huge) madvise(q, bytes, MADV_HUGEPAGE);
  p.reset(q);
  n = m;
}

namespace {

// a table of the plan would pass its bound
struct TooLarge : std::invalid_argument {
  using std::invalid_argument::invalid_argument;
};

IluPlan build(int n, const int* rowptr, const int* col, const int* diag, bool upper,
              const std::function<const std::vector<int>&()>& order, const std::vector<int>& cases, int merge_levels,
              int merge_rows, long most_entries, const std::function<void(const std::vector<int>&)>& known) {
  if (n > kMost / 2) throw std::invalid_argument("ILU(0) sweeps above 32-bit indices");
  if (merge_levels < 1 || merge_levels > kMergeLevels) throw std::invalid_argument("ilu_plan: merge_levels");
  IluPlan out;
  out.n = n;
  auto first = [&](int i) { return upper ? diag[i] + 1 : rowptr[i]; };
  auto last = [&](int i) { return upper ? rowptr[i + 1] : diag[i]; };

  IntArray lev, grp, dep, most, width_of;
  for (IntArray* x : {&lev, &grp, &dep, &most, &width_of}) x->resize(n);
  // most: terms of a row at most, its own input among them
  for (int k = 0; k < n; ++k) {
    const int i = upper ? n - 1 - k : k;
    int l = 0;
    for (int e = first(i); e < last(i); ++e) l = std::max(l, lev[col[e]] + 1);
    lev[i] = l;
  }
  // groups, case by case; dlist: the rows of each depth
  std::vector<std::vector<int>> dlist(merge_levels);
  int ngroup = 0;
  for (size_t c = 0; c + 1 < cases.size(); ++c) {
    const int a = cases[c], e = cases[c + 1];
    if (e <= a) continue;
    int nlev = 0;
    for (int i = a; i < e; ++i) nlev = std::max(nlev, lev[i] + 1);
    std::vector<int> lptr(nlev + 1, 0), lrows(e - a);
    for (int i = a; i < e; ++i) ++lptr[lev[i] + 1];
    for (int l = 0; l < nlev; ++l) lptr[l + 1] += lptr[l];
    {
      std::vector<int> at(lptr.begin(), lptr.end() - 1);
      for (int i = a; i < e; ++i) lrows[at[lev[i]]++] = i;
    }
    int g = -1, begin = 0;  // the open group and its first level
    for (int l = 0; l < nlev; ++l) {
      bool joins = g >= 0 && l - begin < merge_levels && lptr[l + 1] - lptr[begin] <= merge_rows;
      for (int k = lptr[l]; joins && k < lptr[l + 1]; ++k) {
        const int i = lrows[k];
        int m = 1;
        for (int x = first(i); x < last(i); ++x) m += lev[col[x]] >= begin ? most[col[x]] : 1;
        most[i] = m;
        joins = m <= kMergeTerms;
      }
      if (!joins) {
        ++g;
        begin = l;
        for (int k = lptr[l]; k < lptr[l + 1]; ++k) most[lrows[k]] = 1 + last(lrows[k]) - first(lrows[k]);
      }
      const int d = l - begin;
      for (int k = lptr[l]; k < lptr[l + 1]; ++k) {
        grp[lrows[k]] = g;
        dep[lrows[k]] = d;
      }
      dlist[d].insert(dlist[d].end(), lrows.begin() + lptr[l], lrows.begin() + lptr[l + 1]);
    }
    ngroup = std::max(ngroup, g + 1);
  }

  // the terms of every row, depth by depth.  Code j: the input of row j, n + j:
  // the result of row j.  Row i's terms are at its start, count of them; so
  // are, for a row below depth 0, its pairs (term of the row, term of the row
  // referred to, -1 its own input), one run per reference in CSR order.
  // (what another row reads of a row stands together: the loops wait for memory)
  struct Row {
    long start;
    int grp, count;
  };
  std::vector<Row> row(n);
  long entries = 0;
  for (int i = 0; i < n; ++i) {
    row[i] = Row{entries, grp[i], 0};
    entries += most[i];
  }
  if (merge_levels > 1 && entries > most_entries) throw TooLarge("ILU(0) merged rows");
  IntArray code, src, pr, pq;
  for (IntArray* x : {&code, &src, &pr, &pq}) x->resize(entries);
  IntArray nstep, npair, key;  // key: group and class of terms
  for (IntArray* x : {&nstep, &npair, &key}) x->resize(n);
  for (int d = 0; d < merge_levels; ++d) {
    const std::vector<int>& list = dlist[d];
    parallel_for(
        static_cast<long>(list.size()),
        [&](long k) {
          const int i = list[k];
          const long s = row[i].start;
          const int g = row[i].grp;
          int m = 0, pairs = 0, steps = 0;
          int* const codes = code.data() + s;
          // the term of code c, looked for among the first `before` (the codes of
          // one reference differ from each other)
          auto term = [&](int c, int before) {
            int u = -1;
            for (int v = 0; v < before; ++v) u = std::max(u, codes[v] == c ? v : -1);
            if (u >= 0) return u;
            codes[m] = c;
            src[s + m] = -1;
            return m++;
          };
          for (int x = first(i); x < last(i); ++x) {
            const int j = col[x];
            const Row from = row[j];
            if (from.grp != g) {
              src[s + term(n + j, m)] = x;
              continue;
            }
            ++steps;
            const int before = m;
            for (int y = -1; y < from.count; ++y) {  // -1: row j's own input
              pr[s + pairs] = term(y < 0 ? j : code[from.start + y], before);
              pq[s + pairs] = y;
              ++pairs;
            }
          }
          row[i].count = m;
          nstep[i] = steps;
          npair[i] = pairs;
          int c = 0;
          while (m > kTermWidth[c]) ++c;
          key[i] = g * kTermClasses + c;
        },
        1 << 12);
  }

  // sweep order: by (group, class), keeping the order given
  const long nkey = static_cast<long>(ngroup) * kTermClasses;
  std::vector<int> kptr(nkey + 1, 0), width(nkey, 0);
  for (int i = 0; i < n; ++i) {
    const int k = key[i];
    ++kptr[k + 1];
    width[k] = std::max(width[k], row[i].count);
  }
  for (long k = 0; k < nkey; ++k) kptr[k + 1] += kptr[k];
  out.rows.resize(n);
  out.pos.resize(n);
  {
    std::vector<int> at(kptr.begin(), kptr.end() - 1);
    for (int i : order()) {
      const int p = at[key[i]]++;
      out.rows[p] = i;
      out.pos[i] = p;
    }
  }
  if (known) known(out.rows);
  long slots = 0;
  out.group.assign(1, 0);
  out.len.resize(n);
  out.slot0.resize(n);
  out.lanes.resize(n);
  out.stride.resize(n);
  out.depth.resize(n);
  for (int g = 0; g < ngroup; ++g) {
    for (int c = 0; c < kTermClasses; ++c) {
      const long k = static_cast<long>(g) * kTermClasses + c;
      const int p0 = kptr[k], nr = kptr[k + 1] - p0;
      if (nr == 0) continue;
      const int lanes = kTermLanes[c], batch = kTermBatch * lanes;
      if (c + 1 < kTermClasses)
        width[k] = kTermWidth[c];
      else
        width[k] = (width[k] + batch - 1) / batch * batch;
      out.subs.push_back(IluSub{slots, p0, nr, width[k], c});
      if (slots + static_cast<long>(width[k]) * nr > kMost) throw TooLarge("ILU(0) sweep slots above 32-bit indices");
      for (int p = p0; p < p0 + nr; ++p) {
        out.slot0[p] = static_cast<int>(slots + static_cast<long>(p - p0) * lanes);
        out.lanes[p] = lanes;
        width_of[p] = width[k];
        out.stride[p] = nr * lanes;
      }
      slots += static_cast<long>(width[k]) * nr;
    }
    out.group.push_back(static_cast<int>(out.subs.size()));
  }
  out.col.resize(slots);
  out.src.resize(slots);
  struct Place {
    int pos, slot0, stride, shift;  // (lanes: 1 << shift)
    int slot(int u) const { return slot0 + (u >> shift) * stride + (u & ((1 << shift) - 1)); }
  };
  std::vector<Place> place(n);
  parallel_for(
      n,
      [&](long k) {
        const int p = static_cast<int>(k), i = out.rows[p];
        const Row own = row[i];
        const int lanes = out.lanes[p];
        const Place at_p{p, out.slot0[p], out.stride[p], lanes == 1 ? 0 : lanes == 4 ? 2 : 4};
        place[i] = at_p;
        out.len[p] = own.count;
        out.depth[p] = dep[i];
        for (int u = 0; u < width_of[p]; ++u) {
          const int at = at_p.slot(u);
          if (u < own.count) {
            const int c = code[own.start + u];
            out.col[at] = c < n ? out.pos[c] : n + out.pos[c - n];
            out.src[at] = src[own.start + u];
          } else {
            out.col[at] = p;
            out.src[at] = -1;
          }
        }
      },
      1 << 13);

  // the steps of the rows below depth 0
  out.dptr.assign(1, 0);
  for (int d = 1; d < merge_levels; ++d)
    out.dptr.push_back(out.dptr.back() + static_cast<int>(dlist[d].size()));
  out.later.resize(out.dptr.back());
  {
    std::vector<int> at(out.dptr);
    for (int p = 0; p < n; ++p)
      if (out.depth[p]) out.later[at[out.depth[p] - 1]++] = p;
  }
  const size_t nl = out.later.size();
  out.sptr.assign(nl + 1, 0);
  std::vector<long> pairs(nl + 1, 0);
  long steps = 0;
  for (size_t k = 0; k < nl; ++k) {
    const int i = out.rows[out.later[k]];
    steps += nstep[i];
    pairs[k + 1] = pairs[k] + npair[i];
    if (steps > kMost || pairs[k + 1] > kMost) throw TooLarge("ILU(0) sweep steps above 32-bit indices");
    out.sptr[k + 1] = static_cast<int>(steps);
  }
  out.p.resize(steps);
  out.uptr.resize(static_cast<size_t>(steps) + 1);
  out.uptr[0] = 0;
  out.r.resize(pairs[nl]);
  out.q.resize(pairs[nl]);
  parallel_for(
      static_cast<long>(nl),
      [&](long k) {
        const int i = out.rows[out.later[k]];
        const Place to = place[i];
        const int g = row[i].grp;
        int x0 = out.sptr[k];
        long at = pairs[k], from = row[i].start;
        for (int x = first(i); x < last(i); ++x) {
          const int j = col[x];
          if (row[j].grp != g) continue;
          const Place by = place[j];
          out.p[x0] = x;
          for (int y = -1; y < row[j].count; ++y, ++at, ++from) {
            out.r[at] = to.slot(pr[from]);
            out.q[at] = pq[from] < 0 ? -1 - by.pos : by.slot(pq[from]);
          }
          out.uptr[++x0] = static_cast<int>(at);
        }
      },
      1 << 12);
  return out;
}

}  // namespace

IluPlan ilu_plan(int n, const int* rowptr, const int* col, const int* diag, bool upper,
                 const std::function<const std::vector<int>&()>& order, const std::vector<int>& cases, int merge_levels,
                 int merge_rows, long most_entries, const std::function<void(const std::vector<int>&)>& known) {
  try {
    return build(n, rowptr, col, diag, upper, order, cases, merge_levels, merge_rows, most_entries, known);
  } catch (const TooLarge&) {
    if (merge_levels == 1) throw;
    return build(n, rowptr, col, diag, upper, order, cases, 1, merge_rows, most_entries, known);
  }
}

}  // namespace s355

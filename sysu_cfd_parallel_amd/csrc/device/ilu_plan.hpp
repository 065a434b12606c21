// Host plan of the ILU(0) sweeps: which rows go in one launch, and what each
// of them sums.
#pragma once
#include <vector>

namespace s355 {

// A triangular sweep takes its rows level by level (a row depends only on rows
// of earlier levels), and a level of a few thousand rows costs a launch and
// a chain of dependent loads, whatever its bytes.  So up to kMergeLevels
// consecutive levels form a group that one launch completes: a row's
// references to rows of its own group are replaced by what those rows are
// sums of, until every term is an input of the sweep or a result of an
// earlier group,
//
//   z_i = (r_i - sum_j a_ij z_j) / d_i = o_i r_i + sum_t c_t buf[col_t],
//
// buf holding the n inputs followed by the n results, both in sweep order
// (o_i = 1 / d_i; d_i = 1 in the lower sweep).  The coefficients are formed once per
// factorisation, the pattern here once per matrix pattern.
//
// A group ends where it would pass kMergeRows rows (such launches are bound by
// bytes, and merged rows read more of them) or where a row could pass
// kMergeTerms terms (counted without looking for equal ones).  Pressure solves
// (CG, 331,776 tetrahedra, FP64, 54 levels; mixed GMRES, 310,000 hexahedra, 134
// levels) by levels, rows and terms: no merging 131.7 and 162.3 ms; 2, 49152,
// 64: 98.7 and 112.1; 4, 49152, 64: 75.9 and 94.2; 4, 24576, 64: 82.5 and 94.3;
// 6, 49152, 96: 72.3 and 84.7; 6, 131072, 160: 71.9 and 81.2; 8, 131072, 300:
// 74.6 and 74.4.  With 6, 65536, 96 and the row's own input out of the terms:
// 64.8 and 81.8.  Each case of a
// batch is grouped by its own rows, so it sums the same terms in the same
// order as alone.
constexpr int kMergeLevels = 6;
constexpr int kMergeTerms = 96;
constexpr int kMergeRows = 65536;
// Rows of a launch come in classes of term counts, each padded to a width the
// kernel is compiled for; the last takes what is longer, padded to batches.
constexpr int kTermWidth[] = {3, 6, 10, 15, 22, 32, 1 << 30};
constexpr int kTermClasses = 7;
constexpr int kNarrowClasses = 3;  // a launch without wider rows takes a kernel of fewer registers
constexpr int kTermBatch = 16;

// rows of one group and class of term counts
struct IluSub {
  long off;  // first slot; term u of the k-th row at off + u nrows + k
  int p0, nrows, width, cls;
};

struct IluPlan {
  int n = 0;
  std::vector<int> rows;     // sweep order: by group, class, then the order given
  std::vector<int> pos;      // position of each row
  std::vector<IluSub> subs;  // in sweep order
  std::vector<int> group;    // group g: subs group[g] .. group[g + 1] - 1
  std::vector<int> len;      // terms per position (the row's own input, o_i r_i, is not among them)
  std::vector<int> depth;    // per position: 0 where no entry refers to the row's own group
  std::vector<int> slot0, stride;  // per position: its first slot, the distance of its terms
  // per slot: buf index (padding: the row's own input), and where its
  // coefficient starts from: the CSR entry a_ij (coefficient -a_ij) or -1 (0)
  std::vector<int> col, src;
  // rows below depth 0 by depth: positions later[dptr[d - 1]] .. dptr[d] - 1;
  // the k-th has steps sptr[k] .. : entry p of the matrix times the row
  // it refers to, c[r] -= a_p c[q] over pairs uptr[step] .. (q < 0: the own
  // coefficient of position -1 - q)
  std::vector<int> dptr, later, sptr, p, uptr, r, q;
};

// The plan of the lower (strictly lower entries) or upper sweep of a CSR
// pattern with sorted columns; order is the order rows keep inside a group
// and class, cases the first row of each case and n.  Throws
// std::invalid_argument where a table passes 32-bit indices.
IluPlan ilu_plan(int n, const int* rowptr, const int* col, const int* diag, bool upper, const std::vector<int>& order,
                 const std::vector<int>& cases, int merge_levels = kMergeLevels, int merge_rows = kMergeRows);

}  // namespace s355

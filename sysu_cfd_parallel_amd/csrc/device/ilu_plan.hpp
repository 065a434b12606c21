// Host plan of the ILU(0) sweeps: which rows go in one launch, and what each
// of them sums.
#pragma once
#include <cstddef>
#include <cstdlib>
#include <functional>
#include <memory>
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
// kMergeTerms terms (counted without looking for equal ones).  One build, four
// repeated passes: pressure solves by CG on 331,776 tetrahedra in FP64 (54 levels)
// and mixed GMRES(50) on 310,000 hexahedra (134 levels), a momentum phase with its
// factorisation on the tetrahedra, a pressure solve of 512 cavities of 16^3 as a
// batch in FP64, ms:
//   levels, terms   CG     GMRES  momentum  batch
//    1              154.6  139.1  7.7       22.2
//    4,  200         73.6   45.4  4.4       21.1
//    6,  100         62.1   43.1  4.1       21.2
//    8,   60         64.3   52.9  4.1       20.7
//    8,  100         59.7   42.6  4.0       21.2
//    8,  200         56.8   38.1  3.9       22.1
//    8,  300         56.8   35.4  3.9       22.7
//   12,  300         54.0   34.6  3.9       22.7
//   16, 1000         51.7   32.3  4.0       25.1
// (65,536 rows).  Taken: 8, 200; what more terms give a single case a batch loses,
// whose launches are bound by the gathers, and the plan grows (first GMRES solve
// 136 ms at 8, 200, 183 at 16, 1000).  By rows at 8, 200, the same two solves and
// those of 1,119,744 tetrahedra and 1,008,000 hexahedra: 8,192 84.9, 67.1, 191.5,
// 248.0; 16,384 78.3, 43.4, 188.8, 216.4; 32,768 70.1, 38.1, 179.4, 145.0; 65,536
// 56.8, 38.1, 168.6, 127.5; 131,072 56.7, 38.1, 170.7, 127.9; 262,144 54.9, 38.1, 158.3,
// 127.6.  Nothing is gained on hexahedra above 65,536, and the plan of the large
// tetrahedra costs 110 ms more for 10 a solve.
constexpr int kMergeLevels = 8;
constexpr int kMergeTerms = 200;
constexpr int kMergeRows = 65536;
// Entries that the merged rows of one plan may have, counted without looking for
// equal ones: 16 bytes each while the plan is built, so 16 GB, and 32-bit indices
// hold the tables.  Long thin meshes, whose levels are small however many
// rows they have, come there (a duct of 4000 x 32 x 32 hexahedra has 35 entries a row).
constexpr long kMergeEntries = 1L << 30;
// Rows of a launch come in classes of term counts, each padded to a width the
// kernel is compiled for.  A row of many terms is shared by 4 or 16 lanes, so
// that no lane's chain of loads is longer than one batch; the last class takes
// what is longer still, in batches of kTermBatch per lane.
constexpr int kTermWidth[] = {3, 6, 10, 15, 32, 64, 1 << 30};
constexpr int kTermLanes[] = {1, 1, 1, 1, 4, 4, 16};
constexpr int kTermClasses = 7;
constexpr int kNarrowClasses = 3;  // a launch without wider rows takes a kernel of fewer registers
constexpr int kTermBatch = 16;

// rows of one group and class of term counts, lanes = kTermLanes[cls] to a row
struct IluSub {
  long off;  // first slot; term u of the k-th row at off + (u / lanes) lanes nrows + k lanes + u % lanes
  int p0, nrows, width, cls;
};

// n ints that are written before they are read (a vector would first fill them).
// Large ones ask for 2 MiB pages: the plan of 331,776 tetrahedra touches some 80 MB
// for the first time, by 4 KiB pages from many threads at once.
struct IntArray {
  using value_type = int;
  struct Free {
    void operator()(int* q) const { std::free(q); }
  };
  std::unique_ptr<int[], Free> p;
  size_t n = 0;
  void resize(size_t m);
  size_t size() const { return n; }
  bool empty() const { return n == 0; }
  int* data() { return p.get(); }
  const int* data() const { return p.get(); }
  int& operator[](size_t i) { return p[i]; }
  int operator[](size_t i) const { return p[i]; }
};

struct IluPlan {
  int n = 0;
  std::vector<int> rows;     // sweep order: by group, class, then the order given
  std::vector<int> pos;      // position of each row
  std::vector<IluSub> subs;  // in sweep order
  std::vector<int> group;    // group g: subs group[g] .. group[g + 1] - 1
  std::vector<int> len;      // terms per position (the row's own input, o_i r_i, is not among them)
  std::vector<int> depth;    // per position: 0 where no entry refers to the row's own group
  // per position: its first slot, its lanes, the distance of its terms of one lane
  std::vector<int> slot0, lanes, stride;
  int slot(int q, int u) const {  // (lanes: 1, 4 or 16)
    const int shift = lanes[q] == 1 ? 0 : lanes[q] == 4 ? 2 : 4;
    return slot0[q] + (u >> shift) * stride[q] + (u & (lanes[q] - 1));
  }
  // per slot: buf index (padding: the row's own input), and where its
  // coefficient starts from: the CSR entry a_ij (coefficient -a_ij) or -1 (0)
  IntArray col, src;
  // rows below depth 0 by depth: positions later[dptr[d - 1]] .. dptr[d] - 1;
  // the k-th has steps sptr[k] .. : entry p of the matrix times the row
  // it refers to, c[r] -= a_p c[q] over pairs uptr[step] .. (q < 0: the own
  // coefficient of position -1 - q)
  std::vector<int> dptr, later, sptr;
  IntArray p, uptr, r, q;
};

// The plan of the lower (strictly lower entries) or upper sweep of a CSR
// pattern with sorted columns; order is the order rows keep inside a group
// and class (as a function: asked for once the terms are known, so that the upper
// sweep's, the lower plan's rows, can be built at the same time; known is called
// with a plan's rows as soon as they are ordered), cases the first row of each
// case and n.  Where merged rows would take more than
// most_entries entries, or a table passes 32-bit indices, nothing is merged; throws
// std::invalid_argument where a table passes them all the same.
IluPlan ilu_plan(int n, const int* rowptr, const int* col, const int* diag, bool upper,
                 const std::function<const std::vector<int>&()>& order, const std::vector<int>& cases,
                 int merge_levels = kMergeLevels, int merge_rows = kMergeRows, long most_entries = kMergeEntries,
                 const std::function<void(const std::vector<int>&)>& known = {});
inline IluPlan ilu_plan(int n, const int* rowptr, const int* col, const int* diag, bool upper,
                        const std::vector<int>& order, const std::vector<int>& cases,
                        int merge_levels = kMergeLevels, int merge_rows = kMergeRows,
                        long most_entries = kMergeEntries) {
  return ilu_plan(
      n, rowptr, col, diag, upper, [&]() -> const std::vector<int>& { return order; }, cases, merge_levels, merge_rows,
      most_entries);
}

}  // namespace s355

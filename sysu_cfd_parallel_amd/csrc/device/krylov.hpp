// Device Krylov solvers standing in for PETSc KSPSolve (MPIStructure.cpp:273,
// 311, 345, 424, 502): restarted GMRES(m) with left preconditioning and
// classical Gram-Schmidt, and preconditioned CG, both with PETSc's default
// convergence test (KSPConvergedDefault).  Vectors and matrix values are of
// type T (double, or float for the mixed-precision inner solves); the
// Hessenberg least-squares problem is always solved in FP64.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <functional>
#include <map>
#include <vector>

#include "../../../include/simple355.h"
#include "common.hpp"
#include "ilu_plan.hpp"

namespace s355 {

constexpr int kMaxRestart = 64;

// Solver state kept on the device so that kernels can stop themselves once
// the test has passed; the host reads the header every few iterations.
// One state per case of a batched solve, stored contiguously.
struct KState {
  int it;      // completed iterations in the current cycle
  int its;     // completed iterations in total
  int reason;  // 0 running, > 0 converged, < 0 diverged (KSPConvergedReason)
  int maxit;
  int done;    // the case's solve has ended (reason final)
  int cycles;  // restart cycles started
  int ended;   // reason as the last multi-dot found it (see k_orth)
  int pad0;
  double rnorm, rnorm0, ttol, snorm;
  double rtol, abstol, dtol;
  double pad;
  double H[(kMaxRestart + 1) * (kMaxRestart + 1)];  // column-major, H(r,c) = H[c*(m+1)+r]
  double cc[kMaxRestart + 1], ss[kMaxRestart + 1], grs[kMaxRestart + 2];
  double scale[kMaxRestart + 1];  // basis vector k = scale[k] * V[k]
  double hcol[2][kMaxRestart + 1];  // Hessenberg column of step it in hcol[it & 1]
  double y[kMaxRestart + 1];
  // CG scalars
  double beta, betaold, dpi, dpiold, alpha;
};

struct KHeader {
  int it, its, reason, maxit, done, cycles, ended, pad0;
  double rnorm, rnorm0, ttol, snorm;
};
static_assert(offsetof(KState, rnorm) == offsetof(KHeader, rnorm), "KHeader mirrors the head of KState");

// Where the solver kernels leave the headers for the host: coherent pinned memory
// (host, arrived), the count of messages sent (device) and arrived.  One per set
// of states; the solves of a context run one after the other on its stream.
struct Mailbox {
  KHeader* host = nullptr;
  unsigned* arrived = nullptr;
  unsigned* sent = nullptr;
};

template <class T>
struct CsrView {
  int n = 0;
  const int* rowptr = nullptr;
  const int* col = nullptr;
  const int* diag = nullptr;
  const T* val = nullptr;
  int nnz = 0;
};

// Sliced ELL (SELL-64-sigma) copy of a CSR matrix for the SpMV: within each
// window of sigma consecutive rows the rows are ordered by decreasing length
// (stable), then cut into slices of 64, one row per lane; slice s holds
// width_s = its longest row's length columns stored column-major (entry j of
// slot row 64 s + l at ptr[s] + 64 j + l), shorter rows padded with zero
// values and their own column; row[64 s + l] is the matrix row it holds.
// Every lane then has all its row's loads independent and in flight, a
// wave's loads are contiguous, and sorting by length keeps the padding small
// on meshes that mix tetrahedra, hexahedra and polyhedra.  Entries keep the
// CSR order within a row.
template <class T>
struct SellView {
  int n = 0;
  const int* ptr = nullptr;    // nslice + 1 offsets
  const int* row = nullptr;    // n: matrix row of each slot row (null: the slot row itself)
  const int* col = nullptr;
  const int16_t* col16 = nullptr;  // set: column = row + col16 (16-bit offsets, no col)
  const T* val = nullptr;
  const int* scase = nullptr;  // batches: case of each slice, -1 when its rows span two cases
  int two = 0;                 // FP32, one case: two slices per wave
  bool tiled = false;          // the rows of 256 positions are 256 consecutive rows
};

// SELL windows the autotuner chooses from: a short window keeps the rows of
// a slice (and so their gathers of x) close together, a long one removes the
// padding of meshes mixing row lengths.
constexpr int kSellVariants = 3;
constexpr int kSellSigma[kSellVariants] = {64, 512, 4096};
constexpr int kSellDefault = 2;

// one SELL pattern on the device (values live with each precision's workspace)
struct SellPat {
  const int* ptr = nullptr;
  const int* row = nullptr;
  const int* col = nullptr;
  const int16_t* col16 = nullptr;  // the columns as offsets from the slot's row (see sell_offsets16)
  const int* src = nullptr;
  const int* scase = nullptr;  // batches only (see SellView)
  size_t slots = 0;
};

// Host construction of the pattern: ptr, row, col and, for every SELL slot,
// the CSR position it copies (-1 for padding).
void sell_pattern(int n, const int* rowptr, const int* col, int sigma, std::vector<int>& ptr, std::vector<int>& srow,
                  std::vector<int>& scol, std::vector<int>& src);

// The columns of a SELL pattern as 16-bit offsets from each slot's row
// (padding and the slots past the last row: 0).  Returns false when an
// offset does not fit in 16 bits.
bool sell_offsets16(int n, const std::vector<int>& ptr, const std::vector<int>& srow, const std::vector<int>& scol,
                    std::vector<int16_t>& off);

// FP32 values of a CSR by position: entry k of position p's row is
// val[src[k]], divided by the diagonal of the natural row row_nat[p] (its
// Jacobi scaling, 1 for a zero diagonal) when jacobi is set.
void fill_ordered(int n, const int* rowptr, const int* src, const int* row_nat, const int* diag_nat,
                  const double* val, bool jacobi, float* out, hipStream_t s);

// out[q] = csr_val[src[q]] (0 where src[q] < 0), converted to T.
template <class T, class S>
void sell_fill(const int* src, size_t nslots, const S* csr_val, T* out, hipStream_t s);

// The ILU(0) preconditioner (natural ordering).  The factorisation takes
// the rows level by level (rows of a level depend only on rows of earlier
// levels); the sweeps take them by the groups of ilu_plan.hpp, each sweep on a
// buffer of its n inputs and n results in its own row order.  One pass over
// the whole vector moves r into the lower order, one moves the lower
// result into the upper order and one moves z back into the natural order.

// one sweep's plan: what the launches need on the host, the rest on the device
// (names as in IluPlan)
struct IluSweep {
  int n = 0;
  std::vector<IluSub> subs;
  std::vector<int> group, dptr;
  size_t slots = 0;
  const int *len = nullptr, *slot0 = nullptr, *lanes = nullptr, *stride = nullptr, *col = nullptr, *src = nullptr;
  const int *later = nullptr, *sptr = nullptr, *p = nullptr, *uptr = nullptr, *r = nullptr, *q = nullptr;
  // upper sweep: CSR position of the pivot of the row at each position at
  // depth 0, and -1 minus it below
  const int* dsrc = nullptr;
  const int* rcase = nullptr;  // batches: the case of the row at each position
};

// The elimination steps of ILU(0) per row, rows by level: row
// position t has steps ptr[t] .. ptr[t+1]-1; step s divides the lower entry
// p[s] by the pivot d[s] (the diagonal of row col[p]) and then applies the
// slot pairs u[s] .. u[s+1]-1: lu[r] -= l * lu[q].
struct IluSteps {
  const int* ptr = nullptr;
  const int* p = nullptr;
  const int* d = nullptr;
  const int* u = nullptr;  // nsteps + 1
  const int* r = nullptr;
  const int* q = nullptr;
};

struct IluLevels {
  std::vector<int> lptr;        // host: level boundaries of the factorisation's rows
  const int* lpos = nullptr;    // device: lower-sweep position of each row
  const int* l2u = nullptr;     // device: upper-sweep position of the row at each lower position
  const int* upos = nullptr;    // device: upper-sweep position of each row
  IluSweep lower, upper;
  IluSteps steps;
  int nl() const { return static_cast<int>(lptr.size()) - 1; }
};

// Host construction of the elimination steps (rows in the order of rows).
void ilu_steps(int n, const int* rowptr, const int* col, const int* diag, const std::vector<int>& rows,
               std::vector<int>& ptr, std::vector<int>& p, std::vector<int>& d, std::vector<int>& u,
               std::vector<int>& r, std::vector<int>& q);

// Host computation of the factorisation's levels: the rows by level, in their
// natural order inside one.
void ilu_levels(int n, const int* rowptr, const int* col, const int* diag, std::vector<int>& rows,
                std::vector<int>& ptr);

struct KResult {
  int iters = 0, reason = 0;
  double rnorm = 0, rnorm0 = 0;
  int refinements = 0;
};

// Instantiated hipGraphs of GMRES restart cycles, keyed by everything their
// kernel arguments depend on; destroyed with the cache.
struct GraphCache {
  std::map<std::vector<uintptr_t>, hipGraphExec_t> execs;
  ~GraphCache();
  hipGraphExec_t get(const std::vector<uintptr_t>& key, hipStream_t s, const std::function<void()>& record);
};

// Timings taken by autotune(): SpMV per variant v = 2 k + nt (k = 0..4: CSR
// with 1, 2, 4, 8, 16 lanes per row, k = 5..7: SELL-64 with window 64, 512,
// 4096; nt: non-temporal matrix loads) and one Gram-Schmidt step (multi-dot +
// update at iteration gs_it) per rows-per-thread 1, 2, 4, 8, 16; -1 = not timed.
// One case of at most kBlock tiles: the product with its dots, and the rest of
// the step, in the one shape such a system takes.
struct TuneReport {
  // CSR lanes 1, 2, 4, 8, 16 then SELL-64 with windows 64, 512, 4096, each
  // temporal / non-temporal
  double spmv_ms[16] = {-1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1};
  double gs_ms[5] = {-1, -1, -1, -1, -1};
  int gs_it = 0;
};

// Device time of the production SpMV launches inside GMRES solves: every
// `every`-th Arnoldi SpMV is bracketed by a pair of HIP events on the solve's
// stream (no synchronisation is added); harvest() reads the pairs once the
// stream has passed them.  Launch-by-launch solves only.
struct SpmvTimer {
  int every = 4;
  long seen = 0, count = 0;
  double total_ms = 0.0;
  std::vector<hipEvent_t> pool;  // pairs
  size_t used = 0;
  ~SpmvTimer();
  bool take(hipEvent_t& a, hipEvent_t& b);
  void harvest();
};

// Workspace owned by the caller.  ncase independent systems of the same
// type share one launch per kernel: their rows are consecutive, their states
// are st[0..ncase), and tiles[k] splits the rows into tiles of kBlock * 2^k
// rows that never straddle two cases.
//
// rep > 1: the cases are rep right-hand sides of one matrix of n / rep rows, the
// vectors (basis, r, ilu_zl, ilu_zu) one after the other; the matrix, its copies
// and the preconditioner exist once.
struct KWork {
  int n = 0, mmax = 0, ncase = 1, rep = 1;
  bool prepared = false;    // the preconditioner in the workspace is A's already
  size_t ld = 0;            // column stride of V (n rounded up to 8; 0 = n)
  Tiles tiles[5];
  void* V = nullptr;        // (mmax + 1) * ld elements of T
  void* r = nullptr;        // n elements of T: preconditioner input (CG: r, z, p, w use V[0..3])
  void* pcinv = nullptr;    // n elements of T (Jacobi inverse diagonal)
  void* lu = nullptr;       // nnz elements of T (ILU(0) factors), when ilu is set
  void* ilu_lcoef = nullptr;  // coefficients of T per slot of the lower and the upper sweep
  void* ilu_ucoef = nullptr;
  void* ilu_own = nullptr;    // n elements of T: 1 / pivot by upper-sweep position
  void* ilu_zl = nullptr;   // 2 n elements of T each: inputs and results of the lower and the upper sweep
  void* ilu_zu = nullptr;
  const IluLevels* ilu = nullptr;
  double* partial = nullptr;
  size_t partial_len = 0;
  double* norms = nullptr;  // 2 x the tiles of kBlock rows: ||w||^2 per tile of the last two Arnoldi steps
  int lanes = 8;            // CSR SpMV lanes per row (1, 2, 4, 8, 16); 0 = SELL-64 SpMV
  int nt = 0;               // SpMV loads the matrix non-temporally
  int sell_v = kSellDefault;  // SELL window in use (index into kSellSigma) when lanes == 0
  int sell2 = -1;           // FP32 SELL with two slices per wave: 1 / 0 as tuned, -1 above 2^20 rows
  // SELL-64 copies of the matrix being solved: patterns, and values of type T
  SellPat sell[kSellVariants];
  void* sell_vals[kSellVariants] = {nullptr, nullptr, nullptr};
  int rows = 0;             // rows per thread of the Gram-Schmidt kernels; 0: by size
  bool tuned = false;       // lanes / nt / rows chosen by autotune()
  TuneReport report;
  GraphCache* graphs = nullptr;  // set: GMRES cycles (Jacobi / no PC) replay captured graphs
  // mixed GMRES on one case: the FP32 Arnoldi cycle runs on the rows in
  // another order (the matrix and its SELL copies given in that order);
  // ord_pos[i] is the position of natural row i, ord_row[p] the natural row
  // at position p.  The FP64 residual, solution and test stay natural.
  const int* ord_pos = nullptr;
  const int* ord_row = nullptr;
  bool pc_folded = false;  // the FP32 matrix holds M^-1 A (Jacobi): the SpMV scales nothing
  SpmvTimer* timer = nullptr;    // set: time the Arnoldi SpMV launches
  KState* st = nullptr;     // device, ncase states
  KHeader* host = nullptr;  // pinned, ncase headers (the mailbox's)
  Mailbox box;
  unsigned* box_count = nullptr;  // host: messages launched
  std::vector<KResult>* per_case = nullptr;  // filled by a solve when set
};

// Up to this many rows the momentum components are solved together: the launches
// and level groups of small systems are shared, larger ones are bound by the
// vectors' bytes, and three bases of theirs would take gigabytes.  solve_velocity
// one after the other and together, ms: GMRES(50) + Jacobi, mixed and FP64,
// 99,550 rows 1.54 -> 0.80 and 1.27 -> 0.68; 340,215 1.91 -> 1.31 and 1.75 -> 1.38;
// 808,240 3.11 -> 2.18 and 2.63 -> 2.25; 1,566,245 3.71 -> 3.68 and 4.16 -> 4.09.
// GMRES(30) + ILU(0), FP64 and mixed, 331,776 rows 4.26 -> 2.50 and 6.54 -> 3.51;
// 786,432 6.51 -> 3.86 and 9.68 -> 4.96 (1,536,000: 9.25 -> 6.09, 10.6 -> 6.34, left
// out for the memory).
constexpr int kTripleRows = 1 << 20;

// Buffers of the iterative-refinement solve (mixed precision).
struct IrWork {
  double* r64 = nullptr;  // FP64 residual
  float* r32 = nullptr;   // FP32 copy of the residual (inner right-hand side)
  float* e32 = nullptr;   // FP32 correction
  float* inv32 = nullptr; // FP32 Jacobi inverse diagonal of the outer test
  double* partial = nullptr;
  size_t partial_len = 0;
  double* scal = nullptr; // device scalars: [0] ||M^-1 r||^2, [1] ||M^-1 b||^2
  double* host = nullptr; // pinned, 2 doubles
};

// Mixed-precision solve of A64 x = b with FP64 x, b and convergence test
// (PETSc's, on ||M^-1 r||), and FP32 Krylov work on A32 (A64 rounded).
// GMRES(m): every restart cycle is one refinement step — the restart residual
// r = b - A64 x is FP64, the Arnoldi cycle and its basis are FP32, the
// Hessenberg least-squares problem is FP64 and the correction is accumulated
// into the FP64 x; the FP64 residual alone decides convergence.  CG: FP64
// refinement around FP32 CG solves of A32 e = r to relative tolerance
// inner_rtol, at most ir_max of them; the outer test's norm is ||M^-1 r|| with
// M the FP32 Jacobi diagonal or the FP32 ILU(0) factors of A32 (factored once
// per solve and shared with the inner solves), as PETSc's CG tests the
// preconditioned norm.  Taking the residual with A64 keeps the
// exact null space of the pressure-correction matrix (A 1 = 0), which
// rounding breaks.  The iteration cap counts Krylov iterations.
KResult ir_solve(const CsrView<double>& A64, const CsrView<float>& A32, const double* b, double* x,
                 const s355_ksp_opts& o, bool zero_guess, int ir_max, double inner_rtol, KWork& w32, IrWork& ir,
                 hipStream_t s);

// Default rows per thread of the Gram-Schmidt kernels for n rows of elem bytes.
int pick_rows(int n, size_t elem);

// Times the SpMV at 4, 8 and 16 lanes per row with temporal and non-temporal
// matrix loads, and one mid-cycle Gram-Schmidt step (multi-dot + update) at
// 1..16 rows per thread, on A and the workspace; keeps the fastest in
// w.lanes / w.nt / w.rows and the timings in w.report.  The choice is cached per
// process and system shape, so every context of one process that solves
// systems of that shape uses the same kernels (and reproduces its results).
template <class T>
void autotune(const CsrView<T>& A, KWork& w, int m, hipStream_t s);

// Solve A x = b.  x holds the initial guess unless zero_guess.
template <class T>
KResult krylov_solve(const CsrView<T>& A, const T* b, T* x, const s355_ksp_opts& o, bool zero_guess, KWork& w,
                     hipStream_t s);

// x (double) and b (double) with A of type T: r = b - A x  (FP64 accumulate), into r64;
// returns nothing; used by the iterative-refinement outer loop.
template <class T>
void residual64(const CsrView<T>& A, const double* b, const double* x, double* r, hipStream_t s);

// Average device time (ms) of the production SpMV launch y = M^-1 A x (the
// kernel and shape the GMRES solves use, inv = Jacobi inverse or null),
// each of `repeats` launches timed alone with HIP events on stream s after
// `flush_bytes` of `flush` have been overwritten (null: back to back).
template <class T>
double bench_spmv(const CsrView<T>& A, const T* x, T* y, const T* inv, KWork& w, int repeats, void* flush,
                  size_t flush_bytes, hipStream_t s);

// inv = 1 / diag(A) (1 where the diagonal is zero)
template <class T>
void jacobi_inverse(const CsrView<T>& A, T* inv, hipStream_t s);

// Average device time (ms) of a plain copy of `bytes` (a multiple of 16).
double bench_copy(void* dst, const void* src, size_t bytes, int repeats, hipStream_t s);

void convert_to_float(const double* src, float* dst, size_t n, hipStream_t s);

// Zero `bytes` (a multiple of 4) with a fill kernel, which unlike a memset
// node is safe inside a captured graph.
void fill_zero(void* p, size_t bytes, hipStream_t s);

}  // namespace s355

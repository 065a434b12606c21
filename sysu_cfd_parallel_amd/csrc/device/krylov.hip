// Device GMRES(m) / CG for the SIMPLE solves (see krylov.hpp).
//
// One GMRES iteration is four launches: SpMV fused with the Jacobi apply, a
// multi-dot against the basis, the sums of its tiles together with the previous
// step's finalisation (Hessenberg column, Givens rotations, convergence test),
// and the Gram-Schmidt update fused with the norm; two on small systems (see
// k_spmv_dots).  Basis vectors are kept unnormalised (v_k = scale_k V_k); the
// scales are folded into the coefficients, which saves a normalisation pass
// over N and lets a product start before its vector's norm is known.
// Every kernel returns at once when the device state says the solve has
// ended, so the host may launch iterations ahead and read the state back
// only every few iterations.
#include <algorithm>
#include <cmath>
#include <functional>
#include <limits>
#include <map>
#include <mutex>
#include <tuple>
#include <type_traits>

#include "common.hpp"
#include "krylov.hpp"

namespace s355 {
namespace {

constexpr int kConvergedRtol = 2, kConvergedAtol = 3, kDivergedNull = -2, kDivergedIts = -3, kDivergedDtol = -4,
              kDivergedBreakdown = -5, kDivergedIndefinitePc = -8, kDivergedNanorinf = -9,
              kDivergedIndefiniteMat = -10;

__device__ __forceinline__ int conv_check(double ttol, double abstol, double dtol, double rnorm0, double rnorm) {
  if (isnan(rnorm) || isinf(rnorm)) return kDivergedNanorinf;
  if (rnorm <= ttol) return rnorm < abstol ? kConvergedAtol : kConvergedRtol;
  if (rnorm >= dtol * rnorm0) return kDivergedDtol;
  return 0;
}
__device__ __forceinline__ int conv_check(const KState* st, double rnorm) {
  return conv_check(st->ttol, st->abstol, st->dtol, st->rnorm0, rnorm);
}

__device__ __forceinline__ double& Hm(KState* st, int ld, int r, int c) { return st->H[c * ld + r]; }

// ---- preconditioner set-up
template <class T>
__global__ void __launch_bounds__(kBlock) k_jacobi_setup(CsrView<T> A, T* inv) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= A.n) return;
  const double d = static_cast<double>(A.val[A.diag[i]]);
  inv[i] = static_cast<T>(d != 0.0 ? 1.0 / d : 1.0);
}

// Workgroup size of a launch of the ILU(0) factorisation and sweeps: a
// launch below 64 K rows has one-wave workgroups, so its rows spread over
// all CUs (each row is a chain of dependent loads, not a share of bandwidth);
// larger launches keep 256-thread workgroups.
inline int level_block(int nrows) { return nrows < (kBlock << 8) ? kWave : kBlock; }

// ---- ILU(0), natural ordering, one thread per row of a level.  IKJ
// elimination a_ik /= u_kk, a_ij -= l_ik u_kj on the pattern, from the
// precomputed steps of each row (its lower entries p in order, the pivot
// position of each, and the (target, source) slot pairs where row i's pattern
// after p meets the upper part of row k = col[p], in column order): the
// arithmetic and its order are those of merging the two sorted rows.
template <class T>
__global__ void __launch_bounds__(kBlock) k_ilu_factor(T* __restrict__ lu, IluSteps f, int t0, int nrows) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nrows) return;
  const int t = t0 + k;
  const int s0 = f.ptr[t], s1 = f.ptr[t + 1];
  for (int s = s0; s < s1; ++s) {
    const int p = f.p[s];
    lu[p] = lu[p] / lu[f.d[s]];
    const T lik = lu[p];
    const int u1 = f.u[s + 1];
    for (int u = f.u[s]; u < u1; ++u) lu[f.r[u]] -= lik * lu[f.q[u]];
  }
}

// One group of a sweep (see ilu_plan.hpp): each row sums its terms over the
// sweep's inputs and the earlier groups' results, one thread per row, in
// place of a launch per level.  A level of a few thousand rows is bound by
// the launch and the chain slots -> gathers -> store, so all of a row's
// slots load before any is used and all its gathers before any is added: the
// rows of a launch come in classes of term counts, each a run of workgroups
// compiled for its padded width, its loads unconditional (guarded ones wait
// for each other), a long row shared by several lanes.
struct IluLaunch {
  // per class; blk0: its first workgroup (empty classes: nrows 0, where the
  // next class starts)
  long off[kTermClasses];
  int p0[kTermClasses], nrows[kTermClasses], width[kTermClasses], blk0[kTermClasses];
};

// A row's sum in twice T's precision, rounded once at its end.  A merged row adds
// many more terms than a row of a level did (10 on hexahedra, up to 200), and
// the terms of a group replace what levels in between had rounded: summed in T
// the error of an application against the factors' exact solves was 1.3-1.6
// times that of plain solves in T (hexahedra, tetrahedra, both mixed, FP64 and
// FP32), summed so it is 0.7-0.8 of theirs.  The coefficients stay rounded to T; they
// make no difference that can be measured.  The kernel waits for loads most of
// the time, so the sums cost little: a solve with plain sums and with these, CG on
// 331,776 tetrahedra in FP64 54.9 and 53.1 ms, mixed GMRES(50) on 310,000 hexahedra
// 36.4 and 36.2, on 6.0 M hexahedra 828.7 and 841.6 (the conversions of FP32).  They
// cost 3-5 % with the terms tested against the row's length, in place of padding
// coefficients of 0, and the row's input added before the slots were on their way.
template <class T>
struct RowSum;

template <>
struct RowSum<float> {
  double s = 0.0;
  // (the product is exact, so the fused sum rounds as the separate one would)
  __device__ __forceinline__ void add(float c, float x) { s = fma(static_cast<double>(c), static_cast<double>(x), s); }
  __device__ __forceinline__ void join(int mask) { s += __shfl_xor(s, mask, kWave); }
  __device__ __forceinline__ float value() const { return static_cast<float>(s); }
};

// s + e: the products' and the sums' rounding errors go to e
template <>
struct RowSum<double> {
  double s = 0.0, e = 0.0;
  __device__ __forceinline__ void plus(double p) {
    const double t = s + p, z = t - s;
    e += (s - (t - z)) + (p - z);
    s = t;
  }
  __device__ __forceinline__ void add(double c, double x) {
    const double p = c * x;
    e += fma(c, x, -p);
    plus(p);
  }
  __device__ __forceinline__ void join(int mask) {
    const double os = __shfl_xor(s, mask, kWave), oe = __shfl_xor(e, mask, kWave);
    plus(os);
    e += oe;
  }
  __device__ __forceinline__ double value() const {
    const double v = s + e;
    return v == v ? v : s;  // an infinite sum has no error term
  }
};

// adds o x0 and then a row's terms u = lane, lane + Lanes, ... (W of them, slots
// `step` apart; padding: coefficient 0 times the row's own input).  (The additions
// come after the last load: one that waits for x0 first holds the slots up.)
template <class T, int W>
__device__ __forceinline__ void ilu_terms(const int* __restrict__ col, const T* __restrict__ coef, const T* buf,
                                          size_t q0, int step, T o, T x0, RowSum<T>& s) {
  T v[W], x[W];
  int c[W];
#pragma unroll
  for (int u = 0; u < W; ++u) {
    v[u] = coef[q0 + static_cast<size_t>(u) * step];
    c[u] = col[q0 + static_cast<size_t>(u) * step];
  }
#pragma unroll
  for (int u = 0; u < W; ++u) x[u] = buf[c[u]];
  s.add(o, x0);
#pragma unroll
  for (int u = 0; u < W; ++u) s.add(v[u], x[u]);
}

// (own: the coefficient of each row's own input in the upper sweep, 1 in the lower;
// rcase: the case of each row of a batch, whose finished cases' rows are left out)
template <class T, bool Wide, bool Upper>
__global__ void __launch_bounds__(kBlock) k_ilu_group(IluLaunch g, const int* __restrict__ col,
                                                      const T* __restrict__ coef,
                                                      const T* __restrict__ own, T* buf, int n, const KState* st,
                                                      const int* __restrict__ rcase) {
  buf += blockIdx.y * 2 * static_cast<size_t>(n);  // right-hand side blockIdx.y
  // the workgroup's class, by constant indices (the launch stays in registers)
  const int blk = blockIdx.x;
  int cls = 0, p0 = g.p0[0], nrows = g.nrows[0], width = g.width[0], blk0 = 0;
  long off = g.off[0];
#pragma unroll
  for (int c = 1; c < (Wide ? kTermClasses : kNarrowClasses); ++c)
    if (blk >= g.blk0[c]) {
      cls = c;
      p0 = g.p0[c];
      nrows = g.nrows[c];
      width = g.width[c];
      blk0 = g.blk0[c];
      off = g.off[c];
    }
  int lanes = 1;
  if constexpr (Wide) lanes = cls < 4 ? 1 : cls < 6 ? 4 : 16;
  const int i = (blk - blk0) * static_cast<int>(blockDim.x) + threadIdx.x;
  const int k = i / lanes, lane = i % lanes;
  if (k >= nrows) return;  // the lanes of a row together
  const int p = p0 + k;
  if (st && st[rcase ? rcase[p] : blockIdx.y].reason) return;
  const int step = nrows * lanes;
  const size_t q0 = static_cast<size_t>(off) + i;
  T o = T(1), x0 = buf[p];
  if constexpr (Upper) o = own[p];
  if constexpr (Wide) x0 = lane == 0 ? x0 : T(0);
  RowSum<T> z;
  if (cls == 0) {
    ilu_terms<T, 3>(col, coef, buf, q0, step, o, x0, z);
  } else if (cls == 1) {
    ilu_terms<T, 6>(col, coef, buf, q0, step, o, x0, z);
  } else if (cls == 2) {
    ilu_terms<T, 10>(col, coef, buf, q0, step, o, x0, z);
  } else if constexpr (Wide) {
    switch (cls) {
      case 3: ilu_terms<T, 15>(col, coef, buf, q0, step, o, x0, z); break;
      case 4: ilu_terms<T, 8>(col, coef, buf, q0, step, o, x0, z); break;
      case 5: ilu_terms<T, 16>(col, coef, buf, q0, step, o, x0, z); break;
      default:
        for (int j = 0; j < width; j += 16 * kTermBatch)
          ilu_terms<T, kTermBatch>(col, coef, buf, q0 + static_cast<size_t>(j / 16) * step, step, o, j ? T(0) : x0, z);
        break;
    }
    if (lanes > 1) {
      // the lanes' sums, pairs first
      z.join(1);
      z.join(2);
      if (lanes == 16) {
        z.join(4);
        z.join(8);
      }
      if (lane) return;
    }
  }
  buf[static_cast<size_t>(n) + p] = z.value();
}

// The coefficients of a sweep from the factors: those of the rows at depth 0
// (no reference to their own group), and the direct terms of the others.
// (own: 1 / pivot in the upper sweep)
template <class T, bool Upper>
__global__ void __launch_bounds__(kBlock) k_ilu_coef(int n, const int* __restrict__ len, const int* __restrict__ slot0,
                                                     const int* __restrict__ lanes, const int* __restrict__ stride,
                                                     const int* __restrict__ src, const int* __restrict__ dsrc,
                                                     const T* __restrict__ lu, T* __restrict__ coef,
                                                     T* __restrict__ own) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const int L = len[p], nl = lanes[p], step = stride[p];
  const size_t q0 = slot0[p];
  // dsrc < 0: a row below depth 0, divided by its pivot once its terms are complete
  const int dp = Upper ? dsrc[p] : -1;
  const T d = dp >= 0 ? lu[dp] : T(1);
  for (int u = 0; u < L; ++u) {
    const size_t at = q0 + static_cast<size_t>(u / nl) * step + u % nl;
    const int e = src[at];
    const T c = e >= 0 ? -lu[e] : T(0);
    coef[at] = dp >= 0 ? c / d : c;
  }
  if (dp >= 0) own[p] = T(1) / d;
}

// ... and the rows of one depth d > 0, whose references to rows of lower depths
// are replaced by those rows' terms.  The pairs of one reference have different
// targets and are shared by kMergeLanes lanes, the references of a row follow
// one another, so every coefficient is summed in the same order whatever the
// lanes.  One thread per row walked its own run of pairs, a cache line of its
// own per step: 2.6 ms for the widest depth of 512 cavities of 16^3 (2.1 M rows,
// FP64), 3.1 ms of a pressure solve's 18.4.
constexpr int kMergeLanes = 8;
template <class T, bool Upper>
__global__ void __launch_bounds__(kBlock) k_ilu_merge(int k0, int nrows, const int* __restrict__ later,
                                                      const int* __restrict__ sptr, const int* __restrict__ sp,
                                                      const int* __restrict__ uptr, const int* __restrict__ r,
                                                      const int* __restrict__ q, const int* __restrict__ len,
                                                      const int* __restrict__ slot0, const int* __restrict__ lanes,
                                                      const int* __restrict__ stride, const int* __restrict__ dsrc,
                                                      const T* __restrict__ lu, T* coef, T* own) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x, t = i / kMergeLanes, lane = i % kMergeLanes;
  if (t >= nrows) return;  // the lanes of a row together
  const int k = k0 + t, p = later[k];
  for (int x = sptr[k]; x < sptr[k + 1]; ++x) {
    const T a = lu[sp[x]];
    for (int u = uptr[x] + lane; u < uptr[x + 1]; u += kMergeLanes) {
      const int e = q[u];
      coef[r[u]] -= a * (e >= 0 ? coef[e] : (Upper ? own[-1 - e] : T(1)));
    }
    __threadfence_block();  // the next reference's targets may be another lane's
  }
  if constexpr (Upper) {
    const T d = lu[-1 - dsrc[p]];
    const int nl = lanes[p], step = stride[p];
    const size_t q0 = slot0[p];
    for (int u = lane; u < len[p]; u += kMergeLanes) coef[q0 + static_cast<size_t>(u / nl) * step + u % nl] /= d;
    if (lane == 0) own[p] = T(1) / d;
  }
}

// The moves between the natural order and the sweeps' orders (Tag only
// names the move in kernel traces).  Inside one run of a launch's rows (same
// group, depth and class) rows keep their natural order in the lower sweep and
// their lower-sweep order in the upper, so the rows of a range of consecutive
// source positions that fall in one run of the destination order are
// consecutive there: a workgroup reading (or writing) a contiguous range
// writes (reads) one short contiguous piece per run, and consecutive workgroups on one XCD extend the same runs in its L2.
// scatter: dst[pos[q]] = src[q]
// (right-hand side blockIdx.y at src + blockIdx.y * ssrc, dst + blockIdx.y * sdst)
template <class T, int Tag>
__global__ void __launch_bounds__(kBlock) k_scatter(int n, const int* __restrict__ pos, const T* __restrict__ src,
                                                    size_t ssrc, T* __restrict__ dst, size_t sdst, const KState* st) {
  src += blockIdx.y * ssrc;
  dst += blockIdx.y * sdst;
  const int q = xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  if (q >= n) return;
  const int p = pos[q];
  const T v = src[q];
  if (st && st[blockIdx.y].reason) return;
  dst[p] = v;
}

// gather: dst[q] = src[idx[q]].  With Dot (CG with ILU(0): one case, blocks
// of kBlock threads) also the partial sums (dst, dst) and (dst, r) over the
// block's kBlock rows b kBlock .. into partial[2b], partial[2b + 1] (block
// sums in the fixed wave order), which CG's reductions then finish.
template <class T, int Tag, bool Dot = false>
__global__ void __launch_bounds__(kBlock) k_gather_at(int n, const int* __restrict__ idx, const T* __restrict__ src,
                                                      T* __restrict__ dst, const KState* st,
                                                      const T* __restrict__ r = nullptr, double* partial = nullptr) {
  src += blockIdx.y * 2 * static_cast<size_t>(n);
  dst += blockIdx.y * static_cast<size_t>(n);
  const int b = xcd_block(blockIdx.x, gridDim.x);
  const int q = b * blockDim.x + threadIdx.x;
  if constexpr (!Dot) {
    if (q >= n) return;
    const int p = idx[q];
    if (st && st[blockIdx.y].reason) return;
    dst[q] = src[p];
  } else {
    __shared__ double lds[kBlock / kWave];
    if (st && st->reason) return;  // one case: the whole grid leaves together
    double zz = 0.0, zr = 0.0;
    if (q < n) {
      const T v = src[idx[q]];
      dst[q] = v;
      const double zv = static_cast<double>(v);
      zz = zv * zv;
      zr = zv * static_cast<double>(r[q]);
    }
    zz = block_sum(zz, lds);
    zr = block_sum(zr, lds);
    if (threadIdx.x == 0) {
      partial[2 * b] = zz;
      partial[2 * b + 1] = zr;
    }
  }
}

// out[q] = lu[src[q]] (0 where src[q] < 0)
template <class T>
__global__ void __launch_bounds__(kBlock) k_gather(const int* __restrict__ src, size_t n, const T* __restrict__ lu,
                                                   T* __restrict__ out) {
  const size_t q = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (q >= n) return;
  const int p = src[q];
  out[q] = p >= 0 ? lu[p] : T(0);
}

// the coefficients of one sweep from the factors lu
template <class T, bool Upper>
void ilu_coefficients(const IluSweep& w, const T* lu, T* coef, T* own, hipStream_t s) {
  hipLaunchKernelGGL((k_ilu_coef<T, Upper>), dim3(grid_for(w.n)), dim3(kBlock), 0, s, w.n, w.len, w.slot0, w.lanes,
                     w.stride, w.src, w.dsrc, lu, coef, own);
  for (size_t d = 0; d + 1 < w.dptr.size(); ++d) {
    const int nr = w.dptr[d + 1] - w.dptr[d];
    if (nr == 0) continue;
    const int b = level_block(nr);
    hipLaunchKernelGGL((k_ilu_merge<T, Upper>), dim3(grid_for(static_cast<long>(nr) * kMergeLanes, b)), dim3(b), 0, s, w.dptr[d], nr, w.later, w.sptr,
                       w.p, w.uptr, w.r, w.q, w.len, w.slot0, w.lanes, w.stride, w.dsrc, lu, coef, own);
  }
}

// ILU(0) factors of A into lu (CSR), then the sweeps' coefficients
template <class T>
void ilu_factor(const CsrView<T>& A, int nnz, const IluLevels& lv, T* lu, hipStream_t s, const KWork* w) {
  S355_HIP(hipMemcpyAsync(lu, A.val, sizeof(T) * static_cast<size_t>(nnz), hipMemcpyDeviceToDevice, s));
  if (!lv.steps.ptr || !w->ilu_lcoef || !w->ilu_ucoef || !w->ilu_own)
    throw std::invalid_argument("ILU(0) factorisation without its plan");
  for (int l = 0; l < lv.nl(); ++l) {
    const int nr = lv.lptr[l + 1] - lv.lptr[l];
    if (nr == 0) continue;
    const int b = level_block(nr);
    hipLaunchKernelGGL((k_ilu_factor<T>), dim3(grid_for(nr, b)), dim3(b), 0, s, lu, lv.steps, lv.lptr[l], nr);
  }
  ilu_coefficients<T, false>(lv.lower, lu, static_cast<T*>(w->ilu_lcoef), nullptr, s);
  ilu_coefficients<T, true>(lv.upper, lu, static_cast<T*>(w->ilu_ucoef), static_cast<T*>(w->ilu_own), s);
  S355_LAUNCH_CHECK();
}

// one sweep, group by group, on buf: n inputs, then n results
template <class T, bool Upper>
void ilu_sweep(const IluSweep& w, const T* coef, const T* own, T* buf, const KState* st, int rep, hipStream_t s) {
  for (size_t g = 0; g + 1 < w.group.size(); ++g) {
    IluLaunch a{};
    int rows = 0, blocks = 0, k = w.group[g];
    for (int x = k; x < w.group[g + 1]; ++x) rows += w.subs[x].nrows * kTermLanes[w.subs[x].cls];
    const int b = level_block(rows);
    for (int c = 0; c < kTermClasses; ++c) {
      a.blk0[c] = blocks;
      if (k == w.group[g + 1] || w.subs[k].cls != c) continue;
      const IluSub& u = w.subs[k++];
      a.off[c] = u.off;
      a.p0[c] = u.p0;
      a.nrows[c] = u.nrows;
      a.width[c] = u.width;
      blocks += grid_for(static_cast<long>(u.nrows) * kTermLanes[c], b);
    }
    const bool wide = w.subs[w.group[g + 1] - 1].cls >= kNarrowClasses;
    hipLaunchKernelGGL((wide ? k_ilu_group<T, true, Upper> : k_ilu_group<T, false, Upper>), dim3(blocks, rep), dim3(b), 0, s, a,
                       w.col, coef, own, buf, w.n, st, w.rcase);
  }
}

// z = (LU)^-1 r ; r and z distinct (w->rep vectors each, one after the other).
// With a graph cache the sweeps (one
// launch per group) are captured once per (factor, r, z) and replayed.
// With dot (CG) the last move also leaves the partial sums of (z, z) and
// (z, r) per kBlock rows there (see k_gather_at).
template <class T>
void ilu_apply(const CsrView<T>& A, const IluLevels& lv, const T* lu, const T* r, T* z, const KState* st,
               hipStream_t s, GraphCache* graphs = nullptr, const KWork* w = nullptr, double* dot = nullptr) {
  if (graphs) {
    const std::vector<uintptr_t> key = {0x11u, reinterpret_cast<uintptr_t>(lu), reinterpret_cast<uintptr_t>(r),
                                        reinterpret_cast<uintptr_t>(z), reinterpret_cast<uintptr_t>(st),
                                        reinterpret_cast<uintptr_t>(lv.lpos), sizeof(T),
                                        reinterpret_cast<uintptr_t>(w ? w->ilu_lcoef : nullptr),
                                        reinterpret_cast<uintptr_t>(w ? w->ilu_zl : nullptr),
                                        reinterpret_cast<uintptr_t>(dot)};
    hipGraphExec_t g = graphs->get(key, s, [&] { ilu_apply(A, lv, lu, r, z, st, s, nullptr, w, dot); });
    S355_HIP(hipGraphLaunch(g, s));
    return;
  }
  if (!w || !w->ilu_lcoef || !w->ilu_zl || !w->ilu_zu || !lv.lower.col || !lv.lpos || !lv.l2u || !lv.upos)
    throw std::invalid_argument("ILU(0) application without its sweep workspace");
  T* zl = static_cast<T*>(w->ilu_zl);
  T* zu = static_cast<T*>(w->ilu_zu);
  const int n = lv.lptr.back(), rep = w->rep;
  const size_t n1 = n;
  const dim3 gn(grid_for(n), rep);
  const KState* st_move = lv.lower.rcase ? nullptr : st;  // the moves of a batch move every case
  // r into the lower order, the lower sweep, its result into the upper
  // order, the upper sweep, z back into the natural order
  hipLaunchKernelGGL((k_scatter<T, 0>), gn, dim3(kBlock), 0, s, n, lv.lpos, r, n1, zl, 2 * n1, st_move);
  ilu_sweep<T, false>(lv.lower, static_cast<const T*>(w->ilu_lcoef), static_cast<const T*>(nullptr), zl, st, rep, s);
  hipLaunchKernelGGL((k_scatter<T, 1>), gn, dim3(kBlock), 0, s, n, lv.l2u, zl + n, 2 * n1, zu, 2 * n1, st_move);
  ilu_sweep<T, true>(lv.upper, static_cast<const T*>(w->ilu_ucoef), static_cast<const T*>(w->ilu_own), zu, st, rep, s);
  if (dot)
    hipLaunchKernelGGL((k_gather_at<T, 2, true>), gn, dim3(kBlock), 0, s, n, lv.upos, zu + n, z, st, r, dot);
  else
    hipLaunchKernelGGL((k_gather_at<T, 2>), gn, dim3(kBlock), 0, s, n, lv.upos, zu + n, z, st_move, nullptr, nullptr);
  S355_LAUNCH_CHECK();
}

// ---- y = M^-1 A x (of the unnormalised basis vector: its scale goes into the
// coefficients, so a product does not wait for the norm's finalisation)
// L consecutive lanes share a row (L = 4, 8 or 16, picked per matrix): their
// loads of values and column ids are contiguous across the wavefront; a
// shuffle tree in a fixed order sums the lanes.  With NT the matrix streams
// are loaded non-temporally, so that the L2 keeps the gathered x instead.
template <class V, bool NT>
__device__ __forceinline__ V ld_stream(const V* p) {
  if constexpr (NT)
    return __builtin_nontemporal_load(p);
  else
    return *p;
}

// sum over p = p0, p0 + step, ... < p1 of val[p] * x[col[p]] (X: the
// accumulator type), in that order; each batch of 8 entries loads its values
// and column ids before any of its gathers of x
template <class X, class V, bool NT>
__device__ __forceinline__ X csr_dot(const V* __restrict__ val, const int* __restrict__ col, int p0, int p1, int step,
                                     const X* __restrict__ x, X s) {
  constexpr int B = 8;
  for (int pb = p0; pb < p1; pb += B * step) {
    V v[B];
    X xv[B];
    int c[B];
#pragma unroll
    for (int u = 0; u < B; ++u)
      if (pb + u * step < p1) {
        v[u] = ld_stream<V, NT>(val + pb + u * step);
        c[u] = ld_stream<int, NT>(col + pb + u * step);
      }
#pragma unroll
    for (int u = 0; u < B; ++u)
      if (pb + u * step < p1) xv[u] = x[c[u]];
#pragma unroll
    for (int u = 0; u < B; ++u)
      if (pb + u * step < p1) s += static_cast<X>(v[u]) * xv[u];
  }
  return s;
}

template <class T, int L, bool NT>
__device__ __forceinline__ T row_dot(const CsrView<T>& A, const T* __restrict__ x, int row, int lane) {
  T s = T(0);
  if (row < A.n) s = csr_dot<T, T, NT>(A.val, A.col, A.rowptr[row] + lane, A.rowptr[row + 1], L, x, s);
#pragma unroll
  for (int off = L / 2; off > 0; off >>= 1) s += __shfl_down(s, off, L);
  return s;
}

template <class T, int L, bool NT>
__global__ void __launch_bounds__(kBlock) k_spmv_pc(CsrView<T> A, Tiles t, const T* __restrict__ x,
                                                    const T* __restrict__ inv, T* __restrict__ y, const KState* st) {
  x += blockIdx.y * static_cast<size_t>(A.n);  // right-hand side blockIdx.y of the same matrix
  y += blockIdx.y * static_cast<size_t>(A.n);
  st += blockIdx.y;
  const int g = xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  const int row = g / L, lane = g % L;
  // the lanes of one row share its case, so they leave together
  const KState* sc = st + (row < A.n ? t.case_of(row) : 0);
  if (sc->reason) return;
  const T s = row_dot<T, L, NT>(A, x, row, lane);
  if (lane == 0 && row < A.n) {
    double z = static_cast<double>(s);
    if (inv) z *= static_cast<double>(inv[row]);
    y[row] = static_cast<T>(z);
  }
}

// ---- the same product on the SELL-64 copy: one row per lane, the row's
// entries summed in CSR order
constexpr int kSellBatch = 8;

// One row of a slice of width W (1..kSellBatch, a compile-time constant, so
// the W slot loads are unconditional and the compiler issues all of them
// before waiting on any), or of width > kSellBatch for W = 0 (batches of
// kSellBatch slots, the guards wave-uniform).  Every column and value load of
// a batch is issued, then every gather of x, then the products are added in
// slot order.  With one case the first batch loads before the state check,
// in parallel with the row id and the state, which it does not depend on; in
// a batch the state of the row's case is checked first (see sell_row).
// With C16 the columns are 16-bit offsets from the row (SellView::col16):
// half the column bytes, added to the row id once both have loaded.
template <bool NT, bool C16, class V>
__device__ __forceinline__ int sell_col(const V& A, size_t q, int row) {
  if constexpr (C16)
    return row + static_cast<int>(ld_stream<int16_t, NT>(A.col16 + q));
  else
    return ld_stream<int, NT>(A.col + q);
}

template <class T, bool NT, bool PC, int W, bool C16>
__device__ __forceinline__ T sell_row(const SellView<T>& A, const Tiles& t, const T* __restrict__ x,
                                      const T* __restrict__ inv, const KState* st, int sl, int pos, int qa, int q1,
                                      int& row) {
  constexpr int B = W > 0 ? W : kSellBatch;
  row = A.row ? A.row[pos] : pos;
  int q0 = qa + (pos & 63);
  T v[B], xv[B];
  int c[B];
  // the case: one case without a slice table; in batches per slice when the
  // slice lies in one case, else by row.  In a batch the state is read
  // before the slots, so that the rows of cases that have finished load
  // nothing (late in a batch's solve most rows are such); alone, the first
  // batch of slots loads while the state does.
  const KState* sc = st;
  if (A.scase) {
    int cs = A.scase[sl];
    if (cs < 0) cs = t.case_of(row);
    sc = st + cs;
    if (sc->reason) {
      row = -1;
      return T(0);
    }
  }
#pragma unroll
  for (int u = 0; u < B; ++u) {
    v[u] = ld_stream<T, NT>(A.val + q0 + 64 * u);
    c[u] = sell_col<NT, C16>(A, q0 + 64 * u, row);
  }
  if (sc->reason) {
    row = -1;
    return T(0);
  }
  // used after the slots (PC: Jacobi, inv is set)
  T invr = T(1);
  if constexpr (PC) invr = inv[row];
  T acc = T(0);
#pragma unroll
  for (int u = 0; u < B; ++u) xv[u] = x[c[u]];
#pragma unroll
  for (int u = 0; u < B; ++u) acc += v[u] * xv[u];
  if constexpr (W == 0) {
    // rows longer than one batch: the rest, batch by batch
    for (q0 += 64 * kSellBatch; q0 < q1; q0 += 64 * kSellBatch) {
#pragma unroll
      for (int u = 0; u < kSellBatch; ++u)
        if (q0 + 64 * u < q1) {
          v[u] = ld_stream<T, NT>(A.val + q0 + 64 * u);
          c[u] = sell_col<NT, C16>(A, q0 + 64 * u, row);
        }
#pragma unroll
      for (int u = 0; u < kSellBatch; ++u)
        if (q0 + 64 * u < q1) xv[u] = x[c[u]];
#pragma unroll
      for (int u = 0; u < kSellBatch; ++u)
        if (q0 + 64 * u < q1) acc += v[u] * xv[u];
    }
  }
  double z = static_cast<double>(acc);
  if constexpr (PC) z *= static_cast<double>(invr);
  return static_cast<T>(z);
}

// one row of slice sl by the slice's width (wave-uniform); row -1: its case
// has finished, no value
template <class T, bool NT, bool PC, bool C16>
__device__ __forceinline__ T sell_row_any(const SellView<T>& A, const Tiles& t, const T* __restrict__ x,
                                          const T* __restrict__ inv, const KState* st, int sl, int pos, int qa, int q1,
                                          int& row) {
  switch ((q1 - qa) >> 6) {
    case 1: return sell_row<T, NT, PC, 1, C16>(A, t, x, inv, st, sl, pos, qa, q1, row);
    case 2: return sell_row<T, NT, PC, 2, C16>(A, t, x, inv, st, sl, pos, qa, q1, row);
    case 3: return sell_row<T, NT, PC, 3, C16>(A, t, x, inv, st, sl, pos, qa, q1, row);
    case 4: return sell_row<T, NT, PC, 4, C16>(A, t, x, inv, st, sl, pos, qa, q1, row);
    case 5: return sell_row<T, NT, PC, 5, C16>(A, t, x, inv, st, sl, pos, qa, q1, row);
    case 6: return sell_row<T, NT, PC, 6, C16>(A, t, x, inv, st, sl, pos, qa, q1, row);
    case 7: return sell_row<T, NT, PC, 7, C16>(A, t, x, inv, st, sl, pos, qa, q1, row);
    case 8: return sell_row<T, NT, PC, 8, C16>(A, t, x, inv, st, sl, pos, qa, q1, row);
    default: return sell_row<T, NT, PC, 0, C16>(A, t, x, inv, st, sl, pos, qa, q1, row);
  }
}

template <class T, bool NT, bool PC, bool C16 = false>
__global__ void __launch_bounds__(kBlock) k_spmv_sell(SellView<T> A, Tiles t, const T* __restrict__ x,
                                                      const T* __restrict__ inv, T* __restrict__ y, const KState* st) {
  x += blockIdx.y * static_cast<size_t>(A.n);
  y += blockIdx.y * static_cast<size_t>(A.n);
  st += blockIdx.y;
  const int pos = xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  if (pos >= A.n) return;
  // a wave is one slice (64 consecutive positions), so the slice index and
  // width are wave-uniform and the slice bounds load through the scalar cache
  const int sl = __builtin_amdgcn_readfirstlane(pos >> 6);
  int row;
  const T z = sell_row_any<T, NT, PC, C16>(A, t, x, inv, st, sl, pos, A.ptr[sl], A.ptr[sl + 1], row);
  if (row >= 0) y[row] = z;
}

// Two adjacent slices per wave, one row of each per lane (one case, FP32 on
// large systems): twice the loads in flight per wave at the same occupancy.
// Both rows run the one-slice arithmetic: W is the wider slice's width, the
// narrower slice's slots past its width reload the lane's first slot and are
// never added (adjacent slices of a sorted window rarely differ in width).
template <class T, bool NT, bool PC, int W, bool C16>
__device__ __forceinline__ void sell_rows2(const SellView<T>& A, const T* __restrict__ x, const T* __restrict__ inv,
                                           T* __restrict__ y, const KState* st, int sl, int lane, int qa0,
                                           int qa1, int q11) {
  const int w0 = (qa1 - qa0) >> 6, w1 = (q11 - qa1) >> 6;
  const int pos0 = sl * 64 + lane, pos1 = pos0 + 64;
  const bool ok1 = pos1 < A.n;
  const int row0 = A.row ? A.row[pos0] : pos0;
  const int row1 = ok1 ? (A.row ? A.row[pos1] : pos1) : row0;
  T v0[W], v1[W], x0[W], x1[W];
  int c0[W], c1[W];
#pragma unroll
  for (int u = 0; u < W; ++u) {
    const int qa = qa0 + lane + (u < w0 ? 64 * u : 0);
    const int qb = qa1 + lane + (u < w1 ? 64 * u : 0);
    v0[u] = ld_stream<T, NT>(A.val + qa);
    c0[u] = sell_col<NT, C16>(A, qa, row0);
    v1[u] = ld_stream<T, NT>(A.val + qb);
    c1[u] = sell_col<NT, C16>(A, qb, row1);
  }
  if (st->reason) return;
  T i0 = T(1), i1 = T(1);
  if constexpr (PC) {
    i0 = inv[row0];
    i1 = inv[row1];
  }
#pragma unroll
  for (int u = 0; u < W; ++u) {
    x0[u] = x[c0[u]];
    x1[u] = x[c1[u]];
  }
  T a0 = T(0), a1 = T(0);
#pragma unroll
  for (int u = 0; u < W; ++u) {
    if (u < w0) a0 += v0[u] * x0[u];
    if (u < w1) a1 += v1[u] * x1[u];
  }
  double z0 = static_cast<double>(a0), z1 = static_cast<double>(a1);
  if constexpr (PC) {
    z0 *= static_cast<double>(i0);
    z1 *= static_cast<double>(i1);
  }
  y[row0] = static_cast<T>(z0);
  if (ok1) y[row1] = static_cast<T>(z1);
}

template <class T, bool NT, bool PC, bool C16 = false>
__global__ void __launch_bounds__(kBlock) k_spmv_sell2(SellView<T> A, Tiles t, const T* __restrict__ x,
                                                       const T* __restrict__ inv, T* __restrict__ y,
                                                       const KState* st) {
  x += blockIdx.y * static_cast<size_t>(A.n);
  y += blockIdx.y * static_cast<size_t>(A.n);
  st += blockIdx.y;
  // wave w takes slices 2w and 2w + 1
  const int wv = xcd_block(blockIdx.x, gridDim.x) * (kBlock / kWave) + static_cast<int>(threadIdx.x) / kWave;
  const int sl = __builtin_amdgcn_readfirstlane(2 * wv), lane = threadIdx.x & (kWave - 1);
  const int nsl = (A.n + 63) >> 6;
  if (sl >= nsl) return;
  if (sl + 1 >= nsl) {
    // an odd last slice: the one-slice body
    const int pos = sl * 64 + lane;
    if (pos < A.n) {
      int row;
      const T z = sell_row_any<T, NT, PC, C16>(A, t, x, inv, st, sl, pos, A.ptr[sl], A.ptr[sl + 1], row);
      if (row >= 0) y[row] = z;
    }
    return;
  }
  const int qa0 = A.ptr[sl], qa1 = A.ptr[sl + 1], q11 = A.ptr[sl + 2];
  const int wmax = max((qa1 - qa0) >> 6, (q11 - qa1) >> 6);
  switch (wmax) {
    case 1: sell_rows2<T, NT, PC, 1, C16>(A, x, inv, y, st, sl, lane, qa0, qa1, q11); break;
    case 2: sell_rows2<T, NT, PC, 2, C16>(A, x, inv, y, st, sl, lane, qa0, qa1, q11); break;
    case 3: sell_rows2<T, NT, PC, 3, C16>(A, x, inv, y, st, sl, lane, qa0, qa1, q11); break;
    case 4: sell_rows2<T, NT, PC, 4, C16>(A, x, inv, y, st, sl, lane, qa0, qa1, q11); break;
    case 5: sell_rows2<T, NT, PC, 5, C16>(A, x, inv, y, st, sl, lane, qa0, qa1, q11); break;
    case 6: sell_rows2<T, NT, PC, 6, C16>(A, x, inv, y, st, sl, lane, qa0, qa1, q11); break;
    case 7: sell_rows2<T, NT, PC, 7, C16>(A, x, inv, y, st, sl, lane, qa0, qa1, q11); break;
    case 8: sell_rows2<T, NT, PC, 8, C16>(A, x, inv, y, st, sl, lane, qa0, qa1, q11); break;
    default: {
      // a slice wider than one batch: each slice with the one-slice body
      // for its own width
      for (int k = 0; k < 2; ++k) {
        const int s2 = sl + k, pos = s2 * 64 + lane;
        if (pos < A.n) {
          int row;
          const T z = sell_row_any<T, NT, PC, C16>(A, t, x, inv, st, s2, pos, A.ptr[s2], A.ptr[s2 + 1], row);
          if (row >= 0) y[row] = z;
        }
      }
      break;
    }
  }
}

template <class T, class S>
__global__ void __launch_bounds__(kBlock) k_sell_fill(const int* __restrict__ src, size_t nslots,
                                                      const S* __restrict__ csr, T* __restrict__ out) {
  const size_t q = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (q >= nslots) return;
  const int p = src[q];
  out[q] = p >= 0 ? static_cast<T>(csr[p]) : T(0);
}

// SpMV variants: v = 2 k + nt, k = 0..4 CSR with 1, 2, 4, 8, 16 lanes per row,
// k = 5 + s SELL-64 with window kSellSigma[s] (lanes = 0)
constexpr int kSpmvVariants = 16;
inline int spmv_variant(int lanes, int nt, int sell_v) {
  const int k = lanes == 0 ? 5 + sell_v : lanes == 1 ? 0 : lanes == 2 ? 1 : lanes == 4 ? 2 : lanes == 8 ? 3 : 4;
  return 2 * k + (nt ? 1 : 0);
}

template <class T, int L>
void launch_spmv_l(bool nt, const CsrView<T>& A, const Tiles& t, const T* x, const T* inv, T* y, const KState* st,
                   int rep, hipStream_t s) {
  const int g = grid_for(static_cast<long>(A.n) * L);
  if (nt)
    hipLaunchKernelGGL((k_spmv_pc<T, L, true>), dim3(g, rep), dim3(kBlock), 0, s, A, t, x, inv, y, st);
  else
    hipLaunchKernelGGL((k_spmv_pc<T, L, false>), dim3(g, rep), dim3(kBlock), 0, s, A, t, x, inv, y, st);
}

// the SELL-64 product: two slices per wave when the view says so (FP32, one
// case), else one
template <class T, bool NT, bool PC, bool C16>
void launch_sell(const SellView<T>& sell, const Tiles& t, const T* x, const T* inv, T* y, const KState* st, int rep, hipStream_t s) {
  if constexpr (std::is_same<T, float>::value) {
    if (sell.two) {
      // two slices per wave: kBlock / kWave waves per block
      const int nsl = (sell.n + 63) / 64;
      const int g2 = grid_for((nsl + 1) / 2, kBlock / kWave);
      hipLaunchKernelGGL((k_spmv_sell2<T, NT, PC, C16>), dim3(g2, rep), dim3(kBlock), 0, s, sell, t, x, inv, y, st);
      return;
    }
  }
  hipLaunchKernelGGL((k_spmv_sell<T, NT, PC, C16>), dim3(grid_for(sell.n), rep), dim3(kBlock), 0, s, sell, t, x, inv, y,
                     st);
}

template <class T, bool NT, bool PC>
void launch_sell_c(const SellView<T>& sell, const Tiles& t, const T* x, const T* inv, T* y, const KState* st,
                   int rep, hipStream_t s) {
  if (sell.col16) {
    // 16-bit column offsets exist for the FP32 inner order only
    if constexpr (std::is_same<T, float>::value)
      launch_sell<T, NT, PC, true>(sell, t, x, inv, y, st, rep, s);
    else
      throw std::logic_error("16-bit SELL columns in an FP64 product");
  } else {
    launch_sell<T, NT, PC, false>(sell, t, x, inv, y, st, rep, s);
  }
}

// y = M^-1 A x (rep vectors x and y, one after the other) with the CSR kernel at L lanes per row, or with the
// SELL-64 copy for L = 0 (sell must then be set)
template <class T>
void launch_spmv(int L, int nt, const CsrView<T>& A, const SellView<T>& sell, const Tiles& t, const T* x, const T* inv,
                 T* y, const KState* st, hipStream_t s, int rep = 1) {
  switch (L) {
    case 0: {
      if (!sell.ptr) throw std::logic_error("SELL-64 SpMV without a SELL copy");
      if (sell.n != A.n) throw std::logic_error("SELL-64 copy of another size");
      if (nt && inv)
        launch_sell_c<T, true, true>(sell, t, x, inv, y, st, rep, s);
      else if (nt)
        launch_sell_c<T, true, false>(sell, t, x, inv, y, st, rep, s);
      else if (inv)
        launch_sell_c<T, false, true>(sell, t, x, inv, y, st, rep, s);
      else
        launch_sell_c<T, false, false>(sell, t, x, inv, y, st, rep, s);
      break;
    }
    case 1: launch_spmv_l<T, 1>(nt != 0, A, t, x, inv, y, st, rep, s); break;
    case 2: launch_spmv_l<T, 2>(nt != 0, A, t, x, inv, y, st, rep, s); break;
    case 4: launch_spmv_l<T, 4>(nt != 0, A, t, x, inv, y, st, rep, s); break;
    case 16: launch_spmv_l<T, 16>(nt != 0, A, t, x, inv, y, st, rep, s); break;
    default: launch_spmv_l<T, 8>(nt != 0, A, t, x, inv, y, st, rep, s); break;
  }
}

template <class T>
SellView<T> sell_of(const KWork& w, int n, int variant = -1) {
  const int sv = variant < 0 ? w.sell_v : variant;
  SellView<T> v;
  if (w.sell[sv].ptr && w.sell_vals[sv]) {
    v.n = n;
    v.ptr = w.sell[sv].ptr;
    v.row = w.sell[sv].row;
    v.col = w.sell[sv].col;
    v.col16 = w.sell[sv].col16;
    v.val = static_cast<const T*>(w.sell_vals[sv]);
    v.scase = w.sell[sv].scase;
    v.tiled = !v.row || kSellSigma[sv] <= kBlock;
    v.two = std::is_same<T, float>::value && !v.scase && (w.sell2 > 0 || (w.sell2 < 0 && n >= (1 << 20))) ? 1 : 0;
  }
  return v;
}

// ---- Gram-Schmidt kernels.  Thread t of a tile handles R rows in chunks of
// VW consecutive rows (VW = 16 bytes of T, at most R): chunk q covers rows
// a + (q * kBlock + t) * VW ... + VW - 1.  A block whose tile start and
// column stride are multiples of VW loads each chunk with one 16-byte vector
// load; any other block (a tile of a later case in a batch) loads the same
// rows one by one, so the arithmetic and its order never depend on alignment.
template <class T>
struct Vec16;
template <>
struct Vec16<float> {
  using type = float4;
  static constexpr int n = 4;
};
template <>
struct Vec16<double> {
  using type = double2;
  static constexpr int n = 2;
};

// 16 bytes through a non-temporal load (the basis is streamed once per pass)
template <class T>
__device__ __forceinline__ typename Vec16<T>::type load16_nt(const T* p) {
  using E = T __attribute__((ext_vector_type(Vec16<T>::n)));
  const E e = __builtin_nontemporal_load(reinterpret_cast<const E*>(p));
  typename Vec16<T>::type v;
#pragma unroll
  for (int u = 0; u < Vec16<T>::n; ++u) reinterpret_cast<T*>(&v)[u] = e[u];
  return v;
}

template <class T, int VW, bool NT = false>
__device__ __forceinline__ void load_chunk(const T* __restrict__ p, size_t i0, size_t end, bool vec, double* out) {
  if constexpr (VW == Vec16<T>::n) {
    if (vec && i0 + VW <= end) {
      const typename Vec16<T>::type v =
          NT ? load16_nt<T>(p + i0) : *reinterpret_cast<const typename Vec16<T>::type*>(p + i0);
      const T* e = reinterpret_cast<const T*>(&v);
#pragma unroll
      for (int u = 0; u < VW; ++u) out[u] = static_cast<double>(e[u]);
      return;
    }
  }
#pragma unroll
  for (int u = 0; u < VW; ++u) out[u] = i0 + u < end ? static_cast<double>(p[i0 + u]) : 0.0;
}

template <class T, int VW>
__device__ __forceinline__ void store_chunk(T* __restrict__ p, size_t i0, size_t end, bool vec, const T* in) {
  if constexpr (VW == Vec16<T>::n) {
    if (vec && i0 + VW <= end) {
      typename Vec16<T>::type v;
      T* e = reinterpret_cast<T*>(&v);
#pragma unroll
      for (int u = 0; u < VW; ++u) e[u] = in[u];
      *reinterpret_cast<typename Vec16<T>::type*>(p + i0) = v;
      return;
    }
  }
#pragma unroll
  for (int u = 0; u < VW; ++u)
    if (i0 + u < end) p[i0 + u] = in[u];
}

template <class T, int R>
struct GsShape {
  static constexpr int VW = R < Vec16<T>::n ? R : Vec16<T>::n;
  static constexpr int NC = R / VW;
  __device__ static size_t row0(int a, int q) {
    return static_cast<size_t>(a) + (static_cast<size_t>(q) * kBlock + threadIdx.x) * VW;
  }
  __device__ static bool vec_ok(int a, size_t ld) { return (a % Vec16<T>::n) == 0 && (ld % Vec16<T>::n) == 0; }
  // every chunk of this thread lies inside the vector (and, when a chunk is
  // 16 bytes, loads as one aligned 16-byte vector)
  __device__ static bool whole(int a, size_t end, size_t ld) {
    return (VW < Vec16<T>::n || vec_ok(a, ld)) && row0(a, NC - 1) + VW <= end;
  }
  // ... and every chunk is 16 bytes
  __device__ static bool full(int a, size_t end, size_t ld) { return VW == Vec16<T>::n && whole(a, end, ld); }
};

// VW consecutive elements at p, all inside the vector, loaded non-temporally
// as they are (one 16-byte load when VW fills it); nothing waits for them
// until the values are used
template <class T, int VW>
__device__ __forceinline__ void load_raw(const T* p, T (&e)[VW]) {
  if constexpr (VW == Vec16<T>::n) {
    using E = T __attribute__((ext_vector_type(VW)));
    const E v = __builtin_nontemporal_load(reinterpret_cast<const E*>(p));
#pragma unroll
    for (int u = 0; u < VW; ++u) e[u] = v[u];
  } else {
#pragma unroll
    for (int u = 0; u < VW; ++u) e[u] = __builtin_nontemporal_load(p + u);
  }
}

// f(integral_constant<int, c>) for c = rest in 1..7 (nothing for 0): a batch
// of the last rest basis vectors with its size known at compile time
template <class F>
__device__ __forceinline__ void with_rest(int rest, F&& f) {
  switch (rest) {
    case 1: f(std::integral_constant<int, 1>{}); break;
    case 2: f(std::integral_constant<int, 2>{}); break;
    case 3: f(std::integral_constant<int, 3>{}); break;
    case 4: f(std::integral_constant<int, 4>{}); break;
    case 5: f(std::integral_constant<int, 5>{}); break;
    case 6: f(std::integral_constant<int, 6>{}); break;
    case 7: f(std::integral_constant<int, 7>{}); break;
    default: break;
  }
}

// acc[kk] += sum over the thread's whole chunks of w_i V_{k0+kk},i for
// kk < NB: every load issued before any use, the products added chunk by
// chunk and element by element, as the element path adds them
template <class T, class S, int NB>
__device__ __forceinline__ void dot_batch(const T* __restrict__ V, size_t ld, int k0, int a, const double* wr,
                                          double* acc) {
  T e[NB][S::NC][S::VW];
#pragma unroll
  for (int kk = 0; kk < NB; ++kk)
#pragma unroll
    for (int q = 0; q < S::NC; ++q) load_raw<T, S::VW>(V + static_cast<size_t>(k0 + kk) * ld + S::row0(a, q), e[kk][q]);
#pragma unroll
  for (int kk = 0; kk < NB; ++kk)
#pragma unroll
    for (int q = 0; q < S::NC; ++q)
#pragma unroll
      for (int u = 0; u < S::VW; ++u) acc[kk] += wr[q * S::VW + u] * static_cast<double>(e[kk][q][u]);
}

// sacc[u] += sgn * c[k] V_k,i0+u for k = k0 .. k0 + NB - 1 in that order
// (sgn -1: the Gram-Schmidt update, +1: the solution update); the NB loads
// issued before any use
template <class T, int VW, int NB, bool Sub>
__device__ __forceinline__ void axpy_batch(const T* __restrict__ V, size_t ld, int k0, size_t i0, const double* c,
                                           double* sacc) {
  T e[NB][VW];
#pragma unroll
  for (int kk = 0; kk < NB; ++kk) load_raw<T, VW>(V + static_cast<size_t>(k0 + kk) * ld + i0, e[kk]);
#pragma unroll
  for (int kk = 0; kk < NB; ++kk)
#pragma unroll
    for (int u = 0; u < VW; ++u) {
      if constexpr (Sub)
        sacc[u] -= c[k0 + kk] * static_cast<double>(e[kk][u]);
      else
        sacc[u] += c[k0 + kk] * static_cast<double>(e[kk][u]);
    }
}

// the same over k = 0 .. nk - 1: batches of 8, then one of the rest
template <class T, int VW, bool Sub>
__device__ __forceinline__ void axpy_all(const T* __restrict__ V, size_t ld, int nk, size_t i0, const double* c,
                                         double* sacc) {
  int k = 0;
  for (; k + 8 <= nk; k += 8) axpy_batch<T, VW, 8, Sub>(V, ld, k, i0, c, sacc);
  with_rest(nk - k, [&](auto nb) { axpy_batch<T, VW, decltype(nb)::value, Sub>(V, ld, k, i0, c, sacc); });
}

// ---- partial[k][b] = sum over tile b of w_i V_k,i, k = 0..it (k-major, so
// that the per-k reduction over the tiles reads contiguously; the row stride
// is the tile count, pstride only bounds the capacity).  The k run in chunks
// of 8; block (b, g) takes chunks g * cpb .. (g + 1) * cpb - 1 of tile b, so
// a small system spreads its chunks over more blocks (each chunk's sums are
// the same whichever block computes them).  A thread whose chunks are 16
// bytes issues the loads of a chunk of 8 vectors before it uses any; with
// Batch (small grids, see k_maxpy_norm) it does so for every whole chunk and
// for the last chunk's few vectors too.  The sums are the same either way.
template <class T, int R, bool Batch>
__global__ void __launch_bounds__(kBlock) k_mdot(const T* __restrict__ V, size_t ld, Tiles t, int it,
                                                 double* __restrict__ partial, int pstride, KState* st, int cpb) {
  using S = GsShape<T, R>;
  int a, e, c;
  t.range(blockIdx.x, a, e, c);
  const int reason = st[c].reason;
  if (threadIdx.x == 0 && blockIdx.y == 0) {
    // for the next launch, which may change reason while it runs
    int t0, t1;
    t.tiles_of(c, t0, t1);
    if (static_cast<int>(blockIdx.x) == t0) st[c].ended = reason;
  }
  if (reason) return;
  // each wave's sum of every k of the block, reduced over the waves once
  __shared__ double lds[kBlock / kWave][8 * ((kMaxRestart + 8) / 8)];
  const size_t end = static_cast<size_t>(e);
  const bool vec = S::vec_ok(a, ld);
  const T* w = V + static_cast<size_t>(it + 1) * ld;
  double wr[R];
#pragma unroll
  for (int q = 0; q < S::NC; ++q) load_chunk<T, S::VW>(w, S::row0(a, q), end, vec, wr + q * S::VW);
  const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
  const int kbeg = 8 * cpb * static_cast<int>(blockIdx.y);
  const int kend = min(it + 1, 8 * cpb * (static_cast<int>(blockIdx.y) + 1));
  const bool whole = Batch ? S::whole(a, end, ld) : S::full(a, end, ld);
  for (int k0 = kbeg; k0 < kend; k0 += 8) {
    double acc[8];
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) acc[kk] = 0.0;
    if (whole && k0 + 8 <= kend) {
      dot_batch<T, S, 8>(V, ld, k0, a, wr, acc);
    } else if (Batch && whole) {
      with_rest(kend - k0, [&](auto nb) { dot_batch<T, S, decltype(nb)::value>(V, ld, k0, a, wr, acc); });
    } else {
#pragma unroll
      for (int kk = 0; kk < 8; ++kk) {
        const int k = k0 + kk;
        if (k <= it) {
          const T* vk = V + static_cast<size_t>(k) * ld;
#pragma unroll
          for (int q = 0; q < S::NC; ++q) {
            double v[S::VW];
            load_chunk<T, S::VW>(vk, S::row0(a, q), end, vec, v);
#pragma unroll
            for (int u = 0; u < S::VW; ++u) acc[kk] += wr[q * S::VW + u] * v[u];
          }
        }
      }
    }
    const double sk = wave_sum8(acc);
    if ((lane & 7) == 0) lds[wid][k0 - kbeg + (lane >> 3)] = sk;
  }
  __syncthreads();
  for (int j = threadIdx.x; j < kend - kbeg; j += kBlock) {
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < kBlock / kWave; ++q) s += lds[q][j];
    partial[static_cast<size_t>(kbeg + j) * t.ntile + blockIdx.x] = s;
  }
}

// Sum of p[b] over b = b0 + threadIdx.x, + kBlock, ... below b1, added in
// that order; the loads of 8 consecutive terms are issued before any is
// added (indices clamped into the range, the clamped terms never added).
__device__ __forceinline__ double strided_sum(const double* __restrict__ p, int b0, int b1) {
  double v = 0.0;
  for (int b = b0 + static_cast<int>(threadIdx.x); b < b1; b += 8 * kBlock) {
    double x[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) x[u] = p[min(b + u * kBlock, b1 - 1)];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (b + u * kBlock < b1) v += x[u];
  }
  return v;
}

// The same for interleaved pairs: s0 = sum of p[2b], s1 = sum of p[2b + 1].
__device__ __forceinline__ void strided_sum2(const double* __restrict__ p, int n, double& s0, double& s1) {
  s0 = 0.0;
  s1 = 0.0;
  for (int b = static_cast<int>(threadIdx.x); b < n; b += 8 * kBlock) {
    double x0[8], x1[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int q = min(b + u * kBlock, n - 1);
      x0[u] = p[2 * q];
      x1[u] = p[2 * q + 1];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (b + u * kBlock < n) {
        s0 += x0[u];
        s1 += x1[u];
      }
  }
}

// ---- w = scale_it w - sum_k hcol_k scale_k V_k ; ||w||^2 per tile into norms.  With Batch
// (grids too small to hide memory latency with many waves) each thread
// issues the loads of up to 8 basis vectors before it uses any; otherwise it
// streams them one after the other and the resident waves hide the latency
// (batched loads measured slower there).  The subtractions run in the same
// order either way.
template <class T, int R, bool Batch>
__global__ void __launch_bounds__(kBlock) k_maxpy_norm(T* __restrict__ V, size_t ld, Tiles t, int it,
                                                       double* __restrict__ norms, const KState* st) {
  using S = GsShape<T, R>;
  int a, e, c;
  t.range(blockIdx.x, a, e, c);
  const KState* sc = st + c;
  if (sc->reason) return;
  __shared__ double cf[kMaxRestart + 1];
  __shared__ double lds[kBlock / kWave];
  for (int k = threadIdx.x; k <= it; k += kBlock) cf[k] = sc->hcol[it & 1][k] * sc->scale[k];
  const double sw = sc->scale[it];
  __syncthreads();
  const size_t end = static_cast<size_t>(e);
  const bool vec = S::vec_ok(a, ld);
  const bool whole = Batch && S::whole(a, end, ld);
  T* w = V + static_cast<size_t>(it + 1) * ld;
  double nrm = 0.0;
#pragma unroll
  for (int q = 0; q < S::NC; ++q) {
    const size_t i0 = S::row0(a, q);
    double sacc[S::VW];
    load_chunk<T, S::VW>(w, i0, end, vec, sacc);
#pragma unroll
    for (int u = 0; u < S::VW; ++u) sacc[u] *= sw;
    if (whole) {
      axpy_all<T, S::VW, true>(V, ld, it + 1, i0, cf, sacc);
    } else {
      for (int k = 0; k <= it; ++k) {
        double v[S::VW];
        load_chunk<T, S::VW, true>(V + static_cast<size_t>(k) * ld, i0, end, vec, v);
#pragma unroll
        for (int u = 0; u < S::VW; ++u) sacc[u] -= cf[k] * v[u];
      }
    }
    T out[S::VW];
#pragma unroll
    for (int u = 0; u < S::VW; ++u) {
      out[u] = static_cast<T>(sacc[u]);
      if (i0 + u < end) nrm += static_cast<double>(out[u]) * static_cast<double>(out[u]);
    }
    store_chunk<T, S::VW>(w, i0, end, vec, out);
  }
  nrm = block_sum(nrm, lds);
  if (threadIdx.x == 0) norms[blockIdx.x] = nrm;
}

// ---- Hessenberg column, Givens rotations, convergence test of step it of
// one case, by one block, from the norms of its tiles.  The column and the
// previous rotations are staged in LDS and the scalars that thread 0 needs load
// with them, so its serial rotation sweep waits for no global load.
struct ArnoldiScalars {
  double g_it, rnorm, ttol, abstol, dtol, rnorm0;
  int its, maxit;
};

// The rest, once staged and published: s (thread 0) is the squared norm of
// the new basis vector.  Every thread of the block calls it.
__device__ void arnoldi_close(double s, int it, int m, KState* s_, const ArnoldiScalars& q, double* col, double* cc,
                              double* ss) {
  const int ld = m + 1;
  if (threadIdx.x == 0) {
    const double tt = sqrt(s);
    col[it + 1] = tt;
    s_->scale[it + 1] = tt != 0.0 ? 1.0 / tt : 1.0;
    double hapbnd = fabs(tt / q.g_it);
    if (hapbnd > 1.e-30) hapbnd = 1.e-30;
    const bool hapend = tt < hapbnd;
    double carry = col[0];  // col[j] as the rotations before j left it
    double c1 = cc[0], s1 = ss[0], h1 = it > 0 ? col[1] : 0.0;
    for (int j = 1; j <= it; ++j) {
      // the next rotation's operands load while this one's products run
      const int jn = j < it ? j : j - 1;
      const double c2 = cc[jn], s2 = ss[jn], h2 = col[jn + 1];
      col[j - 1] = c1 * carry + s1 * h1;
      carry = c1 * h1 - s1 * carry;
      c1 = c2;
      s1 = s2;
      h1 = h2;
    }
    double res;
    int reason = 0;
    if (!hapend) {
      const double hv = carry, hn = tt;
      const double tr = sqrt(hv * hv + hn * hn);
      if (tr == 0.0) {
        reason = kDivergedNull;
        res = q.rnorm;
        col[it] = carry;
      } else {
        const double c = hv / tr, sn = hn / tr;
        s_->cc[it] = c;
        s_->ss[it] = sn;
        const double g1 = -(sn * q.g_it);
        s_->grs[it + 1] = g1;
        s_->grs[it] = c * q.g_it;
        col[it] = c * hv + sn * hn;
        res = fabs(g1);
      }
    } else {
      res = 0.0;
      col[it] = carry;
    }
    s_->it = it + 1;
    s_->its = q.its + 1;
    s_->rnorm = res;
    if (!reason) {
      reason = conv_check(q.ttol, q.abstol, q.dtol, q.rnorm0, res);
      if (hapend && !reason) reason = kDivergedBreakdown;
    }
    if (!reason && q.its + 1 >= q.maxit) reason = kDivergedIts;
    s_->reason = reason;
  }
  __syncthreads();
  for (int j = threadIdx.x; j <= it + 1; j += kBlock) Hm(s_, ld, j, it) = col[j];
}

// step it of one case from the norms of its tiles, by one block
__device__ void arnoldi_finalize(const double* norms, const Tiles& t, int c, int it, int m, KState* s_) {
  __shared__ double lds[kBlock / kWave];
  __shared__ double col[kMaxRestart + 2], cc[kMaxRestart + 1], ss[kMaxRestart + 1];
  int t0, t1;
  t.tiles_of(c, t0, t1);
  for (int j = threadIdx.x; j <= it; j += kBlock) {
    col[j] = s_->hcol[it & 1][j];
    cc[j] = s_->cc[j];
    ss[j] = s_->ss[j];
  }
  const ArnoldiScalars q = {s_->grs[it], s_->rnorm,  s_->ttol, s_->abstol, s_->dtol,
                            s_->rnorm0,  s_->its, s_->maxit};
  double s = strided_sum(norms, t0, t1);
  s = block_sum(s, lds);  // contains the barrier that publishes col/cc/ss
  arnoldi_close(s, it, m, s_, q, col, cc, ss);
}

// ... as a launch of its own (one block per case)
__global__ void __launch_bounds__(kBlock) k_arnoldi_finalize(const double* norms, Tiles t, int it, int m, KState* st) {
  KState* s_ = st + blockIdx.x;
  if (s_->reason) return;
  arnoldi_finalize(norms, t, blockIdx.x, it, m, s_);
}

// ---- hcol[k] = scale_k scale_it * sum over the case's tiles of dots[k][b]
// (block (k, case), k = 0..it), and with fin the finalisation of step it - 1
// (block (it + 1, case)), which so costs no launch of its own: the product of
// step it and its dots use the unscaled basis vector and do not wait for it.
// The blocks form scale_it themselves from the tile norms (in the
// finalisation's order, the same bits); hcol and the norms alternate between
// two arrays by step, so the finalisation reads what nobody writes here, and
// whether the solve had ended is read from the multi-dot's copy.  Where the
// finalisation ends it now, the column is never used.  With the finalisation
// as a launch between the update and the next product (4.8 us a step) the
// pressure solves of the channel took 374.6 ms (2.53 M rows, FP32 cycles), 98.2
// (748 K), 75.4 (546 K, FP64); beside the sums 361.6, 93.1, 71.0.
__global__ void __launch_bounds__(kBlock) k_orth(const double* dots, const double* norms, Tiles t, int it, int m,
                                                 int fin, KState* st) {
  KState* s = st + blockIdx.y;
  const int ended = s->ended, k = blockIdx.x;
  if (k > it) {
    if (!ended) arnoldi_finalize(norms, t, blockIdx.y, it - 1, m, s);
    return;
  }
  __shared__ double lds[2 * kBlock / kWave];
  int t0, t1;
  t.tiles_of(blockIdx.y, t0, t1);
  // (column k: contiguous over tiles; everything loads before the state is tested)
  double v = strided_sum(dots + static_cast<size_t>(k) * t.ntile, t0, t1);
  double n2 = fin ? strided_sum(norms, t0, t1) : 0.0;
  const double sk = s->scale[k], sit = fin ? 0.0 : s->scale[it];
  if (ended) return;
  // both block sums behind one barrier, in block_sum's order
  v = wave_sum(v);
  if (fin) n2 = wave_sum(n2);
  const int wid = threadIdx.x / kWave;
  if ((threadIdx.x & (kWave - 1)) == 0) {
    lds[wid] = v;
    lds[kBlock / kWave + wid] = n2;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double a = 0.0, b = 0.0;
#pragma unroll
    for (int w = 0; w < kBlock / kWave; ++w) {
      a += lds[w];
      b += lds[kBlock / kWave + w];
    }
    double sw = sit;
    if (fin) {
      const double tt = sqrt(b);
      sw = tt != 0.0 ? 1.0 / tt : 1.0;
    }
    s->hcol[it & 1][k] = a * (k == it ? sw : sk) * sw;
  }
}

// ---- one case of at most kBlock tiles of kBlock rows, without ILU, on the
// SELL-64 copy: an Arnoldi step in two launches.  Such a step moves a few MB
// that the L2s hold, and a launch costs 1.6-2 us before its first load
// returns, so what sets the time is the number of launches and the chain of
// loads in each (32,768 rows, FP64, step 15 of 30: product 5.0 with the
// finalisation, dots 3.8, sums 3.0, update 3.9 us as four launches; 4.5 and 5.9
// as two, and four SIMPLE steps of the cavity 40.3 -> 29.9 ms).  An iteration of
// captured GMRES(30), two launches against four, us: 4,096 rows FP64 10.9 and 13.9,
// mixed 11.6 and 15.0; 32,768 11.0 and 14.2, 11.0 and 14.0; 65,536 12.5 and 15.5, 12.0 and
// 14.9.  kBlock tiles are what the sums below are written for (four 64-tile
// pieces a wave); every block reads all tiles' sums, so the gain ends not far above.

// The product w = M^-1 A V_it, and its dots with V_0..V_it: a block's rows are
// one tile, so each thread still holds its w.  The first 8 basis vectors load
// ahead of the product, each further 8 ahead of the sums before it.  With a
// row map (64-row windows) the rows come back to their own threads through
// LDS.  The sums are those of k_mdot with one row per thread, bit for bit.
template <class T, bool NT, bool PC, bool C16>
__global__ void __launch_bounds__(kBlock) k_spmv_dots(SellView<T> A, Tiles t, T* V, size_t ld,
                                                      const T* __restrict__ inv, KState* st, int it,
                                                      double* __restrict__ dots) {
  const int reason = st->reason;  // (used once the first loads are on their way)
  __shared__ T wrow[kBlock];
  __shared__ double lds[kBlock / kWave][8 * ((kMaxRestart + 8) / 8)];
  const int b = xcd_block(blockIdx.x, gridDim.x);
  const int a = b * kBlock, pos = a + static_cast<int>(threadIdx.x);
  const bool in = pos < A.n;
  const T* vp = V + (in ? pos : A.n - 1);  // past the end: any element, times w = 0
  T e[8];
#pragma unroll
  for (int u = 0; u < 8; ++u) e[u] = vp[static_cast<size_t>(min(u, it)) * ld];
  T w = T(0);
  if (in) {
    const int sl = __builtin_amdgcn_readfirstlane(pos >> 6);
    int row;  // -1 where the solve has ended
    w = sell_row_any<T, NT, PC, C16>(A, t, V + static_cast<size_t>(it) * ld, inv, st, sl, pos, A.ptr[sl],
                                     A.ptr[sl + 1], row);
    if (A.row && row >= 0) wrow[row - a] = w;
  }
  // for the next launch, which may change reason while it runs
  if (blockIdx.x == 0 && threadIdx.x == 0) st->ended = reason;
  if (reason) return;
  if (A.row) {
    __syncthreads();
    w = in ? wrow[threadIdx.x] : T(0);
  }
  if (in) V[static_cast<size_t>(it + 1) * ld + pos] = w;
  const double wd = static_cast<double>(w);
  const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
  for (int k0 = 0; k0 <= it; k0 += 8) {
    T next[8];
    const bool more = k0 + 8 <= it;
    if (more) {
#pragma unroll
      for (int u = 0; u < 8; ++u) next[u] = vp[static_cast<size_t>(min(k0 + 8 + u, it)) * ld];
    }
    double acc[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) acc[u] = k0 + u <= it ? 0.0 + wd * static_cast<double>(e[u]) : 0.0;
    const double sk = wave_sum8(acc);
    if ((lane & 7) == 0) lds[wid][k0 + (lane >> 3)] = sk;
    if (more) {
#pragma unroll
      for (int u = 0; u < 8; ++u) e[u] = next[u];
    }
  }
  __syncthreads();
  for (int j = threadIdx.x; j <= it; j += kBlock) {
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < kBlock / kWave; ++q) s += lds[q][j];
    dots[static_cast<size_t>(j) * t.ntile + b] = s;
  }
}

// wave sums (four 64-tile pieces of up to kBlock tiles each, in tile order) of
// 8 columns of tile values, the columns' sums in lanes 8 k ..; the order is
// that of strided_sum and block_sum
__device__ __forceinline__ double tile_sums8(const double* p, int ntile, int k0, int kn) {
  const int lane = threadIdx.x & (kWave - 1);
  double x[4][8];
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int k = min(k0 + u, kn - 1), b = min(64 * c + lane, ntile - 1);
      x[c][u] = 64 * c < ntile ? p[static_cast<size_t>(k) * ntile + b] : 0.0;
    }
  double s = 0.0;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    if (64 * c >= ntile) break;
#pragma unroll
    for (int u = 0; u < 8; ++u) x[c][u] = 64 * c + lane < ntile ? x[c][u] : 0.0;
    s += wave_sum8(x[c]);
  }
  return s;
}

// the same for one column, its sum in every lane
__device__ __forceinline__ double tile_sum(const double* p, int ntile) {
  const int lane = threadIdx.x & (kWave - 1);
  double x[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) x[c] = c < 4 && 64 * c + lane < ntile ? p[min(64 * c + lane, ntile - 1)] : 0.0;
  const double v = wave_sum8(x);
  double s = 0.0;
#pragma unroll
  for (int c = 0; c < 4; ++c)
    if (64 * c < ntile) s += __shfl(v, 8 * c, kWave);
  return s;
}

// The rest of the step: every block sums the tiles' dots and norms itself (the
// order and bits of k_orth), then updates its tile as k_maxpy_norm does.  The
// block past the tiles finalises step it - 1 (fin).
template <class T>
__global__ void __launch_bounds__(kBlock) k_orth_update(T* V, size_t ld, Tiles t, const double* __restrict__ dots,
                                                        const double* norms, double* norms_out, int it, int m, int fin,
                                                        KState* st) {
  const int ended = st->ended;  // (used once the first loads are on their way)
  if (static_cast<int>(blockIdx.x) == t.ntile) {
    if (!ended) arnoldi_finalize(norms, t, 0, it - 1, m, st);
    return;
  }
  __shared__ double cf[kMaxRestart + 1 + 8];
  __shared__ double lds[kBlock / kWave];
  const int a = blockIdx.x * kBlock, row = a + static_cast<int>(threadIdx.x);
  const bool in = row < t.n;
  T* vp = V + (in ? row : t.n - 1);
  T e[8];
#pragma unroll
  for (int u = 0; u < 8; ++u) e[u] = vp[static_cast<size_t>(min(u, it)) * ld];
  const T wv = in ? vp[static_cast<size_t>(it + 1) * ld] : T(0);
  const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
  double sw;
  if (fin) {
    const double tt = sqrt(tile_sum(norms, t.ntile));
    sw = tt != 0.0 ? 1.0 / tt : 1.0;
  } else {
    sw = st->scale[it];
  }
  for (int k0 = 8 * wid; k0 <= it; k0 += 8 * (kBlock / kWave)) {
    const double v = tile_sums8(dots, t.ntile, k0, it + 1);
    if (ended) return;
    const int k = k0 + (lane >> 3);
    if ((lane & 7) == 0 && k <= it) {
      const double sk = k == it ? sw : st->scale[k];
      const double h = v * sk * sw;
      if (blockIdx.x == 0) st->hcol[it & 1][k] = h;
      cf[k] = h * sk;
    }
  }
  if (ended) return;
  __syncthreads();
  double acc = static_cast<double>(wv) * sw;
  for (int k0 = 0; k0 <= it; k0 += 8) {
    T next[8];
    const bool more = k0 + 8 <= it;
    if (more) {
#pragma unroll
      for (int u = 0; u < 8; ++u) next[u] = vp[static_cast<size_t>(min(k0 + 8 + u, it)) * ld];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (k0 + u <= it) acc -= cf[k0 + u] * static_cast<double>(e[u]);
    if (more) {
#pragma unroll
      for (int u = 0; u < 8; ++u) e[u] = next[u];
    }
  }
  const T out = static_cast<T>(acc);
  double nrm = in ? 0.0 + static_cast<double>(out) * static_cast<double>(out) : 0.0;
  if (in) vp[static_cast<size_t>(it + 1) * ld] = out;
  nrm = block_sum(nrm, lds);
  if (threadIdx.x == 0) norms_out[blockIdx.x] = nrm;
}

template <class T, bool NT, bool PC>
void launch_spmv_dots_c(const SellView<T>& sell, const Tiles& t, T* V, size_t ld, const T* inv, KState* st,
                        int it, double* dots, hipStream_t s) {
  if (sell.col16) {
    if constexpr (std::is_same<T, float>::value)
      hipLaunchKernelGGL((k_spmv_dots<T, NT, PC, true>), dim3(t.ntile), dim3(kBlock), 0, s, sell, t, V, ld, inv, st,
                         it, dots);
    else
      throw std::logic_error("16-bit SELL columns in an FP64 product");
  } else {
    hipLaunchKernelGGL((k_spmv_dots<T, NT, PC, false>), dim3(t.ntile), dim3(kBlock), 0, s, sell, t, V, ld, inv, st,
                       it, dots);
  }
}

// V_it+1 = M^-1 A V_it on the one-slice SELL-64 copy and its dots (t: tiles of kBlock rows)
template <class T>
void launch_spmv_dots(int nt, const SellView<T>& sell, const Tiles& t, T* V, size_t ld, const T* inv,
                      KState* st, int it, double* dots, hipStream_t s) {
  if (!sell.ptr || sell.two || sell.scase || !sell.tiled || t.tile != kBlock || t.ntile > kBlock || t.n != sell.n)
    throw std::logic_error("product with dots on another layout");
  if (nt && inv)
    launch_spmv_dots_c<T, true, true>(sell, t, V, ld, inv, st, it, dots, s);
  else if (nt)
    launch_spmv_dots_c<T, true, false>(sell, t, V, ld, inv, st, it, dots, s);
  else if (inv)
    launch_spmv_dots_c<T, false, true>(sell, t, V, ld, inv, st, it, dots, s);
  else
    launch_spmv_dots_c<T, false, false>(sell, t, V, ld, inv, st, it, dots, s);
}

// ---- the end of a cycle, one block per case: the finalisation of its last step
// it (fin), then the back substitution R y = g on the completed columns, y_j
// scaled by scale_j.  One wavefront solves it, column-oriented: lane i keeps
// t_i, and once y_r is known every lane i < r subtracts H(i,r) y_r; the columns
// are staged in LDS, so its chain is a division and an exchange per column and
// no global load (50 columns: 30 us with the loads in it, 6 without).  The
// number of terms of the update goes to the state's pad word.
__global__ void __launch_bounds__(kBlock) k_build_y(const double* norms, Tiles t, int it, int m, int fin, KState* st) {
  KState* s = st + blockIdx.x;
  constexpr int kCol = kMaxRestart + 1;
  __shared__ double hs[kMaxRestart * kCol], g[kMaxRestart];
  if (fin && !s->reason) arnoldi_finalize(norms, t, blockIdx.x, it, m, s);
  __syncthreads();  // the block's own writes to the state
  int* nupd = reinterpret_cast<int*>(&s->pad);
  const int lane = threadIdx.x;
  const int k = s->it - 1;
  if (k < 0) {
    if (lane == 0) *nupd = 0;
    return;
  }
  for (int j = threadIdx.x; j < (k + 1) * (k + 1); j += kBlock) {
    const int c = j / (k + 1), r = j - c * (k + 1);
    if (r <= c) hs[c * kCol + r] = Hm(s, m + 1, r, c);
  }
  if (lane <= k) g[lane] = s->grs[lane];
  __syncthreads();
  if (lane >= kWave) return;
  double tl = lane <= k ? g[lane] : 0.0;
  double y = 0.0;
  bool broke = false;
  for (int r = k; r >= 0; --r) {
    const double hrr = hs[r * kCol + r], hir = lane < r ? hs[r * kCol + lane] : 0.0;
    if (hrr == 0.0) {
      broke = true;
      break;
    }
    const double yr = __shfl(tl, r, kWave) / hrr;
    if (lane == r) y = yr;
    if (lane < r) tl -= hir * yr;
  }
  if (broke) {
    if (lane == 0) {
      s->reason = kDivergedBreakdown;
      *nupd = 0;
    }
    return;
  }
  if (lane <= k) s->y[lane] = y * s->scale[lane];
  if (lane == 0) *nupd = k + 1;
}

// x += sum_k y_k V_k; with xrow (inner order) position i updates x[xrow[i]]
// (Batch as in k_maxpy_norm)
template <class T, class X, int R, bool Batch>
__global__ void __launch_bounds__(kBlock) k_update_x(const T* __restrict__ V, size_t ld, Tiles t, X* __restrict__ x,
                                                     const KState* st, const int* __restrict__ xrow, int rhs_n) {
  using S = GsShape<T, R>;
  int a, e, c;
  t.range(blockIdx.x, a, e, c);
  const size_t off = static_cast<size_t>(c) * rhs_n;  // as in k_residual_pc
  const KState* sc = st + c;
  const int nk = *reinterpret_cast<const int*>(&sc->pad);
  if (nk == 0) return;
  __shared__ double y[kMaxRestart + 1];
  for (int k = threadIdx.x; k < nk; k += kBlock) y[k] = sc->y[k];
  __syncthreads();
  const size_t end = static_cast<size_t>(e);
  const bool vec = S::vec_ok(a, ld);
  const bool whole = Batch && S::whole(a, end, ld);
#pragma unroll
  for (int q = 0; q < S::NC; ++q) {
    const size_t i0 = S::row0(a, q);
    double sacc[S::VW];
#pragma unroll
    for (int u = 0; u < S::VW; ++u) sacc[u] = 0.0;
    if (whole) {
      axpy_all<T, S::VW, false>(V, ld, nk, i0, y, sacc);
    } else {
      for (int k = 0; k < nk; ++k) {
        double v[S::VW];
        load_chunk<T, S::VW, true>(V + static_cast<size_t>(k) * ld, i0, end, vec, v);
#pragma unroll
        for (int u = 0; u < S::VW; ++u) sacc[u] += y[k] * v[u];
      }
    }
#pragma unroll
    for (int u = 0; u < S::VW; ++u)
      if (i0 + u < end) {
        const size_t r = xrow ? off + static_cast<size_t>(xrow[i0 + u - off]) : i0 + u;
        x[r] = static_cast<X>(static_cast<double>(x[r]) + sacc[u]);
      }
  }
}

// ---- v0 = M^-1 (b - A x); partial ||v0||^2 per tile.  The residual is
// formed in the precision X of the solution and the matrix A (FP64 for the
// mixed solve, whose Arnoldi cycle runs on an FP32 copy); v0 is stored in the
// basis type T and the norm is taken before that rounding when T and X
// differ.  Tiles of finished cases are skipped.
// With vpos (inner order) row i's value goes to v0[vpos[i]].
template <class T, class X>
__global__ void __launch_bounds__(kBlock) k_residual_pc(CsrView<X> A, Tiles t, const X* __restrict__ b,
                                                        const X* __restrict__ x, const X* __restrict__ inv,
                                                        T* __restrict__ v0, double* partial, int zero_guess,
                                                        const KState* st, const int* __restrict__ vpos, int rhs_n) {
  int a, e, c;
  t.range(blockIdx.x, a, e, c);
  if (st[c].done) return;
  // several right-hand sides of one matrix: case c's vectors start at c rhs_n
  const int off = c * rhs_n;
  a -= off;
  e -= off;
  b += off;
  x += off;
  v0 += off;
  __shared__ double lds[kBlock / kWave];
  double nrm = 0.0;
  for (int i = a + threadIdx.x; i < e; i += kBlock) {
    double r = static_cast<double>(b[i]);
    if (!zero_guess) {
      // the matrix streams once per restart: non-temporal, so it does not
      // evict what the cycle's kernels reuse
      const X s = csr_dot<X, X, true>(A.val, A.col, A.rowptr[i], A.rowptr[i + 1], 1, x, X(0));
      r -= static_cast<double>(s);
    }
    if (inv) r *= static_cast<double>(inv[i]);
    const X rx = static_cast<X>(r);
    v0[vpos ? vpos[i] : i] = static_cast<T>(rx);
    nrm += static_cast<double>(rx) * static_cast<double>(rx);
  }
  nrm = block_sum(nrm, lds);
  if (threadIdx.x == 0) partial[blockIdx.x] = nrm;
}

// ---- Jacobi inverses of the mixed solve: FP64 for the restart residual,
// FP32 for the Arnoldi cycle, both from the FP64 diagonal
// (inv32 by position in the inner order when pos32 is set)
__global__ void __launch_bounds__(kBlock) k_jacobi_mixed(CsrView<double> A, double* inv64, float* inv32,
                                                         const int* __restrict__ pos32) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= A.n) return;
  const double d = A.val[A.diag[i]];
  const double v = d != 0.0 ? 1.0 / d : 1.0;
  inv64[i] = v;
  inv32[pos32 ? pos32[i] : i] = static_cast<float>(v);
}

// ---- partial ||M^-1 b||^2 per tile (reference norm for a nonzero guess)
template <class T>
__global__ void __launch_bounds__(kBlock) k_pc_norm(Tiles t, const T* __restrict__ b, const T* __restrict__ inv,
                                                    double* partial, const KState* st, int rhs_n = 0) {
  int a, e, c;
  t.range(blockIdx.x, a, e, c);
  if (st[c].done) return;
  const int off = c * rhs_n;
  a -= off;
  e -= off;
  b += off;
  __shared__ double lds[kBlock / kWave];
  double nrm = 0.0;
  for (int i = a + threadIdx.x; i < e; i += kBlock) {
    double r = static_cast<double>(b[i]);
    if (inv) r *= static_cast<double>(inv[i]);
    const T rv = static_cast<T>(r);
    nrm += static_cast<double>(rv) * static_cast<double>(rv);
  }
  nrm = block_sum(nrm, lds);
  if (threadIdx.x == 0) partial[blockIdx.x] = nrm;
}

__global__ void __launch_bounds__(kBlock) k_snorm_final(const double* partial, Tiles t, KState* st) {
  __shared__ double lds[kBlock / kWave];
  int t0, t1;
  t.tiles_of(blockIdx.x, t0, t1);
  double s = 0.0;
  s = strided_sum(partial, t0, t1);
  s = block_sum(s, lds);
  if (threadIdx.x == 0) st[blockIdx.x].snorm = sqrt(s);
}

// ---- start of a GMRES cycle (one block per case).  The restart residual is
// the true one, so a passed test here ends the case's solve; in the mixed
// solve the iteration cap is applied here too, after the FP64 test.
__global__ void __launch_bounds__(kBlock) k_restart_finalize(const double* partial, Tiles t, KState* st, int first,
                                                             int guess_zero, int mixed) {
  KState* s_ = st + blockIdx.x;
  if (s_->done) {
    if (threadIdx.x == 0) s_->it = 0;
    return;
  }
  __shared__ double lds[kBlock / kWave];
  int t0, t1;
  t.tiles_of(blockIdx.x, t0, t1);
  double s = 0.0;
  s = strided_sum(partial, t0, t1);
  s = block_sum(s, lds);
  if (threadIdx.x != 0) return;
  const double res = sqrt(s);
  s_->grs[0] = res;
  s_->scale[0] = res != 0.0 ? 1.0 / res : 1.0;
  s_->it = 0;
  s_->cycles += 1;
  s_->rnorm = res;
  if (first) {
    s_->rnorm0 = guess_zero ? res : (s_->snorm != 0.0 ? s_->snorm : res);
    s_->ttol = fmax(s_->rtol * s_->rnorm0, s_->abstol);
  }
  int reason = res == 0.0 ? kConvergedAtol : conv_check(s_, res);
  if (mixed && !reason && s_->its >= s_->maxit) reason = kDivergedIts;
  s_->reason = reason;
  if (reason) s_->done = 1;
}

// ---- the headers of all cases to the host: stores into coherent pinned memory,
// then the count of such messages, which the host polls (one block)
__device__ __forceinline__ void publish(const KState* st, int ncase, const Mailbox& box) {
  for (int c = threadIdx.x; c < ncase; c += blockDim.x) {
    KHeader h;
    h.it = st[c].it;
    h.its = st[c].its;
    h.reason = st[c].reason;
    h.maxit = st[c].maxit;
    h.done = st[c].done;
    h.cycles = st[c].cycles;
    h.ended = st[c].ended;
    h.pad0 = 0;
    h.rnorm = st[c].rnorm;
    h.rnorm0 = st[c].rnorm0;
    h.ttol = st[c].ttol;
    h.snorm = st[c].snorm;
    box.host[c] = h;
  }
  __threadfence_system();
  __syncthreads();
  if (threadIdx.x == 0) {
    const unsigned n = *box.sent + 1;
    *box.sent = n;
    __hip_atomic_store(box.arrived, n, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

__global__ void __launch_bounds__(kBlock) k_publish(const KState* st, int ncase, Mailbox box) {
  publish(st, ncase, box);
}

// ---- end of a GMRES cycle, after the update of x (one thread per case).
// Plain solve: a set reason ends the case, then the iteration cap.  Mixed
// solve: a passed estimate, a breakdown of the FP32 cycle after which x was
// still updated, or the cap met inside the cycle is cleared and goes back to
// the FP64 residual, which applies the cap after its own test; a divergence
// ends the case, and so does a breakdown of the back substitution (no
// update: the next cycle would start from the same residual and break down
// the same way).  One block, which then publishes the headers.
__global__ void __launch_bounds__(kBlock) k_cycle_end(KState* st, int ncase, int mixed, Mailbox box) {
  for (int c = threadIdx.x; c < ncase; c += blockDim.x) {
    KState* s = st + c;
    if (s->done) continue;
    const int r = s->reason;
    if (!mixed) {
      if (r) {
        s->done = 1;
      } else if (s->its >= s->maxit) {
        s->reason = kDivergedIts;
        s->done = 1;
      }
    } else {
      const int nupd = *reinterpret_cast<const int*>(&s->pad);
      if ((r < 0 && r != kDivergedBreakdown && r != kDivergedIts) || (r == kDivergedBreakdown && nupd == 0))
        s->done = 1;
      else
        s->reason = 0;
    }
  }
  // (a thread publishes the cases it has just ended)
  publish(st, ncase, box);
}

// ---- solver state of every case at the start of a solve
__global__ void k_init_states(KState* st, int ncase, int maxit, double rtol, double abstol, double dtol) {
  for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < ncase; c += gridDim.x * blockDim.x) {
    KState* s = st + c;
    s->it = 0;
    s->its = 0;
    s->reason = 0;
    s->maxit = maxit;
    s->done = 0;
    s->ended = 0;
    s->cycles = 0;
    s->rnorm = s->rnorm0 = s->ttol = s->snorm = 0.0;
    s->rtol = rtol;
    s->abstol = abstol;
    s->dtol = dtol;
    s->pad = 0.0;
    s->beta = s->betaold = s->dpi = s->dpiold = s->alpha = 0.0;
  }
}

// ---- CG pieces (left-preconditioned, preconditioned residual norm)
template <class T>
__global__ void __launch_bounds__(kBlock) k_cg_start(CsrView<T> A, const T* b, T* x, const T* inv, T* r, T* z,
                                                     double* partial, int zero_guess) {
  __shared__ double lds[kBlock / kWave];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double zz = 0.0, zr = 0.0;
  if (i < A.n) {
    double rv = static_cast<double>(b[i]);
    if (zero_guess) {
      x[i] = T(0);
    } else {
      const T s = csr_dot<T, T, false>(A.val, A.col, A.rowptr[i], A.rowptr[i + 1], 1, x, T(0));
      rv -= static_cast<double>(s);
    }
    const T rt = static_cast<T>(rv);
    const T zt = inv ? static_cast<T>(static_cast<double>(rt) * static_cast<double>(inv[i])) : rt;
    r[i] = rt;
    z[i] = zt;
    zz = static_cast<double>(zt) * static_cast<double>(zt);
    zr = static_cast<double>(zt) * static_cast<double>(rt);
  }
  zz = block_sum(zz, lds);
  zr = block_sum(zr, lds);
  if (threadIdx.x == 0) {
    partial[2 * blockIdx.x] = zz;
    partial[2 * blockIdx.x + 1] = zr;
  }
}

__global__ void __launch_bounds__(kBlock) k_cg_start_final(const double* partial, int nblk, KState* st, int guess_zero) {
  __shared__ double lds[kBlock / kWave];
  double zz = 0.0, zr = 0.0;
  strided_sum2(partial, nblk, zz, zr);
  zz = block_sum(zz, lds);
  zr = block_sum(zr, lds);
  if (threadIdx.x != 0) return;
  const double dp = sqrt(zz);
  st->rnorm = dp;
  st->rnorm0 = guess_zero ? dp : (st->snorm != 0.0 ? st->snorm : dp);
  st->ttol = fmax(st->rtol * st->rnorm0, st->abstol);
  st->its = 0;
  st->beta = zr;
  st->reason = conv_check(st, dp);
}

// p = z + (beta/betaold) p  (p = z on the first iteration); checks on beta
template <class T>
__global__ void __launch_bounds__(kBlock) k_cg_p(int n, const T* z, T* p, KState* st, int i_it) {
  if (st->reason) return;
  const double beta = st->beta, betaold = st->betaold;
  if (beta == 0.0 || (i_it > 0 && beta * betaold < 0.0)) return;  // the finaliser records the reason
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  if (i_it == 0)
    p[i] = z[i];
  else
    p[i] = static_cast<T>(static_cast<double>(z[i]) + (beta / betaold) * static_cast<double>(p[i]));
}

template <class T>
__global__ void __launch_bounds__(kBlock) k_cg_spmv_dot(CsrView<T> A, const T* p, T* w, double* partial,
                                                        const KState* st, int i_it) {
  if (st->reason) return;
  const double beta = st->beta;
  if (beta == 0.0 || (i_it > 0 && beta * st->betaold < 0.0)) return;
  __shared__ double lds[kBlock / kWave];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double d = 0.0;
  if (i < A.n) {
    // the row's slots loaded in batches ahead of their gathers, summed in order
    const T s = csr_dot<T, T, false>(A.val, A.col, A.rowptr[i], A.rowptr[i + 1], 1, p, T(0));
    w[i] = s;
    d = static_cast<double>(p[i]) * static_cast<double>(s);
  }
  d = block_sum(d, lds);
  if (threadIdx.x == 0) partial[blockIdx.x] = d;
}

__global__ void __launch_bounds__(kBlock) k_cg_alpha(const double* partial, int nblk, KState* st, int i_it) {
  if (st->reason) return;
  __shared__ double lds[kBlock / kWave];
  double s = 0.0;
  s = strided_sum(partial, 0, nblk);
  s = block_sum(s, lds);
  if (threadIdx.x != 0) return;
  const double beta = st->beta;
  if (beta == 0.0) {
    st->reason = kConvergedAtol;
    return;
  }
  if (i_it > 0 && beta * st->betaold < 0.0) {
    st->reason = kDivergedIndefinitePc;
    return;
  }
  const double dpi = s;
  if (dpi == 0.0 || (i_it > 0 && dpi * st->dpiold <= 0.0)) {
    st->reason = kDivergedIndefiniteMat;
    return;
  }
  st->dpi = dpi;
  st->alpha = beta / dpi;
}

template <class T>
__global__ void __launch_bounds__(kBlock) k_cg_update(int n, T* x, T* r, T* z, const T* p, const T* w, const T* inv,
                                                      double* partial, const KState* st) {
  if (st->reason) return;
  __shared__ double lds[kBlock / kWave];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const double a = st->alpha;
  double zz = 0.0, zr = 0.0;
  if (i < n) {
    x[i] = static_cast<T>(static_cast<double>(x[i]) + a * static_cast<double>(p[i]));
    const T rt = static_cast<T>(static_cast<double>(r[i]) - a * static_cast<double>(w[i]));
    r[i] = rt;
    const T zt = inv ? static_cast<T>(static_cast<double>(rt) * static_cast<double>(inv[i])) : rt;
    z[i] = zt;
    zz = static_cast<double>(zt) * static_cast<double>(zt);
    zr = static_cast<double>(zt) * static_cast<double>(rt);
  }
  zz = block_sum(zz, lds);
  zr = block_sum(zr, lds);
  if (threadIdx.x == 0) {
    partial[2 * blockIdx.x] = zz;
    partial[2 * blockIdx.x + 1] = zr;
  }
}

__global__ void __launch_bounds__(kBlock) k_cg_final(const double* partial, int nblk, KState* st) {
  if (st->reason) return;
  __shared__ double lds[kBlock / kWave];
  double zz = 0.0, zr = 0.0;
  strided_sum2(partial, nblk, zz, zr);
  zz = block_sum(zz, lds);
  zr = block_sum(zr, lds);
  if (threadIdx.x != 0) return;
  const double dp = sqrt(zz);
  st->its += 1;
  st->rnorm = dp;
  st->dpiold = st->dpi;
  st->betaold = st->beta;
  st->beta = zr;
  st->reason = conv_check(st, dp);
}

// ---- FP64 residual of a T matrix for iterative refinement
template <class T>
__global__ void __launch_bounds__(kBlock) k_residual64(CsrView<T> A, const double* b, const double* x, double* r) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= A.n) return;
  const double s = csr_dot<double, T, false>(A.val, A.col, A.rowptr[i], A.rowptr[i + 1], 1, x, 0.0);
  r[i] = b[i] - s;
}

// Rows per thread of the multi-dot, Gram-Schmidt and update kernels: enough
// that each block's fixed reduction work is amortised over its loads, while
// the grid keeps several blocks per CU.  FP32 halves the bytes per row, so it
// takes twice the rows per thread on large systems.
int pick_r(int n, size_t elem) {
  if (elem == 4 && n >= 16 * kBlock * 1024) return 16;
  if (n >= 8 * kBlock * 1024) return 8;
  if (n >= 4 * kBlock * 1024) return 4;
  if (n >= 2 * kBlock * 1024) return 2;
  return 1;
}

// blocks a multi-dot launch aims at before splitting its dot products
constexpr int kMdotBlocks = 1024;

int log2_r(int R) { return R == 16 ? 4 : R == 8 ? 3 : R == 4 ? 2 : R == 2 ? 1 : 0; }

// Below this many tiles (blocks of 256 threads) a Gram-Schmidt update or a
// solution update has too few resident waves to hide its loads' latency, and
// each thread batches its basis loads
constexpr int kBatchTiles = 1024;

template <class T>
struct Dispatch {
  template <int R>
  static void mdot_r(const T* V, size_t ld, const Tiles& t, int it, double* partial, int pstride, KState* st,
                     hipStream_t s) {
    // below kMdotBlocks tiles, the chunks of 8 dot products go to separate blocks
    const int chunks = (it + 8) / 8;
    const int groups = std::max(1, std::min(chunks, (kMdotBlocks + t.ntile - 1) / t.ntile));
    const int cpb = (chunks + groups - 1) / groups;
    const int gy = (chunks + cpb - 1) / cpb;
    if (t.ntile * gy < kBatchTiles)
      hipLaunchKernelGGL((k_mdot<T, R, true>), dim3(t.ntile, gy), dim3(kBlock), 0, s, V, ld, t, it, partial, pstride,
                         st, cpb);
    else
      hipLaunchKernelGGL((k_mdot<T, R, false>), dim3(t.ntile, gy), dim3(kBlock), 0, s, V, ld, t, it, partial, pstride,
                         st, cpb);
  }
  template <int R>
  static void maxpy_r(T* V, size_t ld, const Tiles& t, int it, double* norms, const KState* st, hipStream_t s) {
    if (t.ntile < kBatchTiles)
      hipLaunchKernelGGL((k_maxpy_norm<T, R, true>), dim3(t.ntile), dim3(kBlock), 0, s, V, ld, t, it, norms, st);
    else
      hipLaunchKernelGGL((k_maxpy_norm<T, R, false>), dim3(t.ntile), dim3(kBlock), 0, s, V, ld, t, it, norms, st);
  }
  template <int R, class X>
  static void update_r(const T* V, size_t ld, const Tiles& t, X* x, const KState* st, const int* xrow,
                       int rhs_n, hipStream_t s) {
    if (t.ntile < kBatchTiles)
      hipLaunchKernelGGL((k_update_x<T, X, R, true>), dim3(t.ntile), dim3(kBlock), 0, s, V, ld, t, x, st, xrow, rhs_n);
    else
      hipLaunchKernelGGL((k_update_x<T, X, R, false>), dim3(t.ntile), dim3(kBlock), 0, s, V, ld, t, x, st, xrow, rhs_n);
  }
  static void mdot(int R, const T* V, size_t ld, const Tiles& t, int it, double* partial, int pstride,
                   KState* st, hipStream_t s) {
    switch (R) {
      case 16: mdot_r<16>(V, ld, t, it, partial, pstride, st, s); break;
      case 8: mdot_r<8>(V, ld, t, it, partial, pstride, st, s); break;
      case 4: mdot_r<4>(V, ld, t, it, partial, pstride, st, s); break;
      case 2: mdot_r<2>(V, ld, t, it, partial, pstride, st, s); break;
      default: mdot_r<1>(V, ld, t, it, partial, pstride, st, s); break;
    }
  }
  static void maxpy(int R, T* V, size_t ld, const Tiles& t, int it, double* norms, const KState* st,
                    hipStream_t s) {
    switch (R) {
      case 16: maxpy_r<16>(V, ld, t, it, norms, st, s); break;
      case 8: maxpy_r<8>(V, ld, t, it, norms, st, s); break;
      case 4: maxpy_r<4>(V, ld, t, it, norms, st, s); break;
      case 2: maxpy_r<2>(V, ld, t, it, norms, st, s); break;
      default: maxpy_r<1>(V, ld, t, it, norms, st, s); break;
    }
  }
  template <class X>
  static void update(int R, const T* V, size_t ld, const Tiles& t, X* x, const KState* st, const int* xrow,
                     int rhs_n, hipStream_t s) {
    switch (R) {
      case 16: update_r<16>(V, ld, t, x, st, xrow, rhs_n, s); break;
      case 8: update_r<8>(V, ld, t, x, st, xrow, rhs_n, s); break;
      case 4: update_r<4>(V, ld, t, x, st, xrow, rhs_n, s); break;
      case 2: update_r<2>(V, ld, t, x, st, xrow, rhs_n, s); break;
      default: update_r<1>(V, ld, t, x, st, xrow, rhs_n, s); break;
    }
  }
};

// Waits for the last message of w's mailbox launched on s.  A copy of the
// headers and a stream synchronisation took 36-40 us between a cycle's last
// kernel and the next one's first; the poll takes about half of that.  It ends
// with the stream: a stream that is idle or in error without the message throws.
void await_headers(KWork& w, hipStream_t s) {
  const unsigned want = *w.box_count;
  auto here = [&] { return __atomic_load_n(w.box.arrived, __ATOMIC_ACQUIRE) == want; };
  for (int n = 0; !here(); ++n) {
    if ((n & 4095) != 4095) continue;
    const hipError_t e = hipStreamQuery(s);
    if (e == hipErrorNotReady) continue;
    S355_HIP(e);
    if (!here()) throw HipError("solver state not received from the device");
  }
}

// headers of every case
void read_headers(KWork& w, hipStream_t s) {
  hipLaunchKernelGGL(k_publish, dim3(1), dim3(kBlock), 0, s, w.st, w.ncase, w.box);
  S355_LAUNCH_CHECK();
  ++*w.box_count;
  await_headers(w, s);
}

bool all_done(const KWork& w) {
  for (int c = 0; c < w.ncase; ++c)
    if (!w.host[c].done) return false;
  return true;
}

bool all_stopped(const KWork& w) {
  for (int c = 0; c < w.ncase; ++c)
    if (!w.host[c].done && !w.host[c].reason) return false;
  return true;
}

// the fewest iterations a running case has completed (device count); int
// max when none runs
int running_its(const KWork& w) {
  int its = std::numeric_limits<int>::max();
  for (int c = 0; c < w.ncase; ++c)
    if (!w.host[c].done) its = std::min(its, w.host[c].its);
  return its;
}

void init_states(KWork& w, const s355_ksp_opts& o, hipStream_t s) {
  if (__atomic_load_n(w.box.arrived, __ATOMIC_ACQUIRE) != *w.box_count) {
    // an earlier solve ended in an exception with a message under way or not sent
    S355_HIP(hipStreamSynchronize(s));
    *w.box_count = __atomic_load_n(w.box.arrived, __ATOMIC_ACQUIRE);
  }
  hipLaunchKernelGGL(k_init_states, dim3(grid_for(w.ncase)), dim3(kBlock), 0, s, w.st, w.ncase, o.maxit, o.rtol,
                     o.abstol, o.dtol);
  S355_LAUNCH_CHECK();
}

// Per-case results from the headers; the aggregate is the worst case: the
// first divergence if any, the largest iteration count, the largest
// relative residual.
KResult collect(KWork& w, bool mixed) {
  KResult agg;
  double worst = -1.0;
  if (w.per_case) w.per_case->assign(w.ncase, KResult{});
  for (int c = 0; c < w.ncase; ++c) {
    const KHeader& h = w.host[c];
    KResult r;
    r.iters = h.its;
    r.reason = h.reason;
    r.rnorm = h.rnorm;
    r.rnorm0 = h.rnorm0;
    r.refinements = mixed ? h.cycles : 0;
    if (w.per_case) (*w.per_case)[c] = r;
    agg.iters = std::max(agg.iters, r.iters);
    agg.refinements = std::max(agg.refinements, r.refinements);
    if (r.reason < 0 && agg.reason >= 0) agg.reason = r.reason;
    if (agg.reason >= 0 && (agg.reason == 0 || r.reason < agg.reason)) agg.reason = r.reason;
    const double rel = r.rnorm0 > 0.0 ? r.rnorm / r.rnorm0 : r.rnorm;
    if (rel > worst) {
      worst = rel;
      agg.rnorm = r.rnorm;
      agg.rnorm0 = r.rnorm0;
    }
  }
  return agg;
}

// Restarted GMRES(m) over the w.ncase systems stored one after the other.
// The Arnoldi cycle runs on A (values and basis of type T); each restart
// forms the residual b - Ares x in the solution type X.  With T = X and
// Ares = A this is the plain solve.  With T = float, X = double it is the
// mixed solve: every cycle is one step of FP64 iterative refinement (FP64
// residual with the FP64 matrix, FP32 Krylov correction accumulated into the
// FP64 x), so refinement costs no restarts beyond GMRES(m)'s own, and
// convergence is accepted only on the FP64 residual: a cycle whose Givens
// estimate passes the test ends early and the restart residual decides.
// inv_x (mixed Jacobi only) holds the FP64 inverse diagonal.  Cases run their
// cycles in lockstep; a case that has finished drops out of every kernel.
// Whether a solve without ILU takes the two launches of k_spmv_dots per step:
// one case of at most kBlock tiles of one row per thread on a SELL-64 copy
// whose windows lie inside a tile.
template <class T>
bool two_launch_steps(const KWork& w, const SellView<T>& sell, int L, int R) {
  return w.ncase == 1 && w.tiles[0].ntile <= kBlock && L == 0 && R == 1 && sell.ptr && sell.tiled && !sell.two &&
         !sell.scase;
}

template <class T, class X>
KResult gmres(const CsrView<T>& A, const CsrView<X>& Ares, const X* b, X* x, const s355_ksp_opts& o, bool zero_guess,
              KWork& w, X* inv_x, hipStream_t s) {
  constexpr bool mixed = !std::is_same<T, X>::value;
  const int n = A.n;
  const int m = o.restart < 1 ? 1 : (o.restart > kMaxRestart ? kMaxRestart : o.restart);
  if (m > w.mmax) throw std::invalid_argument("gmres: restart above workspace size");
  // rep right-hand sides of one matrix: cases whose rows are n each
  const int rep = w.rep, rhs_n = rep > 1 ? n : 0;
  if (Ares.n != n || w.n != n * rep || (rep > 1 && w.ncase != rep))
    throw std::invalid_argument("gmres: operator sizes differ");
  const size_t ld = w.ld ? w.ld : static_cast<size_t>(w.n);
  const int R = w.rows ? w.rows : pick_r(n, sizeof(T));
  const SellView<T> sell = sell_of<T>(w, n);
  const int L = (w.lanes == 0 && !sell.ptr) ? 8 : w.lanes;
  const Tiles& tl = w.tiles[log2_r(R)];
  if (tl.tile != kBlock * R || tl.n != w.n) throw std::runtime_error("gmres: tile table missing");
  const int nc = w.ncase;
  // the inner order (mixed, no ILU): the FP32 basis, the matrix A and its
  // SELL copies are by position (each case of a batch keeps its own position
  // range); the restart residual goes to its positions and the correction
  // back to the natural rows
  const bool ordered = w.ord_pos != nullptr;
  if (ordered && (!mixed || o.pc == S355_PC_ILU0 || !w.ord_row))
    throw std::invalid_argument("gmres: the inner order serves mixed solves without ILU(0)");
  T* V = static_cast<T*>(w.V);
  T* inv = nullptr;
  const X* invr = nullptr;
  T* lu = nullptr;
  T* tmp = static_cast<T*>(w.r);
  if (o.pc == S355_PC_JACOBI) {
    inv = static_cast<T*>(w.pcinv);
    if constexpr (mixed) {
      if (!inv_x) throw std::invalid_argument("gmres: mixed Jacobi needs an FP64 inverse buffer");
      if (!w.prepared)
        hipLaunchKernelGGL(k_jacobi_mixed, dim3(grid_for(n)), dim3(kBlock), 0, s, Ares, inv_x, inv, w.ord_pos);
      invr = inv_x;
      if (w.pc_folded) inv = nullptr;  // A is M^-1 A already
    } else {
      if (!w.prepared) hipLaunchKernelGGL((k_jacobi_setup<T>), dim3(grid_for(n)), dim3(kBlock), 0, s, A, inv);
      invr = inv;
    }
  } else if (o.pc == S355_PC_ILU0) {
    if (!w.ilu || !w.lu || !w.r) throw std::invalid_argument("gmres: ILU(0) workspace missing");
    lu = static_cast<T*>(w.lu);
    if (!w.prepared) ilu_factor(A, A.nnz, *w.ilu, lu, s, &w);
  } else if (o.pc != S355_PC_NONE) {
    throw std::invalid_argument("gmres: unknown preconditioner");
  }
  init_states(w, o, s);
  const int pstride = m + 1;
  if (!w.norms) throw std::runtime_error("gmres: no norm buffer");
  if (static_cast<size_t>(tl.ntile) * pstride > w.partial_len) throw std::runtime_error("gmres: partial buffer too small");
  if (!zero_guess) {
    if (lu) {
      const T* bt;
      if constexpr (mixed) {
        convert_to_float(b, tmp, w.n, s);
        bt = tmp;
      } else {
        bt = b;
      }
      ilu_apply(A, *w.ilu, lu, bt, V, w.st, s, nullptr, &w);
      hipLaunchKernelGGL((k_pc_norm<T>), dim3(tl.ntile), dim3(kBlock), 0, s, tl, V, static_cast<const T*>(nullptr),
                         w.partial, w.st, rhs_n);
    } else {
      hipLaunchKernelGGL((k_pc_norm<X>), dim3(tl.ntile), dim3(kBlock), 0, s, tl, b, invr, w.partial, w.st, rhs_n);
    }
    hipLaunchKernelGGL(k_snorm_final, dim3(nc), dim3(kBlock), 0, s, w.partial, tl, w.st);
  } else {
    fill_zero(x, sizeof(X) * static_cast<size_t>(w.n), s);
  }
  auto enqueue_restart = [&](bool first_c, bool gz_c) {
    if (lu) {
      hipLaunchKernelGGL((k_residual_pc<T, X>), dim3(tl.ntile), dim3(kBlock), 0, s, Ares, tl, b, x,
                         static_cast<const X*>(nullptr), tmp, w.partial, gz_c ? 1 : 0, w.st,
                         static_cast<const int*>(nullptr), rhs_n);
      ilu_apply(A, *w.ilu, lu, tmp, V, w.st, s, w.graphs, &w);
      hipLaunchKernelGGL((k_pc_norm<T>), dim3(tl.ntile), dim3(kBlock), 0, s, tl, V, static_cast<const T*>(nullptr),
                         w.partial, w.st, rhs_n);
    } else {
      hipLaunchKernelGGL((k_residual_pc<T, X>), dim3(tl.ntile), dim3(kBlock), 0, s, Ares, tl, b, x, invr, V,
                         w.partial, gz_c ? 1 : 0, w.st, w.ord_pos, rhs_n);
    }
    hipLaunchKernelGGL(k_restart_finalize, dim3(nc), dim3(kBlock), 0, s, w.partial, tl, w.st, first_c ? 1 : 0,
                       zero_guess ? 1 : 0, mixed ? 1 : 0);
    S355_LAUNCH_CHECK();
  };
  // One case on a small system without ILU: two launches per step (see
  // k_spmv_dots), the same bits as the four.  An SpMV that is timed on its own
  // takes the four.
  const bool small = two_launch_steps<T>(w, sell, L, R) && !lu;
  // the tile norms of the newest basis vector alternate between two arrays; the
  // finalisation of step it - 1 runs beside step it, the cycle's last on its own
  double* const norms[2] = {w.norms, w.norms + w.tiles[0].ntile};
  int fin_pending = -1;
  auto flush_fin = [&] {
    if (fin_pending < 0) return;
    hipLaunchKernelGGL(k_arnoldi_finalize, dim3(nc), dim3(kBlock), 0, s, norms[fin_pending & 1], tl, fin_pending, m,
                       w.st);
    S355_LAUNCH_CHECK();
    fin_pending = -1;
  };
  auto enqueue_iteration = [&](int it, bool timed) {
    hipEvent_t e0 = nullptr, e1 = nullptr;
    const bool rec = timed && w.timer && (w.timer->seen++ % w.timer->every) == 0 && w.timer->take(e0, e1);
    const int fin = fin_pending >= 0 && fin_pending == it - 1 ? 1 : 0;
    const double* before = norms[(it + 1) & 1];
    if (small && !rec) {
      launch_spmv_dots<T>(w.nt, sell, tl, V, ld, inv, w.st, it, w.partial, s);
      hipLaunchKernelGGL((k_orth_update<T>), dim3(tl.ntile + fin), dim3(kBlock), 0, s, V, ld, tl, w.partial, before,
                         norms[it & 1], it, m, fin, w.st);
    } else {
      if (rec) S355_HIP(hipEventRecord(e0, s));
      if (lu)
        launch_spmv<T>(L, w.nt, A, sell, tl, V + it * ld, static_cast<const T*>(nullptr), tmp, w.st, s, rep);
      else
        launch_spmv<T>(L, w.nt, A, sell, tl, V + it * ld, inv, V + (it + 1) * ld, w.st, s, rep);
      if (rec) S355_HIP(hipEventRecord(e1, s));
      if (lu) ilu_apply(A, *w.ilu, lu, tmp, V + (it + 1) * ld, w.st, s, w.graphs, &w);
      Dispatch<T>::mdot(R, V, ld, tl, it, w.partial, pstride, w.st, s);
      hipLaunchKernelGGL(k_orth, dim3(it + 1 + fin, nc), dim3(kBlock), 0, s, w.partial, before, tl, it, m, fin, w.st);
      Dispatch<T>::maxpy(R, V, ld, tl, it, norms[it & 1], w.st, s);
    }
    fin_pending = it;
    S355_LAUNCH_CHECK();
  };
  auto enqueue_end = [&] {
    hipLaunchKernelGGL(k_build_y, dim3(nc), dim3(kBlock), 0, s, norms[fin_pending & 1], tl, fin_pending, m,
                       fin_pending >= 0 ? 1 : 0, w.st);
    fin_pending = -1;
    Dispatch<T>::update(R, V, ld, tl, x, w.st, w.ord_row, rhs_n, s);
    hipLaunchKernelGGL(k_cycle_end, dim3(1), dim3(kBlock), 0, s, w.st, nc, mixed ? 1 : 0, w.box);
    S355_LAUNCH_CHECK();
  };

  if (w.graphs && !lu) {
    // every restart cycle is one captured graph (the first cycle has its own:
    // it sets the reference norm and may skip the product with a zero
    // guess); a cycle always runs m iterations, the kernels of a finished
    // case returning at once, and the iteration cap is applied on the device.
    // The first cycle runs as two graphs, its first ksplit steps and the
    // rest, with a state read between: a solve that has ended by then (the
    // momentum solves often do) runs only the cycle's end, not m - ksplit
    // steps of kernels that would return at once.  The same kernels run in
    // the same order either way.
    const int ksplit = m >= 8 ? (2 * m) / 5 : m;
    for (bool first_c = true;; first_c = false) {
      std::vector<uintptr_t> key = {reinterpret_cast<uintptr_t>(A.val), reinterpret_cast<uintptr_t>(Ares.val),
                                          reinterpret_cast<uintptr_t>(b), reinterpret_cast<uintptr_t>(x),
                                          reinterpret_cast<uintptr_t>(inv), reinterpret_cast<uintptr_t>(invr),
                                          reinterpret_cast<uintptr_t>(V), reinterpret_cast<uintptr_t>(w.st),
                                          reinterpret_cast<uintptr_t>(w.partial),
                                          static_cast<uintptr_t>(m), static_cast<uintptr_t>(R),
                                          static_cast<uintptr_t>(L), static_cast<uintptr_t>(w.nt),
                                          static_cast<uintptr_t>(w.sell_v),
                                          static_cast<uintptr_t>(w.sell2 + 1), sizeof(T), sizeof(X),
                                          reinterpret_cast<uintptr_t>(w.ord_row),
                                          reinterpret_cast<uintptr_t>(sell.col16),
                                          static_cast<uintptr_t>(rep), static_cast<uintptr_t>(first_c),
                                          static_cast<uintptr_t>(zero_guess), 0};
      // segment: 0 a whole cycle, 1 the first ksplit steps, 2 the rest and
      // the end, 3 the end alone
      auto launch = [&](uintptr_t seg, const std::function<void()>& record) {
        key.back() = seg;
        S355_HIP(hipGraphLaunch(w.graphs->get(key, s, record), s));
      };
      if (first_c && ksplit < m) {
        launch(1, [&] {
          enqueue_restart(true, zero_guess);
          fin_pending = -1;
          for (int it = 0; it < ksplit; ++it) enqueue_iteration(it, false);
          flush_fin();
          hipLaunchKernelGGL(k_publish, dim3(1), dim3(kBlock), 0, s, w.st, nc, w.box);
          S355_LAUNCH_CHECK();
        });
        ++*w.box_count;
        await_headers(w, s);
        if (all_stopped(w)) {
          launch(3, [&] { enqueue_end(); });
        } else {
          launch(2, [&] {
            for (int it = ksplit; it < m; ++it) enqueue_iteration(it, false);
            enqueue_end();
          });
        }
      } else {
        launch(0, [&] {
          enqueue_restart(first_c, first_c && zero_guess);
          for (int it = 0; it < m; ++it) enqueue_iteration(it, false);
          enqueue_end();
        });
      }
      ++*w.box_count;
      await_headers(w, s);
      if (all_done(w)) break;
    }
    return collect(w, mixed);
  }

  // its: iterations launched, an upper bound on a running case's count that
  // only saves launches; it goes back to the device count at every header
  // read, so cycles that end early (the device applies the cap) never stop
  // the launches before the device has ended the solve
  bool first = true, gz = zero_guess;
  int its = 0;
  const int check_every = n >= (1 << 20) ? 4 : 8;
  for (;;) {
    enqueue_restart(first, gz);
    if (mixed && !first) {
      // the FP64 residual decides whether the solve has ended
      read_headers(w, s);
      if (all_done(w)) break;
      its = running_its(w);
    }
    first = false;
    gz = false;
    int it = 0;
    while (it < m && its < o.maxit) {
      enqueue_iteration(it, true);
      ++it;
      ++its;
      if (it % check_every == 0 && it < m) {
        // (the state lags a step: its last finalisation runs beside the next step)
        read_headers(w, s);
        if (all_stopped(w)) break;
      }
    }
    enqueue_end();
    ++*w.box_count;
    await_headers(w, s);
    if (all_done(w)) break;
    its = running_its(w);
  }
  if (w.timer) {
    S355_HIP(hipStreamSynchronize(s));
    w.timer->harvest();
  }
  return collect(w, mixed);
}

// With factored (ILU(0) only) the factors already in w.lu are those of A and
// are used as they are.
template <class T>
KResult cg(const CsrView<T>& A, const T* b, T* x, const s355_ksp_opts& o, bool zero_guess, KWork& w, hipStream_t s,
           bool factored = false) {
  const int n = A.n;
  T* V = static_cast<T*>(w.V);
  const size_t ld = static_cast<size_t>(n);
  if (w.mmax < 3) throw std::invalid_argument("cg: workspace needs 4 vectors");
  if (w.ncase != 1) throw std::invalid_argument("cg: batched systems are solved with GMRES");
  const Tiles& t1 = w.tiles[0];
  T *r = V, *z = V + ld, *p = V + 2 * ld, *wv = V + 3 * ld;
  T* inv = nullptr;
  T* lu = nullptr;
  if (o.pc == S355_PC_JACOBI) {
    inv = static_cast<T*>(w.pcinv);
    hipLaunchKernelGGL((k_jacobi_setup<T>), dim3(grid_for(n)), dim3(kBlock), 0, s, A, inv);
  } else if (o.pc == S355_PC_ILU0) {
    if (!w.ilu || !w.lu) throw std::invalid_argument("cg: ILU(0) workspace missing");
    lu = static_cast<T*>(w.lu);
    if (!factored) ilu_factor(A, A.nnz, *w.ilu, lu, s, &w);
  } else if (o.pc != S355_PC_NONE) {
    throw std::invalid_argument("cg: unknown preconditioner");
  }
  init_states(w, o, s);
  const int g1 = grid_for(n);
  if (2 * static_cast<size_t>(g1) > w.partial_len || t1.ntile != g1)
    throw std::runtime_error("cg: partial buffer too small");
  if (!zero_guess) {
    if (lu) {
      ilu_apply(A, *w.ilu, lu, b, z, w.st, s, nullptr, &w);
      hipLaunchKernelGGL((k_pc_norm<T>), dim3(g1), dim3(kBlock), 0, s, t1, z, static_cast<const T*>(nullptr),
                         w.partial, w.st);
    } else {
      hipLaunchKernelGGL((k_pc_norm<T>), dim3(g1), dim3(kBlock), 0, s, t1, b, inv, w.partial, w.st);
    }
    hipLaunchKernelGGL(k_snorm_final, dim3(1), dim3(kBlock), 0, s, w.partial, t1, w.st);
  }
  hipLaunchKernelGGL((k_cg_start<T>), dim3(g1), dim3(kBlock), 0, s, A, b, x, inv, r, z, w.partial, zero_guess ? 1 : 0);
  if (lu) ilu_apply(A, *w.ilu, lu, r, z, w.st, s, w.graphs, &w, w.partial);  // with the (z, z), (z, r) partials
  hipLaunchKernelGGL(k_cg_start_final, dim3(1), dim3(kBlock), 0, s, w.partial, g1, w.st, zero_guess ? 1 : 0);
  S355_LAUNCH_CHECK();
  const int check_every = n >= (1 << 20) ? 4 : 8;
  KResult res;
  int i = 0;
  for (; i < o.maxit; ++i) {
    hipLaunchKernelGGL((k_cg_p<T>), dim3(g1), dim3(kBlock), 0, s, n, z, p, w.st, i);
    hipLaunchKernelGGL((k_cg_spmv_dot<T>), dim3(g1), dim3(kBlock), 0, s, A, p, wv, w.partial, w.st, i);
    hipLaunchKernelGGL(k_cg_alpha, dim3(1), dim3(kBlock), 0, s, w.partial, g1, w.st, i);
    hipLaunchKernelGGL((k_cg_update<T>), dim3(g1), dim3(kBlock), 0, s, n, x, r, z, p, wv, inv, w.partial, w.st);
    if (lu) ilu_apply(A, *w.ilu, lu, r, z, w.st, s, w.graphs, &w, w.partial);
    hipLaunchKernelGGL(k_cg_final, dim3(1), dim3(kBlock), 0, s, w.partial, g1, w.st);
    S355_LAUNCH_CHECK();
    if ((i + 1) % check_every == 0) {
      read_headers(w, s);
      if (w.host->reason) break;
    }
  }
  read_headers(w, s);
  res.iters = w.host->its;
  res.reason = w.host->reason;
  if (res.reason == 0) res.reason = kDivergedIts;
  res.rnorm = w.host->rnorm;
  res.rnorm0 = w.host->rnorm0;
  return res;
}

__global__ void k_bench_init(KState* st, int ncase) {
  for (int c = threadIdx.x; c < ncase; c += blockDim.x) {
    st[c].reason = st[c].ended = 0;
    st[c].scale[0] = 1.0;
    st[c].scale[1] = 1.0;
  }
}

__global__ void __launch_bounds__(kBlock) k_to_float(const double* src, float* dst, size_t n) {
  const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = static_cast<float>(src[i]);
}

__global__ void __launch_bounds__(kBlock) k_fill_u32(uint32_t* p, size_t n, uint32_t v) {
  const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// ---- iterative refinement pieces
__global__ void __launch_bounds__(kBlock) k_inv_diag32(CsrView<float> A, float* inv, int jacobi) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= A.n) return;
  const double d = static_cast<double>(A.val[A.diag[i]]);
  inv[i] = jacobi ? static_cast<float>(d != 0.0 ? 1.0 / d : 1.0) : 1.0f;
}

// r = b - A x (FP64 matrix and accumulation), r32 = (float) r,
// partial ||M^-1 r||^2 ; with b_only the residual of x = 0
__global__ void __launch_bounds__(kBlock) k_ir_residual(CsrView<double> A, const double* __restrict__ b,
                                                        const double* __restrict__ x, const float* __restrict__ inv,
                                                        double* __restrict__ r, float* __restrict__ r32,
                                                        double* partial, int b_only) {
  __shared__ double lds[kBlock / kWave];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double nrm = 0.0;
  if (i < A.n) {
    double rv = b[i];
    if (!b_only) {
      const double s = csr_dot<double, double, false>(A.val, A.col, A.rowptr[i], A.rowptr[i + 1], 1, x, 0.0);
      rv -= s;
    }
    r[i] = rv;
    r32[i] = static_cast<float>(rv);
    const double z = rv * static_cast<double>(inv[i]);
    nrm = z * z;
  }
  nrm = block_sum(nrm, lds);
  if (threadIdx.x == 0) partial[blockIdx.x] = nrm;
}

__global__ void __launch_bounds__(kBlock) k_sum_to(const double* partial, int nblk, double* out) {
  __shared__ double lds[kBlock / kWave];
  double s = 0.0;
  s = strided_sum(partial, 0, nblk);
  s = block_sum(s, lds);
  if (threadIdx.x == 0) *out = s;
}

// partial ||z||^2 per block (FP64 sums of the FP32 values)
__global__ void __launch_bounds__(kBlock) k_sq_partial(int n, const float* __restrict__ z, double* partial) {
  __shared__ double lds[kBlock / kWave];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double v = 0.0;
  if (i < n) {
    const double zi = static_cast<double>(z[i]);
    v = zi * zi;
  }
  v = block_sum(v, lds);
  if (threadIdx.x == 0) partial[blockIdx.x] = v;
}

__global__ void __launch_bounds__(kBlock) k_add_correction(int n, double* x, const float* e) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] += static_cast<double>(e[i]);
}

}  // namespace

SpmvTimer::~SpmvTimer() {
  for (hipEvent_t e : pool) hipEventDestroy(e);
}

bool SpmvTimer::take(hipEvent_t& a, hipEvent_t& b) {
  if (used + 2 > pool.size()) {
    if (pool.size() >= 8192) return false;  // bounded: the rest go untimed until harvest
    for (int k = 0; k < 2; ++k) {
      hipEvent_t e;
      if (hipEventCreate(&e) != hipSuccess) return false;
      pool.push_back(e);
    }
  }
  a = pool[used];
  b = pool[used + 1];
  used += 2;
  return true;
}

void SpmvTimer::harvest() {
  for (size_t k = 0; k + 1 < used; k += 2) {
    float ms = 0.f;
    if (hipEventElapsedTime(&ms, pool[k], pool[k + 1]) == hipSuccess) {
      total_ms += ms;
      ++count;
    }
  }
  used = 0;
}

GraphCache::~GraphCache() {
  for (auto& kv : execs) hipGraphExecDestroy(kv.second);
}

hipGraphExec_t GraphCache::get(const std::vector<uintptr_t>& key, hipStream_t s, const std::function<void()>& record) {
  auto it = execs.find(key);
  if (it != execs.end()) return it->second;
  hipGraph_t graph = nullptr;
  S355_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
  try {
    record();
  } catch (...) {
    hipStreamEndCapture(s, &graph);
    if (graph) hipGraphDestroy(graph);
    throw;
  }
  S355_HIP(hipStreamEndCapture(s, &graph));
  hipGraphExec_t exec = nullptr;
  const hipError_t e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
  hipGraphDestroy(graph);
  S355_HIP(e);
  execs.emplace(key, exec);
  return exec;
}

namespace {
struct TuneKey {
  int n, nnz, ncase, elem, m, ordered;
  bool operator<(const TuneKey& o) const {
    return std::tie(n, nnz, ncase, elem, m, ordered) < std::tie(o.n, o.nnz, o.ncase, o.elem, o.m, o.ordered);
  }
};
std::mutex g_tune_mu;
struct TuneResult {
  int lanes, nt, rows, sell_v, sell2;
  TuneReport report;
};
std::map<TuneKey, TuneResult> g_tuned;

template <class F>
double time_ms(F&& launch, int reps, hipStream_t s) {
  launch();
  hipEvent_t e0, e1;
  S355_HIP(hipEventCreate(&e0));
  S355_HIP(hipEventCreate(&e1));
  S355_HIP(hipEventRecord(e0, s));
  for (int r = 0; r < reps; ++r) launch();
  S355_HIP(hipEventRecord(e1, s));
  S355_HIP(hipEventSynchronize(e1));
  float ms = 0.f;
  S355_HIP(hipEventElapsedTime(&ms, e0, e1));
  S355_HIP(hipEventDestroy(e0));
  S355_HIP(hipEventDestroy(e1));
  return static_cast<double>(ms) / reps;
}
}  // namespace

template <class T>
void autotune(const CsrView<T>& A, KWork& w, int m, hipStream_t s) {
  const TuneKey key{A.n, A.nnz, w.ncase, static_cast<int>(sizeof(T)), m, w.ord_row ? 1 : 0};
  {
    std::lock_guard<std::mutex> g(g_tune_mu);
    auto it = g_tuned.find(key);
    if (it != g_tuned.end()) {
      w.lanes = it->second.lanes;
      w.nt = it->second.nt;
      w.rows = it->second.rows;
      w.sell_v = it->second.sell_v;
      w.sell2 = it->second.sell2;
      w.report = it->second.report;
      w.tuned = true;
      return;
    }
  }
  const int n = A.n;
  if (n <= 0 || m < 1 || m > w.mmax) return;
  const size_t ld = w.ld ? w.ld : static_cast<size_t>(n);
  T* V = static_cast<T*>(w.V);
  // a zero basis: the timings do not depend on the values
  fill_zero(V, sizeof(T) * ld * (static_cast<size_t>(m) + 1), s);
  s355_ksp_opts o{};
  o.maxit = 1 << 30;
  o.rtol = 0.0;
  o.dtol = 1e300;
  init_states(w, o, s);
  hipLaunchKernelGGL(k_bench_init, dim3(1), dim3(kBlock), 0, s, w.st, w.ncase);
  S355_LAUNCH_CHECK();
  const T* none = nullptr;
  // One small case takes the SELL-64 copy with windows inside a tile and one
  // row per thread, two launches a step, whatever the four launches of other
  // shapes measure here: only the matrix loads are left to choose.  (The
  // shapes serve every solve of the context, ILU(0) solves too.)
  int tiled = -1;
  if (w.ncase == 1 && w.tiles[0].ntile <= kBlock)
    for (int sv = kSellVariants - 1; sv >= 0; --sv)
      if (two_launch_steps<T>(w, sell_of<T>(w, n, sv), 0, 1)) tiled = sv;
  TuneReport rep;
  int best_l = 8, best_nt = 0;
  double best = 1e300;
  int best_sv = w.sell_v;
  for (int L : {1, 2, 4, 8, 16, 0})
    for (int sv = 0; sv < (L == 0 ? kSellVariants : 1); ++sv) {
      const SellView<T> sell = sell_of<T>(w, n, sv);
      if (L == 0 && !sell.ptr) continue;
      if (tiled >= 0 && (L != 0 || sv != tiled)) continue;
      if (L == 0) {
        // values of this window's copy from the CSR matrix being tuned on
        const SellPat& pt = w.sell[sv];
        hipLaunchKernelGGL((k_gather<T>), dim3(grid_for(static_cast<long>(pt.slots))), dim3(kBlock), 0, s, pt.src,
                           pt.slots, A.val, static_cast<T*>(w.sell_vals[sv]));
      }
      for (int nt : {0, 1}) {
        const double ms = time_ms(
            [&] {
              if (tiled >= 0)
                launch_spmv_dots<T>(nt, sell, w.tiles[0], V, ld, none, w.st, m / 2, w.partial, s);
              else
                launch_spmv<T>(L, nt, A, sell, w.tiles[0], V, none, V + ld, w.st, s);
            },
            5, s);
        rep.spmv_ms[spmv_variant(L, nt, sv)] = ms;
        if (ms < best) {
          best = ms;
          best_l = L;
          best_nt = nt;
          best_sv = sv;
        }
      }
    }
  // FP32 SELL on one case: the best window with one and with two slices per
  // wave (twice the loads in flight per wave; it pays where the product is
  // bound by its loads' latency, not where it already streams at the copy rate)
  if constexpr (std::is_same<T, float>::value) {
    if (best_l == 0 && w.ncase == 1 && n >= (1 << 18)) {
      SellView<T> sell = sell_of<T>(w, n, best_sv);
      if (sell.ptr && !sell.scase) {
        double ms2[2];
        for (int two = 0; two < 2; ++two) {
          sell.two = two;
          ms2[two] = time_ms([&] { launch_spmv<T>(0, best_nt, A, sell, w.tiles[0], V, none, V + ld, w.st, s); },
                             5, s);
        }
        w.sell2 = ms2[1] < ms2[0] ? 1 : 0;
      }
    }
  }
  // the Gram-Schmidt launches of three Arnoldi steps across the cycle (a
  // quarter, half and three quarters of the restart length) at every tile
  // size; the tile count also sets the work of the final reduction
  const int it = m / 2;
  int best_r = pick_r(n, sizeof(T));
  best = 1e300;
  for (int R : {1, 2, 4, 8, 16}) {
    const Tiles& t = w.tiles[log2_r(R)];
    if (static_cast<size_t>(t.ntile) * (m + 1) > w.partial_len) continue;
    if (tiled >= 0 && R != 1) continue;
    const double ms = time_ms(
        [&] {
          for (int j : {m / 4, m / 2, (3 * m) / 4}) {
            if (tiled >= 0) {
              hipLaunchKernelGGL((k_orth_update<T>), dim3(t.ntile), dim3(kBlock), 0, s, V, ld, t, w.partial, w.norms,
                                 w.norms + t.ntile, j, m, 0, w.st);
              continue;
            }
            Dispatch<T>::mdot(R, V, ld, t, j, w.partial, m + 1, w.st, s);
            hipLaunchKernelGGL(k_orth, dim3(j + 1, w.ncase), dim3(kBlock), 0, s, w.partial, w.norms, t, j, m, 0, w.st);
            Dispatch<T>::maxpy(R, V, ld, t, j, w.norms, w.st, s);
          }
        },
        5, s) / 3.0;
    rep.gs_ms[log2_r(R)] = ms;
    if (ms < best) {
      best = ms;
      best_r = R;
    }
  }
  rep.gs_it = it;
  w.lanes = best_l;
  w.nt = best_nt;
  w.rows = best_r;
  w.sell_v = best_sv;
  w.report = rep;
  w.tuned = true;
  std::lock_guard<std::mutex> g(g_tune_mu);
  g_tuned[key] = TuneResult{best_l, best_nt, best_r, best_sv, w.sell2, rep};
}

int pick_rows(int n, size_t elem) { return pick_r(n, elem); }

template void autotune<double>(const CsrView<double>&, KWork&, int, hipStream_t);
template void autotune<float>(const CsrView<float>&, KWork&, int, hipStream_t);

template <class T>
KResult krylov_solve(const CsrView<T>& A, const T* b, T* x, const s355_ksp_opts& o, bool zero_guess, KWork& w,
                     hipStream_t s) {
  if (A.n <= 0) return KResult{0, kConvergedAtol, 0.0, 0.0};
  if (o.maxit < 0 || !(o.rtol >= 0.0)) throw std::invalid_argument("krylov: bad tolerances");
  if (o.type == S355_KSP_CG) return cg(A, b, x, o, zero_guess, w, s);
  return gmres<T, T>(A, A, b, x, o, zero_guess, w, nullptr, s);
}

template <class T>
void residual64(const CsrView<T>& A, const double* b, const double* x, double* r, hipStream_t s) {
  hipLaunchKernelGGL((k_residual64<T>), dim3(grid_for(A.n)), dim3(kBlock), 0, s, A, b, x, r);
  S355_LAUNCH_CHECK();
}

template KResult krylov_solve<double>(const CsrView<double>&, const double*, double*, const s355_ksp_opts&, bool,
                                      KWork&, hipStream_t);
template KResult krylov_solve<float>(const CsrView<float>&, const float*, float*, const s355_ksp_opts&, bool, KWork&,
                                     hipStream_t);
template void residual64<double>(const CsrView<double>&, const double*, const double*, double*, hipStream_t);
template void residual64<float>(const CsrView<float>&, const double*, const double*, double*, hipStream_t);

KResult ir_solve(const CsrView<double>& A64, const CsrView<float>& A, const double* b, double* x,
                 const s355_ksp_opts& o, bool zero_guess, int ir_max, double inner_rtol, KWork& w32, IrWork& ir,
                 hipStream_t s) {
  const int n = A.n;
  KResult res;
  if (n <= 0) {
    res.reason = kConvergedAtol;
    return res;
  }
  if (o.maxit < 0 || !(o.rtol >= 0.0)) throw std::invalid_argument("krylov: bad tolerances");
  if (o.type != S355_KSP_CG) return gmres<float, double>(A, A64, b, x, o, zero_guess, w32, ir.r64, s);
  const int g = grid_for(n);
  if (static_cast<size_t>(g) > ir.partial_len) throw std::runtime_error("ir_solve: partial buffer too small");
  hipLaunchKernelGGL(k_inv_diag32, dim3(g), dim3(kBlock), 0, s, A, ir.inv32, o.pc == S355_PC_JACOBI ? 1 : 0);
  // ILU(0): the outer test takes ||(LU)^-1 r|| as PETSc's CG does, with the
  // FP32 factors of A32 (factored once here; the inner solves reuse them)
  float* lu = nullptr;
  if (o.pc == S355_PC_ILU0) {
    if (!w32.ilu || !w32.lu) throw std::invalid_argument("ir_solve: ILU(0) workspace missing");
    lu = static_cast<float*>(w32.lu);
    ilu_factor(A, A.nnz, *w32.ilu, lu, s, &w32);
  }
  // partial ||M^-1 r||^2 of the residual just formed (Jacobi: inside k_ir_residual)
  auto pc_norm = [&](double* out) {
    if (lu) {
      ilu_apply(A, *w32.ilu, lu, ir.r32, ir.e32, static_cast<const KState*>(nullptr), s, nullptr, &w32);
      hipLaunchKernelGGL(k_sq_partial, dim3(g), dim3(kBlock), 0, s, n, ir.e32, ir.partial);
    }
    hipLaunchKernelGGL(k_sum_to, dim3(1), dim3(kBlock), 0, s, ir.partial, g, out);
  };
  if (zero_guess) fill_zero(x, sizeof(double) * static_cast<size_t>(n), s);
  // ||M^-1 b|| for the reference norm of a nonzero initial guess
  hipLaunchKernelGGL(k_ir_residual, dim3(g), dim3(kBlock), 0, s, A64, b, x, ir.inv32, ir.r64, ir.r32, ir.partial, 1);
  pc_norm(ir.scal + 1);
  S355_LAUNCH_CHECK();
  s355_ksp_opts inner = o;
  inner.rtol = inner_rtol;
  inner.abstol = 0.0;
  inner.dtol = 1e30;
  int total = 0;
  double rnorm0 = 0.0, ttol = 0.0;
  for (int k = 0;; ++k) {
    hipLaunchKernelGGL(k_ir_residual, dim3(g), dim3(kBlock), 0, s, A64, b, x, ir.inv32, ir.r64, ir.r32, ir.partial,
                       zero_guess && k == 0 ? 1 : 0);
    pc_norm(ir.scal);
    S355_LAUNCH_CHECK();
    S355_HIP(hipMemcpyAsync(ir.host, ir.scal, 2 * sizeof(double), hipMemcpyDeviceToHost, s));
    S355_HIP(hipStreamSynchronize(s));
    const double rn = std::sqrt(ir.host[0]);
    if (k == 0) {
      const double snorm = std::sqrt(ir.host[1]);
      rnorm0 = zero_guess ? rn : (snorm != 0.0 ? snorm : rn);
      ttol = std::max(o.rtol * rnorm0, o.abstol);
    }
    res.rnorm = rn;
    res.rnorm0 = rnorm0;
    res.refinements = k;
    if (std::isnan(rn) || std::isinf(rn)) {
      res.reason = kDivergedNanorinf;
      break;
    }
    if (rn <= ttol) {
      res.reason = rn < o.abstol ? kConvergedAtol : kConvergedRtol;
      break;
    }
    if (rn >= o.dtol * rnorm0) {
      res.reason = kDivergedDtol;
      break;
    }
    if (total >= o.maxit || k >= ir_max) {
      res.reason = kDivergedIts;
      break;
    }
    inner.maxit = o.maxit - total;
    KResult r = cg<float>(A, ir.r32, ir.e32, inner, true, w32, s, lu != nullptr);
    total += r.iters;
    if (r.iters == 0 && r.reason < 0) {
      res.reason = r.reason;
      break;
    }
    hipLaunchKernelGGL(k_add_correction, dim3(g), dim3(kBlock), 0, s, n, x, ir.e32);
    S355_LAUNCH_CHECK();
  }
  res.iters = total;
  return res;
}

template <class T>
double bench_spmv(const CsrView<T>& A, const T* x, T* y, const T* inv, KWork& w, int repeats, void* flush,
                  size_t flush_bytes, hipStream_t s) {
  hipLaunchKernelGGL(k_bench_init, dim3(1), dim3(kBlock), 0, s, w.st, w.ncase);
  const Tiles& t = w.tiles[0];
  const SellView<T> sell = sell_of<T>(w, A.n);
  const int L = (w.lanes == 0 && !sell.ptr) ? 8 : w.lanes;
  launch_spmv<T>(L, w.nt, A, sell, t, x, inv, y, w.st, s);
  S355_LAUNCH_CHECK();
  hipEvent_t e0, e1;
  S355_HIP(hipEventCreate(&e0));
  S355_HIP(hipEventCreate(&e1));
  double total = 0.0;
  for (int r = 0; r < repeats; ++r) {
    // overwrite the Infinity Cache so that every launch starts cold, as it
    // does inside a Krylov iteration whose other kernels stream the basis
    if (flush) fill_zero(flush, flush_bytes, s);
    S355_HIP(hipEventRecord(e0, s));
    launch_spmv<T>(L, w.nt, A, sell, t, x, inv, y, w.st, s);
    S355_HIP(hipEventRecord(e1, s));
    S355_HIP(hipEventSynchronize(e1));
    float ms = 0.f;
    S355_HIP(hipEventElapsedTime(&ms, e0, e1));
    total += ms;
  }
  S355_HIP(hipEventDestroy(e0));
  S355_HIP(hipEventDestroy(e1));
  return total / repeats;
}

namespace {
// plain copy, U 16-byte loads in flight per lane before the stores: the
// reference point for bandwidth and for scaling hardware byte counters
template <int U>
__global__ void __launch_bounds__(kBlock) k_stream_copy(const uint4* __restrict__ src, uint4* __restrict__ dst,
                                                        size_t n) {
  const size_t stride = static_cast<size_t>(gridDim.x) * blockDim.x;
  size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  for (; i + (U - 1) * stride < n; i += U * stride) {
    uint4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = src[i + u * stride];
#pragma unroll
    for (int u = 0; u < U; ++u) dst[i + u * stride] = v[u];
  }
  for (; i < n; i += stride) dst[i] = src[i];
}
}  // namespace

double bench_copy(void* dst, const void* src, size_t bytes, int repeats, hipStream_t s) {
  if (bytes % sizeof(uint4)) throw std::invalid_argument("bench_copy: size must be a multiple of 16 bytes");
  const size_t n = bytes / sizeof(uint4);
  const uint4* a = static_cast<const uint4*>(src);
  uint4* b = static_cast<uint4*>(dst);
  // the best of a few launch shapes: the measured peak, not one kernel's
  double best = 1e300;
  for (int g : {2048, 4096, 8192, 16384})
    for (int unroll : {1, 4}) {
      const int grid = static_cast<int>(std::min<size_t>(g, (n + kBlock - 1) / kBlock));
      const double ms = time_ms(
          [&] {
            if (unroll == 4)
              hipLaunchKernelGGL(k_stream_copy<4>, dim3(grid), dim3(kBlock), 0, s, a, b, n);
            else
              hipLaunchKernelGGL(k_stream_copy<1>, dim3(grid), dim3(kBlock), 0, s, a, b, n);
          },
          repeats, s);
      best = std::min(best, ms);
    }
  S355_LAUNCH_CHECK();
  return best;
}

void sell_pattern(int n, const int* rowptr, const int* col, int sigma, std::vector<int>& ptr, std::vector<int>& srow,
                  std::vector<int>& scol, std::vector<int>& src) {
  if (sigma < 64 || sigma % 64) throw std::invalid_argument("SELL sigma must be a positive multiple of 64");
  // slot-row order: each window of sigma rows by decreasing length, stable
  srow.resize(n);
  for (int w0 = 0; w0 < n; w0 += sigma) {
    const int w1 = std::min(n, w0 + sigma);
    for (int r = w0; r < w1; ++r) srow[r] = r;
    std::stable_sort(srow.begin() + w0, srow.begin() + w1, [&](int a, int b) {
      return rowptr[a + 1] - rowptr[a] > rowptr[b + 1] - rowptr[b];
    });
  }
  auto len = [&](int pos) { return pos < n ? rowptr[srow[pos] + 1] - rowptr[srow[pos]] : 0; };
  const int ns = (n + 63) / 64;
  ptr.assign(ns + 1, 0);
  for (int sl = 0; sl < ns; ++sl) {
    int w = 0;
    for (int pos = 64 * sl; pos < std::min(n, 64 * sl + 64); ++pos) w = std::max(w, len(pos));
    const long next = static_cast<long>(ptr[sl]) + 64L * w;
    if (next > 0x7fffffffL) throw std::invalid_argument("SELL-64 copy above 32-bit indices");
    ptr[sl + 1] = static_cast<int>(next);
  }
  scol.assign(ptr[ns], 0);
  src.assign(ptr[ns], -1);
  for (int sl = 0; sl < ns; ++sl) {
    const int w = (ptr[sl + 1] - ptr[sl]) / 64;
    for (int l = 0; l < 64; ++l) {
      const int pos = 64 * sl + l;
      const int r = pos < n ? srow[pos] : 0;
      const int lr = len(pos);
      for (int j = 0; j < w; ++j) {
        const size_t q = static_cast<size_t>(ptr[sl]) + 64 * static_cast<size_t>(j) + l;
        if (j < lr) {
          scol[q] = col[rowptr[r] + j];
          src[q] = rowptr[r] + j;
        } else {
          scol[q] = r;  // a valid column; the value is zero
        }
      }
    }
  }
}

namespace {
// out[k] = (float) (val[src[k]] / d) over the entries of position p's row,
// d the diagonal of its natural row (1 without Jacobi, 1 for a zero diagonal)
__global__ void __launch_bounds__(kBlock) k_fill_ordered(int n, const int* __restrict__ rowptr,
                                                         const int* __restrict__ src, const int* __restrict__ row_nat,
                                                         const int* __restrict__ diag_nat,
                                                         const double* __restrict__ val, int jacobi,
                                                         float* __restrict__ out) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  double inv = 1.0;
  if (jacobi) {
    const double d = val[diag_nat[row_nat[p]]];
    inv = d != 0.0 ? 1.0 / d : 1.0;
  }
  for (int k = rowptr[p]; k < rowptr[p + 1]; ++k) out[k] = static_cast<float>(val[src[k]] * inv);
}
}  // namespace

void fill_ordered(int n, const int* rowptr, const int* src, const int* row_nat, const int* diag_nat,
                  const double* val, bool jacobi, float* out, hipStream_t s) {
  hipLaunchKernelGGL(k_fill_ordered, dim3(grid_for(n)), dim3(kBlock), 0, s, n, rowptr, src, row_nat, diag_nat, val,
                     jacobi ? 1 : 0, out);
  S355_LAUNCH_CHECK();
}

bool sell_offsets16(int n, const std::vector<int>& ptr, const std::vector<int>& srow, const std::vector<int>& scol,
                    std::vector<int16_t>& off) {
  off.assign(scol.size(), 0);
  const int ns = static_cast<int>(ptr.size()) - 1;
  for (int sl = 0; sl < ns; ++sl) {
    const int w = (ptr[sl + 1] - ptr[sl]) / 64;
    for (int l = 0; l < 64; ++l) {
      const int pos = 64 * sl + l;
      if (pos >= n) continue;  // past the last row: offset 0 from the row the kernel substitutes
      const long r = srow[pos];
      for (int j = 0; j < w; ++j) {
        const size_t q = static_cast<size_t>(ptr[sl]) + 64 * static_cast<size_t>(j) + l;
        const long d = static_cast<long>(scol[q]) - r;
        if (d < INT16_MIN || d > INT16_MAX) return false;
        off[q] = static_cast<int16_t>(d);
      }
    }
  }
  return true;
}

template <class T, class S>
void sell_fill(const int* src, size_t nslots, const S* csr_val, T* out, hipStream_t s) {
  hipLaunchKernelGGL((k_sell_fill<T, S>), dim3(grid_for(static_cast<long>(nslots))), dim3(kBlock), 0, s, src, nslots,
                     csr_val, out);
  S355_LAUNCH_CHECK();
}
template void sell_fill<double, double>(const int*, size_t, const double*, double*, hipStream_t);
template void sell_fill<float, double>(const int*, size_t, const double*, float*, hipStream_t);
template void sell_fill<float, float>(const int*, size_t, const float*, float*, hipStream_t);

void convert_to_float(const double* src, float* dst, size_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_to_float, dim3(grid_for(static_cast<long>(n))), dim3(kBlock), 0, s, src, dst, n);
  S355_LAUNCH_CHECK();
}

void fill_zero(void* p, size_t bytes, hipStream_t s) {
  const size_t n = bytes / 4;
  if (n == 0) return;
  hipLaunchKernelGGL(k_fill_u32, dim3(grid_for(static_cast<long>(n))), dim3(kBlock), 0, s, static_cast<uint32_t*>(p),
                     n, 0u);
  S355_LAUNCH_CHECK();
}

template double bench_spmv<double>(const CsrView<double>&, const double*, double*, const double*, KWork&, int, void*,
                                   size_t, hipStream_t);
template double bench_spmv<float>(const CsrView<float>&, const float*, float*, const float*, KWork&, int, void*, size_t,
                                  hipStream_t);

template <class T>
void jacobi_inverse(const CsrView<T>& A, T* inv, hipStream_t s) {
  hipLaunchKernelGGL((k_jacobi_setup<T>), dim3(grid_for(A.n)), dim3(kBlock), 0, s, A, inv);
  S355_LAUNCH_CHECK();
}
template void jacobi_inverse<double>(const CsrView<double>&, double*, hipStream_t);
template void jacobi_inverse<float>(const CsrView<float>&, float*, hipStream_t);

void ilu_steps(int n, const int* rowptr, const int* col, const int* diag, const std::vector<int>& rows,
               std::vector<int>& ptr, std::vector<int>& p, std::vector<int>& d, std::vector<int>& u,
               std::vector<int>& r, std::vector<int>& q) {
  ptr.assign(1, 0);
  p.clear();
  d.clear();
  u.assign(1, 0);
  r.clear();
  q.clear();
  for (int t = 0; t < n; ++t) {
    const int i = rows[t];
    const int pd = diag[i], pe = rowptr[i + 1];
    for (int pp = rowptr[i]; pp < pd; ++pp) {
      const int k = col[pp];
      p.push_back(pp);
      d.push_back(diag[k]);
      // the merge of row i after pp with the upper part of row k
      int a = diag[k] + 1, b = pp + 1;
      const int ae = rowptr[k + 1];
      while (a < ae && b < pe) {
        if (col[a] == col[b]) {
          r.push_back(b);
          q.push_back(a);
          ++a;
          ++b;
        } else if (col[a] < col[b]) {
          ++a;
        } else {
          ++b;
        }
      }
      if (r.size() > 0x7fffffffUL) throw std::invalid_argument("ILU(0) elimination steps above 32-bit indices");
      u.push_back(static_cast<int>(r.size()));
    }
    if (p.size() > 0x7fffffffUL) throw std::invalid_argument("ILU(0) elimination steps above 32-bit indices");
    ptr.push_back(static_cast<int>(p.size()));
  }
}

void ilu_levels(int n, const int* rowptr, const int* col, const int* diag, std::vector<int>& rows,
                std::vector<int>& ptr) {
  std::vector<int> lev(n, 0);
  int nl = 0;
  for (int i = 0; i < n; ++i) {
    int l = 0;
    for (int p = rowptr[i]; p < diag[i]; ++p) l = std::max(l, lev[col[p]] + 1);
    lev[i] = l;
    nl = std::max(nl, l + 1);
  }
  ptr.assign(nl + 1, 0);
  for (int i = 0; i < n; ++i) ptr[lev[i] + 1]++;
  for (int l = 0; l < nl; ++l) ptr[l + 1] += ptr[l];
  rows.assign(n, 0);
  std::vector<int> pos(ptr.begin(), ptr.end() - 1);
  for (int i = 0; i < n; ++i) rows[pos[lev[i]]++] = i;
}

}  // namespace s355

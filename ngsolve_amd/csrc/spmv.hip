// CSR sparse matrix-vector product on gfx950.
//
// Replaces SparseMatrix<double>::MultAdd (linalg/sparsematrix_impl.hpp:264-306,
// row kernel RowTimesVector linalg/sparsematrix.hpp:625-632) and the
// reference's cuSPARSE call (ngscuda/cuda_linalg.cpp:243-275).
//
// Three kernels:
//
// runs (default when it saves at least a quarter of the column numbers): up
// to 8 consecutive rows with the same column list (the dofs of one edge, face
// or cell of an H1 space) form a run that stores the list once and its values
// column by column.  Values still stream once (8 B per nonzero) but the column
// numbers drop to 4 B per run entry and each gathered x entry serves the
// whole run.  A group of lanes per run keeps the run's row sums in registers.
//
// stream: int32 row pointers, int32 column numbers, FP64 values (12 B per
// nonzero streamed once); the rows are cut on the host into blocks of consecutive
// rows holding at most 2048 nonzeros (NGSAMD_SPMV_NNZ=1024/4096 selects other
// sizes; a single longer row is a block of its own).  A 256-thread workgroup streams a block's column and value
// ranges with fully coalesced non-temporal loads (they are read once and
// must not evict x from L2), multiplies by the gathered x entries into LDS,
// and then reduces each row from LDS with a power-of-two group of lanes sized
// to the block's row count.  Every lane is busy whatever the row lengths.
//
// rowgroup: a group of G lanes works on one row, lane l of the group reading
// nonzeros l, l+G, ...; the partial sums are combined with cross-lane
// shuffles.  Kept for comparison (NGSAMD_SPMV=rowgroup).
//
// All three walk contiguous row ranges that are grouped per XCD (workgroup i runs
// on XCD i mod 8), so the x entries a row range gathers stay in one XCD's L2.
#include <algorithm>
#include <cstdlib>
#include <string>
#include <type_traits>

#include "common.hpp"
#include "csr.hpp"
#include "runs.hpp"
#include "runsdev.hpp"
#include "reduce.hpp"
#include "runtime_state.hpp"

namespace ngsamd {

constexpr int kSpmvBlock = 256;

// y[r] = (ACCUM ? y[r] : 0) + s * (A x)[r]; optionally the per-workgroup
// partial sums of x[r]*(A x)[r] (the <s, A s> of CG) into partials[].
template <int G, bool ACCUM, bool DOT>
__global__ __launch_bounds__(kSpmvBlock) void CsrSpmvKernel(
    const int* __restrict__ rowptr, const int* __restrict__ cols, const double* __restrict__ vals,
    const double* __restrict__ x, double* __restrict__ y, int n, double s, int iters_per_wg,
    double* __restrict__ partials, const int* __restrict__ stop_flag) {
  if (stop_flag && *stop_flag) return;
  constexpr int RPB = kSpmvBlock / G;  // rows per workgroup pass
  const int lb = XcdContiguousBlock(blockIdx.x, gridDim.x);
  const int g = threadIdx.x / G;
  const int l = threadIdx.x % G;
  double dotacc = 0.0;
  const int row_begin = lb * iters_per_wg * RPB;
  for (int it = 0; it < iters_per_wg; it++) {
    const int r = row_begin + it * RPB + g;
    if (r < n) {
      const int k0 = rowptr[r], k1 = rowptr[r + 1];
      double a0 = 0.0, a1 = 0.0;
      int k = k0 + l;
      for (; k + G < k1; k += 2 * G) {
        const int c0 = cols[k], c1 = cols[k + G];
        const double v0 = vals[k], v1 = vals[k + G];
        a0 += v0 * x[c0];
        a1 += v1 * x[c1];
      }
      if (k < k1) a0 += vals[k] * x[cols[k]];
      double sum = a0 + a1;
#pragma unroll
      for (int off = G / 2; off > 0; off >>= 1) sum += __shfl_xor(sum, off, G);
      if (l == 0) {
        const double val = s * sum;
        if (ACCUM) y[r] += val; else y[r] = val;
        if (DOT) dotacc += x[r] * sum;
      }
    }
  }
  if (DOT) {
    __shared__ double lds[kSpmvBlock / 64];
    StorePartial<kSpmvBlock>(dotacc, partials, lds);
  }
}


constexpr int kStreamBlock = 256;
constexpr int kRunWaves = kStreamBlock / 64;  // tasks of the runs kernel in flight per workgroup

// y[r] = (ACCUM ? y[r] : 0) + s * (A x)[r] over the row blocks
// [blk_row[b], blk_row[b+1]) of at most NNZ nonzeros; DOT as in CsrSpmvKernel.
template <int NNZ, bool ACCUM, bool DOT>
__global__ __launch_bounds__(kStreamBlock) void CsrStreamKernel(
    const int* __restrict__ rowptr, const int* __restrict__ cols, const double* __restrict__ vals,
    const double* __restrict__ x, double* __restrict__ y, const int* __restrict__ blk_row, int nblocks,
    int blocks_per_wg, double s, double* __restrict__ partials, const int* __restrict__ stop_flag) {
  if (stop_flag && *stop_flag) return;
  __shared__ double prod[NNZ];
  __shared__ double lds[kStreamBlock / 64];
  const int tid = threadIdx.x;
  const int lb = XcdContiguousBlock(blockIdx.x, gridDim.x);
  const int b0 = lb * blocks_per_wg;
  const int b1 = min(b0 + blocks_per_wg, nblocks);
  double dotacc = 0.0;
  for (int b = b0; b < b1; b++) {
    const int r0 = blk_row[b], r1 = blk_row[b + 1];
    const int k0 = rowptr[r0], k1 = rowptr[r1];
    const int nz = k1 - k0;
    if (nz > NNZ) {
      // one long row: the whole workgroup strides over it
      double a = 0.0;
      for (int k = k0 + tid; k < k1; k += kStreamBlock)
        a += __builtin_nontemporal_load(&vals[k]) * x[__builtin_nontemporal_load(&cols[k])];
      a = BlockSum<kStreamBlock>(a, lds);
      if (tid == 0) {
        if (ACCUM) y[r0] += s * a; else y[r0] = s * a;
        if (DOT) dotacc += x[r0] * a;
      }
      continue;
    }
    // every load is unconditional (lanes past the block read entry k0,
    // which the padding keeps in bounds, and contribute 0) so all of them
    // are in flight at once instead of one round trip per branch
    constexpr int PER = NNZ / kStreamBlock;
    int c[PER];
    double v[PER], xv[PER];
#pragma unroll
    for (int i = 0; i < PER; i++) {
      const int k = tid + i * kStreamBlock;
      const int kk = k0 + (k < nz ? k : 0);
      c[i] = __builtin_nontemporal_load(&cols[kk]);
      v[i] = __builtin_nontemporal_load(&vals[kk]);
    }
#pragma unroll
    for (int i = 0; i < PER; i++) xv[i] = x[c[i]];
#pragma unroll
    for (int i = 0; i < PER; i++) {
      const int k = tid + i * kStreamBlock;
      prod[k] = k < nz ? v[i] * xv[i] : 0.0;
    }
    __syncthreads();
    const int nr = r1 - r0;
    int tpr = 64;
    while (tpr > 1 && tpr * nr > kStreamBlock) tpr >>= 1;
    const int l = tid & (tpr - 1);
    for (int j0 = 0; j0 < nr; j0 += kStreamBlock / tpr) {
      const int j = j0 + tid / tpr;
      double sum = 0.0;
      if (j < nr) {
        const int s0 = rowptr[r0 + j] - k0, s1 = rowptr[r0 + j + 1] - k0;
        double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
        int k = s0 + l;
        for (; k + 3 * tpr < s1; k += 4 * tpr) {
          a0 += prod[k];
          a1 += prod[k + tpr];
          a2 += prod[k + 2 * tpr];
          a3 += prod[k + 3 * tpr];
        }
        for (; k < s1; k += tpr) a0 += prod[k];
        sum = (a0 + a1) + (a2 + a3);
      }
      for (int off = tpr / 2; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
      if (j < nr && l == 0) {
        if (ACCUM) y[r0 + j] += s * sum; else y[r0 + j] = s * sum;
        if (DOT) dotacc += x[r0 + j] * sum;
      }
    }
    __syncthreads();
  }
  if (DOT) StorePartial<kStreamBlock>(dotacc, partials, lds);
}


// ------------------------------------------------------------- runs kernel
// A task is up to 64 / G consecutive runs of R rows each, one wavefront's
// work: a group of G lanes per run (RunGroup: 8 to 64 by the run's length).
// Lane l of a group takes the column slots l, l + G, ... of its run: one
// column number and one x entry per slot serve the R values of the slot
// (adjacent in memory), and the R row sums stay in the lane's registers until
// a butterfly over the group ends them.  No LDS and no barrier: every
// wavefront runs on its own, so the loads of one cover the sums of another.

// The single vector x of the runs kernel: plain, or formed from {s, z} pairs
// (CgDirection) as beta s + z.
struct PlainX {
  const double* __restrict__ x;
  __device__ __forceinline__ double operator()(int i) const { return x[i]; }
};
struct PairX {
  const double2* __restrict__ pair;
  double beta;
  __device__ __forceinline__ double operator()(int i) const {
    const double2 t = pair[i];
    return CgFma(beta, t.x, t.y);
  }
};

// A task and, per lane, the first column, first value and length of its run.
// The walk loads the record two tasks ahead and the run pointers one task
// ahead, so that a task starts with its value and column loads.
struct RunHead {
  int4 t;
  int c0, c1, base;
};
__device__ __forceinline__ void LoadRunHead(RunHead& h, const int* __restrict__ run_ptr) {
  const int n = h.t.w & 0xff, lg = (h.t.w >> 16) & 0xff;
  const int u = h.t.x + min((int)(threadIdx.x & 63) >> lg, n - 1);
  h.c0 = run_ptr[u];
  h.c1 = run_ptr[u + 1];
  h.base = run_ptr[h.t.x];
}
// Calls f(head) for the wavefront's tasks of workgroup lb of grid: every
// kRunWaves-th of the workgroup's contiguous share (reverse: downwards).
template <class F>
__device__ __forceinline__ void WalkRunTasks(const int4* __restrict__ tasks, int ntasks,
                                             const int* __restrict__ run_ptr, int lb, int grid, int reverse, F f) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int first = (int)((int64_t)lb * ntasks / grid) + wave;
  const int end = (int)((int64_t)(lb + 1) * ntasks / grid);
  if (first >= end) return;
  const int cnt = (end - first + kRunWaves - 1) / kRunWaves;
  auto at = [&](int i) {
    const int k = min(i, cnt - 1);
    return tasks[first + (reverse ? cnt - 1 - k : k) * kRunWaves];
  };
  RunHead h, next;
  h.t = at(0);
  LoadRunHead(h, run_ptr);
  next = h;
  if (cnt > 1) next.t = at(1);
  for (int i = 0; i < cnt; i++) {
    int4 t2 = next.t;
    if (i + 1 < cnt) {
      t2 = at(i + 2);
      LoadRunHead(next, run_ptr);
    }
    f(h);
    h = next;
    next.t = t2;
  }
}

// The task's rows: y[r] = (ACCUM ? y[r] : 0) + s * (A x)[r]; with DOT the
// lane's sum of x[r] * (A x)[r] is added to dotacc.
template <int R, int U, bool ACCUM, bool DOT, class X>
__device__ __forceinline__ void RunTaskRows(const RunHead& h, const int* __restrict__ rcols,
                                            const double* __restrict__ rvals, const X& x,
                                            double* __restrict__ y, double s, double& dotacc,
                                            double* __restrict__ next) {
  const int4 t = h.t;
  const int n = t.w & 0xff, lg = (t.w >> 16) & 0xff;
  const int lane = threadIdx.x & 63, G = 1 << lg;
  const int g = lane >> lg, l = lane & (G - 1);
  const int c0 = h.c0, L = h.c1 - h.c0;
  const int v0 = t.y + (c0 - h.base) * R;
  double acc[R][1];
  RunPartials<R, 1, U>(rcols, rvals, x, 1, 0, c0, v0, L, l, G, acc);
  double mine = 0.0;
#pragma unroll
  for (int q = 0; q < R; q++) {
    const double sum = GroupSum(acc[q][0], lg);
    mine = l == q ? sum : mine;
  }
  if (g < n && l < R) {
    const int r = t.z + g * R + l;
    if (ACCUM) y[r] += s * mine; else y[r] = s * mine;
    if (DOT) {
      const double xr = x(r);
      dotacc += xr * mine;
      if (std::is_same<X, PairX>::value) next[2 * (int64_t)r] = xr;
    }
  }
}

// y = (ACCUM ? y : 0) + s * A x over the tasks (see above); DOT as in
// CsrSpmvKernel.  Each workgroup takes 4 * rounds consecutive tasks, its wavefronts
// in turn.
// Consecutive plain applies (Mult / MultAdd) alternate the direction of the
// walk (reverse), so that each apply starts on the values the previous one
// read last, which the 256 MB Infinity Cache still holds.  Every row is
// summed by the same code in the same order either way.  Inside CG (DOT) the
// vector kernels between two applies take that cache: it keeps the forward
// walk.  (Non-temporal value loads are slower here: the loads of one slot's
// R values share lines that L1 has to keep; CG on 64^2 p=3 17.2 -> 19.5 us an
// iteration.)
//
// Bound by the value stream and the loads per byte of it.  Against the former
// kernel (products of 2048-value blocks through LDS, one column and x load
// per value), us per apply: 32^3 p=4 (159M nonzeros) 389 -> 298 (4.3 TB/s of
// values alone, 5.2 TB/s with the shared columns), 20x16x24 p=4 97 -> 64,
// 61x67 p=3 7.8 -> 4.7.
// DIR (with DOT): x is the new search direction, formed from the pairs of D
// and stored by the rows' owners (CgDirection, which holds the stop flag).
template <bool ACCUM, bool DOT, bool DIR>
__global__ __launch_bounds__(kStreamBlock, DIR ? 4 : 6) void CsrRunsKernel(
    const int4* __restrict__ tasks, int ntasks, const int* __restrict__ run_ptr,
    const int* __restrict__ rcols, const double* __restrict__ rvals, const double* __restrict__ xv,
    double* __restrict__ y, double s, double* __restrict__ partials, const int* __restrict__ stop_flag, int reverse,
    CgDirection D) {
  static_assert(kStreamBlock == kCgBlock, "DirectionBeta");
  __shared__ double lds[kStreamBlock / 64 + 2];
  typename std::conditional<DIR, PairX, PlainX>::type x;
  if constexpr (DIR) {
    bool stopped;
    x.beta = DirectionBeta(D, stopped, lds);
    if (stopped) return;
    x.pair = reinterpret_cast<const double2*>(D.pair);
  } else {
    if (stop_flag && *stop_flag) return;
    x.x = xv;
  }
  const int lx = XcdContiguousBlock(blockIdx.x, gridDim.x);
  double dotacc = 0.0;
  WalkRunTasks(tasks, ntasks, run_ptr, reverse ? (int)gridDim.x - 1 - lx : lx, gridDim.x, reverse, [&](const RunHead& h) __attribute__((always_inline)) {
    ForRunShape<1>((h.t.w >> 8) & 0xff, h.t.w >> 24, [&](auto r, auto u) __attribute__((always_inline)) {
      RunTaskRows<decltype(r)::value, decltype(u)::value, ACCUM, DOT>(h, rcols, rvals, x, y, s, dotacc, D.next);
    });
  });
  if (DOT) {
    __syncthreads();
    StorePartial<kStreamBlock>(dotacc, partials, lds);
  }
}

template <int R, int U, int KC>
__device__ __forceinline__ void RunTaskRowsMulti(const RunHead& h, const int* __restrict__ rcols,
                                                 const double* __restrict__ rvals, const double* __restrict__ x,
                                                 double* __restrict__ y, int K, int j0) {
  const int4 t = h.t;
  const int n = t.w & 0xff, lg = (t.w >> 16) & 0xff;
  const int lane = threadIdx.x & 63, G = 1 << lg;
  const int g = lane >> lg, l = lane & (G - 1);
  const int c0 = h.c0, L = h.c1 - h.c0;
  const int v0 = t.y + (c0 - h.base) * R;
  double acc[R][KC];
  RunPartials<R, KC, U>(rcols, rvals, x, K, j0, c0, v0, L, l, G, acc);
  double mine[KC];
#pragma unroll
  for (int j = 0; j < KC; j++) mine[j] = 0.0;
#pragma unroll
  for (int q = 0; q < R; q++)
#pragma unroll
    for (int j = 0; j < KC; j++) {
      const double sum = GroupSum(acc[q][j], lg);
      mine[j] = l == q ? sum : mine[j];
    }
  if (g < n && l < R) {
    double* yp = y + ((int64_t)(t.z + g * R + l) * K + j0);
#pragma unroll
    for (int j = 0; j < KC; j++) yp[j] = mine[j];
  }
}

// Y = A X for K vectors stored interleaved (entry j of dof i at i K + j, the
// layout of a BaseVector with K components): the runs kernel with KC row sums
// per value (the KC components of a column's x are adjacent), the components
// in passes of KC = 4, 2, 1.  Each component is summed in the single kernel's
// order: bit-identical to a single apply.
__global__ __launch_bounds__(kStreamBlock, 3) void CsrRunsMultiKernel(
    const int4* __restrict__ tasks, int ntasks, const int* __restrict__ run_ptr,
    const int* __restrict__ rcols, const double* __restrict__ rvals, const double* __restrict__ x,
    double* __restrict__ y, int K, const int* __restrict__ stop) {
  if (stop && *stop) return;
  WalkRunTasks(tasks, ntasks, run_ptr, XcdContiguousBlock(blockIdx.x, gridDim.x), gridDim.x, 0, [&](const RunHead& h) __attribute__((always_inline)) {
    const int R = (h.t.w >> 8) & 0xff;
    int j0 = 0;
    while (j0 < K) {
      // 8 components at once up to 3 rows: 48 registers of sums
      const int rem = K - j0, kc = rem >= 8 && R <= 3 ? 8 : rem >= 4 ? 4 : rem >= 2 ? 2 : 1;
      auto go = [&](auto comps) __attribute__((always_inline)) {
        constexpr int KC = decltype(comps)::value;
        ForRunShape<KC>(R, h.t.w >> 24, [&](auto r, auto u) __attribute__((always_inline)) {
          RunTaskRowsMulti<decltype(r)::value, decltype(u)::value, KC>(h, rcols, rvals, x, y, K, j0);
        });
      };
      if (kc == 8) go(std::integral_constant<int, 8>{});
      else if (kc == 4) go(std::integral_constant<int, 4>{});
      else if (kc == 2) go(std::integral_constant<int, 2>{});
      else go(std::integral_constant<int, 1>{});
      j0 += kc;
    }
  });
}

// Component j of an interleaved K-vector to a plain vector and back (the
// other layouts apply the single-vector kernel per component).
__global__ void GatherComponentKernel(const double* __restrict__ x, int K, int j, double* __restrict__ out,
                                      int64_t n, const int* __restrict__ stop) {
  if (stop && *stop) return;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    out[i] = x[i * K + j];
}
__global__ void ScatterComponentKernel(const double* __restrict__ in, int K, int j, double* __restrict__ y,
                                       int64_t n, const int* __restrict__ stop) {
  if (stop && *stop) return;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    y[i * K + j] = in[i];
}

template <bool ACCUM, bool DOT>
static int LaunchSpmv(const CsrOp& A, double s, const double* x, double* y, hipStream_t st, double* partials,
                      const int* stop, int reverse = 0);

// Workgroups of a runs launch: one task per wavefront if cap allows, a
// multiple of 8 beyond 8 (the XCD mapping).
static int RunsGrid(const CsrOp& A, int cap) {
  const int wg = A.nblocks <= 8 ? A.nblocks : (A.nblocks + 7) & ~7;
  return std::max(1, std::min(wg, cap > 8 ? cap & ~7 : cap));
}

// The runs kernel with partial sums: a fold kernel (4.4 us) follows a grid of
// over 1024 workgroups, so up to 7168 workgroups' worth of tasks run on 1024
// and, with Jacobi, form the direction (us per CG iteration, wide grid / 1024:
// 14^3 p=4, 6,150 workgroups, 40.1 / 37.0; 128^2 p=5, 6,193, 42.7 / 40.1; 16^3
// p=3, 6,303, 33.7 / 29.1; 140^2 p=5, 7,403, 44.9 / 46.2; 200^2 p=3, 7,526, 37.4
// / 34.7; 150^2 p=5, 8,513, 49.3 / 51.6; 23x19x27 p=3, 17,964, 58.8 / 64.1).
static int RunsDotCap(const CsrOp& A) {
  return std::min(A.walk_grid, A.nblocks <= 7168 ? 1024 : kMaxWideBlocks);
}

void CsrOp::MultMulti(int K, const double* x, double* y, hipStream_t st, const int* stop) {
  NGSAMD_REQUIRE(K >= 1 && K <= 64, "multi-vector apply: 1 <= K <= 64 vectors");
  if (height == 0) return;
  if (width == 0) {
    // no columns: Y = 0
    LaunchFill(y, height * K, 0.0, st);
    return;
  }
  if (algo == 2) {
    CsrRunsMultiKernel<<<RunsGrid(*this, walk_grid), kStreamBlock, 0, st>>>(tasks.p, ntasks, run_ptr.p, rcols.p,
                                                                           rvals.p, x, y, K, stop);
    NGSAMD_CHECK_LAUNCH();
    return;
  }
  if (xcomp.n < (size_t)width) xcomp.alloc(width);
  if (ycomp.n < (size_t)height) ycomp.alloc(height);
  for (int j = 0; j < K; j++) {
    GatherComponentKernel<<<GridFor(width, 256, 8192), 256, 0, st>>>(x, K, j, xcomp.p, width, stop);
    NGSAMD_CHECK_LAUNCH();
    LaunchSpmv<false, false>(*this, 1.0, xcomp.p, ycomp.p, st, nullptr, stop);
    ScatterComponentKernel<<<GridFor(height, 256, 8192), 256, 0, st>>>(ycomp.p, K, j, y, height, stop);
    NGSAMD_CHECK_LAUNCH();
  }
}

__global__ void RunsDiagKernel(const int* __restrict__ run_row, const int* __restrict__ run_ptr,
                               const int* __restrict__ val_ptr, const int* __restrict__ rcols,
                               const double* __restrict__ rvals, double* __restrict__ d, int nruns) {
  for (int u = blockIdx.x * blockDim.x + threadIdx.x; u < nruns; u += gridDim.x * blockDim.x) {
    const int r0 = run_row[u], R = run_row[u + 1] - r0;
    const int c0 = run_ptr[u], L = run_ptr[u + 1] - c0;
    for (int q = 0; q < R; q++) {
      double val = 0.0;
      for (int j = 0; j < L; j++)
        if (rcols[c0 + j] == r0 + q) { val = rvals[val_ptr[u] + j * R + q]; break; }
      d[r0 + q] = val;
    }
  }
}

// The runs kernel's tasks: consecutive runs of equal length (rows) and group
// size, at most one wavefront's lanes; slots per lane are those of the
// task's longest run.
static std::vector<int4> RunTasks(const std::vector<int>& rr, const std::vector<int>& rpp, const std::vector<int>& vp) {
  std::vector<int4> tk;
  const int nruns = (int)rr.size() - 1;
  for (int u = 0; u < nruns;) {
    const int R = rr[u + 1] - rr[u], lg = RunGroupLog2(R, rpp[u + 1] - rpp[u]);
    int n = 1, len = rpp[u + 1] - rpp[u];
    while (n < (64 >> lg) && u + n < nruns && rr[u + n + 1] - rr[u + n] == R &&
           RunGroupLog2(R, rpp[u + n + 1] - rpp[u + n]) == lg) {
      len = std::max(len, rpp[u + n + 1] - rpp[u + n]);
      n++;
    }
    const int m = std::max(1, std::min(127, (len + (1 << lg) - 1) >> lg));
    tk.push_back(make_int4(u, vp[u], rr[u], n | R << 8 | lg << 16 | m << 24));
    u += n;
  }
  return tk;
}

CsrOp::CsrOp(int64_t h, int64_t w, const int64_t* rp, const int* c, const double* v)
    : ngsamd_op_s(OpKind::CSR) {
  height = h;
  width = w;
  NGSAMD_REQUIRE(h >= 0 && w >= 0, "ngsamd_csr_create: negative size");
  NGSAMD_REQUIRE(h < (int64_t(1) << 31) && w < (int64_t(1) << 31), "ngsamd_csr_create: size exceeds int32");
  nnz = rp[h];
  NGSAMD_REQUIRE(rp[0] == 0 && nnz >= 0, "ngsamd_csr_create: row pointer must start at 0");
  NGSAMD_REQUIRE(nnz < (int64_t(1) << 31), "ngsamd_csr_create: nnz exceeds int32");
  std::vector<int> rp32(h + 1);
  for (int64_t i = 0; i <= h; i++) {
    if (i > 0) NGSAMD_REQUIRE(rp[i] >= rp[i - 1], "ngsamd_csr_create: row pointer not monotone");
    rp32[i] = (int)rp[i];
  }
  for (int64_t k = 0; k < nnz; k++)
    NGSAMD_REQUIRE(c[k] >= 0 && c[k] < w, "ngsamd_csr_create: column number out of range");
  for (int64_t i = 0; i < h; i++) max_row_len = std::max<int64_t>(max_row_len, rp[i + 1] - rp[i]);
  if (w == 0) {
    static const double z = 0.0;
    xpad.alloc(1);
    xpad.upload(&z, 1);
  }
  const char* nnz_env = getenv("NGSAMD_SPMV_NNZ");
  block_nnz = nnz_env ? atoi(nnz_env) : 0;
  NGSAMD_REQUIRE(block_nnz == 0 || block_nnz == 1024 || block_nnz == 2048 || block_nnz == 4096,
                 "NGSAMD_SPMV_NNZ must be 1024, 2048 or 4096");
  // largest grid of the stream applies: 16384 measured best at 32^3 p=4
  max_grid = 16384;
  const char* grid_env = getenv("NGSAMD_SPMV_GRID");
  if (grid_env) {
    max_grid = atoi(grid_env);
    NGSAMD_REQUIRE(max_grid >= 8 && max_grid <= 65536, "NGSAMD_SPMV_GRID must be 8..65536");
  }
  const char* algo_env = getenv("NGSAMD_SPMV");
  const std::string algo_name = algo_env ? algo_env : "";
  NGSAMD_REQUIRE(algo_name.empty() || algo_name == "rowgroup" || algo_name == "stream" || algo_name == "runs",
                 "NGSAMD_SPMV must be rowgroup, stream or runs");
  if (algo_name.empty() || algo_name == "runs") {
    // in the runs layout block_nnz bounds the values of one run
    const int saved = block_nnz;
    if (block_nnz == 0) block_nnz = nnz < (int64_t(1) << 20) ? 1024 : 2048;
    // the runs layout pays when it saves at least a quarter of the column
    // numbers (H1 matrices of order >= 2 share patterns between the dofs of
    // an edge, a face or a cell)
    std::vector<int> rr, rpp, vp, rc, br, bl;
    std::vector<double> rv;
    rc.reserve(nnz);
    rv.reserve(nnz);
    nshared = BuildRuns(h, rp, c, v, block_nnz, rr, rpp, vp, rc, rv, br, bl);
    if (algo_name == "runs" || 4 * nshared <= 3 * nnz) {
      algo = 2;
      nruns = (int64_t)rr.size() - 1;
      std::vector<int4> tk = RunTasks(rr, rpp, vp);
      ntasks = (int)tk.size();
      tasks.alloc(std::max<size_t>(tk.size(), 1));
      if (!tk.empty()) tasks.upload(tk.data(), tk.size());
      nblocks = (ntasks + kRunWaves - 1) / kRunWaves;
      // One task per wavefront (32^3 p=4, 53K workgroups: 298 us per apply;
      // 16,384 workgroups 327, 2,048, the resident ones, 361).  Several
      // vectors' sums fill the registers: there a wavefront of 16,384
      // workgroups walks its tasks, each one's records loaded ahead (4
      // vectors 563 us against 650 with one task each).
      if (!grid_env) {
        max_grid = 1 << 28;
        walk_grid = 16384;
        if (nblocks > 4096) walk_grid = std::max(4096, std::min(16384, nblocks / 3));
      } else {
        walk_grid = max_grid;
      }
      run_row.alloc(rr.size());
      run_ptr.alloc(rpp.size());
      val_ptr.alloc(vp.size());
      rcols.alloc(std::max<int64_t>(nshared, 1));
      rvals.alloc(std::max<int64_t>(nnz, 1));
      run_row.upload(rr.data(), rr.size());
      run_ptr.upload(rpp.data(), rpp.size());
      val_ptr.upload(vp.data(), vp.size());
      if (nshared) rcols.upload(rc.data(), nshared);
      if (nnz && v) rvals.upload(rv.data(), nnz);
      if (nnz && !v) NGSAMD_HIP(hipMemsetAsync(rvals.p, 0, sizeof(double) * nnz, Stream()));
      if (!v) {
        std::vector<int> rrun(std::max<int64_t>(h, 1), 0);
        for (int64_t u = 0; u < nruns; u++)
          for (int r = rr[u]; r < rr[u + 1]; r++) rrun[r] = (int)u;
        row_run.alloc(rrun.size());
        row_run.upload(rrun.data(), rrun.size());
        NGSAMD_HIP(hipStreamSynchronize(Stream()));
      }
      NGSAMD_HIP(hipStreamSynchronize(Stream()));
      return;
    }
    block_nnz = saved;
  }
  // stream kernel: 2048 values per block (443.8 us on the 32^3 p=4 matrix,
  // 4096 443.4 us, 1024 470.7 us)
  if (block_nnz == 0) block_nnz = 2048;
  rowptr.alloc(h + 1);
  // 4 padding entries (column 0, value 0) behind the last nonzero: lanes
  // past the last block read entry nnz
  cols.alloc(nnz + 4);
  vals.alloc(nnz + 4);
  rowptr.upload(rp32.data(), h + 1);
  cols.upload(c, nnz);
  if (v) vals.upload(v, nnz);
  else if (nnz) NGSAMD_HIP(hipMemsetAsync(vals.p, 0, sizeof(double) * nnz, Stream()));
  {
    const int zc[4] = {0, 0, 0, 0};
    const double zv[4] = {0, 0, 0, 0};
    NGSAMD_HIP(hipMemcpyAsync(cols.p + nnz, zc, sizeof(zc), hipMemcpyHostToDevice, Stream()));
    NGSAMD_HIP(hipMemcpyAsync(vals.p + nnz, zv, sizeof(zv), hipMemcpyHostToDevice, Stream()));
    NGSAMD_HIP(hipStreamSynchronize(Stream()));
  }
  NGSAMD_HIP(hipStreamSynchronize(Stream()));
  double mean = h ? double(nnz) / double(h) : 0.0;
  group = mean > 48 ? 32 : mean > 20 ? 16 : mean > 9 ? 8 : 4;
  // row blocks of at most block_nnz nonzeros (or one longer row)
  std::vector<int> br;
  br.push_back(0);
  int64_t acc = 0;
  for (int64_t r = 0; r < h; r++) {
    const int64_t len = rp[r + 1] - rp[r];
    if (r > br.back() && acc + len > block_nnz) {
      br.push_back((int)r);
      acc = 0;
    }
    acc += len;
  }
  if (br.back() != h || h == 0) br.push_back((int)h);
  nblocks = (int)br.size() - 1;
  // about two blocks per workgroup (P1 matrices: 1024^2 triangles, 3.6K
  // blocks, 24.7 us on 2048 workgroups against 39.1 us on one block each;
  // 96^3 tets, 6.6K blocks, 45 vs 64 us on 4096), 1024 to 16384 workgroups
  if (!grid_env && nblocks > 1024) max_grid = std::max(1024, std::min(16384, nblocks / 2));
  blk_row.alloc(br.size());
  blk_row.upload(br.data(), br.size());
  NGSAMD_HIP(hipStreamSynchronize(Stream()));
  algo = algo_name == "rowgroup" ? 0 : 1;
}

void CsrOp::Values(double* host_vals) const {
  NGSAMD_HIP(hipStreamSynchronize(Stream()));
  if (nnz == 0) return;
  if (algo != 2) {
    NGSAMD_HIP(hipMemcpy(host_vals, vals.p, sizeof(double) * nnz, hipMemcpyDeviceToHost));
    return;
  }
  // runs layout: run u holds rows run_row[u].. with values [L][R]
  std::vector<int> rr(nruns + 1), vp(nruns + 1);
  std::vector<double> rv(nnz);
  NGSAMD_HIP(hipMemcpy(rr.data(), run_row.p, sizeof(int) * (nruns + 1), hipMemcpyDeviceToHost));
  NGSAMD_HIP(hipMemcpy(vp.data(), val_ptr.p, sizeof(int) * (nruns + 1), hipMemcpyDeviceToHost));
  NGSAMD_HIP(hipMemcpy(rv.data(), rvals.p, sizeof(double) * nnz, hipMemcpyDeviceToHost));
  int64_t k = 0;  // CSR position: rows in order
  for (int64_t u = 0; u < nruns; u++) {
    const int R = rr[u + 1] - rr[u];
    const int64_t L = R ? (vp[u + 1] - vp[u]) / R : 0;
    for (int q = 0; q < R; q++)
      for (int64_t j = 0; j < L; j++) host_vals[k++] = rv[vp[u] + j * R + q];
  }
}

template <int G, bool ACCUM, bool DOT>
static int LaunchSpmvG(const CsrOp& A, double s, const double* x, double* y, hipStream_t st, double* partials,
                       const int* stop) {
  constexpr int RPB = kSpmvBlock / G;
  const int64_t n = A.height;
  const int64_t passes = (n + RPB - 1) / RPB;
  // enough workgroups to fill the chip several times over; DOT variants are
  // limited by the size of the partials workspace
  const int64_t max_wg = DOT ? kMaxReduceBlocks : 65536;
  int64_t wg = passes < max_wg ? passes : max_wg;
  if (wg > 8) wg &= ~int64_t(7);
  if (wg < 1) wg = 1;
  const int iters = (int)((passes + wg - 1) / wg);
  CsrSpmvKernel<G, ACCUM, DOT><<<(int)wg, kSpmvBlock, 0, st>>>(A.rowptr.p, A.cols.p, A.vals.p, x, y, (int)n, s,
                                                               iters, partials, stop);
  NGSAMD_CHECK_LAUNCH();
  return (int)wg;
}

template <bool ACCUM, bool DOT>
static int LaunchStream(const CsrOp& A, double s, const double* x, double* y, hipStream_t st, double* partials,
                        const int* stop) {
  auto kern = A.block_nnz == 1024   ? CsrStreamKernel<1024, ACCUM, DOT>
              : A.block_nnz == 4096 ? CsrStreamKernel<4096, ACCUM, DOT>
                                    : CsrStreamKernel<2048, ACCUM, DOT>;
  // a wide grid (many more workgroups than resident slots) lets the hardware
  // balance blocks of uneven cost: measured faster than one workgroup per
  // resident slot (412 vs 452 us for the runs kernel at 32^3 p=4); the
  // variant with partial sums stays within the partials workspace
  const int cap = DOT ? std::min(A.max_grid, kMaxWideBlocks) : A.max_grid;
  int wg = A.nblocks < cap ? A.nblocks : cap;
  if (wg > 8) wg &= ~7;
  if (wg < 1) wg = 1;
  const int per = (A.nblocks + wg - 1) / wg;
  kern<<<(int)wg, kStreamBlock, 0, st>>>(A.rowptr.p, A.cols.p, A.vals.p, x, y, A.blk_row.p, A.nblocks, per, s,
                                         partials, stop);
  NGSAMD_CHECK_LAUNCH();
  return (int)wg;
}

template <bool ACCUM, bool DOT>
static int LaunchRuns(const CsrOp& A, double s, const double* x, double* y, hipStream_t st, double* partials,
                      const int* stop, int reverse) {
  const int wg = RunsGrid(A, DOT ? RunsDotCap(A) : A.max_grid);
  CsrRunsKernel<ACCUM, DOT, false><<<wg, kStreamBlock, 0, st>>>(A.tasks.p, A.ntasks, A.run_ptr.p, A.rcols.p,
                                                                A.rvals.p, x, y, s, partials, stop, reverse, {});
  NGSAMD_CHECK_LAUNCH();
  return wg;
}

template <bool ACCUM, bool DOT>
static int LaunchSpmv(const CsrOp& A, double s, const double* x, double* y, hipStream_t st, double* partials,
                      const int* stop, int reverse) {
  if (A.width == 0) x = A.xpad.p;
  if (A.algo == 2) return LaunchRuns<ACCUM, DOT>(A, s, x, y, st, partials, stop, reverse);
  if (A.algo == 1) return LaunchStream<ACCUM, DOT>(A, s, x, y, st, partials, stop);
  switch (A.group) {
    case 4: return LaunchSpmvG<4, ACCUM, DOT>(A, s, x, y, st, partials, stop);
    case 8: return LaunchSpmvG<8, ACCUM, DOT>(A, s, x, y, st, partials, stop);
    case 16: return LaunchSpmvG<16, ACCUM, DOT>(A, s, x, y, st, partials, stop);
    default: return LaunchSpmvG<32, ACCUM, DOT>(A, s, x, y, st, partials, stop);
  }
}

void CsrOp::MultAdd(double s, const double* x, double* y, hipStream_t st) {
  if (height == 0) return;
  LaunchSpmv<true, false>(*this, s, x, y, st, nullptr, nullptr, flip);
  flip ^= 1;
}

void CsrOp::Mult(const double* x, double* y, hipStream_t st) {
  if (height == 0) return;
  LaunchSpmv<false, false>(*this, 1.0, x, y, st, nullptr, nullptr, flip);
  flip ^= 1;
}

// Workgroups of the DOT variant's launch (one partial each), as LaunchRuns,
// LaunchStream and LaunchSpmvG choose them.
static int DotWorkgroups(const CsrOp& A) {
  if (A.algo == 0) return kMaxReduceBlocks;  // at most this many (LaunchSpmvG)
  if (A.algo == 2) return RunsGrid(A, RunsDotCap(A));
  const int cap = std::min(A.max_grid, kMaxWideBlocks);
  int wg = A.nblocks < cap ? A.nblocks : cap;
  if (wg > 8) wg &= ~7;
  return wg < 1 ? 1 : wg;
}

int CsrOp::MultDot(const double* x, double* y, double* partials, const int* d_stop, hipStream_t st,
                   double* wide) {
  // a small grid (at most 1,024 workgroups, e.g. 2D 64^2 p=3) writes its
  // partials straight to CG's, whose update kernel sums them: one launch
  // less per iteration
  if (DotWorkgroups(*this) <= 1024) return LaunchSpmv<false, true>(*this, 1.0, x, y, st, partials, d_stop);
  // the operator on its wide grid writes one partial per workgroup; a
  // 64-workgroup kernel folds them so that CG's kernels read 64 values
  if (!wide) wide = State().wide_partials;
  const int np = LaunchSpmv<false, true>(*this, 1.0, x, y, st, wide, d_stop);
  LaunchFoldPartials(wide, np, partials, d_stop, st);
  return kFoldedPartials;
}

bool CsrOp::FormsDirection() const { return algo == 2 && width > 0 && DotWorkgroups(*this) <= 1024; }

int CsrOp::MultDotDirection(const CgDirection& D, double* w, double* partials, hipStream_t st) {
  const int wg = RunsGrid(*this, RunsDotCap(*this));
  CsrRunsKernel<false, true, true><<<wg, kStreamBlock, 0, st>>>(tasks.p, ntasks, run_ptr.p, rcols.p, rvals.p, nullptr,
                                                                w, 1.0, partials, nullptr, 0, D);
  NGSAMD_CHECK_LAUNCH();
  return wg;
}

__global__ void CsrDiagKernel(const int* __restrict__ rowptr, const int* __restrict__ cols,
                              const double* __restrict__ vals, double* __restrict__ d, int n) {
  for (int r = blockIdx.x * blockDim.x + threadIdx.x; r < n; r += gridDim.x * blockDim.x) {
    double v = 0.0;
    for (int k = rowptr[r]; k < rowptr[r + 1]; k++)
      if (cols[k] == r) { v = vals[k]; break; }
    d[r] = v;
  }
}

void CsrOp::Diagonal(double* d, hipStream_t st) {
  if (height == 0) return;
  if (algo == 2) {
    RunsDiagKernel<<<GridFor(nruns, 256, 8192), 256, 0, st>>>(run_row.p, run_ptr.p, val_ptr.p, rcols.p, rvals.p, d,
                                                              (int)nruns);
    NGSAMD_CHECK_LAUNCH();
    return;
  }
  CsrDiagKernel<<<GridFor(height, 256, 8192), 256, 0, st>>>(rowptr.p, cols.p, vals.p, d, (int)height);
  NGSAMD_CHECK_LAUNCH();
}

}  // namespace ngsamd

using namespace ngsamd;

extern "C" int ngsamd_csr_create(ngsamd_op_t* op, int64_t height, int64_t width, const int64_t* rp,
                                 const int* cols, const double* vals) {
  return Guard([&] {
    RequireInit();
    NGSAMD_REQUIRE(height >= 0 && width >= 0, "ngsamd_csr_create: negative size");
    NGSAMD_REQUIRE(op && rp && (rp[height] == 0 || (cols && vals)), "ngsamd_csr_create: null argument");
    *op = nullptr;
    *op = new CsrOp(height, width, rp, cols, vals);
  });
}

extern "C" int ngsamd_csr_values(ngsamd_op_t op, double* h_vals) {
  return Guard([&] {
    RequireInit();
    NGSAMD_REQUIRE(op && op->kind == OpKind::CSR, "ngsamd_csr_values: not a CSR operator");
    CsrOp* A = static_cast<CsrOp*>(op);
    NGSAMD_REQUIRE(h_vals || A->nnz == 0, "ngsamd_csr_values: null argument");
    A->Values(h_vals);
  });
}

extern "C" int ngsamd_csr_info(ngsamd_op_t op, int64_t* h_info) {
  return Guard([&] {
    RequireInit();
    NGSAMD_REQUIRE(op && op->kind == OpKind::CSR, "ngsamd_csr_info: not a CSR operator");
    NGSAMD_REQUIRE(h_info, "ngsamd_csr_info: null argument");
    const CsrOp* A = static_cast<CsrOp*>(op);
    h_info[0] = A->algo;
    h_info[1] = DotWorkgroups(*A);
    h_info[2] = A->FormsDirection() ? 1 : 0;
    h_info[3] = 8 * (A->nnz + A->width + A->height) +
                (A->algo == 2 ? 4 * (A->nshared + A->nruns + 1) + 16 * (int64_t)A->ntasks
                              : 4 * (A->nnz + A->height + 1));
  });
}

extern "C" int ngsamd_csr_diagonal(ngsamd_op_t op, double* d) {
  return Guard([&] {
    RequireInit();
    NGSAMD_REQUIRE(op && op->kind == OpKind::CSR, "ngsamd_csr_diagonal: not a CSR operator");
    static_cast<CsrOp*>(op)->Diagonal(d, Stream());
  });
}

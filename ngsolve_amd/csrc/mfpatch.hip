// Matrix-free apply over element patches: the gather scatter of the factored
// kernels with most of the summation done in LDS.
//
// The elements are cut into patches of WAVES tiles of 16 (mfpart.hpp), one
// workgroup's work at a time.  A workgroup stages the x entries of the
// patch's dofs in LDS, each wavefront forms the element results of one tile
// (the factored contraction of MfFacKernel / MfFac16Kernel) into LDS, and then
// each of the patch's dofs is summed from LDS by one thread, in a fixed order:
// a dof inside the patch goes straight to y, a dof shared with other patches
// leaves one FP64 partial sum, and the gather kernel adds those up.  Element
// results never go to memory: at 32^3 p=4 with 128-element patches 1.4M
// partial sums of 8 B remain of 6.9M contributions, and x is read 1,900
// entries a patch instead of 4,480.
//
// All vertex orders use one reference class (ClassMap: the dofs of the other
// classes permuted, some with their signs turned, the metric transformed), so that a
// patch's tiles are full whatever the classes of its elements and one D block
// stays in LDS.  Where a class's 16-bit D is other numbers than the reference's
// (BF16 / FP16, 3D p=4) there are two, both in LDS, and a tile has one of them:
// patches of 112 elements in 8 tiles, 48 in 4 (32^3 p=4 BF16 43.8 us per apply
// with FP64 vectors, 40.9 with FP32; the general gather 71.1, 50.7).  Signs ride
// in bit 15 of the 16-bit LDS indices.
//
// What bounds it: per patch two barriers and the chain dof list -> x -> LDS
// -> MFMA -> LDS -> sums, overlapped between the workgroups of a CU.
#include <algorithm>
#include <memory>
#include <type_traits>
#include <vector>

#include "common.hpp"
#include "half.hpp"
#include "matfree.hpp"
#include "mfdev.hpp"
#include "mfpart.hpp"
#include "reduce.hpp"
#include "runtime_state.hpp"

namespace ngsamd {

// Table arguments of the kernels:
//   hdr     per patch: first group, groups of inner dofs, groups, first partial sum
//   xdof    [groups][64] dof, -1: padding
//   js      [groups][64][4] LDS position of the dof's first 4 contributions | sign << 15
//           (padding: a position that holds 0)
//   grp     per group: first further row of jx, contributions per dof
//   jx      [rows][64][4] the contributions after the fourth
//   lidx    [tile][64][KI] LDS position of an x entry | sign << 15
//   metric  [tile][NC][16], elnr [tile][16]
// nx: LDS x entries, the last one 0
#define NGSAMD_PATCH_PARAMS                                                                                     \
  const int4 *__restrict__ hdr, const int *__restrict__ xdof, const ushort4v *__restrict__ js,                  \
      const int2 *__restrict__ grp_tab, const ushort4v *__restrict__ jx, const uint16_t *__restrict__ lidx,     \
      const double *__restrict__ metric, const int *__restrict__ elnr, int npatch, int nx

typedef uint16_t ushort4v __attribute__((ext_vector_type(4)));

// v with the sign of bit 15 of idx
__device__ __forceinline__ double Signed(double v, int idx) {
  return __hiloint2double(__double2hiint(v) ^ ((idx & 0x8000) << 16), __double2loint(v));
}
__device__ __forceinline__ float Signed(float v, int idx) {
  return __int_as_float(__float_as_int(v) ^ ((idx & 0x8000) << 16));
}

// A wavefront's groups of a patch: wave, wave + WAVES, ...  The first NG are
// held in registers; the next patch's dofs are loaded during the contraction
// and their x entries during the sums.  (Loading the next patch's metric,
// coefficients and indices there as well measured slower, split FP16 at 32^3
// p=4 43.2 -> 45.5 us: it re-reads the dofs for the sums, and the kernel is
// bound by its tables' bytes more than by these latencies.)
template <int NG, class V>
struct PatchRegs {
  int xd[NG];      // dofs
  V v[NG];         // their x entries
  ushort4v j[NG];  // positions of their first contributions
  int2 gr[NG];     // grp_tab
};

template <int WAVES, int NG>
__device__ __forceinline__ void LoadDofs(int (&xd)[NG], const int4 h, const int* __restrict__ xdof, int wave, int lane) {
#pragma unroll
  for (int i = 0; i < NG; i++) xd[i] = xdof[(int64_t)(h.x + min(wave + i * WAVES, h.z - 1)) * 64 + lane];
}

// Sum of a dof's contributions cs in slot order, w of them (uniform), the
// first 4 at j, the others from row `more` of jx, 20 positions at a time.
template <class T>
__device__ __forceinline__ double SumSlots(const T* cs, const ushort4v j, int w, const ushort4v* __restrict__ jx,
                                           int more, int lane) {
  constexpr int U = 5;
  double acc = 0.0;
#pragma unroll
  for (int i = 0; i < 4; i++)
    if (i < w) acc += (double)Signed(cs[j[i] & 0x7fff], j[i]);
  for (int k = 4; k < w; k += 4 * U, more += U) {
    const int rows = (w - k + 3) / 4;
    ushort4v a[U];
#pragma unroll
    for (int r = 0; r < U; r++) a[r] = jx[(int64_t)(more + min(r, rows - 1)) * 64 + lane];
#pragma unroll
    for (int r = 0; r < U; r++)
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (k + 4 * r + i < w) acc += (double)Signed(cs[a[r][i] & 0x7fff], a[r][i]);
  }
  return acc;
}

// The sum of group g's dof d: an inner one into y, a shared one into part.
template <class V>
__device__ __forceinline__ void StoreSum(const int4 h, int g, int d, double acc, V* __restrict__ y,
                                         double* __restrict__ part, double s, int accumulate, int lane) {
  if (d < 0) return;
  if (g < h.y) {
    const double v = s * acc;
    y[d] = accumulate ? (V)((double)y[d] + v) : (V)v;
  } else {
    part[(int64_t)h.w + (g - h.y) * 64 + lane] = acc;
  }
}

template <int WAVES, int NG, class T, class V>
__device__ __forceinline__ void SumPatch(const PatchRegs<NG, V>& R, const int4 h, const T* cs,
                                         const int* __restrict__ xdof, const ushort4v* __restrict__ js,
                                         const int2* __restrict__ grp_tab, const ushort4v* __restrict__ jx,
                                         V* __restrict__ y, double* __restrict__ part, double s, int accumulate,
                                         int wave, int lane) {
#pragma unroll
  for (int i = 0; i < NG; i++) {
    const int g = wave + i * WAVES;
    if (g < h.z)
      StoreSum(h, g, R.xd[i], SumSlots(cs, R.j[i], R.gr[i].y, jx, R.gr[i].x, lane), y, part, s, accumulate, lane);
  }
  for (int g = wave + NG * WAVES; g < h.z; g += WAVES) {
    const int2 gr = grp_tab[h.x + g];
    const int64_t at = (int64_t)(h.x + g) * 64 + lane;
    const int d = xdof[at];
    StoreSum(h, g, d, SumSlots(cs, js[at], gr.y, jx, gr.x, lane), y, part, s, accumulate, lane);
  }
}

// An x entry as the contraction holds it in LDS.  For BF16 operands an FP64 entry
// goes to FP32 by rounding to odd, so that its rounding to BF16 is that of the
// FP64 value (one rounding, as in the general kernel; two differ in one of 1e4
// entries, 1e-5 of the result).
template <class T, bool ODD, class V>
__device__ __forceinline__ T PatchX(V v) {
  const T t = (T)v;
  if constexpr (ODD && sizeof(V) == 8) {
    const double r = (double)t;
    const int b = __float_as_int(t) - (fabs(r) > fabs(v) ? 1 : 0);  // toward 0
    return r < v || r > v ? __int_as_float(b | 1) : t;
  }
  return t;
}

// The start of a patch, whose dofs and x entries R holds: when the other
// wavefronts have finished the previous patch (its contributions share the
// LDS), the x entries go into LDS.  The first contributions' positions are
// loaded for the sums.
template <int WAVES, bool ODD, int NG, class T, class V>
__device__ __forceinline__ void StageX(PatchRegs<NG, V>& R, const int4 h, const V* __restrict__ x, T* xs, int nx,
                                       const int* __restrict__ xdof, const ushort4v* __restrict__ js,
                                       const int2* __restrict__ grp_tab, int wave, int lane) {
#pragma unroll
  for (int i = 0; i < NG; i++) {
    const int g = h.x + min(wave + i * WAVES, h.z - 1);
    R.j[i] = js[(int64_t)g * 64 + lane];
    const int2 gr = grp_tab[g];
    R.gr[i] = make_int2(__builtin_amdgcn_readfirstlane(gr.x), __builtin_amdgcn_readfirstlane(gr.y));
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NG; i++)
    if (wave + i * WAVES < h.z) xs[(wave + i * WAVES) * 64 + lane] = PatchX<T, ODD>(R.v[i]);
  for (int g = wave + NG * WAVES; g < h.z; g += WAVES)
    xs[g * 64 + lane] = PatchX<T, ODD>(x[max(xdof[(int64_t)(h.x + g) * 64 + lane], 0)]);
  if (threadIdx.x == 0) xs[nx - 1] = (T)0;
  __syncthreads();
}

// FP64 / FP32 contraction; D in LDS in the layout of MfFacKernel
template <class T, int DIM, int NDP, int ND, int KG, class V, int WAVES>
__global__ __launch_bounds__(64 * WAVES, 4) void MfPatchKernel(const T* __restrict__ fmat, int64_t fstride, NGSAMD_PATCH_PARAMS,
                                                            const double* __restrict__ kappa,
                                                            const V* __restrict__ x, V* __restrict__ y,
                                                            double* __restrict__ part, double s, int accumulate,
                                                            const int* __restrict__ stop,
                                                            double* __restrict__ partials) {
  if (stop && *stop) return;
  typedef typename Acc4<T>::type acc_t;
  constexpr int NC = DIM * (DIM + 1) / 2;
  constexpr int NG = ND >= 20 ? 4 : 2;
  constexpr int KS = NDP / 4;
  constexpr int KI = (KS + 3) / 4 * 4;
  constexpr int MT = (NDP + 15) / 16;
  constexpr int NSL = DIM * KG;
  constexpr int TT = (NSL + 3) / 4;
  constexpr int VW = 16 / (int)sizeof(T);
  constexpr int KSP = (KS + VW - 1) / VW * VW;
  constexpr int JP = (NSL + VW - 1) / VW * VW;
  typedef T vec_t __attribute__((ext_vector_type(VW)));
  typedef ushort4v Idx;  // 4 LDS indices of a lane
  constexpr int NI = KI / 4;
  extern __shared__ __align__(16) unsigned char lds_raw[];
  T* ls = reinterpret_cast<T*>(lds_raw);
  T* xs = ls + fstride;
  T* cs = xs;  // after the x entries have been read
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int col = lane & 15, grp = lane >> 4;
  CopyToLds<64 * WAVES>(ls, fmat, (int)(fstride * sizeof(T) / 16));
  const T* a1 = ls + lane * KSP;
  const T* a2 = ls + TT * 64 * KSP + lane * JP;
  double dacc = 0.0;
  const int wg = XcdContiguousBlock(blockIdx.x, gridDim.x);
  const int p0 = (int)((int64_t)wg * npatch / gridDim.x), p1 = (int)((int64_t)(wg + 1) * npatch / gridDim.x);
  PatchRegs<NG, V> R;
  int4 h = hdr[min(p0, npatch - 1)], hn = hdr[min(p0 + 1, npatch - 1)];
  LoadDofs<WAVES>(R.xd, h, xdof, wave, lane);
#pragma unroll
  for (int i = 0; i < NG; i++) R.v[i] = x[max(R.xd[i], 0)];
  for (int p = p0; p < p1; p++) {
    const int64_t tile = (int64_t)p * WAVES + wave;
    Idx li[NI];
#pragma unroll
    for (int q = 0; q < NI; q++) li[q] = reinterpret_cast<const Idx*>(lidx)[(tile * 64 + lane) * NI + q];
    double mv[NC];
#pragma unroll
    for (int c = 0; c < NC; c++) mv[c] = metric[(tile * NC + c) * 16 + col];
    const double kap = kappa[elnr[tile * 16 + col]];
    StageX<WAVES, false>(R, h, x, xs, nx, xdof, js, grp_tab, wave, lane);
    int xn[NG];  // the next patch's dofs
    LoadDofs<WAVES>(xn, hn, xdof, wave, lane);
    T xk[KS];
#pragma unroll
    for (int st = 0; st < KS; st++) {
      const int j = li[st / 4][st % 4];
      xk[st] = Signed(xs[j & 0x7fff], j);
    }
    __syncthreads();  // all x entries are read: the contributions may take their place
    // U = D^T X
    acc_t u[TT];
#pragma unroll
    for (int t = 0; t < TT; t++) u[t] = acc_t{0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < KSP / VW; q++) {
      vec_t a[TT];
#pragma unroll
      for (int t = 0; t < TT; t++) a[t] = *reinterpret_cast<const vec_t*>(a1 + t * 64 * KSP + VW * q);
#pragma unroll
      for (int j = 0; j < VW; j++)
        if (VW * q + j < KS)
#pragma unroll
          for (int t = 0; t < TT; t++) u[t] = Mfma(a[t][j], xk[VW * q + j], u[t]);
    }
    // V = (kappa G) U
    T g[NC];
#pragma unroll
    for (int c = 0; c < NC; c++) g[c] = (T)(kap * mv[c]);
    T v[JP];
#pragma unroll
    for (int j = 0; j < JP; j++) v[j] = (T)0;
#pragma unroll
    for (int kl = 0; kl < KG; kl++) {
      T uu[DIM], vv[DIM];
#pragma unroll
      for (int d = 0; d < DIM; d++) uu[d] = u[(kl * DIM + d) / 4][(kl * DIM + d) % 4];
      ApplyMetric<DIM, T>(g, uu, vv);
#pragma unroll
      for (int d = 0; d < DIM; d++) v[kl * DIM + d] = vv[d];
    }
    if (partials) {
      T ld = (T)0;
#pragma unroll
      for (int j = 0; j < NSL; j++) ld += u[j / 4][j % 4] * v[j];
      dacc += (double)ld;
    }
    // Y = D V
    acc_t yacc[MT];
#pragma unroll
    for (int m = 0; m < MT; m++) yacc[m] = acc_t{0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < JP / VW; q++) {
      vec_t a[MT];
#pragma unroll
      for (int m = 0; m < MT; m++) a[m] = *reinterpret_cast<const vec_t*>(a2 + m * 64 * JP + VW * q);
#pragma unroll
      for (int j = 0; j < VW; j++)
        if (VW * q + j < NSL)
#pragma unroll
          for (int m = 0; m < MT; m++) yacc[m] = Mfma(a[m][j], v[VW * q + j], yacc[m]);
    }
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int dof = 16 * m + AccRow<T>(grp, r);
        // FP32 rows of a full tile in the order 4 r + grp: a store covers 64 adjacent words
        const int pos = sizeof(T) == 4 && 16 * m + 16 <= ND ? 16 * m + 4 * r + grp : dof;
        if (dof < ND) cs[(wave * ND + pos) * 16 + col] = yacc[m][r];
      }
    if (threadIdx.x == 0) cs[16 * WAVES * ND] = (T)0;
#pragma unroll
    for (int i = 0; i < NG; i++) R.v[i] = x[max(xn[i], 0)];
    __syncthreads();
    SumPatch<WAVES>(R, h, cs, xdof, js, grp_tab, jx, y, part, s, accumulate, wave, lane);
#pragma unroll
    for (int i = 0; i < NG; i++) R.xd[i] = xn[i];
    h = hn;
    hn = hdr[min(p + 2, npatch - 1)];
  }
  if (partials) {
    __shared__ double s_dot[WAVES];
    StorePartial<64 * WAVES>(dacc, partials, s_dot);
  }
}

// 16-bit contraction (BF16, FP16, split FP16); D in LDS in the layout of MfFac16Kernel
// TWO: the factors of two reference classes, tile_rep the one of each tile
template <class H, int DIM, int KS1, int MT, int KG, int ND, class V, bool SPLIT, int WAVES, bool TWO>
__global__ __launch_bounds__(64 * WAVES, 4) void MfPatch16Kernel(const uint16_t* __restrict__ fmat, int64_t fstride,
                                                              NGSAMD_PATCH_PARAMS, const double* __restrict__ kappa,
                                                              const V* __restrict__ x, V* __restrict__ y,
                                                              double* __restrict__ part, double s, int accumulate,
                                                              const int* __restrict__ stop,
                                                              double* __restrict__ partials,
                                                              const int* __restrict__ tile_rep) {
  if (stop && *stop) return;
  typedef typename Vec8<H>::type h8;
  typedef uint16_t Idx __attribute__((ext_vector_type(8)));  // 8 LDS indices of a lane
  constexpr int NI = KS1;
  constexpr int NC = DIM * (DIM + 1) / 2;
  constexpr int NG = ND >= 20 ? 4 : 2;
  constexpr int NSL = DIM * KG;
  constexpr int TT = ((NSL + 3) / 4 + 1) / 2 * 2;
  constexpr int KS2 = TT / 2;
  extern __shared__ __align__(16) unsigned char lds_raw[];
  float* xs = reinterpret_cast<float*>(lds_raw + fstride * (TWO ? 4 : 2));
  float* cs = xs;  // after the x entries have been read
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int col = lane & 15, grp = lane >> 4;
  CopyToLds<64 * WAVES>(lds_raw, fmat, (int)(fstride / (TWO ? 4 : 8)));
  const h8* a1 = reinterpret_cast<const h8*>(lds_raw) + lane;
  const h8* a2 = a1 + TT * KS1 * 64;
  const h8* a1l = a1 + (TT * KS1 + MT * KS2) * 64;
  const h8* a2l = a1l + TT * KS1 * 64;
  int rep = 0;
  double dacc = 0.0;
  const int wg = XcdContiguousBlock(blockIdx.x, gridDim.x);
  const int p0 = (int)((int64_t)wg * npatch / gridDim.x), p1 = (int)((int64_t)(wg + 1) * npatch / gridDim.x);
  PatchRegs<NG, V> R;
  int4 h = hdr[min(p0, npatch - 1)], hn = hdr[min(p0 + 1, npatch - 1)];
  LoadDofs<WAVES>(R.xd, h, xdof, wave, lane);
#pragma unroll
  for (int i = 0; i < NG; i++) R.v[i] = x[max(R.xd[i], 0)];
  for (int p = p0; p < p1; p++) {
    const int64_t tile = (int64_t)p * WAVES + wave;
    Idx li[NI];
#pragma unroll
    for (int q = 0; q < NI; q++) li[q] = reinterpret_cast<const Idx*>(lidx)[(tile * 64 + lane) * NI + q];
    double mv[NC];
#pragma unroll
    for (int c = 0; c < NC; c++) mv[c] = metric[(tile * NC + c) * 16 + col];
    const double kap = kappa[elnr[tile * 16 + col]];
    if constexpr (TWO) {
      const int r = __builtin_amdgcn_readfirstlane(tile_rep[tile]);
      a1 += (r - rep) * (int)(fstride / 8);
      a2 += (r - rep) * (int)(fstride / 8);
      rep = r;
    }
    StageX<WAVES, std::is_same<H, __bf16>::value>(R, h, x, xs, nx, xdof, js, grp_tab, wave, lane);
    int xn[NG];  // the next patch's dofs
    LoadDofs<WAVES>(xn, hn, xdof, wave, lane);
    float xf[KS1][8];
#pragma unroll
    for (int ks = 0; ks < KS1; ks++)
#pragma unroll
      for (int j = 0; j < 8; j++) {
        // (ks, j) beyond ND is padding in every lane group
        const int k = li[ks][j];
        xf[ks][j] = 32 * ks + j < ND ? Signed(xs[k & 0x7fff], k) : 0.0f;
      }
    __syncthreads();  // all x entries are read: the contributions may take their place
    float g[NC];
#pragma unroll
    for (int c = 0; c < NC; c++) g[c] = (float)(kap * mv[c]);
    // FP16: powers of two out of x and the metric, as in MfFac16Kernel
    int escale = 0, edot = 0;
    if constexpr (!std::is_same<H, __bf16>::value) {
      float xm = 0.0f, gm = 0.0f;
#pragma unroll
      for (int ks = 0; ks < KS1; ks++)
#pragma unroll
        for (int j = 0; j < 8; j++) xm = fmaxf(xm, fabsf(xf[ks][j]));
      xm = fmaxf(xm, __shfl_xor(xm, 16, 64));
      xm = fmaxf(xm, __shfl_xor(xm, 32, 64));
#pragma unroll
      for (int c = 0; c < NC; c++) gm = fmaxf(gm, fabsf(g[c]));
      int ex = 0, eg = 0;
      (void)frexpf(xm, &ex);
      (void)frexpf(gm, &eg);
#pragma unroll
      for (int ks = 0; ks < KS1; ks++)
#pragma unroll
        for (int j = 0; j < 8; j++) xf[ks][j] = ldexpf(xf[ks][j], -ex);
#pragma unroll
      for (int c = 0; c < NC; c++) g[c] = ldexpf(g[c], -eg);
      escale = ex + eg;
      edot = 2 * ex + eg;
    }
    h8 xg[KS1], xl[KS1];
#pragma unroll
    for (int ks = 0; ks < KS1; ks++)
#pragma unroll
      for (int j = 0; j < 8; j++) {
        xg[ks][j] = (H)xf[ks][j];
        if (SPLIT) xl[ks][j] = (H)(xf[ks][j] - (float)xg[ks][j]);
      }
    float4v u[TT];
#pragma unroll
    for (int t = 0; t < TT; t++) u[t] = float4v{0, 0, 0, 0};
#pragma unroll
    for (int ks = 0; ks < KS1; ks++)
#pragma unroll
      for (int t = 0; t < TT; t++) {
        u[t] = Mfma16(a1[(t * KS1 + ks) * 64], xg[ks], u[t]);
        if (SPLIT) {
          u[t] = Mfma16(a1[(t * KS1 + ks) * 64], xl[ks], u[t]);
          u[t] = Mfma16(a1l[(t * KS1 + ks) * 64], xg[ks], u[t]);
        }
      }
    float v[4 * TT];
#pragma unroll
    for (int j = 0; j < 4 * TT; j++) v[j] = 0.0f;
#pragma unroll
    for (int kl = 0; kl < KG; kl++) {
      float uu[DIM], vv[DIM];
#pragma unroll
      for (int d = 0; d < DIM; d++) uu[d] = u[(kl * DIM + d) / 4][(kl * DIM + d) % 4];
      ApplyMetric<DIM, float>(g, uu, vv);
#pragma unroll
      for (int d = 0; d < DIM; d++) v[kl * DIM + d] = vv[d];
    }
    h8 vb[KS2], vl[KS2];
#pragma unroll
    for (int k2 = 0; k2 < KS2; k2++)
#pragma unroll
      for (int j = 0; j < 8; j++) {
        vb[k2][j] = (H)v[8 * k2 + j];
        if (SPLIT) vl[k2][j] = (H)(v[8 * k2 + j] - (float)vb[k2][j]);
      }
    if (partials) {
      float ld = 0.0f;
#pragma unroll
      for (int j = 0; j < NSL; j++)
        ld += u[j / 4][j % 4] * (SPLIT ? (float)vb[j / 8][j % 8] + (float)vl[j / 8][j % 8] : (float)vb[j / 8][j % 8]);
      dacc += ldexp((double)ld, edot);
    }
    float4v yacc[MT];
#pragma unroll
    for (int m = 0; m < MT; m++) yacc[m] = float4v{0, 0, 0, 0};
#pragma unroll
    for (int k2 = 0; k2 < KS2; k2++)
#pragma unroll
      for (int m = 0; m < MT; m++) {
        yacc[m] = Mfma16(a2[(m * KS2 + k2) * 64], vb[k2], yacc[m]);
        if (SPLIT) {
          yacc[m] = Mfma16(a2[(m * KS2 + k2) * 64], vl[k2], yacc[m]);
          yacc[m] = Mfma16(a2l[(m * KS2 + k2) * 64], vb[k2], yacc[m]);
        }
      }
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int dof = 16 * m + 4 * grp + r;
        const int pos = 16 * m + 16 <= ND ? 16 * m + 4 * r + grp : dof;  // as in MfPatchKernel
        if (dof < ND) cs[(wave * ND + pos) * 16 + col] = ldexpf(yacc[m][r], escale);
      }
    if (threadIdx.x == 0) cs[16 * WAVES * ND] = 0.0f;
#pragma unroll
    for (int i = 0; i < NG; i++) R.v[i] = x[max(xn[i], 0)];
    __syncthreads();
    SumPatch<WAVES>(R, h, cs, xdof, js, grp_tab, jx, y, part, s, accumulate, wave, lane);
#pragma unroll
    for (int i = 0; i < NG; i++) R.xd[i] = xn[i];
    h = hn;
    hn = hdr[min(p + 2, npatch - 1)];
  }
  if (partials) {
    __shared__ double s_dot[WAVES];
    StorePartial<64 * WAVES>(dacc, partials, s_dot);
  }
}

// ----------------------------------------------------------------- host side

// A table that its loop fills whole: not cleared first, so that the threads that
// write it take its pages in.
template <class T>
class HostTable {
 public:
  explicit HostTable(size_t n) : n_(n), p_(new T[n]) {}
  T& operator[](size_t i) { return p_[i]; }
  T* data() { return p_.get(); }
  const T* data() const { return p_.get(); }
  size_t size() const { return n_; }

 private:
  size_t n_;
  std::unique_ptr<T[]> p_;
};

// whether the one-term 16-bit kernels have an instance for two reference
// classes: tetrahedra of order 4, the first order whose classes round apart
static bool PatchShapeOfTwo(int dim, int nd) { return dim == 3 && nd == 35; }

bool MfPatchPlan::Build(int dim, int nd, int64_t ndof, int prec, int ks1_, int64_t fbytes,
                        const std::vector<MfClass>& classes, const std::vector<double>& S,
                        const std::vector<double>& D, int rank, const int* dofs, const double* metric, const int* elnr,
                        int max_lds, int64_t min_elements) {
  const bool f64_ = prec == NGSAMD_PREC_F64;
  const bool half_ = prec == NGSAMD_PREC_BF16 || prec == NGSAMD_PREC_F16 || prec == NGSAMD_PREC_F16X3;
  const int nclass = (int)classes.size(), nc = dim * (dim + 1) / 2;
  const int64_t nel = nclass ? classes.back().end : 0;
  // on few patches a patch's chain of phases is longer than the two wide
  // kernels (MatFreeOp's rule gives the number)
  if (nel < min_elements) return false;
  // Each class as a relabelling of a reference class, the first one where that can be.
  // One 16-bit term: a class's results change with the rounding of its factor (3D
  // p=4 structured meshes: one class of three maps with A = (1 0 0; -1 -1 -1;
  // 0 1 0), BF16 results 4e-4 apart), so that the reference class's must be the
  // same rounded numbers, and a class without one becomes the second.  Split FP16
  // and FP32 differ by less than their sums' rounding.
  const bool one_term = half_ && prec != NGSAMD_PREC_F16X3;
  std::vector<ClassMap> map(nclass);
  std::vector<int> rep(nclass, -1);  // index among reps
  const size_t ssz = (size_t)nc * nd * nd, dsz = (size_t)dim * nd * rank;
  reps.clear();
  for (int c = 0; c < nclass; c++) {
    auto maps_to = [&](int r) {
      return MapClass(dim, nd, S.data() + r * ssz, S.data() + c * ssz, map[c]) &&
             (!one_term || SameRoundedFactor(dim, nd, rank, D.data() + r * dsz, D.data() + c * dsz, map[c],
                                             prec == NGSAMD_PREC_F16 ? ToF16 : ToBf16));
    };
    for (size_t r = 0; r < reps.size() && rep[c] < 0; r++)
      if (maps_to(reps[r])) rep[c] = (int)r;
    if (rep[c] >= 0) continue;
    if (reps.size() >= (one_term && PatchShapeOfTwo(dim, nd) ? 2 : 1) || !maps_to(c)) return false;
    rep[c] = (int)reps.size();
    reps.push_back(c);
  }
  // elements by number: neighbours in the mesh are mostly near each other
  int64_t kmax = 0;
  for (int64_t e = 0; e < nel; e++) kmax = std::max<int64_t>(kmax, elnr[e]);
  if (kmax >= 8 * nel + 1024) return false;
  Workers workers(16);
  std::vector<int> cnt(kmax + 2, 0), cls(nel);
  for (int c = 0; c < nclass; c++)
    for (int64_t e = classes[c].begin; e < classes[c].end; e++) cls[e] = c;
  for (int64_t e = 0; e < nel; e++) cnt[elnr[e] + 1]++;
  for (int64_t k = 0; k <= kmax; k++) cnt[k + 1] += cnt[k];
  std::vector<int> row(nel);
  for (int64_t e = 0; e < nel; e++) row[cnt[elnr[e]]++] = (int)e;
  // 8 tiles a patch (fewer shared dofs), 4 (more and smaller workgroups) where
  // 8 leave fewer than four patches per CU: 32^3 p=4 (1,536 patches of 8) FP64
  // 72 us against 89 with 4, split FP16 43 against 48 with FP32 vectors; 181x203
  // triangles p=5 (574) FP32 18.6 against 16.2, 23x19x27 p=3 (553) split FP16
  // 19.4 against 18.1
  waves = nel >= (int64_t)4 * 128 * DeviceCUs() ? 8 : 4;
  // A tile's elements have one reference class: with two of them, 16 elements
  // less always fit.
  const int size = 16 * waves, fill = size - 16 * ((int)reps.size() - 1);
  npatch = (int)((nel + fill - 1) / fill);
  // grown in chunks of 128 patches (whatever the number of threads)
  std::vector<int> order(nel);  // element rows, patch by patch
  {
    const int nv = std::min(dim + 1, nd);
    std::vector<int> vptr, vadj, vd((size_t)nel * nv);  // vd: the elements' vertex dofs
    for (int64_t i = 0; i < nel; i++) std::copy_n(dofs + (int64_t)row[i] * nd, nv, &vd[(size_t)i * nv]);
    VertexElements(nel, nv, nv, vd.data(), vptr, vadj);
    const int64_t chunk = (int64_t)128 * fill;
    workers.Run((nel + chunk - 1) / chunk, 1, [&](Workers::Ranges& r) {
      std::vector<int> stamp(vptr.size(), 0);
      int patch = 0;
      for (int64_t c, c1; r.Next(c, c1);)
        GrowPatches(c * chunk, std::min(nel, c1 * chunk), nv, nv, vd.data(), vptr, vadj, fill, stamp, patch, order.data());
    });
    for (int64_t i = 0; i < nel; i++) order[i] = row[order[i]];
  }

  // the element row of every tile column, -1: none
  std::vector<int> slot((size_t)npatch * size, -1), trep((size_t)npatch * waves, 0);
  for (int64_t p = 0; p < npatch; p++) {
    int64_t at = p * size;
    for (int r = 0; r < (int)reps.size(); r++) {
      at = (at + 15) / 16 * 16;
      for (int64_t i = p * fill; i < std::min(nel, (p + 1) * fill); i++)
        if (rep[cls[order[i]]] == r) {
          trep[at / 16] = r;
          slot[at++] = order[i];
        }
    }
  }

  // dofs of more than one patch (whichever thread meets a dof first owns it,
  // the flags come out the same)
  std::vector<int> owner(ndof, -1);
  std::vector<unsigned char> shared(ndof, 0);
  workers.Run(npatch, 32, [&](Workers::Ranges& r) {
    r.Each([&](int64_t p) {
      for (int64_t i = p * size; i < (p + 1) * size; i++)
        for (int k = 0; k < nd && slot[i] >= 0; k++) {
          const int d = dofs[(int64_t)slot[i] * nd + k];
          int was = __atomic_load_n(&owner[d], __ATOMIC_RELAXED);
          if (was < 0 && __atomic_compare_exchange_n(&owner[d], &was, (int)p, false, __ATOMIC_RELAXED, __ATOMIC_RELAXED))
            continue;
          if (was != p) __atomic_store_n(&shared[d], (unsigned char)1, __ATOMIC_RELAXED);
        }
    });
  });
  for (int64_t d = 0; d < ndof; d++)
    if (owner[d] < 0) return false;  // a dof of no element: the general gather writes its 0

  // per patch: its dofs (inner, then shared; by falling count, then number),
  // the groups and slot rows
  struct Patch {
    std::vector<int> xdof;
    std::vector<int2> grp;
    std::vector<uint16_t> js, jx;  // first 4 slots of each dof, the others
    int nig = 0;
  };
  std::vector<Patch> pt(npatch);
  const int ki = half_ ? 8 * ks1_ : ((nd + 3) / 4 + 3) / 4 * 4;
  const int ntile = npatch * waves;
  HostTable<uint16_t> lidx((size_t)ntile * 64 * ki);
  HostTable<double> tm((size_t)ntile * nc * 16);
  HostTable<int> te((size_t)ntile * 16);
  HostTable<uint16_t> local((size_t)npatch * size * nd);  // position of each element dof in its patch's list
  const int zero_cs = 16 * waves * nd;
  auto pos_of = [&](int k) {  // row order of the contributions in LDS (see the kernels)
    if (f64_ || (k & ~15) + 16 > nd) return k;
    const int r = k & 15;
    return (k & ~15) + 4 * (r % 4) + r / 4;
  };
  std::vector<int> max_local(npatch, 0);
  workers.Run(npatch, 8, [&](Workers::Ranges& r) {
    Numbering number((size_t)size * nd);
    std::vector<int> at((size_t)size * nd), dl, c, place;  // at: number of each element dof among the patch's dl
    std::vector<int> width, rows, filled;
    std::vector<uint64_t> key;
    std::vector<int> o;
    KeySort sort;
    r.Each([&](int64_t p) {
      Patch& P = pt[p];
      const int64_t i0 = p * size, i1 = i0 + size;
      dl.clear();
      c.clear();
      number.Clear();
      for (int64_t i = i0; i < i1; i++)
        for (int k = 0; k < nd && slot[i] >= 0; k++) {
          const int d = dofs[(int64_t)slot[i] * nd + k], a = number.Add(d);
          at[(size_t)(i - i0) * nd + k] = a;
          if (a == (int)dl.size()) {
            dl.push_back(d);
            c.push_back(0);
          }
          c[a]++;
        }
      // inner before shared, then by falling count, then by number
      key.resize(dl.size());
      for (size_t q = 0; q < dl.size(); q++)
        key[q] = (uint64_t)shared[dl[q]] << 63 | (uint64_t)(0x7fffffff - c[q]) << 32 | (uint32_t)dl[q];
      sort(key, o);
      size_t q = 0;
      place.resize(dl.size());  // padded position
      for (int part = 0; part < 2; part++) {
        while (P.xdof.size() % 64) P.xdof.push_back(-1);
        if (part == 1) P.nig = (int)P.xdof.size() / 64;
        for (; q < o.size() && shared[dl[o[q]]] == part; q++) {
          place[o[q]] = (int)P.xdof.size();
          P.xdof.push_back(dl[o[q]]);
        }
      }
      while (P.xdof.size() % 64) P.xdof.push_back(-1);
      max_local[p] = (int)P.xdof.size();
      const int ng = (int)P.xdof.size() / 64;
      width.assign(ng, 0);
      rows.assign(ng + 1, 0);
      for (size_t a = 0; a < dl.size(); a++) width[place[a] / 64] = std::max(width[place[a] / 64], c[a]);
      for (int g = 0; g < ng; g++) rows[g + 1] = rows[g] + std::max(0, (width[g] - 1) / 4);
      for (int g = 0; g < ng; g++) P.grp.push_back(make_int2(rows[g], width[g]));
      P.js.assign((size_t)ng * 256, (uint16_t)zero_cs);
      P.jx.assign((size_t)rows[ng] * 256, (uint16_t)zero_cs);
      filled.assign(dl.size(), 0);
      for (int64_t i = i0; i < i1; i++) {
        const int e = slot[i];
        if (e < 0) continue;
        const ClassMap& m = map[cls[e]];
        for (int k = 0; k < nd; k++) {
          const int a = at[(size_t)(i - i0) * nd + k], pl = place[a];
          const uint16_t sg = m.sign[k] < 0 ? 0x8000 : 0;
          const int li = (int)(i - i0);
          const int sl = filled[a]++;
          uint16_t& to = sl < 4 ? P.js[(size_t)pl * 4 + sl]
                                : P.jx[((size_t)(rows[pl / 64] + sl / 4 - 1) * 64 + pl % 64) * 4 + sl % 4];
          to = (uint16_t)(((li / 16) * nd + pos_of(m.perm[k])) * 16 + li % 16) | sg;
          local[(size_t)i * nd + m.perm[k]] = (uint16_t)pl | sg;
        }
      }
    });
  });
  nx = *std::max_element(max_local.begin(), max_local.end()) + 1;
  if (nx > 0x7fff || zero_cs > 0x7fff) return false;
  nx = (nx + 3) / 4 * 4;
  const size_t ts = f64_ ? 8 : 4;
  lds = (size_t)fbytes * reps.size() + ts * (size_t)std::max(nx, zero_cs + 1);  // the contributions take the x entries' place
  lds = (lds + 15) / 16 * 16;
  if (lds + 1024 > (size_t)max_lds) return false;

  workers.Run(ntile, 64, [&](Workers::Ranges& r) {
    r.Each([&](int64_t t) {
      for (int l = 0; l < 64; l++) {
        const int64_t i = t * 16 + l % 16;
        const int g = l / 16, e = slot[i];
        uint16_t* out = &lidx[((size_t)t * 64 + l) * ki];
        for (int q = 0; q < ki; q++) {
          const int k = half_ ? 32 * (q / 8) + 8 * g + q % 8 : 4 * q + g;
          out[q] = e >= 0 && k < nd ? local[(size_t)i * nd + k] : (uint16_t)(nx - 1);
        }
        if (g) continue;
        if (e < 0) {  // lanes without an element: metric 0, some element's coefficient
          for (int q = 0; q < nc; q++) tm[((size_t)t * nc + q) * 16 + l % 16] = 0.0;
          te[(size_t)t * 16 + l % 16] = elnr[order[nel - 1]];
          continue;
        }
        const double* A = map[cls[e]].A;
        const double* m = metric + (int64_t)e * nc;
        const double G3[9] = {m[0], m[nc > 3 ? 3 : 0], m[nc > 3 ? 4 : 0], m[nc > 3 ? 3 : 0], m[1], m[nc > 3 ? 5 : 0],
                              m[nc > 3 ? 4 : 0], m[nc > 3 ? 5 : 0], m[2]};
        const double G2[4] = {m[0], m[2], m[2], m[1]};
        const double* G = dim == 3 ? G3 : G2;
        double R[9];
        for (int a = 0; a < dim; a++)
          for (int b = 0; b < dim; b++) {
            double sum = 0.0;
            for (int c = 0; c < dim; c++)
              for (int d = 0; d < dim; d++) sum += A[a * dim + c] * G[c * dim + d] * A[b * dim + d];
            R[a * dim + b] = sum;
          }
        const double r3[6] = {R[0], R[4], R[8], R[1], R[2], R[5]}, r2[3] = {R[0], R[3], R[1]};
        for (int q = 0; q < nc; q++) tm[((size_t)t * nc + q) * 16 + l % 16] = dim == 3 ? r3[q] : r2[q];
        te[(size_t)t * 16 + l % 16] = elnr[e];
      }
    });
  });

  // concatenated tables, and the shared dofs' partial sums in patch order
  std::vector<int4> hdr(npatch);
  int64_t g0 = 0, r0 = 0, b0 = 0;
  for (int p = 0; p < npatch; p++) {
    const int ng = (int)pt[p].grp.size();
    hdr[p] = make_int4((int)g0, pt[p].nig, ng, (int)b0);
    for (auto& g : pt[p].grp) g.x += (int)r0;
    g0 += ng;
    r0 += (int64_t)pt[p].jx.size() / 256;
    b0 += (int64_t)(ng - pt[p].nig) * 64;
  }
  if (g0 * 64 >= (int64_t(1) << 31) || b0 >= (int64_t(1) << 31) || r0 >= (int64_t(1) << 31)) return false;
  HostTable<int> xd((size_t)g0 * 64);
  HostTable<int2> gp(g0);
  HostTable<uint16_t> js((size_t)g0 * 256), jx((size_t)r0 * 256);
  std::vector<int64_t> roff(npatch + 1, 0);
  for (int p = 0; p < npatch; p++) roff[p + 1] = roff[p] + (int64_t)pt[p].jx.size();
  workers.Run(npatch, 64, [&](Workers::Ranges& r) {
    r.Each([&](int64_t p) {
      std::copy(pt[p].xdof.begin(), pt[p].xdof.end(), xd.data() + (size_t)hdr[p].x * 64);
      std::copy(pt[p].grp.begin(), pt[p].grp.end(), gp.data() + hdr[p].x);
      std::copy(pt[p].js.begin(), pt[p].js.end(), js.data() + (size_t)hdr[p].x * 256);
      std::copy(pt[p].jx.begin(), pt[p].jx.end(), jx.data() + roff[p]);
    });
  });
  // gather of the shared dofs: in the order their first partial sum appears
  std::vector<int> pc(ndof, 0), gorder, grow(1, 0), gslot(0);
  for (int p = 0; p < npatch; p++)
    for (int q = pt[p].nig * 64; q < (int)pt[p].xdof.size(); q++) {
      const int d = pt[p].xdof[q];
      if (d < 0) continue;
      if (pc[d]++ == 0) gorder.push_back(d);
    }
  nshared = (int64_t)gorder.size();
  std::vector<int>& first = owner;  // reused: first slot of each shared dof
  int64_t tot = 0;
  for (int64_t i = 0; i < nshared; i++) {
    first[gorder[i]] = (int)tot;
    tot += pc[gorder[i]];
    grow.push_back((int)tot);
  }
  gslot.resize(tot);
  for (int p = 0; p < npatch; p++)
    for (int q = pt[p].nig * 64; q < (int)pt[p].xdof.size(); q++)
      if (pt[p].xdof[q] >= 0) gslot[first[pt[p].xdof[q]]++] = hdr[p].w + q - pt[p].nig * 64;

  auto up = [](auto& dev, const auto& host) {
    dev.alloc(std::max<size_t>(host.size(), 1));
    if (host.size()) dev.upload(host.data(), host.size());
  };
  up(d_hdr, hdr);
  up(d_xdof, xd);
  up(d_grp, gp);
  up(d_js, js);
  up(d_jx, jx);
  up(d_lidx, lidx);
  up(d_metric, tm);
  up(d_elnr, te);
  if (reps.size() > 1) up(d_tile_rep, trep);
  up(s_rowptr, grow);
  up(s_slots, gslot);
  up(s_order, gorder);
  part.alloc(std::max<int64_t>(b0, 1));
  NGSAMD_HIP(hipStreamSynchronize(Stream()));
  return true;
}

// prepare: enable the dynamic LDS size and record the occupancy
template <class K, class F, class V, class... More>
static void LaunchPatch(const MatFreeOp& A, K kern, const F* fmat, const V* x, V* y, double s, int accumulate,
                        const int* stop, hipStream_t st, double* partials, bool prepare, More... more) {
  const MfPatchPlan& L = A.patch;
  if (prepare) {
    NGSAMD_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)L.lds));
    int nb = 0;
    NGSAMD_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kern, 64 * L.waves, L.lds));
    L.occ[sizeof(V) == 8] = std::max(1, nb);
    return;
  }
  kern<<<L.Grid(sizeof(V) == 8), 64 * L.waves, L.lds, st>>>(
      fmat, A.fstride, L.d_hdr.p, L.d_xdof.p, reinterpret_cast<const ushort4v*>(L.d_js.p), L.d_grp.p,
      reinterpret_cast<const ushort4v*>(L.d_jx.p), L.d_lidx.p, L.d_metric.p, L.d_elnr.p, L.npatch, L.nx, A.Kappa(), x,
      y, L.part.p, s, accumulate, stop, partials, more...);
  NGSAMD_CHECK_LAUNCH();
}

template <class T, int DIM, class V>
static void DispatchPatch(const MatFreeOp& A, const T* fm, const V* x, V* y, double s, int accumulate, const int* stop,
                          hipStream_t st, double* partials, bool prepare) {
#define NGSAMD_PATCH(NDP, ND, KG)                                                                                    \
  if (A.nd == ND && A.fac_kg == KG)                                                                                  \
    return A.patch.waves == 8                                                                                        \
               ? LaunchPatch(A, MfPatchKernel<T, DIM, NDP, ND, KG, V, 8>, fm, x, y, s, accumulate, stop, st, partials, prepare) \
               : LaunchPatch(A, MfPatchKernel<T, DIM, NDP, ND, KG, V, 4>, fm, x, y, s, accumulate, stop, st, partials, prepare);
  if constexpr (DIM == 2) {
    NGSAMD_PATCH(8, 6, 1) NGSAMD_PATCH(12, 10, 2) NGSAMD_PATCH(16, 15, 3) NGSAMD_PATCH(24, 21, 4)
  } else {
    NGSAMD_PATCH(4, 4, 1) NGSAMD_PATCH(12, 10, 1) NGSAMD_PATCH(20, 20, 3) NGSAMD_PATCH(36, 35, 5)
  }
#undef NGSAMD_PATCH
  throw Error(NGSAMD_E_STATE, "matrix-free: unsupported patch shape");
}

template <class H, int DIM, bool SPLIT, class V>
static void DispatchPatch16(const MatFreeOp& A, const V* x, V* y, double s, int accumulate, const int* stop,
                            hipStream_t st, double* partials, bool prepare) {
  const uint16_t* fm = A.patch.reps.size() > 1 ? A.patch.d_reps.p : A.fmat16.p;
  const int* tile_rep = A.patch.d_tile_rep.p;
#define NGSAMD_PATCH(KS1, MT, KG, ND, TWO)                                                                           \
  if (A.nd == ND && A.fac_kg == KG && TWO == (A.patch.reps.size() > 1))                                              \
    return A.patch.waves == 8                                                                                        \
               ? LaunchPatch(A, MfPatch16Kernel<H, DIM, KS1, MT, KG, ND, V, SPLIT, 8, TWO>, fm, x, y, s, accumulate, stop, st, partials, prepare, tile_rep) \
               : LaunchPatch(A, MfPatch16Kernel<H, DIM, KS1, MT, KG, ND, V, SPLIT, 4, TWO>, fm, x, y, s, accumulate, stop, st, partials, prepare, tile_rep);
  if constexpr (DIM == 2) {
    NGSAMD_PATCH(1, 1, 1, 6, false) NGSAMD_PATCH(1, 1, 2, 10, false) NGSAMD_PATCH(1, 1, 3, 15, false)
    NGSAMD_PATCH(1, 2, 4, 21, false)
  } else {
    NGSAMD_PATCH(1, 1, 1, 4, false) NGSAMD_PATCH(1, 1, 1, 10, false) NGSAMD_PATCH(1, 2, 3, 20, false)
    NGSAMD_PATCH(2, 3, 5, 35, false)
    if constexpr (!SPLIT) {
      NGSAMD_PATCH(2, 3, 5, 35, true)
    }
  }
#undef NGSAMD_PATCH
  throw Error(NGSAMD_E_STATE, "matrix-free: unsupported 16-bit patch shape");
}

bool PatchShape(int dim, int nd, int kg) {
  auto is = [&](int n, int k) { return nd == n && kg == k; };
  return dim == 2 ? is(6, 1) || is(10, 2) || is(15, 3) || is(21, 4)
                  : is(4, 1) || is(10, 1) || is(20, 3) || is(35, 5);
}

template <class V>
void PatchApply(const MatFreeOp& A, const V* x, V* y, double s, int accumulate, const int* stop, hipStream_t st,
                double* partials, bool prepare) {
  auto half = [&](auto h, auto split) {
    typedef decltype(h) H;
    constexpr bool S = decltype(split)::value;
    if (A.dim == 2) DispatchPatch16<H, 2, S, V>(A, x, y, s, accumulate, stop, st, partials, prepare);
    else DispatchPatch16<H, 3, S, V>(A, x, y, s, accumulate, stop, st, partials, prepare);
  };
  if (A.precision == NGSAMD_PREC_BF16) half(__bf16{}, std::false_type{});
  else if (A.precision == NGSAMD_PREC_F16) half(_Float16{}, std::false_type{});
  else if (A.precision == NGSAMD_PREC_F16X3) half(_Float16{}, std::true_type{});
  else if (A.precision == NGSAMD_PREC_F64) {
    if (A.dim == 2) DispatchPatch<double, 2, V>(A, A.fmat64.p, x, y, s, accumulate, stop, st, partials, prepare);
    else DispatchPatch<double, 3, V>(A, A.fmat64.p, x, y, s, accumulate, stop, st, partials, prepare);
  } else {
    if (A.dim == 2) DispatchPatch<float, 2, V>(A, A.fmat32.p, x, y, s, accumulate, stop, st, partials, prepare);
    else DispatchPatch<float, 3, V>(A, A.fmat32.p, x, y, s, accumulate, stop, st, partials, prepare);
  }
}
template void PatchApply<double>(const MatFreeOp&, const double*, double*, double, int, const int*, hipStream_t, double*, bool);
template void PatchApply<float>(const MatFreeOp&, const float*, float*, double, int, const int*, hipStream_t, double*, bool);

}  // namespace ngsamd

// Newton + FGMRES + upper block-triangular preconditioner (Badia2024Solver,
// src/Solvers/badia2024.jl:2-48) on the GPU.
//
// Unknowns are numbered in the Badia2024 block style [u; j], p, phi
// (src/fespaces.jl:8), so the [u,j] block A11 is the leading n1 x n1 block and,
// with rows' columns sorted, every row of A11 is a prefix of its CSR row.
//
// Preconditioner, applied to v = (v1, vp, vphi):
//   z_phi = S_phi^-1 v_phi,  S_phi = alpha_phi M_phi,  alpha_phi = -1/(1 + zeta_j)
//   z_p   = S_p^-1 v_p,      S_p   = alpha_p M_p,      alpha_p   = -1/(beta + zeta_u)
//   z1    ~ A11^-1 (v1 - A12 z_p - A13 z_phi)
// M_p (dP1) and M_phi (dQ1) are cell-block diagonal, so their inverses are
// exact cell-local 4x4 / 8x8 blocks (the reference reaches the same fixed point
// with CG-Jacobi).  A11^-1 is approximated by `inner_iters` steps of GMRES on
// A11, right-preconditioned by additive Schwarz over vertex-star patches (the
// patch of a vertex holds every u / j dof whose support lies in the cells
// around it); the dense patch inverses come from a batched Gauss-Jordan kernel.
//
// Precision: precision 0 runs everything in FP64.  Precisions 1 to 3 keep
// FP64 for the residual assembly, the outer FGMRES (the refinement residual,
// its classical Gram-Schmidt with reorthogonalisation, the Newton update) and
// the p / phi Schur solves, and run the inner A11 GMRES in FP32 with an FP32
// copy of A11; the patch inverses are stored in FP32 (1), BF16 (2) or FP16
// scaled by a power of two per patch (3).  Patch products sum in FP64.
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>
#include <rocblas/rocblas.h>
#include <rocsolver/rocsolver.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <type_traits>

#include "mhd_cell.h"

using namespace mhd;

namespace {

constexpr int TB = 256;

inline int nblocks(int64_t n, int per = TB) { return (int)std::min<int64_t>((n + per - 1) / per, 1 << 20); }

template <class T>
__device__ inline double todbl(T v) { return (double)v; }
template <>
__device__ inline double todbl<__hip_bfloat16>(__hip_bfloat16 v) { return (double)__bfloat162float(v); }
template <>
__device__ inline double todbl<__half>(__half v) { return (double)__half2float(v); }

// ---------------------------------------------------------------- vectors
template <class T>
__global__ void k_fill(int64_t n, T v, T *__restrict__ x) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) x[i] = v;
}
template <class T>
__global__ void k_axpy(int64_t n, double a, const T *__restrict__ x, T *__restrict__ y) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    y[i] = (T)((double)y[i] + a * (double)x[i]);
}
template <class T>
__global__ void k_scale_copy(int64_t n, double a, const T *__restrict__ x, T *__restrict__ y) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    y[i] = (T)(a * (double)x[i]);
}
template <class S, class D>
__global__ void k_convert(int64_t n, const S *__restrict__ x, D *__restrict__ y) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    y[i] = (D)x[i];
}

__device__ inline double block_sum(double v) {
  __shared__ double red[TB / 64];
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  if (lane == 0) red[wv] = v;
  __syncthreads();
  double s = 0.0;
  if (threadIdx.x == 0)
    for (int k = 0; k < TB / 64; ++k) s += red[k];
  __syncthreads();
  return s;
}

// part[k * gridDim.x + b] = sum over block b's slice of V_k . w   (grid: x = slices, y = k)
template <class T>
__global__ __launch_bounds__(TB) void k_mdot(const T *__restrict__ V, int64_t ldv, const T *__restrict__ w, int64_t n,
                                             double *__restrict__ part) {
  const int k = blockIdx.y;
  const T *v = V + (int64_t)k * ldv;
  double acc = 0.0;
  for (int64_t i = blockIdx.x * (int64_t)TB + threadIdx.x; i < n; i += (int64_t)gridDim.x * TB)
    acc += (double)v[i] * (double)w[i];
  acc = block_sum(acc);
  if (threadIdx.x == 0) part[(int64_t)k * gridDim.x + blockIdx.x] = acc;
}
__global__ __launch_bounds__(TB) void k_mdot_final(int nb, const double *__restrict__ part, double *__restrict__ out) {
  const int k = blockIdx.x;
  double acc = 0.0;
  for (int b = threadIdx.x; b < nb; b += TB) acc += part[(int64_t)k * nb + b];
  acc = block_sum(acc);
  if (threadIdx.x == 0) out[k] = acc;
}
// w -= sum_k h[k] V_k  (h on device; K doubles of dynamic LDS)
template <class T>
__global__ __launch_bounds__(TB) void k_gs_update(int K, const T *__restrict__ V, int64_t ldv,
                                                  const double *__restrict__ h, T *__restrict__ w, int64_t n) {
  extern __shared__ double hs[];
  for (int k = threadIdx.x; k < K; k += TB) hs[k] = h[k];
  __syncthreads();
  for (int64_t i = blockIdx.x * (int64_t)TB + threadIdx.x; i < n; i += (int64_t)gridDim.x * TB) {
    double acc = (double)w[i];
    for (int k = 0; k < K; ++k) acc -= hs[k] * (double)V[(int64_t)k * ldv + i];
    w[i] = (T)acc;
  }
}
// x = beta * x + sum_k y[k] Z_k  (y on device; K doubles of dynamic LDS)
template <class T>
__global__ __launch_bounds__(TB) void k_lincomb(int K, const T *__restrict__ Z, int64_t ldz, const double *__restrict__ y,
                                                double beta, T *__restrict__ x, int64_t n) {
  extern __shared__ double ys[];
  for (int k = threadIdx.x; k < K; k += TB) ys[k] = y[k];
  __syncthreads();
  for (int64_t i = blockIdx.x * (int64_t)TB + threadIdx.x; i < n; i += (int64_t)gridDim.x * TB) {
    double acc = beta == 0.0 ? 0.0 : beta * (double)x[i];
    for (int k = 0; k < K; ++k) acc += ys[k] * (double)Z[(int64_t)k * ldz + i];
    x[i] = (T)acc;
  }
}

// ---------------------------------------------------------------- SpMV
// One lane's share of a CSR row dot product: entries p0, p0 + LPR, ... < e,
// four independent accumulators so that four value / column / x loads are in
// flight per lane (1.4x over a single accumulator at 64 x 64 x 8, measured).
template <int LPR, class MV, class TX>
__device__ inline double csr_row_dot(int64_t p0, int64_t e, const int32_t *__restrict__ colind,
                                     const MV *__restrict__ val, const TX *__restrict__ x) {
  double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
  int64_t p = p0;
  for (; p + 3 * LPR < e; p += 4 * LPR) {
    a0 += (double)val[p] * (double)x[colind[p]];
    a1 += (double)val[p + LPR] * (double)x[colind[p + LPR]];
    a2 += (double)val[p + 2 * LPR] * (double)x[colind[p + 2 * LPR]];
    a3 += (double)val[p + 3 * LPR] * (double)x[colind[p + 3 * LPR]];
  }
  for (; p < e; p += LPR) a0 += (double)val[p] * (double)x[colind[p]];
  return (a0 + a1) + (a2 + a3);
}

// y = v - (the columns from split on) . x: the p and phi columns of the [u,j] rows
template <int LPR>
__global__ __launch_bounds__(256) void k_spmv_suffix(int64_t nrows, const int64_t *__restrict__ rowptr,
                                                     const int64_t *__restrict__ split,
                                                     const int32_t *__restrict__ colind,
                                                     const double *__restrict__ val, const double *__restrict__ x,
                                                     const double *__restrict__ v, double *__restrict__ y) {
  const int64_t gid = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  const int64_t row = gid / LPR;
  const int lane = threadIdx.x % LPR;
  double acc = 0.0;
  if (row < nrows) acc = csr_row_dot<LPR>(split[row] + lane, rowptr[row + 1], colind, val, x);
#pragma unroll
  for (int off = LPR / 2; off > 0; off >>= 1) acc += __shfl_down(acc, off, LPR);
  if (row < nrows && lane == 0) y[row] = v[row] - acc;
}

// Rows that share one column list (the 3 components of a velocity node, the 4
// flux dofs of a face, the 12 interior current dofs, the 4 pressure and 8
// potential dofs of a cell) form a group: its columns are stored once, its
// values stay where the CSR has them (row i of the group at rowptr[r0] +
// i * len).  `LPG` lanes per group; each column's x value is loaded once for
// all rows of the group.  MODE 0: y = A x (full rows); 1: y = A11 x (the
// prefix up to split); 3: y = v - A11 x.
constexpr int GMAX = 12;
template <class MV, class TX, class TY, int LPG, int MODE>
__global__ __launch_bounds__(256) void k_spmv_grp(int64_t ngroups, const int64_t *__restrict__ grow,
                                                  const int64_t *__restrict__ gcp, const int32_t *__restrict__ gcol,
                                                  const int64_t *__restrict__ rowptr, const int64_t *__restrict__ split,
                                                  const MV *__restrict__ val, const TX *__restrict__ x,
                                                  const TY *__restrict__ v, TY *__restrict__ y) {
  const int64_t gid = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  const int64_t g = gid / LPG;
  const int lane = threadIdx.x % LPG;
  double acc[GMAX];
#pragma unroll
  for (int i = 0; i < GMAX; ++i) acc[i] = 0.0;
  int m = 0;
  int64_t r0 = 0;
  if (g < ngroups) {
    r0 = grow[g];
    m = (int)(grow[g + 1] - r0);
    const int64_t b = rowptr[r0];
    const int64_t len = rowptr[r0 + 1] - b;
    const int64_t e = MODE == 0 ? len : split[r0] - b;
    const int32_t *__restrict__ cols = gcol + gcp[g];
    const MV *__restrict__ vb = val + b;
    int64_t k = lane;
    // four columns per step: four independent column -> x load chains in flight
    for (; k + 3 * LPG < e; k += 4 * LPG) {
      const double x0 = (double)x[cols[k]], x1 = (double)x[cols[k + LPG]];
      const double x2 = (double)x[cols[k + 2 * LPG]], x3 = (double)x[cols[k + 3 * LPG]];
#pragma unroll
      for (int i = 0; i < GMAX; ++i)
        if (i < m) {
          const MV *__restrict__ vr = vb + i * len + k;
          acc[i] += ((double)vr[0] * x0 + (double)vr[LPG] * x1) + ((double)vr[2 * LPG] * x2 + (double)vr[3 * LPG] * x3);
        }
    }
    for (; k < e; k += LPG) {
      const double xv = (double)x[cols[k]];
#pragma unroll
      for (int i = 0; i < GMAX; ++i)
        if (i < m) acc[i] += (double)vb[i * len + k] * xv;
    }
  }
#pragma unroll
  for (int i = 0; i < GMAX; ++i) {
    double sm = acc[i];
#pragma unroll
    for (int off = LPG / 2; off > 0; off >>= 1) sm += __shfl_down(sm, off, LPG);
    if (lane == 0 && i < m) {
      const int64_t row = r0 + i;
      y[row] = MODE == 3 ? (TY)((double)v[row] - sm) : (TY)sm;
    }
  }
}

// y (+)= A x for a plain CSR matrix (prolongation / restriction)
template <class MV, class T, int LPR, bool ACC>
__global__ __launch_bounds__(256) void k_csr(int64_t nrows, const int64_t *__restrict__ rowptr,
                                             const int32_t *__restrict__ colind, const MV *__restrict__ val,
                                             const T *__restrict__ x, T *__restrict__ y) {
  const int64_t gid = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  const int64_t row = gid / LPR;
  const int lane = threadIdx.x % LPR;
  double acc = 0.0;
  if (row < nrows) acc = csr_row_dot<LPR>(rowptr[row] + lane, rowptr[row + 1], colind, val, x);
#pragma unroll
  for (int off = LPR / 2; off > 0; off >>= 1) acc += __shfl_down(acc, off, LPR);
  if (row < nrows && lane == 0) y[row] = ACC ? (T)((double)y[row] + acc) : (T)acc;
}

// minimal-residual coarse correction: a = (rr . w) / (w . w) from dots[0..1],
// y += a yc, rr -= a w  (w = A yc); a = 0 when w vanishes
template <class T>
__global__ void k_cc_update(int64_t n, const double *__restrict__ dots, const T *__restrict__ yc,
                            const T *__restrict__ w, T *__restrict__ y, T *__restrict__ rr) {
  const double a = dots[1] > 0.0 ? dots[0] / dots[1] : 0.0;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    y[i] = (T)((double)y[i] + a * (double)yc[i]);
    rr[i] = (T)((double)rr[i] - a * (double)w[i]);
  }
}

// Adjoint scaling D^-1 A^T D with D = 1 on u, p and s on j, phi (block
// numbering [u; j], p, phi): A^T carries A's Lorentz couplings swapped, sigma X
// in the u rows and -gamma X^T in the j rows; with s = gamma / sigma the scaled
// operator has A's coupling magnitudes again, which the Schur and Krylov parts
// of the preconditioner are tuned to (row weights of the 2-norm residual).
__device__ inline double adj_d(int64_t i, int64_t nu, int64_t n1, int64_t np, double s) {
  return ((i >= nu && i < n1) || i >= n1 + np) ? s : 1.0;
}
__global__ void k_adj_scale(int64_t n, const int64_t *__restrict__ rowptr, const int32_t *__restrict__ colind,
                            double *__restrict__ val, int64_t nu, int64_t n1, int64_t np, double s) {
  for (int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; r < n; r += (int64_t)gridDim.x * blockDim.x) {
    const double ir = 1.0 / adj_d(r, nu, n1, np, s);
    for (int64_t p = rowptr[r]; p < rowptr[r + 1]; ++p) val[p] *= adj_d(colind[p], nu, n1, np, s) * ir;
  }
}
__global__ void k_adj_scale_vec(int64_t n, int64_t nu, int64_t n1, int64_t np, double f, double *__restrict__ x) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    if ((i >= nu && i < n1) || i >= n1 + np) x[i] *= f;
}

// D = diag(v) on an n x n column-major matrix (off-diagonal untouched)
__global__ void k_set_diag(int64_t n, double v, double *__restrict__ D) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    D[i + i * n] = v;
}

// ---------------------------------------------------------------------------
// Dense inverse of the condensed coarsest [u,j] block by block Gauss-Jordan: for
// each block column K of width BGJ_B, P = A_KK^-1 (one workgroup, pivoting
// inside its 32 x 32 diagonal blocks), then the rank-BGJ_B update
//   A <- A - A[:,K] P A[K,:],  A[K,:] <- P A[K,:],  A[:,K] <- -A[:,K] P,  A_KK <- P
// (2 n^3 flops in all, like an LU plus triangular solves).  Pivoting is inside
// the diagonal blocks only; the result is checked by a residual and redone with
// the row-pivoted LU if it fails.
// Two launches a block column: k_gj_panel writes C = -A[:,K] and R = P A[K,:]
// with R[:,K] = P, so that k_gj_update is A += C R with zero for A[:,K] and R
// for A[K,:].  The next diagonal block needs only its own part of the update,
// so the first workgroup of k_gj_update forms and inverts it while the others
// update: the chain of pivots (73 us a block) hides behind the update.  A block
// column of a 4144-block takes 95 + 20 us; with library products, the copies
// between them and the inverse in its turn it took 181 (8.0 -> 5.1 ms in all).
constexpr int BGJ_B = 96;

typedef double d4_t __attribute__((ext_vector_type(4)));

__device__ inline double read_lane(double v, int lane) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), lane);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), lane);
  return __hiloint2double(hi, lo);
}

// One wave inverts the 32 x 32 block A (LDS) in place: Gauss-Jordan with the
// block in registers (lane = row + 32 half, 16 columns each), no workgroup
// barrier.  A diagonal pivot is taken unless an unused row holds an entry ten
// times larger, then the largest.
constexpr int SB = 32;
__device__ inline void wave_inverse(double *A, int lda, double *prow, int *pk, int lane,
                                    int32_t *__restrict__ flag) {
  const int r = lane & 31, h = lane >> 5;
  double a[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) a[j] = A[r * lda + 16 * h + j];
  bool used = false;
  uint32_t mask = 0;
  int kof = 0;
#pragma unroll
  for (int k = 0; k < SB; ++k) {
    const int hk = k >> 4, kk = k & 15;
    const double f = __shfl(a[kk], r + 32 * hk, 64);  // column k on both halves
    const double dk = read_lane(f, k);
    int p = k;
    if (__ballot(!used && !(fabs(f) <= 10.0 * fabs(dk))) || (mask >> k & 1u) || !(dk != 0.0)) {
      double best = used ? -1.0 : fabs(f);
      int bi = r;
      for (int off = 16; off > 0; off >>= 1) {
        const double ob = __shfl_xor(best, off, 32);
        const int oi = __shfl_xor(bi, off, 32);
        if (ob > best || (ob == best && oi < bi)) {
          best = ob;
          bi = oi;
        }
      }
      p = __builtin_amdgcn_readfirstlane(bi);
    }
    const double piv = read_lane(f, p);
    if (!(fabs(piv) > 0.0) && lane == 0) *flag = 1;
    const double inv = 1.0 / piv;
    if (r == p) {
#pragma unroll
      for (int j = 0; j < 16; ++j) prow[16 * h + j] = (j == kk && h == hk) ? inv : a[j] * inv;
      used = true;
      kof = k;
    }
    mask |= 1u << p;
    if (lane == 0) pk[k] = p;
    if (h == hk) a[kk] = 0.0;
    wave_order();
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const double pr = prow[16 * h + j];
      a[j] = r == p ? pr : fma(-f, pr, a[j]);
    }
    wave_order();
  }
  // A^-1[k][pk[c]] = S[pk[k]][c]
#pragma unroll
  for (int j = 0; j < 16; ++j) A[kof * lda + pk[16 * h + j]] = a[j];
}

// One workgroup inverts a kb x kb (kb <= BGJ_B = 96) block in LDS by block
// Gauss-Jordan with 32 x 32 diagonal blocks (wave_inverse) and FP64 MFMA tiles
// for their updates.  The chain of pivots is what bounds it: a step of one wave
// in registers costs a sixth of a step of the whole workgroup with its four
// barriers (a 96-block took 200 us, now 60).  The block is src (leading
// dimension ld); P [96 x 96] is padded by the identity.
constexpr int GJ_T = 512;
struct GJBlock {
  double A[BGJ_B][BGJ_B + 1];
  double prow[SB];
  int pk[SB];
};
__device__ __forceinline__ void invert_block(GJBlock &S, const double *__restrict__ src, int64_t ld, int kb,
                                             double *__restrict__ Pout, int32_t *__restrict__ flag) {
  static_assert(BGJ_B == 96 && SB == 32 && GJ_T == 512, "4 x 4 tiles outside a 32-block, two for each of 8 waves");
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, li = lane & 15, lk = lane >> 4;
#pragma unroll
  for (int u = 0; u < BGJ_B * BGJ_B / GJ_T; ++u) {
    const int e = tid + u * GJ_T, i = e % BGJ_B, j = e / BGJ_B;
    S.A[i][j] = i < kb && j < kb ? src[i + (int64_t)j * ld] : (i == j ? 1.0 : 0.0);
  }
  __syncthreads();
  for (int s0 = 0; s0 < kb; s0 += SB) {
    if (wave == 0) wave_inverse(&S.A[s0][s0], BGJ_B + 1, S.prow, S.pk, lane, flag);
    __syncthreads();
    // tile t = 0..3 of the 16-wide tiles outside the block
    auto outside = [&](int t) { return 16 * t + (16 * t >= s0 ? SB : 0); };
    {  // A[s][:] <- P A[s][:]
      const int i0 = s0 + 16 * (wave & 1), j0 = outside(wave >> 1);
      d4_t acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int k = 0; k < SB; k += 4)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(S.A[i0 + li][s0 + k + lk], S.A[s0 + k + lk][j0 + li], acc, 0, 0, 0);
      __syncthreads();
#pragma unroll
      for (int q = 0; q < 4; ++q) S.A[i0 + lk + 4 * q][j0 + li] = acc[q];
    }
    __syncthreads();
#pragma unroll
    for (int h = 0; h < 2; ++h) {  // A[i][j] -= A[i][s] A[s][j] outside the block
      const int i0 = outside(wave & 3), j0 = outside((wave >> 2) + 2 * h);
      d4_t acc;
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[q] = S.A[i0 + lk + 4 * q][j0 + li];
#pragma unroll
      for (int k = 0; k < SB; k += 4)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(-S.A[i0 + li][s0 + k + lk], S.A[s0 + k + lk][j0 + li], acc, 0, 0,
                                                   0);
#pragma unroll
      for (int q = 0; q < 4; ++q) S.A[i0 + lk + 4 * q][j0 + li] = acc[q];
    }
    // A[i][s] <- -A[i][s] P, written once every wave has read A[i][s]
    d4_t col = {0.0, 0.0, 0.0, 0.0};
    const int ci = outside(wave & 3), cj = s0 + 16 * (wave >> 2);
#pragma unroll
    for (int k = 0; k < SB; k += 4)
      col = __builtin_amdgcn_mfma_f64_16x16x4f64(-S.A[ci + li][s0 + k + lk], S.A[s0 + k + lk][cj + li], col, 0, 0, 0);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; ++q) S.A[ci + lk + 4 * q][cj + li] = col[q];
    __syncthreads();
  }
  for (int e = tid; e < BGJ_B * BGJ_B; e += GJ_T) Pout[e] = S.A[e % BGJ_B][e / BGJ_B];
}

__global__ __launch_bounds__(GJ_T) void k_block_inv(int64_t m, int kb, const double *__restrict__ M,
                                                    double *__restrict__ P, int32_t *__restrict__ flag) {
  __shared__ GJBlock S;
  invert_block(S, M, m, kb, P, flag);
}

// C = -M[:,K], R = P M[K,:] with R[:,K] = P (both [k][m], zero for k >= kb); 32
// columns (and rows of C) per workgroup.  The workgroups of the next block's
// columns also form that block after the update, D (kd x kd in [96 x 96]).
constexpr int GJ_PC = 32;
__global__ __launch_bounds__(GJ_T) void k_gj_panel(int64_t m, int64_t k0, int kb, int kd, const double *__restrict__ M,
                                                  const double *__restrict__ P, double *__restrict__ C,
                                                  double *__restrict__ R, double *__restrict__ D) {
  __shared__ double S[GJ_PC][BGJ_B + 1], Q[BGJ_B][BGJ_B + 1];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, li = lane & 15, lk = lane >> 4;
  const int64_t j0 = (int64_t)blockIdx.x * GJ_PC;
  const int64_t k1 = k0 + BGJ_B;
#pragma unroll
  for (int u = 0; u < BGJ_B * BGJ_B / GJ_T; ++u) {
    const int e = tid + u * GJ_T;
    Q[e / BGJ_B][e % BGJ_B] = P[e];
  }
#pragma unroll
  for (int u = 0; u < GJ_PC * BGJ_B / GJ_T; ++u) {
    const int e = tid + u * GJ_T, k = e % BGJ_B, j = e / BGJ_B;
    S[j][k] = k < kb && j0 + j < m ? M[k0 + k + (j0 + j) * m] : 0.0;
  }
#pragma unroll
  for (int u = 0; u < GJ_PC * BGJ_B / GJ_T; ++u) {
    const int e = tid + u * GJ_T, k = e / GJ_PC;
    const int64_t i = j0 + e % GJ_PC;
    if (i < m) C[k * m + i] = k < kb ? -M[i + (k0 + k) * m] : 0.0;
  }
  double ck[BGJ_B * BGJ_B / GJ_T];
  const bool next = j0 >= k1 && j0 < k1 + kd;
  if (next) {
#pragma unroll
    for (int u = 0; u < BGJ_B * BGJ_B / GJ_T; ++u) {
      const int e = tid + u * GJ_T, i = e % BGJ_B, k = e / BGJ_B;
      ck[u] = i < kd && k < kb ? -M[k1 + i + (k0 + k) * m] : 0.0;
    }
  }
  __syncthreads();
  d4_t rt[2] = {};
#pragma unroll
  for (int q = 0; q < 2; ++q) {  // 6 x 2 tiles
    const int t = wave + q * (GJ_T / 64), i0 = 16 * (t >> 1), c0 = 16 * (t & 1);
    if (t >= 12) break;
    d4_t acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 8
    for (int k = 0; k < BGJ_B; k += 4)
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(Q[k + lk][i0 + li], S[c0 + li][k + lk], acc, 0, 0, 0);
    rt[q] = acc;
    const int64_t j = j0 + c0 + li;
    if (j >= m) continue;
    const bool in = j >= k0 && j < k0 + kb;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int k = i0 + lk + 4 * r;
      R[k * m + j] = in ? Q[j - k0][k] : acc[r];
    }
  }
  if (!next) return;
  static_assert(BGJ_B % GJ_PC == 0, "a workgroup's columns lie inside or outside the next block");
  __syncthreads();
  // D = M[K1, j] + C[K1, :] R[:, j]: C's rows take P's place, R's columns M's
#pragma unroll
  for (int u = 0; u < BGJ_B * BGJ_B / GJ_T; ++u) Q[(tid + u * GJ_T) / BGJ_B][(tid + u * GJ_T) % BGJ_B] = ck[u];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int t = wave + q * (GJ_T / 64);
    if (t < 12) {
#pragma unroll
      for (int r = 0; r < 4; ++r) S[16 * (t & 1) + li][16 * (t >> 1) + lk + 4 * r] = rt[q][r];
    }
  }
  __syncthreads();
  for (int t = wave; t < 12; t += GJ_T / 64) {
    const int i0 = 16 * (t >> 1), c0 = 16 * (t & 1);
    const int64_t j = j0 + c0 + li;
    d4_t acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = i0 + lk + 4 * r;
      if (i < kd && j < m) acc[r] = M[k1 + i + j * m];
    }
#pragma unroll 8
    for (int k = 0; k < BGJ_B; k += 4)
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(Q[k + lk][i0 + li], S[c0 + li][k + lk], acc, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 4; ++r) D[i0 + lk + 4 * r + BGJ_B * (j - k1)] = acc[r];
  }
}

// M += C R outside [K,:], M[:,K] counted as zero and M[K,:] = R; one 48 x 48 tile
// per wave, straight from L2 (9 matrix instructions, 576 cycles, for 6 loads of
// 512 bytes); 4 x 2 waves of a workgroup share its rows and columns in L1.  At
// 4144 it takes 86 us, 95 with the inverse: 47 to move M in and out (275 MB, as
// measured with one k step) and the products, 43 at the matrix unit's rate,
// which overlap little (starting half of the waves with the products changed
// nothing).  Workgroup 0 inverts the next block (kd > 0).
constexpr int GJ_W = 48;
__global__ __launch_bounds__(GJ_T, 4) void k_gj_update(int64_t m, int64_t k0, int kb, int kd,
                                                       const double *__restrict__ C, const double *__restrict__ R,
                                                       const double *__restrict__ D, double *__restrict__ P,
                                                       int32_t *__restrict__ flag, double *__restrict__ M) {
  __shared__ GJBlock S;
  static_assert(BGJ_B % GJ_W == 0, "a wave's tile lies inside or outside K");
  if (blockIdx.x == 0) {
    __builtin_amdgcn_s_setprio(3);
    if (kd > 0) invert_block(S, D, BGJ_B, kd, P, flag);
    return;
  }
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int li = lane & 15, lk = lane >> 4;
  const unsigned ni = (unsigned)((m + 4 * GJ_W - 1) / (4 * GJ_W)), b = blockIdx.x - 1;
  const int64_t i0 = ((int64_t)(b % ni) * 4 + (wave & 3)) * GJ_W, j0 = ((int64_t)(b / ni) * 2 + (wave >> 2)) * GJ_W;
  if (i0 >= m || j0 >= m) return;
  if (i0 >= k0 && i0 < k0 + BGJ_B) {
    for (int e = lane; e < GJ_W * GJ_W; e += 64) {
      const int64_t i = i0 + e % GJ_W, j = j0 + e / GJ_W;
      if (i < m && j < m) M[i + j * m] = R[(i - k0) * m + j];
    }
    return;
  }
  // the tile transposed: D row (l / 16 + 4 r) is a column of M, its 16 lanes rows
  const bool skip = j0 >= k0 && j0 < k0 + BGJ_B;
  int64_t ii[3], jj[3];
#pragma unroll
  for (int t = 0; t < 3; ++t) {
    ii[t] = min(i0 + 16 * t + li, m - 1);
    jj[t] = min(j0 + 16 * t + li, m - 1);
  }
  d4_t acc[3][3];
#pragma unroll
  for (int t = 0; t < 3; ++t)
#pragma unroll
    for (int u = 0; u < 3; ++u)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        acc[t][u][r] = skip ? 0.0 : M[ii[u] + min(j0 + 16 * t + lk + 4 * r, m - 1) * m];
  // operands one step ahead; the barriers keep the compiler from moving the
  // loads down to their use
  const double *Ck = C + lk * m, *Rk = R + lk * m;
  double a[2][3], c[2][3];
  auto load = [&](int h) {
#pragma unroll
    for (int t = 0; t < 3; ++t) {
      a[h][t] = Rk[jj[t]];
      c[h][t] = Ck[ii[t]];
    }
    Ck += 4 * m;
    Rk += 4 * m;
    __builtin_amdgcn_sched_barrier(0);
  };
  auto multiply = [&](int h) {
#pragma unroll
    for (int t = 0; t < 3; ++t)
#pragma unroll
      for (int u = 0; u < 3; ++u)
        acc[t][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[h][t], c[h][u], acc[t][u], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  load(0);
  for (int k = 0; k < kb; k += 8) {  // C and R are zero in [kb, BGJ_B)
    load(1);
    multiply(0);
    if (k + 8 < kb) load(0);
    multiply(1);
  }
#pragma unroll
  for (int t = 0; t < 3; ++t) {
#pragma unroll
    for (int u = 0; u < 3; ++u)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t i = i0 + 16 * u + li, j = j0 + 16 * t + lk + 4 * r;
        if (i < m && j < m) M[i + j * m] = acc[t][u][r];
      }
  }
}

// b_i = deterministic values in [-1/2, 1/2) + 1 (the check's right-hand side)
__global__ void k_check_rhs(int64_t n, double *__restrict__ b) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    b[i] = 1.0 + (double)((uint64_t)(i * 2654435761ull) % 1000ull) / 1000.0 - 0.5;
}

// max that keeps a NaN (fmax would drop it): a NaN in the check fails it
__device__ inline double nan_max(double a, double b) { return (b > a || b != b) ? b : a; }

// out[0] = max |z - b|, out[1] = max |b| (one workgroup); NaN if z has one
__global__ __launch_bounds__(1024) void k_check_residual(int64_t n, const double *__restrict__ z,
                                                         const double *__restrict__ b, double *__restrict__ out) {
  __shared__ double r0[16], r1[16];
  double m0 = 0.0, m1 = 0.0;
  for (int64_t i = threadIdx.x; i < n; i += blockDim.x) {
    m0 = nan_max(m0, fabs(z[i] - b[i]));
    m1 = nan_max(m1, fabs(b[i]));
  }
  for (int off = 32; off > 0; off >>= 1) {
    m0 = nan_max(m0, __shfl_down(m0, off, 64));
    m1 = nan_max(m1, __shfl_down(m1, off, 64));
  }
  if ((threadIdx.x & 63) == 0) {
    r0[threadIdx.x >> 6] = m0;
    r1[threadIdx.x >> 6] = m1;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w) {
      m0 = nan_max(m0, r0[w]);
      m1 = nan_max(m1, r1[w]);
    }
    out[0] = m0;
    out[1] = m1;
  }
}

// coarse state: u by injection from the fine state, everything else zero
// coarse state: xc_u = R xf_u (the fine velocity at the coarse u nodes), the
// other coarse fields zero
__global__ void k_state_restrict(int64_t nc, int64_t nuc, const int64_t *__restrict__ rrow,
                                 const int32_t *__restrict__ rcol, const double *__restrict__ rval,
                                 const double *__restrict__ xf, double *__restrict__ xc) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < nc; i += (int64_t)gridDim.x * blockDim.x) {
    double s = 0.0;
    if (i < nuc)
      for (int64_t k = rrow[i]; k < rrow[i + 1]; ++k) s += rval[k] * xf[rcol[k]];
    xc[i] = s;
  }
}

__global__ void k_split(int64_t n1, const int64_t *__restrict__ rowptr, const int32_t *__restrict__ colind,
                        int64_t *__restrict__ split) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n1; i += (int64_t)gridDim.x * blockDim.x) {
    int64_t lo = rowptr[i], hi = rowptr[i + 1];
    while (lo < hi) {
      const int64_t mid = (lo + hi) >> 1;
      if (colind[mid] < n1) lo = mid + 1;
      else hi = mid;
    }
    split[i] = lo;
  }
}

// ---------------------------------------------------------------- Schur blocks
// x_p = Sp_c r_p and x_phi = Sphi_c r_phi for every cell (thread per (cell, row)).
template <class T>
__global__ void k_schur(int ncells, const int32_t *__restrict__ pfirst, const int32_t *__restrict__ phifirst,
                        const double *__restrict__ Sp, const double *__restrict__ Sphi, const T *__restrict__ r,
                        T *__restrict__ x) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t >= (int64_t)ncells * 12) return;
  const int c = (int)(t / 12), k = (int)(t % 12);
  if (k < 4) {
    const int32_t p0 = pfirst[c];
    const double *S = Sp + (int64_t)c * 16 + 4 * k;
    double acc = 0.0;
    for (int l = 0; l < 4; ++l) acc += S[l] * (double)r[p0 + l];
    x[p0 + k] = (T)acc;
  } else {
    const int kk = k - 4;
    const int32_t f0 = phifirst[c];
    const double *S = Sphi + (int64_t)c * 64 + 8 * kk;
    double acc = 0.0;
    for (int l = 0; l < 8; ++l) acc += S[l] * (double)r[f0 + l];
    x[f0 + kk] = (T)acc;
  }
}

// ---------------------------------------------------------------- patches

// Thread grid TR x TC, register tile RI x RJ: matrices of up to N = TR RI + 1
// rows, the last row and column in LDS.
template <int TR_, int TC_, int RI_, int RJ_>
struct GJTile {
  static constexpr int TR = TR_, TC = TC_, RI = RI_, RJ = RJ_;
  static constexpr int T = TR * TC;       // threads per patch
  static constexpr int NL = TR * RI;      // the row / column held in LDS
  static constexpr int NMAX = NL + 1;
  static_assert(TR == 16 && TC * RJ == TR * RI && TC % TR == 0 && TC <= 64, "square register part, row blocks of 16 lanes");
};
using GJLarge = GJTile<16, 32, 14, 7>;    // up to 225 rows, 512 threads
using GJSmall = GJTile<16, 16, 8, 8>;     // up to 129 rows, 256 threads
constexpr int PATCH_MAX = GJLarge::NMAX;  // unknowns of the largest vertex star (all dofs)


// Static condensation of the vertex patches.  The 12 interior RT1 dofs of a
// cell couple to the cell's own dofs only, and the star of a vertex that holds
// one of a cell's other [u,j] dofs holds the whole cell (cells of which that is
// not so are left out, see build_condensation).  With D the 12 x 12
// interior block of cell c (the RT1 mass plus zeta_j div-div: symmetric
// positive definite for zeta_j >= 0), eliminating the interior dofs of every
// patch therefore gives exactly
//   rt = r - sum_c A_bi D^-1 r_i                (one vector for all patches)
//   yb = sum_P R_P^T S_P^-1 R_P rt,             S = A_bb - sum_c A_bi D^-1 A_ib
//   yi = N D^-1 r_i - D^-1 A_ib yb              (N: patches that hold the cell)
// for y = sum_P R_P^T A_P^-1 R_P r.  An interior star has 225 dofs, 129 of
// them not interior to a cell: 129^2 / 225^2 = 33 % of the patch entries are
// left, and 2 x 105 x 12 + 12^2 coupling entries per cell.  One FP32 application
// at 64 x 64 x 8 (33,800 stars) went from 1.21 ms (6.5 GB of 225 x 225 inverses)
// to 0.56 ms (2.5 GB in all), FP64 on 13 x 11 x 5 cells from 67 to 39 us.
constexpr int NI = 12, NB = NU + 24;   // interior dofs of a cell; its other [u,j] dofs, local index l
__device__ inline int bdof_local(int l) { return l < NU ? l : l + (OFF_J - NU); }
// row of F: the three components of a node side by side, as their dofs are
__device__ inline int frow(int l) { return l < NU ? (l % 27) * 3 + l / 27 : l; }

// Per cell: Gauss-Jordan with partial pivoting on [D | I | A_ib] gives D^-1 and
// E = D^-1 A_ib (stored [l][i]); F = A_bi D^-1 ([frow(l)][i]) and G = N D^-1.  E is
// eliminated, not multiplied by the explicit D^-1: the grad-div part of D makes
// A_bi (D^-1 A_ib) lose 1.5 digits of the condensed matrix, the elimination
// none.  E and A_bi in FP64 for the patch matrices (k_patch_build), E, F, G in
// the precision of the smoother.  Entries are found through the rank map.  One
// workgroup per cell, a thread per column; 23 KB of values are read and 31 to
// 42 KB written per cell, small beside the patches (0.97 ms at 32,768 cells).
constexpr int CND_T = 192, CND_W = 2 * NI + NB;  // threads; columns of [D | I | A_ib]
template <class TE>
__global__ __launch_bounds__(CND_T) void k_condense(int ncells, const int32_t *__restrict__ dofs,
                                                    const int32_t *__restrict__ ifirst,
                                                    const int32_t *__restrict__ npat, int dups,
                                                    const int64_t *__restrict__ rowptr,
                                                    const uint16_t *__restrict__ rank, const double *__restrict__ val,
                                                    double *__restrict__ E64, double *__restrict__ B64,
                                                    TE *__restrict__ E32, TE *__restrict__ F, TE *__restrict__ G,
                                                    int32_t *__restrict__ flag) {
  __shared__ double M[NI][CND_W + 1];
  __shared__ double Abi[NB][NI + 1];
  __shared__ double colk[NI];
  __shared__ int32_t g[NB];
  __shared__ int64_t rp[NB];
  __shared__ int piv;
  const int c = blockIdx.x, t = threadIdx.x;
  const int64_t oc = (int64_t)c * NB * NI;
  const int32_t f0 = ifirst[c];
  if (f0 < 0) {  // not condensed: no couplings (uniform over the block)
    for (int e = t; e < NB * NI; e += CND_T) {
      E64[oc + e] = B64[oc + e] = 0.0;
      if (E32) E32[oc + e] = (TE)0;
      F[oc + e] = (TE)0;
    }
    for (int e = t; e < NI * NI; e += CND_T) G[(int64_t)c * NI * NI + e] = (TE)0;
    return;
  }
  const uint16_t *rk = rank + (int64_t)c * NENT;
  if (t < NB) {
    const int32_t *cd = dofs + (int64_t)c * NDOF;
    int32_t id = cd[bdof_local(t)];
    if (dups && id >= 0)  // a dof listed twice in the cell counts once
      for (int l = 0; l < t; ++l)
        if (cd[bdof_local(l)] == id) id = -1;
    g[t] = id;
    rp[t] = id >= 0 ? rowptr[id] : 0;
  }
  __syncthreads();
  const int r0 = 24;  // RT1 row of the first interior dof
  for (int e = t; e < NI * NI; e += CND_T) {
    const int i = e / NI, k = e % NI;
    M[i][k] = val[rowptr[f0 + i] + rk[E_J + (r0 + i) * ROWS_J_LEN + NU + r0 + k]];
    M[i][NI + k] = i == k ? 1.0 : 0.0;
  }
  for (int e = t; e < NI * NB; e += CND_T) {
    const int i = e / NB, l = e % NB;
    M[i][2 * NI + l] = g[l] >= 0 ? val[rowptr[f0 + i] + rk[E_J + (r0 + i) * ROWS_J_LEN + l]] : 0.0;
    const int lb = e / NI, k = e % NI;
    const int row = lb < NU ? lb * ROWS_U_LEN + OFF_J + r0 : E_J + (lb - NU) * ROWS_J_LEN + NU + r0;
    Abi[lb][k] = g[lb] >= 0 ? val[rp[lb] + rk[row + k]] : 0.0;
  }
  __syncthreads();
  for (int k = 0; k < NI; ++k) {
    if (t < 16) {
      double best = t >= k && t < NI ? fabs(M[t][k]) : -1.0;
      int bi = t;
      for (int off = 8; off > 0; off >>= 1) {
        const double ob = __shfl_xor(best, off, 16);
        const int oi = __shfl_xor(bi, off, 16);
        if (ob > best || (ob == best && oi < bi)) {
          best = ob;
          bi = oi;
        }
      }
      if (t == 0) {
        piv = bi;
        if (!(best > 0.0)) *flag = c + 1;
      }
    }
    __syncthreads();
    const int p = piv;
    const double inv = 1.0 / M[p][k];
    if (t < NI) colk[t] = t == p ? M[k][k] : M[t][k];
    __syncthreads();
    if (t < CND_W) {  // column t: rows k and p exchanged, then eliminated
      const double a = M[k][t], rkk = M[p][t] * inv;
      if (p != k) M[p][t] = a;
#pragma unroll
      for (int i = 0; i < NI; ++i)
        if (i != k) M[i][t] -= colk[i] * rkk;
      M[k][t] = rkk;
    }
    __syncthreads();
  }
  for (int e = t; e < NB * NI; e += CND_T) {
    const int l = e / NI, i = e % NI;
    double sf = 0.0;
#pragma unroll
    for (int k = 0; k < NI; ++k) sf += Abi[l][k] * M[k][NI + i];
    const double ev = M[i][2 * NI + l];
    E64[oc + e] = ev;
    B64[oc + e] = Abi[l][i];
    if (E32) E32[oc + e] = (TE)ev;
    F[oc + frow(l) * NI + i] = (TE)sf;
  }
  const double nc = (double)npat[c];
  for (int e = t; e < NI * NI; e += CND_T) G[(int64_t)c * NI * NI + e] = (TE)(nc * M[e / NI][NI + e % NI]);
}

// Condensed patch matrices S_P (column-major, identity on the padding): the
// entries of A between the patch's dofs, minus A_bi E of every condensed cell
// around the vertex, cell by cell in a fixed order.  Two dofs of a patch couple
// only through cells that hold both, and those are around the vertex, so the
// entries are taken cell by cell through the rank map, without a search (10 K
// entries per patch, where scanning the CSR rows visits 32 K columns).  SCAN:
// the skeleton term, or an unusual dof or vertex table, couples dofs of a patch
// beyond those cells; the rows are scanned then, each by a wave whose lanes
// binary-search the columns among the sorted ids.  One 1024-thread workgroup
// per patch.  LDSM: the matrix is built in LDS (129 x 129 FP64, 133 of the CU's
// 160 KB) and written once, coalesced; larger patches are built in place in A.  5.1 ms for 33,800 patches; with the rows scanned and the
// cells taken one after another, each waiting for its loads, 7.5 ms (the full
// 225 x 225 matrices, scattered into cleared memory, 18 ms).
template <bool LDSM, bool SCAN>
__global__ __launch_bounds__(1024) void k_patch_build(int PS, const int32_t *__restrict__ psize,
                                                      const int32_t *__restrict__ pidx,
                                                      const int32_t *__restrict__ pcptr,
                                                      const int32_t *__restrict__ pcell,
                                                      const int64_t *__restrict__ rowptr,
                                                      const int32_t *__restrict__ colind,
                                                      const uint16_t *__restrict__ rank,
                                                      const double *__restrict__ val,
                                                      const int32_t *__restrict__ dofs,
                                                      const int32_t *__restrict__ ifirst, int dups,
                                                      const double *__restrict__ E64,
                                                      const double *__restrict__ B64, double *__restrict__ A) {
  constexpr int NS = LDSM ? GJSmall::NMAX : 1;
  constexpr int NUJ = NB + NI;  // [u,j] dofs of a cell
  constexpr int CB = 8;         // cells in work together: 128 threads each
  __shared__ double lmat[NS * NS];
  __shared__ double Bs[NB][NI + 1], Es[NB][NI + 1];
  __shared__ int32_t sid[256];
  __shared__ uint8_t lpos[CB][NUJ], lsel[CB][NUJ];
  __shared__ int m[CB];
  const int pch = blockIdx.x, t = threadIdx.x;
  const int sz = psize[pch];
  const int32_t *ids = pidx + (int64_t)pch * PS;
  double *Ap = A + (int64_t)pch * PS * PS;
  double *M = LDSM ? lmat : Ap;
  if (t < sz) sid[t] = ids[t];
  for (int e = t; e < PS * PS; e += 1024) M[e] = 0.0;
  __syncthreads();
  for (int k = sz + t; k < PS; k += 1024) M[k + k * PS] = 1.0;
  const int32_t first = sz > 0 ? sid[0] : 0, last = sz > 0 ? sid[sz - 1] : -1;
  auto find = [&](int32_t id) {
    if (id < first || id > last) return -1;
    int lo = 0, hi = sz;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (sid[mid] < id) lo = mid + 1;
      else hi = mid;
    }
    return lo < sz && sid[lo] == id ? lo : -1;
  };
  if (SCAN) {
    const int wave = t >> 6, lane = t & 63;
    for (int a = wave; a < sz; a += 16) {
      const int32_t row = sid[a];
      const int64_t e = rowptr[row + 1];
      for (int64_t p = rowptr[row] + lane; p < e; p += 64) {
        const int b = find(colind[p]);
        if (b >= 0) M[a + b * PS] = val[p];
      }
    }
  }
  const int q0 = pcptr[pch], q1 = pcptr[pch + 1];
  // the dofs of the cells qb .. qb + CB - 1 that the patch holds: local index
  // and position (the order of the lists changes no result)
  auto locate = [&](int qb) {
    __syncthreads();  // the previous lists are done with
    if (t < CB) m[t] = 0;
    __syncthreads();
    const int k = t >> 7, l = t & 127;
    if (qb + k < q1) {
      const int c = pcell[qb + k];
      if (l < (ifirst[c] >= 0 ? NB : NUJ)) {
        const int32_t *cd = dofs + (int64_t)c * NDOF;
        const int32_t id = cd[bdof_local(l)];
        int pos = id >= 0 ? find(id) : -1;
        if (dups && pos >= 0)
          for (int o = 0; o < l; ++o)
            if (cd[bdof_local(o)] == id) pos = -1;
        if (pos >= 0) {
          const int at = atomicAdd(&m[k], 1);
          lpos[k][at] = (uint8_t)pos;
          lsel[k][at] = (uint8_t)l;
        }
      }
    }
    __syncthreads();
  };
  // entries of A, all cells at once (an entry of two cells is written twice,
  // with the same value)
  if (!SCAN)
    for (int qb = q0; qb < q1; qb += CB) {
      locate(qb);
      const int k = t >> 7, mk = m[k];
      if (qb + k < q1) {
        const uint16_t *rk = rank + (int64_t)pcell[qb + k] * NENT;
        for (int e = t & 127; e < mk * mk; e += 128) {
          const int ka = e / mk, kb = e - ka * mk;
          const int la = lsel[k][ka], lb = lsel[k][kb], pa = lpos[k][ka], pb = lpos[k][kb];
          // u rows hold [u p j], j rows [u j phi]
          const int ent = la < NU ? la * ROWS_U_LEN + (lb < NU ? lb : lb + NP) : E_J + (la - NU) * ROWS_J_LEN + lb;
          M[pa + pb * PS] = val[rowptr[sid[pa]] + rk[ent]];
        }
      }
    }
  // minus A_bi E, cell after cell; the next cell's couplings are loaded meanwhile
  for (int qb = q0; qb < q1; qb += CB) {
    if (SCAN || q1 - q0 > CB) locate(qb);
    else __syncthreads();  // the entries are in place, the lists still hold
    const int nk = min(CB, q1 - qb);
    constexpr int PF = (NB * NI + 1023) / 1024;
    double bn[PF], en[PF];
    auto fetch = [&](int k) {
      const int64_t oc = (int64_t)pcell[qb + k] * NB * NI;
      const int n = ifirst[pcell[qb + k]] >= 0 ? m[k] * NI : 0;
#pragma unroll
      for (int u = 0; u < PF; ++u) {
        const int e = t + 1024 * u;
        if (e < n) {
          const int64_t at = oc + lsel[k][e / NI] * NI + e % NI;
          bn[u] = B64[at];
          en[u] = E64[at];
        }
      }
    };
    fetch(0);
    for (int k = 0; k < nk; ++k) {
      const int mk = ifirst[pcell[qb + k]] >= 0 ? m[k] : 0;  // uniform
#pragma unroll
      for (int u = 0; u < PF; ++u) {
        const int e = t + 1024 * u;
        if (e < mk * NI) {
          Bs[e / NI][e % NI] = bn[u];
          Es[e / NI][e % NI] = en[u];
        }
      }
      __syncthreads();
      if (k + 1 < nk) fetch(k + 1);
      for (int e = t; e < mk * mk; e += 1024) {
        const int kb = e / mk, ka = e - kb * mk;
        double s = 0.0;
#pragma unroll
        for (int i = 0; i < NI; ++i) s += Bs[ka][i] * Es[kb][i];
        M[lpos[k][ka] + lpos[k][kb] * PS] -= s;
      }
      __syncthreads();
    }
  }
  if (LDSM) {
    __syncthreads();
    for (int e = t; e < PS * PS; e += 1024) Ap[e] = M[e];
  }
}

// rt_b = r_b - sum over the cells holding b of F_c[b] . r_i(c), FP64 sums;
// interior dofs of condensed cells are skipped (`map`: where the others go, or
// null).  Four lanes per dof share its (up to eight) cells, so the chain of
// dependent loads is at most two cells long: a level of 200 cells takes 5 us
// (one lane per dof: 11 us), 32,768 cells 60 us (F read once, 138 MB).
template <class T, class TE>
__global__ __launch_bounds__(256) void k_cond_rhs(int64_t n1, const int32_t *__restrict__ crow,
                                                  const int32_t *__restrict__ centry,
                                                  const uint8_t *__restrict__ elim,
                                                  const int32_t *__restrict__ ifirst, const TE *__restrict__ F,
                                                  const T *__restrict__ r, double *__restrict__ rt,
                                                  const int32_t *__restrict__ map) {
  const int64_t gid = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, i = gid >> 2;
  const int sub = (int)(gid & 3);
  double s = 0.0;
  const bool on = i < n1 && !elim[i];
  if (on) {
    const int32_t e = crow[i + 1];
    for (int32_t h = crow[i] + sub; h < e; h += 4) {
      const int32_t ce = centry[h];
      const int c = ce / NDOF, a = ce - c * NDOF;
      const int l = a < NU ? a : a - (OFF_J - NU);
      const int32_t f0 = ifirst[c];
      if (l >= NB || f0 < 0) continue;
      // a row of F is 12 TE, 16-byte aligned: three to six wide loads
      constexpr int V = 16 / (int)sizeof(TE);
      const uint4 *Fr = reinterpret_cast<const uint4 *>(F + ((int64_t)c * NB + frow(l)) * NI);
      union {
        uint4 raw[NI / V];
        TE v[NI];
      } f;
#pragma unroll
      for (int k = 0; k < NI / V; ++k) f.raw[k] = Fr[k];
#pragma unroll
      for (int k = 0; k < NI; ++k) s += (double)f.v[k] * (double)r[f0 + k];
    }
  }
  s += __shfl_xor(s, 1, 4);
  s += __shfl_xor(s, 2, 4);
  if (on && sub == 0) rt[map ? map[i] : i] = (double)r[i] - s;
}

// y_b (+)= w yb with yb = sum over the patches P holding b of part[P][b] (FP64,
// in patch order: no atomics, the same result in every run), and
// y_i (+)= w (G r_i - E yb) on the interior dofs of the condensed cells.  One
// wave per cell: it gathers yb of its dofs into LDS (the cell that is the first
// holder of a dof writes it), then takes the E rows l = s, s + 5, ... on lanes
// i + 12 s, coalesced.  One launch and no yb vector; the product sums are read
// 2.7 times (75 MB at 32,768 cells), E once: 94 us there, 9 us on 200 cells,
// where two launches (sums, then interiors) took 26 + 72 and 6 + 11 us.  Small
// levels are one chain of dependent loads: a dof at a time took 11 us, all
// eight products of two dofs 8, but 110 on the large one (registers).
constexpr int CG_CELLS = 4;
template <class T, class TE>
__global__ __launch_bounds__(64 * CG_CELLS) void k_cond_gather(
    int ncells, int64_t n1, const int32_t *__restrict__ dofs, const int32_t *__restrict__ ifirst,
    const int32_t *__restrict__ crow, const int32_t *__restrict__ centry, const int32_t *__restrict__ dptr,
    const int32_t *__restrict__ dent, const double *__restrict__ part, const TE *__restrict__ E,
    const TE *__restrict__ G, const T *__restrict__ r, double w, T *__restrict__ y, int accumulate) {
  __shared__ double yb[CG_CELLS][NB + 1];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int c = blockIdx.x * CG_CELLS + wave;
  const int32_t f0 = c < ncells ? ifirst[c] : -1;
  const int i = lane % NI, sl = lane / NI;
  TE ev[NB / 5];  // this lane's E entries, in flight during the gather
  if (f0 >= 0 && sl < 5) {
    const TE *Ec = E + ((int64_t)c * NB + sl) * NI + i;
#pragma unroll
    for (int k = 0; k < NB / 5; ++k) ev[k] = Ec[5 * k * NI];
  }
  if (c < ncells) {
    const int32_t *cd = dofs + (int64_t)c * NDOF;
    const int nl = f0 < 0 ? NB + NI : NB;
    for (int k0 = lane; k0 < nl; k0 += 128) {
      // two dofs a lane and four products of each (only the cell's central node
      // lies in more stars) requested together: one chain of dependent loads
      int32_t id[2], b[2], n[2], h[2], at[2][4];
      double pv[2][4];
      int loc[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int k = min(k0 + 64 * u, nl - 1);
        const int l = k < NU ? (k % 3) * 27 + k / 3 : k;  // node by node: neighbouring lanes read neighbouring sums
        loc[u] = l;
        const int32_t g = cd[bdof_local(l)];
        id[u] = k0 + 64 * u < nl && g >= 0 && g < n1 ? g : -1;
      }
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        b[u] = n[u] = 0;
        h[u] = -1;
        if (id[u] >= 0) {
          b[u] = dptr[id[u]];
          n[u] = dptr[id[u] + 1] - b[u];
          h[u] = crow[id[u]];
        }
      }
#pragma unroll
      for (int u = 0; u < 2; ++u) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (q < n[u]) at[u][q] = dent[b[u] + q];
        if (h[u] >= 0) h[u] = centry[h[u]];
      }
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int q = 0; q < 4; ++q) pv[u][q] = q < n[u] ? part[at[u][q]] : 0.0;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        if (k0 + 64 * u >= nl) continue;
        double s = 0.0;
#pragma unroll
        for (int q = 0; q < 4; ++q) s += pv[u][q];
        for (int32_t q = b[u] + 4, e = b[u] + n[u]; q < e; q += 4) {
          const double p0 = part[dent[q]], p1 = q + 1 < e ? part[dent[q + 1]] : 0.0;
          const double p2 = q + 2 < e ? part[dent[q + 2]] : 0.0, p3 = q + 3 < e ? part[dent[q + 3]] : 0.0;
          s = (((s + p0) + p1) + p2) + p3;
        }
        const int32_t g = id[u];
        if (g >= 0 && h[u] == c * NDOF + bdof_local(loc[u]))
          y[g] = accumulate ? (T)((double)y[g] + w * s) : (T)(w * s);
        if (loc[u] < NB) yb[wave][loc[u]] = s;
      }
    }
  }
  __syncthreads();
  if (f0 < 0) return;  // uniform over the wave
  double acc = 0.0;
  if (sl < 5) {
#pragma unroll
    for (int k = 0; k < NB / 5; ++k) acc -= (double)ev[k] * yb[wave][sl + 5 * k];
    const TE *Gc = G + ((int64_t)c * NI + i) * NI;
    for (int k = sl; k < NI; k += 5) acc += (double)Gc[k] * (double)r[f0 + k];
  }
  double s = acc;
#pragma unroll
  for (int k = 1; k < 5; ++k) s += __shfl(acc, (i + NI * k) & 63, 64);
  if (lane < NI) {
    T *yp = y + f0 + i;
    *yp = accumulate ? (T)((double)*yp + w * s) : (T)(w * s);
  }
}

// Row b of the condensed coarsest [u,j] block, dense and row-major: the CSR
// entries of the dofs that are not eliminated, minus A_bi E of the cells that
// hold the row's dof, in increasing cell order.  One workgroup per row; every
// entry of the row is written.
__global__ __launch_bounds__(256) void k_dense_cond(int64_t nb, const int32_t *__restrict__ bidx,
                                                    const int32_t *__restrict__ bmap,
                                                    const int64_t *__restrict__ rowptr,
                                                    const int64_t *__restrict__ split,
                                                    const int32_t *__restrict__ colind,
                                                    const double *__restrict__ val, const int32_t *__restrict__ crow,
                                                    const int32_t *__restrict__ centry,
                                                    const int32_t *__restrict__ dofs,
                                                    const int32_t *__restrict__ ifirst, int dups,
                                                    const double *__restrict__ E64, const double *__restrict__ B64,
                                                    double *__restrict__ D) {
  const int t = threadIdx.x;
  const int32_t i = bidx[blockIdx.x];
  double *row = D + (int64_t)blockIdx.x * nb;
  for (int64_t e = t; e < nb; e += 256) row[e] = 0.0;
  __syncthreads();
  for (int64_t p = rowptr[i] + t; p < split[i]; p += 256) {
    const int32_t b = bmap[colind[p]];
    if (b >= 0) row[b] = val[p];
  }
  for (int32_t h = crow[i]; h < crow[i + 1]; ++h) {
    const int32_t ce = centry[h], c = ce / NDOF, a = ce - c * NDOF;
    const int l = a < NU ? a : a - (OFF_J - NU);
    if (l >= NB || ifirst[c] < 0) continue;  // uniform
    __syncthreads();
    if (t < NB) {
      const int32_t *cd = dofs + (int64_t)c * NDOF;
      int32_t id = cd[bdof_local(t)];
      if (dups && id >= 0)  // a dof listed twice in the cell has its couplings at the first place
        for (int k = 0; k < t; ++k)
          if (cd[bdof_local(k)] == id) id = -1;
      if (id >= 0) {
        const double *B = B64 + ((int64_t)c * NB + l) * NI, *E = E64 + ((int64_t)c * NB + t) * NI;
        double s = 0.0;
#pragma unroll
        for (int k = 0; k < NI; ++k) s += B[k] * E[k];
        row[bmap[id]] -= s;
      }
    }
  }
}

// y = A^-1 x with the explicit inverse stored row-major: one workgroup per row,
// coalesced 8-byte loads, eight in flight per lane, FP64 accumulation.  The
// result goes to yd[row], or to yd[bidx[row]] and y[bidx[row]].  (One wave per
// row left 137 MB, 4,144 rows, at 3.4 TB/s: 40 us.)
template <class T>
__global__ __launch_bounds__(TB) void k_dense_rowdot(int64_t m, const double *__restrict__ Ainv,
                                                      const double *__restrict__ x, const int32_t *__restrict__ bidx,
                                                      double *__restrict__ yd, T *__restrict__ y) {
  const int64_t row = blockIdx.x;
  const double *a = Ainv + row * m;
  double s[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  int64_t j = threadIdx.x;
  for (; j + 7 * TB < m; j += 8 * TB) {
#pragma unroll
    for (int u = 0; u < 8; ++u) s[u] += a[j + u * TB] * x[j + u * TB];
  }
#pragma unroll
  for (int u = 0; u < 8; ++u)
    if (j + u * TB < m) s[u] += a[j + u * TB] * x[j + u * TB];
  const double v = block_sum(((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7])));
  if (threadIdx.x == 0) {
    const int64_t i = bidx ? bidx[row] : row;
    yd[i] = v;
    if (y) y[i] = (T)v;
  }
}

// interior dofs of the condensed cells, y_i = G r_i - E yb: one wave per cell,
// lane = i + 12 s as in k_cond_gather
template <class T>
__global__ __launch_bounds__(256) void k_cond_inner(int ncells, const int32_t *__restrict__ dofs,
                                                    const int32_t *__restrict__ ifirst, const double *__restrict__ E,
                                                    const double *__restrict__ G, const T *__restrict__ r,
                                                    const double *__restrict__ yb, T *__restrict__ y) {
  const int c = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (c >= ncells) return;  // uniform over the wave
  const int32_t f0 = ifirst[c];
  if (f0 < 0) return;
  const int i = lane % NI, sl = lane / NI;
  double acc = 0.0;
  if (sl < 5) {
    const double *Ec = E + ((int64_t)c * NB + sl) * NI + i;
    const int32_t *cd = dofs + (int64_t)c * NDOF;
#pragma unroll
    for (int k = 0; k < NB / 5; ++k) {
      const int32_t id = cd[bdof_local(sl + 5 * k)];
      acc -= Ec[5 * k * NI] * (id >= 0 ? yb[id] : 0.0);
    }
    const double *Gc = G + ((int64_t)c * NI + i) * NI;
    for (int k = sl; k < NI; k += 5) acc += Gc[k] * (double)r[f0 + k];
  }
  double s = acc;
#pragma unroll
  for (int k = 1; k < 5; ++k) s += __shfl(acc, (i + NI * k) & 63, 64);
  if (lane < NI) y[f0 + i] = (T)s;
}

// ---------------------------------------------------------------------------
// Batched inversion of the vertex patches: in-place Gauss-Jordan elimination,
// one workgroup per patch, the matrix held in registers.  The condensed
// matrix of a vertex star has at most 129 = 128 + 1 unknowns (27 Q2 nodes x 3
// components + 48 RT1 face dofs; GJSmall); stars of unusual valence, or whose
// cells cannot be condensed, have up to 225 (GJLarge).  Thread (tr, tc) =
// (t mod 16, t / 16) holds an RI x RJ tile: RI rows (one of every block of 16
// rows) and RJ columns (one of every block of TC columns); the last row and
// column live in LDS.  GJSmall's FP64 tile is 64 values (128 VGPRs) on 256
// threads, so two to three workgroups share a CU and hide each other's
// barriers (one per step): 10.6 ms for 33,800 patches (12.1 with the diagonal
// read in a step before the matrix, a millisecond more with three barriers per
// step), where the full stars took 61 ms on GJLarge's 98 values on 512 threads,
// one workgroup per CU.
//
// Elimination step k, with the pivot column saved as f and zeroed and the
// pivot row p saved as r = a_p,: / a_pk (r_k = 1 / a_pk) and zeroed, updates
// every entry as
//   a_ij <- a_ij - f'_i r_j,   f'_i = f_i (i != p), f'_p = -1,
// the in-place Gauss-Jordan step of [A | I] with column p of the right-hand
// block stored in column k.
//
// k_patch_gjd pivots on the diagonal (p = k).  The tile then rotates one row
// after every 16 steps and one column after every TC, so that the pivot row
// and column always sit in register row 0 and column 0 and every register
// index is a compile-time constant.  It accepts a diagonal pivot only if
// |a_kk| >= tau max_{i > k} |a_ik| (threshold pivoting) and otherwise
// flags the patch.  The rows are first scaled by powers of two to a diagonal in
// [1, 2) (exactly; the columns of the inverse take the scale back), so that the
// penalty rows of thin-wall faces do not fail the test against rows of another
// magnitude; a row whose diagonal is too small for that is scaled by its
// largest entry (gj_row_scale) and fails.  Flagged patches are inverted again by k_patch_gj, with
// partial pivoting (the unused row of largest |a_ik|, lowest row on ties).
// Rows are not swapped there: A^-1[k][j] = S[p_k][q_j] with q = p^-1, and the
// smoother applies it without un-permuting: z = S x' with x'_c = x_{p_c}, and
// z_r is the patch product of local dof q_r (p is the identity after
// k_patch_gjd).  Patches smaller than the padded size are padded with
// identity rows and columns, whose pivots are their own rows.
template <class T>
__device__ inline T from_dbl(double v) { return (T)v; }
template <>
__device__ inline __hip_bfloat16 from_dbl<__hip_bfloat16>(double v) { return __float2bfloat16((float)v); }
template <>
__device__ inline __half from_dbl<__half>(double v) { return __float2half((float)v); }

template <class G>
struct GJShared {
  double colbuf[G::NMAX], rowbuf[G::NMAX], Rl[G::NMAX], Cl[G::NL];
  double rs[G::NMAX];  // powers of two: the scale of row r (gj_row_scale)
  int used[G::NMAX];
  int16_t pk[G::NMAX];
  int p, bad;
  double piv;
  double wmax[G::T / 64];
};

// Scale of a row with diagonal |d| and largest |entry| m: d into [1, 2), or, if
// d is smaller than 2^-8 m, that.  A row scaled by a vanishing diagonal would
// pass the threshold test with entries of any size and carry them into the
// others.  (The u rows' Lorentz entries are up to 800 times the diagonal at
// Ha = 500, where both lines accept the same patches.)
__device__ inline double gj_row_scale(double d, double m) {
  const double v = fmax(d, ldexp(m, -8));
  return v > 0.0 && v < INFINITY ? ldexp(1.0, -max(-1000, min(1000, ilogb(v)))) : 1.0;
}

template <class G>
__device__ __forceinline__ void gj_load(double (&S)[G::RI][G::RJ], GJShared<G> &L, const double *__restrict__ Ap, int PS,
                                        int t, int tr, int tc) {
  double d = 0.0;
  if (t < G::NMAX) {
    d = t < PS ? fabs(Ap[(int64_t)t * PS + t]) : 1.0;
    L.rs[t] = 0.0;
    L.used[t] = 0;
  }
#pragma unroll
  for (int i = 0; i < G::RI; ++i)
#pragma unroll
    for (int j = 0; j < G::RJ; ++j) {
      const int r = tr + G::TR * i, c = tc + G::TC * j;
      S[i][j] = (r < PS && c < PS) ? Ap[(int64_t)c * PS + r] : (r == c ? 1.0 : 0.0);
    }
  const double rl = t < PS && G::NL < PS ? Ap[(int64_t)t * PS + G::NL] : (t == G::NL ? 1.0 : 0.0);
  const double cl = t < PS && t < G::NL && G::NL < PS ? Ap[(int64_t)G::NL * PS + t] : 0.0;
  __syncthreads();
  // largest |entry| of every row, as the bits of non-negative doubles, which
  // order as integers
  auto row_max = [&](int r, double m) {
    atomicMax(reinterpret_cast<unsigned long long *>(&L.rs[r]), (unsigned long long)__double_as_longlong(m));
  };
#pragma unroll
  for (int i = 0; i < G::RI; ++i) {
    double m = 0.0;
#pragma unroll
    for (int j = 0; j < G::RJ; ++j) m = fmax(m, fabs(S[i][j]));
    m = fmax(m, __shfl_xor(m, 16, 64));
    m = fmax(m, __shfl_xor(m, 32, 64));
    if ((t & 63) < G::TR) row_max(tr + G::TR * i, m);
  }
  double m = fabs(rl);
  for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off, 64));
  if ((t & 63) == 0) row_max(G::NL, m);
  if (t < G::NL) row_max(t, fabs(cl));
  __syncthreads();
  if (t < G::NMAX) L.rs[t] = gj_row_scale(d, L.rs[t]);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < G::RI; ++i)
#pragma unroll
    for (int j = 0; j < G::RJ; ++j) S[i][j] *= L.rs[tr + G::TR * i];
  if (t < G::NMAX) L.Rl[t] = rl * L.rs[G::NL];
  if (t < G::NL) L.Cl[t] = cl * L.rs[t];
  if (t == 0) L.bad = 0;
}

// A^-1 from the inverse of the row-scaled matrix: column c times the scale of
// the row its slot takes (row_of: identity, or the pivot rows).
template <class G, class RowOf>
__device__ __forceinline__ void gj_unscale(double (&S)[G::RI][G::RJ], GJShared<G> &L, int t, int tc, RowOf row_of) {
  __syncthreads();
#pragma unroll
  for (int j = 0; j < G::RJ; ++j) {
    const double f = L.rs[row_of(tc + G::TC * j)];
#pragma unroll
    for (int i = 0; i < G::RI; ++i) S[i][j] *= f;
  }
  if (t < G::NMAX) L.Rl[t] *= L.rs[row_of(t)];
  if (t < G::NL) L.Cl[t] *= L.rs[row_of(G::NL)];
  __syncthreads();
}

// FP16 inverses are stored scaled by a power of two per patch, so that the
// largest |entry| lies in [2^14, 2^15) (FP16 reaches 65504): pscale[pch] is the
// factor the product is multiplied by again.  Other types store unscaled.
template <class G, class OutT>
__device__ __forceinline__ double gj_scale(const double (&S)[G::RI][G::RJ], GJShared<G> &L, int PS, int t, int tr,
                                           int tc, float *__restrict__ pscale, int64_t pch) {
  if constexpr (!std::is_same<OutT, __half>::value) {
    return 1.0;
  } else {
    double m = 0.0;
#pragma unroll
    for (int i = 0; i < G::RI; ++i)
#pragma unroll
      for (int j = 0; j < G::RJ; ++j) {
        const int r = tr + G::TR * i, c = tc + G::TC * j;
        if (r < PS && c < PS) m = fmax(m, fabs(S[i][j]));
      }
    if (PS > G::NL) {
      if (t < PS) m = fmax(m, fabs(L.Rl[t]));
      if (t < G::NL) m = fmax(m, fabs(L.Cl[t]));
    }
    for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off, 64));
    if ((t & 63) == 0) L.wmax[t >> 6] = m;
    __syncthreads();
    m = L.wmax[0];
    for (int w = 1; w < G::T / 64; ++w) m = fmax(m, L.wmax[w]);
    const int e = m > 0.0 ? ilogb(m) : 0;
    if (t == 0) pscale[pch] = ldexpf(1.0f, e - 14);
    return ldexp(1.0, 14 - e);
  }
}

template <class G, class OutT>
__device__ __forceinline__ void gj_store(const double (&S)[G::RI][G::RJ], const GJShared<G> &L, OutT *__restrict__ Op,
                                         int PS, int ld, int t, int tr, int tc, double sc) {
#pragma unroll
  for (int i = 0; i < G::RI; ++i)
#pragma unroll
    for (int j = 0; j < G::RJ; ++j) {
      const int r = tr + G::TR * i, c = tc + G::TC * j;
      if (r < PS && c < PS) Op[(int64_t)c * ld + r] = from_dbl<OutT>(S[i][j] * sc);
    }
  if (PS > G::NL) {
    if (t < PS) Op[(int64_t)t * ld + G::NL] = from_dbl<OutT>(L.Rl[t] * sc);
    if (t < G::NL) Op[(int64_t)G::NL * ld + t] = from_dbl<OutT>(L.Cl[t] * sc);
  }
}

// Pivot search over (best |value|, lowest row) candidates of a lane group.
__device__ __forceinline__ void gj_argmax(double &best, double &bval, int &bi, int width) {
  for (int off = width >> 1; off > 0; off >>= 1) {
    const double ob = __shfl_xor(best, off, width), ov = __shfl_xor(bval, off, width);
    const int oi = __shfl_xor(bi, off, width);
    if (ob > best || (ob == best && oi < bi)) {
      best = ob;
      bval = ov;
      bi = oi;
    }
  }
}

// ---- diagonal pivots, rotating tile ----------------------------------------

// Step k = 16 rb + tq (column block cb = k / TC).  col and row hold the pivot
// column and row of the step in register order (slot tr + 16 i: the row of
// register row i; slot tc + TC j: the column of register column j; slot NL: row
// / column NL), unscaled.  The lanes that own the next step's column and row
// write them to the other buffer as soon as they have updated them, so a step
// has one barrier; the pivot's reciprocal is taken by every thread, and the
// threshold test of the next pivot is off that path.  rot_r / rot_c: the tile
// rotates after this step, so the next row / column block is the second one.
template <class G>
__device__ __forceinline__ void gjd_step(double (&S)[G::RI][G::RJ], GJShared<G> &L, const double *col,
                                         const double *row, double *ncol, double *nrow, int t, int tr, int tc, int rb,
                                         int cb, int tq, bool rot_r, bool rot_c) {
  const int k = G::TR * rb + tq, kc = k & (G::TC - 1);
  const double piv = col[tq];
  const double inv = piv != 0.0 ? 1.0 / piv : 0.0;
  // f'_i = f_i (pivot row: -1), r_j = a_kj / a_kk (pivot column: 1 / a_kk);
  // a_ij <- a_ij - f'_i r_j with the pivot row and column of a zeroed
  double rv[G::RJ];
#pragma unroll
  for (int j = 0; j < G::RJ; ++j) rv[j] = row[tc + G::TC * j] * inv;
  const bool mycol = tc == kc, myrow = tr == tq;
  if (mycol) rv[0] = inv;
#pragma unroll
  for (int i = 0; i < G::RI; ++i) {
    const double f = i == 0 && myrow ? -1.0 : col[tr + G::TR * i];
#pragma unroll
    for (int j = 0; j < G::RJ; ++j) {
      const double a = (j == 0 && mycol) || (i == 0 && myrow) ? 0.0 : S[i][j];
      S[i][j] = fma(-f, rv[j], a);
    }
  }
  const double fl = col[G::NL], rl = row[G::NL] * inv;
  if (t < G::NMAX) {  // row NL, physical column t
    int slot = G::NL;
    if (t < G::NL) {
      const int blk = t / G::TC - cb;
      slot = (t & (G::TC - 1)) + G::TC * (blk < 0 ? blk + G::RJ : blk);
    }
    L.Rl[t] = fma(-fl, t == k ? inv : row[slot] * inv, t == k ? 0.0 : L.Rl[t]);
  }
  if (t < G::NL) {  // column NL, physical row t
    const int blk = t / G::TR - rb;
    const int slot = (t & (G::TR - 1)) + G::TR * (blk < 0 ? blk + G::RI : blk);
    L.Cl[t] = fma(t == k ? 1.0 : -col[slot], rl, t == k ? 0.0 : L.Cl[t]);
  }
  // next step: its column (register column 0, or 1 before a rotation) and row
  const int kn = k + 1;
  if (kn < G::NL) {
    if (tc == (kn & (G::TC - 1))) {
#pragma unroll
      for (int i = 0; i < G::RI; ++i) {
        const int i1 = i + 1 < G::RI ? i + 1 : 0;  // every register index a compile-time constant
        ncol[tr + G::TR * i] = rot_r ? (rot_c ? S[i1][1] : S[i1][0]) : S[i][0];
      }
    }
    if (tr == (kn & (G::TR - 1))) {
#pragma unroll
      for (int j = 0; j < G::RJ; ++j) {
        const int j1 = j + 1 < G::RJ ? j + 1 : 0;
        nrow[tc + G::TC * j] = rot_r ? (rot_c ? S[1][j1] : S[1][j]) : S[0][j];
      }
    }
    // entries of row / column NL: the threads that have just updated them
    if (t == kn) {
      ncol[G::NL] = L.Rl[t];
      nrow[G::NL] = L.Cl[t];
    }
  }
  __syncthreads();
}

// The threshold test of step k's pivot on the column in `col`: 16 lanes.
// Register row i holds row block (i + rb) mod RI: unused rows are the blocks
// after rb, the rows of block rb after tq, and row NL.
template <class G>
__device__ __forceinline__ void gjd_test(GJShared<G> &L, const double *col, int tr, int rb, int tq, double tau) {
  double cmax = tr == 0 ? fabs(col[G::NL]) : 0.0;
#pragma unroll
  for (int i = 0; i < G::RI; ++i)
    if (i < G::RI - rb && (i > 0 || tr > tq)) cmax = fmax(cmax, fabs(col[tr + G::TR * i]));
  for (int off = G::TR >> 1; off > 0; off >>= 1) cmax = fmax(cmax, __shfl_xor(cmax, off, G::TR));
  const double dia = col[tq];
  if (tr == tq && (!(fabs(dia) >= tau * cmax) || dia == 0.0)) atomicCAS(&L.bad, 0, G::TR * rb + tq + 1);
}

template <class G, class OutT>
__global__ __launch_bounds__(G::T) void k_patch_gjd(int PS, int ld, double tau, const double *__restrict__ A,
                                                     OutT *__restrict__ out, int16_t *__restrict__ perm,
                                                     int32_t *__restrict__ status, float *__restrict__ pscale) {
  __shared__ GJShared<G> L;
  __shared__ double buf[2][2][G::NMAX];  // [parity][column, row]
  const int t = threadIdx.x, tr = t % G::TR, tc = t / G::TR;
  const int64_t pch = blockIdx.x;
  double S[G::RI][G::RJ];
  gj_load<G>(S, L, A + pch * PS * PS, PS, t, tr, tc);
  __syncthreads();
  if (tc == 0)
#pragma unroll
    for (int i = 0; i < G::RI; ++i) buf[0][0][tr + G::TR * i] = S[i][0];
  if (tr == 0)
#pragma unroll
    for (int j = 0; j < G::RJ; ++j) buf[0][1][tc + G::TC * j] = S[0][j];
  if (t == 0) {
    buf[0][0][G::NL] = L.Rl[0];
    buf[0][1][G::NL] = L.Cl[0];
  }
  __syncthreads();
  for (int cb = 0; cb < G::RJ; ++cb) {
    for (int h = 0; h < G::TC / G::TR; ++h) {
      const int rb = G::TC / G::TR * cb + h;
#pragma unroll 2
      for (int tq = 0; tq < G::TR; ++tq) {
        const int par = tq & 1;
        if (tc == G::TC - 1) gjd_test<G>(L, buf[par][0], tr, rb, tq, tau);  // one 16-lane group
        const bool lr = tq == G::TR - 1;
        gjd_step<G>(S, L, buf[par][0], buf[par][1], buf[par ^ 1][0], buf[par ^ 1][1], t, tr, tc, rb, cb, tq, lr,
                    lr && h == G::TC / G::TR - 1);
      }
      // next row block into register row 0
#pragma unroll
      for (int j = 0; j < G::RJ; ++j) {
        const double r0 = S[0][j];
#pragma unroll
        for (int i = 0; i + 1 < G::RI; ++i) S[i][j] = S[i + 1][j];
        S[G::RI - 1][j] = r0;
      }
    }
    // next column block into register column 0
#pragma unroll
    for (int i = 0; i < G::RI; ++i) {
      const double c0 = S[i][0];
#pragma unroll
      for (int j = 0; j + 1 < G::RJ; ++j) S[i][j] = S[i][j + 1];
      S[i][G::RJ - 1] = c0;
    }
  }
  // last step: row and column NL (LDS); the tile is back in place
  if (t < G::NL) L.colbuf[t] = L.Cl[t];
  if (t == 0) {
    const double v = L.Rl[G::NL];
    L.colbuf[G::NL] = v;
    L.piv = v;
    if (v == 0.0) atomicCAS(&L.bad, 0, G::NL + 1);
  }
  __syncthreads();
  {
    const double piv = L.piv;
    const double inv = piv != 0.0 ? 1.0 / piv : 0.0;
    if (t < G::NMAX) L.rowbuf[t] = t == G::NL ? inv : L.Rl[t] * inv;
    __syncthreads();
    if (t == 0) L.colbuf[G::NL] = -1.0;
    __syncthreads();
    double rv[G::RJ];
#pragma unroll
    for (int j = 0; j < G::RJ; ++j) rv[j] = L.rowbuf[tc + G::TC * j];
#pragma unroll
    for (int i = 0; i < G::RI; ++i) {
      const double f = L.colbuf[tr + G::TR * i];
#pragma unroll
      for (int j = 0; j < G::RJ; ++j) S[i][j] = fma(-f, rv[j], S[i][j]);
    }
    __syncthreads();
    if (t < G::NMAX) L.Rl[t] = L.rowbuf[t];
    if (t < G::NL) L.Cl[t] = -L.colbuf[t] * L.rowbuf[G::NL];
    __syncthreads();
  }
  gj_unscale<G>(S, L, t, tc, [](int c) { return c; });
  const double sc = gj_scale<G, OutT>(S, L, PS, t, tr, tc, pscale, pch);
  gj_store<G, OutT>(S, L, out + pch * PS * ld, PS, ld, t, tr, tc, sc);
  int16_t *pp = perm + pch * 2 * PS;
  if (t < PS) {
    pp[t] = (int16_t)t;
    pp[PS + t] = (int16_t)t;
  }
  if (t == 0) status[pch] = L.bad;
}

// ---- partial pivoting (patches the diagonal pivots rejected) ---------------

// One Gauss-Jordan step on column k with the row of largest |a_ik| among the
// unused rows.  Register column 0 is the column block in work (jk < RJ: columns
// tc + TC jk; the tile rotates one column after every block, so register
// column j holds column tc + TC ((j + jk) mod RJ)); jk = RJ is column NL (LDS).
template <class G>
__device__ __forceinline__ void gj_step(double (&S)[G::RI][G::RJ], GJShared<G> &L, int t, int tr, int tc, int jk,
                                        int tk) {
  const int k = tk + G::TC * jk;
  if (jk < G::RJ) {
    if (tc == tk) {  // 16 lanes of one wave
      double best = -1.0, bval = 0.0;
      int bi = 0x7fffffff;
#pragma unroll
      for (int i = 0; i < G::RI; ++i) {
        const int r = tr + G::TR * i;
        const double v = S[i][0];
        L.colbuf[r] = v;
        S[i][0] = 0.0;
        const double a = L.used[r] ? -1.0 : fabs(v);
        if (a > best) {
          best = a;
          bval = v;
          bi = r;
        }
      }
      if (tr == 0) {
        const double v = L.Rl[k];
        L.colbuf[G::NL] = v;
        const double a = L.used[G::NL] ? -1.0 : fabs(v);
        if (a > best) {
          best = a;
          bval = v;
          bi = G::NL;
        }
      }
      gj_argmax(best, bval, bi, G::TR);
      if (tr == 0) {
        L.p = bi;
        L.piv = bval;
        if (!(best > 0.0) && L.bad == 0) L.bad = k + 1;
      }
    }
  } else if (t < 64) {  // k = NL: the column lives in LDS
    double best = -1.0, bval = 0.0;
    int bi = 0x7fffffff;
    for (int r = t; r < G::NMAX; r += 64) {
      const double v = r < G::NL ? L.Cl[r] : L.Rl[G::NL];
      L.colbuf[r] = v;
      const double a = L.used[r] ? -1.0 : fabs(v);
      if (a > best) {
        best = a;
        bval = v;
        bi = r;
      }
    }
    gj_argmax(best, bval, bi, 64);
    if (t == 0) {
      L.p = bi;
      L.piv = bval;
      if (!(best > 0.0) && L.bad == 0) L.bad = k + 1;
    }
  }
  __syncthreads();
  const int p = __builtin_amdgcn_readfirstlane(L.p);
  const double piv = L.piv;
  const double inv = piv != 0.0 ? 1.0 / piv : 0.0;
  if (p < G::NL) {
    // the lanes holding row p: one test per register row keeps every
    // register index a compile-time constant
#pragma unroll
    for (int i = 0; i < G::RI; ++i)
      if (tr + G::TR * i == p) {
#pragma unroll
        for (int j = 0; j < G::RJ; ++j) {
          const int jj = j + jk;
          const int c = tc + G::TC * (jj >= G::RJ ? jj - G::RJ : jj);
          L.rowbuf[c] = c == k ? inv : S[i][j] * inv;
          S[i][j] = 0.0;
        }
        if (tc == 0) L.rowbuf[G::NL] = k == G::NL ? inv : L.Cl[p] * inv;
      }
  } else if (t < G::NMAX) {
    L.rowbuf[t] = t == k ? inv : L.Rl[t] * inv;
  }
  if (t == 0) {
    L.pk[k] = (int16_t)p;
    L.used[p] = 1;
    L.colbuf[p] = -1.0;
  }
  __syncthreads();
  double rv[G::RJ];
#pragma unroll
  for (int j = 0; j < G::RJ; ++j) {
    const int jj = j + jk;
    rv[j] = L.rowbuf[tc + G::TC * (jj >= G::RJ ? jj - G::RJ : jj)];
  }
#pragma unroll
  for (int i = 0; i < G::RI; ++i) {
    const double f = L.colbuf[tr + G::TR * i];
#pragma unroll
    for (int j = 0; j < G::RJ; ++j) S[i][j] = fma(-f, rv[j], S[i][j]);
  }
  if (t < G::NMAX) {
    const double old = (t == k || p == G::NL) ? 0.0 : L.Rl[t];
    L.Rl[t] = fma(-L.colbuf[G::NL], L.rowbuf[t], old);
  }
  if (t < G::NL) {
    const double old = (t == p || k == G::NL) ? 0.0 : L.Cl[t];
    L.Cl[t] = fma(-L.colbuf[t], L.rowbuf[G::NL], old);
  }
  __syncthreads();
}

template <class G, class OutT>
__global__ __launch_bounds__(G::T) void k_patch_gj(int PS, int ld, const int32_t *__restrict__ list,
                                                    const double *__restrict__ A, OutT *__restrict__ out,
                                                    int16_t *__restrict__ perm, int32_t *__restrict__ status,
                                                    float *__restrict__ pscale) {
  __shared__ GJShared<G> L;
  const int t = threadIdx.x, tr = t % G::TR, tc = t / G::TR;
  const int64_t pch = list[blockIdx.x];
  double S[G::RI][G::RJ];
  gj_load<G>(S, L, A + pch * PS * PS, PS, t, tr, tc);
  __syncthreads();
  for (int jk = 0; jk < G::RJ; ++jk) {
    for (int tk = 0; tk < G::TC; ++tk) gj_step<G>(S, L, t, tr, tc, jk, tk);
#pragma unroll
    for (int i = 0; i < G::RI; ++i) {
      const double c0 = S[i][0];
#pragma unroll
      for (int j = 0; j + 1 < G::RJ; ++j) S[i][j] = S[i][j + 1];
      S[i][G::RJ - 1] = c0;
    }
  }
  gj_step<G>(S, L, t, tr, tc, G::RJ, 0);
  gj_unscale<G>(S, L, t, tc, [&](int c) { return (int)L.pk[c]; });
  const double sc = gj_scale<G, OutT>(S, L, PS, t, tr, tc, pscale, pch);
  gj_store<G, OutT>(S, L, out + pch * PS * ld, PS, ld, t, tr, tc, sc);
  int16_t *pp = perm + pch * 2 * PS;
  if (t < PS) {
    pp[t] = L.pk[t];
    pp[PS + L.pk[t]] = (int16_t)t;
  }
  if (t == 0) status[pch] = L.bad;
}

// The products of the patch inverses with the condensed residual.  The inverse
// is stored column-major as Gauss-Jordan leaves it (see k_patch_gj): slot c of
// the input takes the residual of local dof perm[c], and row t of the product
// belongs to local dof perm[PS + t].  Columns are padded to `ld`, a multiple of
// the VEC = 16 bytes / sizeof(MP) rows that a lane loads at once, so the
// ld / VEC lanes of a column and the next columns' lanes read one linear
// stream; the NG column groups of the workgroup are summed through LDS.  The
// kernel is bound by that stream: 2.36 GB of traffic for the FP32 inverses of
// 33,800 stars in 0.40 ms, 5.9 TB/s.
template <class MP>
struct MatVec {
  static constexpr int VEC = 16 / (int)sizeof(MP);
  union {
    uint4 raw;
    MP v[VEC];
  };
  __device__ MatVec() {}
};
template <class MP>
__global__ __launch_bounds__(512) void k_patch_apply(int PS, int ld, const int32_t *__restrict__ psize,
                                                     const int32_t *__restrict__ pidx, const int16_t *__restrict__ perm,
                                                     const MP *__restrict__ Ainv, const double *__restrict__ r,
                                                     double *__restrict__ part, const float *__restrict__ pscale) {
  constexpr int VEC = MatVec<MP>::VEC;
  extern __shared__ double red[];  // [NG][ld]
  __shared__ double rl[256];
  const int pch = blockIdx.x;
  const int sz = psize[pch];
  const int32_t *ids = pidx + (int64_t)pch * PS;
  const int16_t *pp = perm + (int64_t)pch * 2 * PS;
  const int t = threadIdx.x;
  if (t < sz) rl[t] = r[ids[pp[t]]];
  __syncthreads();
  const int lc = ld / VEC, ng = blockDim.x / lc;
  const int grp = t / lc, r0 = (t - grp * lc) * VEC;
  if (grp < ng && r0 < sz) {
    const MP *Ap = Ainv + ((int64_t)pch * PS + grp) * ld + r0;
    const int64_t st = (int64_t)ng * ld;
    double acc[VEC];
#pragma unroll
    for (int v = 0; v < VEC; ++v) acc[v] = 0.0;
    int b = grp;
    for (; b + 3 * ng < sz; b += 4 * ng, Ap += 4 * st) {  // four loads in flight
      MatVec<MP> m[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) m[u].raw = *reinterpret_cast<const uint4 *>(Ap + u * st);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const double x = rl[b + u * ng];
#pragma unroll
        for (int v = 0; v < VEC; ++v) acc[v] += todbl(m[u].v[v]) * x;
      }
    }
    for (; b < sz; b += ng, Ap += st) {
      MatVec<MP> m;
      m.raw = *reinterpret_cast<const uint4 *>(Ap);
      const double x = rl[b];
#pragma unroll
      for (int v = 0; v < VEC; ++v) acc[v] += todbl(m.v[v]) * x;
    }
#pragma unroll
    for (int v = 0; v < VEC; ++v) red[grp * ld + r0 + v] = acc[v];
  }
  __syncthreads();
  if (t < sz) {
    double sum = 0.0;
    for (int k = 0; k < ng; ++k) sum += red[k * ld + t];
    part[(int64_t)pch * PS + pp[PS + t]] = pscale ? sum * (double)pscale[pch] : sum;
  }
}

}  // namespace

// ==================================================================== host side
struct Solver {
  int64_t n = 0, n1 = 0, np = 0, nphi = 0;
  int64_t *d_split = nullptr;
  int32_t *d_pfirst = nullptr, *d_phifirst = nullptr;
  std::vector<double> h_Mp, h_Mphi;   // cell mass inverses (unscaled)
  double *d_Sp = nullptr, *d_Sphi = nullptr;
  double alpha_p = 0.0, alpha_phi = 0.0;
  // patches, with the interior dofs of condensed cells eliminated: PS unknowns
  // at most, columns of the inverses padded to ld (a multiple of 16 bytes)
  int npatch = 0, PS = 0, ld = 0;
  int32_t *d_psize = nullptr, *d_pidx = nullptr;
  int PS_all = 0;                     // all dofs of the largest vertex star
  int64_t pent_all = 0;               // sum over the stars of (all dofs)^2
  int32_t *d_pcptr = nullptr, *d_pcell = nullptr;  // cells around each patch's vertex
  // condensed cells: first interior dof (-1: the cell is not condensed),
  // patches holding them, eliminated [u,j] dofs
  int32_t *d_ifirst = nullptr, *d_npat = nullptr;
  uint8_t *d_elim = nullptr;
  double *d_cE64 = nullptr, *d_cB64 = nullptr;     // [ncells][NB][NI] D^-1 A_ib, A_bi (set-up; E of precision 0)
  double *d_cF64 = nullptr, *d_cG64 = nullptr;     // A_bi D^-1, N D^-1 (precision 0)
  float *d_cE32 = nullptr, *d_cF32 = nullptr, *d_cG32 = nullptr;  // the same for the FP32 inner solve
  int32_t *d_cflag = nullptr;
  double *d_rt = nullptr;             // [n1] condensed residual
  // dof -> patch rows holding it (patch * PS + local index), in patch order
  int32_t *d_dptr = nullptr, *d_dent = nullptr;
  double *d_ppart = nullptr;  // [npatch * PS] per-patch products
  double *d_pA = nullptr;             // FP64 inverses (precision 0)
  float *d_pA32 = nullptr;            // FP32 inverses (precision 1)
  __hip_bfloat16 *d_pA16 = nullptr;   // BF16 inverses (precision 2)
  __half *d_pAh = nullptr;            // FP16 inverses scaled per patch (precision 3)
  float *d_pscale = nullptr;          // [npatch] their scale factors
  int16_t *d_pperm = nullptr;         // [npatch][2][PS] Gauss-Jordan pivot rows and their inverse
  int32_t *d_pstatus = nullptr;       // [npatch] 0, or 1 + the step of a zero pivot
  double *d_pscratch = nullptr;       // FP64 patch matrices of one chunk
  int pchunk = 0;                     // patches per chunk
  int64_t nflagged = 0;               // patches of the last set-up inverted with partial pivoting
  rocblas_handle rb = nullptr;
  // mixed precision copy of A11 values
  float *d_val32 = nullptr;
  // Krylov workspace
  int m = 0, kin = 0;
  double *V = nullptr, *Z = nullptr, *w = nullptr, *b = nullptr, *dx = nullptr, *t1 = nullptr;
  void *V1 = nullptr, *Z1 = nullptr, *w1 = nullptr, *x1 = nullptr, *r1 = nullptr;  // inner, n1-long, FP64 or FP32
  int inner_prec = -1;
  bool transposed = false;  // adjoint solve: every level holds its transposed Jacobian
  double *d_part = nullptr, *d_dots = nullptr, *d_y = nullptr;
  double *h_dots = nullptr;  // pinned, 3 * ldots + 1
  int ldots = 0;             // stride of the reduction slots: max(m, kin) + 1
  int nb_dot = 0;
  // operation counts (mhd_op_counts): nonzeros of the A11 block and of the
  // A12 / A13 columns of the [u,j] rows, sum of dim^2 and dim^3 over patches
  int64_t nnz11 = 0, nnz1x = 0;
  double pent = 0.0, pcube = 0.0;
  double ops[MHD_NOPS] = {};
  // products without the matrix (mhd_cellop_apply); with a skeleton term, or
  // with u or j dofs numbered outside of the [u,j] block, they stream it
  // instead, through the row groups below.  Their element results have a buffer
  // of their own: the context's belongs to mhd_residual_d, which may be pending
  // on a caller's stream.
  bool matfree = true;
  bool scan = false;                  // patch entries from the rows, not cell by cell
  bool unheld = false;                // some [u,j] dof is in no cell
  bool condense = true;               // cells' interior current dofs eliminated where they can be
  double *d_prod = nullptr;           // [ncells][NDOF]
  // row groups sharing a column list (k_spmv_grp): all rows, and the first
  // ngroups11 groups cover the [u,j] rows exactly
  int64_t ngroups = 0, ngroups11 = 0;
  int64_t *d_grow = nullptr, *d_gcp = nullptr;
  int32_t *d_gcol = nullptr;
};

namespace {

inline void count(mhd_ctx *c, int k, double v) {
  if (c->solver) c->solver->ops[k] += v;
}

// s = gamma / sigma of the adjoint scaling (1 when either vanishes)
double adjoint_scale(const mhd_ctx *c) {
  const double g = c->phys.gamma, sg = c->phys.sigma;
  return (g > 0.0 && sg > 0.0) ? g / sg : 1.0;
}

// the scaling of the products: of the transposed ones only
double op_scale(const mhd_ctx *c) { return c->solver->transposed ? adjoint_scale(c) : 1.0; }

// FGMRES Krylov dimension for a requested restart length
int krylov_dim(int restart) { return std::max(2, std::min(restart, 2000)); }

template <class T>
int dmalloc(mhd_ctx *c, T **p, size_t count) {
  MHD_HIP(hipMalloc(reinterpret_cast<void **>(p), sizeof(T) * std::max<size_t>(count, 1)));
  return 0;
}

// Gauss-Jordan inverse of a small SPD matrix (host, no pivoting needed).
void inv_spd(int n, const double *A, double *Ai) {
  std::vector<double> M(n * 2 * n);
  for (int i = 0; i < n; ++i)
    for (int j = 0; j < 2 * n; ++j) M[i * 2 * n + j] = j < n ? A[i * n + j] : (j - n == i ? 1.0 : 0.0);
  for (int c = 0; c < n; ++c) {
    double d = 1.0 / M[c * 2 * n + c];
    for (int j = 0; j < 2 * n; ++j) M[c * 2 * n + j] *= d;
    for (int r = 0; r < n; ++r)
      if (r != c) {
        double f = M[r * 2 * n + c];
        if (f != 0.0)
          for (int j = 0; j < 2 * n; ++j) M[r * 2 * n + j] -= f * M[c * 2 * n + j];
      }
  }
  for (int i = 0; i < n; ++i)
    for (int j = 0; j < n; ++j) Ai[i * n + j] = M[i * 2 * n + n + j];
}

// Cell mass matrices of dP1 and dQ1 (3x3x3 Gauss, the degree-4/5 measures of
// Badia2024Solver, src/Solvers/badia2024.jl:8-15) and their inverses.
void cell_mass_inverses(mhd_ctx *c, std::vector<double> &Mp, std::vector<double> &Mphi) {
  mhd::RefTables *T = new mhd::RefTables;
  mhd::build_ref_tables(T);
  Mp.assign((size_t)c->ncells * 16, 0.0);
  Mphi.assign((size_t)c->ncells * 64, 0.0);
  for (int32_t cc = 0; cc < c->ncells; ++cc) {
    const double *X = &c->h_xyz[(size_t)cc * 24];
    double mp[16] = {0}, mf[64] = {0};
    for (int q = 0; q < NQ; ++q) {
      double J[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
      for (int v = 0; v < 8; ++v)
        for (int i = 0; i < 3; ++i)
          for (int l = 0; l < 3; ++l) J[i][l] += X[3 * v + i] * T->dq1[q][v][l];
      const double det = J[0][0] * (J[1][1] * J[2][2] - J[1][2] * J[2][1]) -
                         J[0][1] * (J[1][0] * J[2][2] - J[1][2] * J[2][0]) +
                         J[0][2] * (J[1][0] * J[2][1] - J[1][1] * J[2][0]);
      const double W = T->w[q] * std::fabs(det);
      for (int k = 0; k < 4; ++k)
        for (int l = 0; l < 4; ++l) mp[4 * k + l] += W * T->p1[q][k] * T->p1[q][l];
      for (int k = 0; k < 8; ++k)
        for (int l = 0; l < 8; ++l) mf[8 * k + l] += W * T->q1[q][k] * T->q1[q][l];
    }
    inv_spd(4, mp, &Mp[(size_t)cc * 16]);
    inv_spd(8, mf, &Mphi[(size_t)cc * 64]);
  }
  delete T;
}

// Vertex-star patches: dofs of u and j (A11 numbering) whose entity contains
// the vertex.  `all` lists every vertex that has any (sorted dofs), `cells`
// the cells around it in increasing order.
void build_patches(mhd_ctx *c, std::vector<std::vector<int32_t>> &all, std::vector<std::vector<int32_t>> &cells) {
  const int64_t n1 = (int64_t)c->nfree[0] + c->nfree[2];
  std::vector<std::vector<int32_t>> lists(c->nverts), around(c->nverts);
  for (int32_t cc = 0; cc < c->ncells; ++cc) {
    const int32_t *cd = &c->h_dofs[(size_t)cc * NDOF];
    for (int lv = 0; lv < 8; ++lv) {
      const int vi = lv & 1, vj = (lv >> 1) & 1, vk = lv >> 2;
      const int32_t v = c->h_verts[(size_t)cc * 8 + lv];
      auto &L = lists[v];
      if (around[v].empty() || around[v].back() != cc) around[v].push_back(cc);
      for (int a = 0; a < 27; ++a) {
        const int i = a % 3, j = (a / 3) % 3, k = a / 9;
        if (std::abs(i - 2 * vi) > 1 || std::abs(j - 2 * vj) > 1 || std::abs(k - 2 * vk) > 1) continue;
        for (int comp = 0; comp < 3; ++comp) {
          const int32_t g = cd[comp * 27 + a];
          if (g >= 0 && g < n1) L.push_back(g);
        }
      }
      for (int r = 0; r < 36; ++r) {
        bool in = true;
        if (r < 24) {
          const int f = r >> 2, d = 2 - f / 2, side = f & 1;
          const int vc = d == 0 ? vi : (d == 1 ? vj : vk);
          in = vc == side;
        }
        if (!in) continue;
        const int32_t g = cd[OFF_J + r];
        if (g >= 0 && g < n1) L.push_back(g);
      }
    }
  }
  all.clear();
  cells.clear();
  for (int32_t v = 0; v < c->nverts; ++v) {
    auto &L = lists[v];
    if (L.empty()) continue;
    std::sort(L.begin(), L.end());
    L.erase(std::unique(L.begin(), L.end()), L.end());
    all.push_back(std::move(L));
    cells.push_back(std::move(around[v]));
  }
}

// The vertices of a cell (bit lv) whose stars hold the local [u,j] dof l.
uint8_t star_vertices(int l) {
  uint8_t m = 0;
  for (int lv = 0; lv < 8; ++lv) {
    const int at[3] = {lv & 1, (lv >> 1) & 1, lv >> 2};
    bool in = true;
    if (l < NU) {
      const int a = l % 27, x[3] = {a % 3, (a / 3) % 3, a / 9};
      for (int d = 0; d < 3; ++d) in = in && std::abs(x[d] - 2 * at[d]) <= 1;
    } else if (l < NB) {
      const int f = (l - NU) >> 2;
      in = at[2 - f / 2] == (f & 1);
    }
    if (in) m |= (uint8_t)(1 << lv);
  }
  return m;
}

// Cells whose interior current dofs can be eliminated: 12 consecutive free
// [u,j] dofs that no other cell and no other place of the cell lists, no u or j
// dof of the cell numbered outside of the [u,j] block, and every star that
// holds a dof of the cell holds the whole cell.  That fails where two cells
// share dofs of an entity but not its vertices (a periodic direction glued in
// the dof table only): a dof then lies in more stars (`stars`) than its entity
// has vertices in the cell.  regular: false if any cell fails the last test.
void build_condensation(const mhd_ctx *c, const std::vector<std::vector<int32_t>> &stars, std::vector<int32_t> &ifirst,
                        std::vector<uint8_t> &elim, bool &regular, bool condense) {
  const int64_t n1 = (int64_t)c->nfree[0] + c->nfree[2];
  std::vector<uint8_t> held(std::max<int64_t>(n1, 1), 0);  // places listing the dof, 2 = more than one
  for (int32_t g : c->h_dofs)
    if (g >= 0 && g < n1) held[g] = (uint8_t)std::min(2, held[g] + 1);
  std::vector<int32_t> nstars(std::max<int64_t>(n1, 1), 0);
  for (const auto &L : stars)
    for (int32_t g : L) ++nstars[g];
  uint8_t mask[NB];
  int local[NB], size[NB];
  for (int l = 0; l < NB; ++l) {
    local[l] = l < NU ? l : l + (OFF_J - NU);
    mask[l] = star_vertices(l);
    size[l] = __builtin_popcount(mask[l]);
  }
  ifirst.assign(c->ncells, -1);
  elim.assign(std::max<int64_t>(n1, 1), 0);
  regular = true;
  for (int32_t cc = 0; cc < c->ncells; ++cc) {
    const int32_t *uj = &c->h_dofs[(size_t)cc * NDOF], *cd = uj + OFF_J + 24, *v = &c->h_verts[(size_t)cc * 8];
    bool ok = cd[0] >= 0 && (int64_t)cd[0] + NI <= n1, whole = true;
    for (int k = 0; k < NI && ok; ++k) ok = cd[k] == cd[0] + k && held[cd[k]] == 1;
    uint8_t first = 0xff;  // local vertices that are not a repetition of an earlier one
    for (int a = 1; a < 8; ++a)
      for (int b = 0; b < a; ++b)
        if (v[a] == v[b]) first &= (uint8_t)~(1 << a);
    for (int l = 0; l < NB; ++l) {
      const int32_t g = uj[local[l]];
      if (g >= n1) ok = false;
      if (g < 0 || g >= n1) continue;
      int n = size[l];
      if (first != 0xff) {
        n = 0;
        for (int a = 0; a < 8; ++a) {
          bool seen = !(mask[l] >> a & 1);
          for (int b = 0; b < a && !seen; ++b) seen = (mask[l] >> b & 1) && v[a] == v[b];
          n += !seen;
        }
      }
      whole = whole && nstars[g] == n;
    }
    regular = regular && whole;
    if (!condense || !ok || !whole) continue;
    ifirst[cc] = cd[0];
    for (int k = 0; k < NI; ++k) elim[cd[k]] = 1;
  }
}

// The interior block of a cell is the RT1 mass plus zeta_j div-div: for a
// negative zeta_j it may be singular where no patch is, so nothing is eliminated.
bool may_condense(const mhd_ctx *c) {
  return !(c->phys.zeta_j < 0.0 || (c->jac_valid && c->jac_phys.zeta_j < 0.0));
}

int solver_build(mhd_ctx *c, const mhd_solver_opts *o, bool condense);

// The solver of a context, built if it has none for this choice.  A solver that
// was refused half-way is not kept: the next call would take it for whole.
int solver_init(mhd_ctx *c, const mhd_solver_opts *o, bool condense) {
  if (c->solver && c->solver->condense == condense) return 0;
  if (c->solver) mhd_solver_free(c);
  const int rc = solver_build(c, o, condense);
  if (rc) mhd_solver_free(c);
  return rc;
}

int solver_build(mhd_ctx *c, const mhd_solver_opts *o, bool condense) {
  if (c->block_style != 1) {
    c->err = "mhd_newton_solve needs the Badia2024 block numbering (spaces.block_style = 1)";
    return -1;
  }
  if (c->h_verts.empty()) {
    c->err = "mhd_newton_solve needs mesh.cell_verts for the vertex-star smoother";
    return -1;
  }
  Solver *S = new Solver();
  c->solver = S;
  S->condense = condense;
  S->n = c->n;
  S->n1 = (int64_t)c->nfree[0] + c->nfree[2];
  S->np = c->nfree[1];
  S->nphi = c->nfree[3];
  S->matfree = c->nskel == 0;
  // p / phi dofs: consecutive per cell
  std::vector<int32_t> pf(c->ncells), ff(c->ncells);
  for (int32_t cc = 0; cc < c->ncells; ++cc) {
    const int32_t *cd = &c->h_dofs[(size_t)cc * NDOF];
    pf[cc] = cd[OFF_P];
    ff[cc] = cd[OFF_PHI];
    for (int k = 0; k < 4; ++k)
      if (cd[OFF_P + k] != pf[cc] + k || pf[cc] < S->n1 || pf[cc] + 4 > S->n1 + S->np) {
        c->err = "p dofs of a cell must be consecutive and inside the p block";
        return -1;
      }
    for (int k = 0; k < 8; ++k)
      if (cd[OFF_PHI + k] != ff[cc] + k || ff[cc] < S->n1 + S->np || ff[cc] + 8 > S->n) {
        c->err = "phi dofs of a cell must be consecutive and inside the phi block";
        return -1;
      }
    for (int l = 0; l < NU + NJ; ++l)
      if (cd[l < NU ? l : l + NP] >= S->n1) S->matfree = false;  // A11 is a block of the matrix, not of the form
  }
  int rc;
  if ((rc = dmalloc(c, &S->d_pfirst, c->ncells))) return rc;
  if ((rc = dmalloc(c, &S->d_phifirst, c->ncells))) return rc;
  MHD_HIP(hipMemcpy(S->d_pfirst, pf.data(), sizeof(int32_t) * c->ncells, hipMemcpyHostToDevice));
  MHD_HIP(hipMemcpy(S->d_phifirst, ff.data(), sizeof(int32_t) * c->ncells, hipMemcpyHostToDevice));
  cell_mass_inverses(c, S->h_Mp, S->h_Mphi);
  if ((rc = dmalloc(c, &S->d_Sp, S->h_Mp.size()))) return rc;
  if ((rc = dmalloc(c, &S->d_Sphi, S->h_Mphi.size()))) return rc;
  if ((rc = dmalloc(c, &S->d_split, S->n1))) return rc;
  for (int64_t i = 0; i < S->n1; ++i) {
    const int32_t *b = c->h_colind.data() + c->h_rowptr[i], *e = c->h_colind.data() + c->h_rowptr[i + 1];
    const int64_t k = std::lower_bound(b, e, (int32_t)S->n1) - b;
    S->nnz11 += k;
    S->nnz1x += (e - b) - k;
  }
  if (!S->matfree) {
    // runs of consecutive rows with one column list (at most GMAX rows; no run
    // crosses the end of the [u,j] rows)
    std::vector<int64_t> grow, gcp;
    std::vector<int32_t> gcol;
    const int64_t *rp = c->h_rowptr.data();
    const int32_t *ci = c->h_colind.data();
    int64_t r = 0;
    while (r < S->n) {
      const int64_t len = rp[r + 1] - rp[r];
      int64_t m = 1;
      while (r + m < S->n && m < GMAX && (r + m != S->n1) && rp[r + m + 1] - rp[r + m] == len &&
             std::equal(ci + rp[r], ci + rp[r] + len, ci + rp[r + m]))
        ++m;
      grow.push_back(r);
      gcp.push_back((int64_t)gcol.size());
      gcol.insert(gcol.end(), ci + rp[r], ci + rp[r] + len);
      if (r < S->n1) S->ngroups11 = (int64_t)grow.size();
      r += m;
    }
    grow.push_back(S->n);
    gcp.push_back((int64_t)gcol.size());
    S->ngroups = (int64_t)grow.size() - 1;
    if ((rc = dmalloc(c, &S->d_grow, grow.size()))) return rc;
    if ((rc = dmalloc(c, &S->d_gcp, gcp.size()))) return rc;
    if ((rc = dmalloc(c, &S->d_gcol, gcol.size()))) return rc;
    MHD_HIP(hipMemcpy(S->d_grow, grow.data(), sizeof(int64_t) * grow.size(), hipMemcpyHostToDevice));
    MHD_HIP(hipMemcpy(S->d_gcp, gcp.data(), sizeof(int64_t) * gcp.size(), hipMemcpyHostToDevice));
    MHD_HIP(hipMemcpy(S->d_gcol, gcol.data(), sizeof(int32_t) * gcol.size(), hipMemcpyHostToDevice));
  }
  hipLaunchKernelGGL(k_split, dim3(nblocks(S->n1)), dim3(TB), 0, c->stream, S->n1, c->d_rowptr, c->d_colind,
                     S->d_split);
  MHD_HIP(hipGetLastError());
  // patches
  {
    std::vector<std::vector<int32_t>> stars, around;
    std::vector<int32_t> ifirst, npat(c->ncells, 0);
    std::vector<uint8_t> elim;
    build_patches(c, stars, around);
    bool regular;
    build_condensation(c, stars, ifirst, elim, regular, S->condense);
    S->scan = !S->matfree || !regular;
    std::vector<uint8_t> in_cell(std::max<int64_t>(S->n1, 1), 0);
    for (int32_t g : c->h_dofs)
      if (g >= 0 && g < S->n1) in_cell[g] = 1;
    S->unheld = std::count(in_cell.begin(), in_cell.begin() + S->n1, (uint8_t)0) > 0;
    S->npatch = (int)stars.size();
    for (const auto &L : stars) {
      S->PS_all = std::max<int>(S->PS_all, (int)L.size());
      S->pent_all += (int64_t)L.size() * (int64_t)L.size();
    }
    if (S->PS_all > PATCH_MAX) {
      c->err = S->PS_all > 256 ? std::string("vertex patch larger than 256 dofs")
                               : "vertex patch larger than " + std::to_string(PATCH_MAX) + " dofs";
      return -1;
    }
    for (auto &L : stars) {
      L.erase(std::remove_if(L.begin(), L.end(), [&](int32_t g) { return elim[g] != 0; }), L.end());
      S->PS = std::max<int>(S->PS, (int)L.size());
    }
    S->PS = std::max(S->PS, 1);
    const int PS = S->PS;
    std::vector<int32_t> psize(S->npatch), pidx((size_t)S->npatch * PS, -1), pcptr(S->npatch + 1, 0), pcell;
    std::vector<int32_t> dptr(S->n1 + 1, 0), dent;
    for (int p = 0; p < S->npatch; ++p) {
      psize[p] = (int32_t)stars[p].size();
      std::copy(stars[p].begin(), stars[p].end(), pidx.begin() + (size_t)p * PS);
      for (int32_t g : stars[p]) ++dptr[g + 1];
      for (int32_t cc : around[p]) {
        pcell.push_back(cc);
        ++npat[cc];
      }
      pcptr[p + 1] = (int32_t)pcell.size();
      S->pent += (double)psize[p] * psize[p];
      S->pcube += (double)psize[p] * psize[p] * psize[p];
    }
    for (int32_t f : ifirst)
      if (f >= 0) S->pent += 2.0 * NB * NI + NI * NI;
    // the smoother sums the patch products of a dof in this fixed order, so
    // its result does not depend on the order the patches finish in
    for (int64_t i = 0; i < S->n1; ++i) dptr[i + 1] += dptr[i];
    dent.resize(dptr[S->n1]);
    std::vector<int32_t> fill(dptr.begin(), dptr.end() - 1);
    for (int p = 0; p < S->npatch; ++p)
      for (int a = 0; a < psize[p]; ++a) dent[fill[pidx[(size_t)p * PS + a]]++] = p * PS + a;
    auto up = [&](auto **dst, const auto &v) -> int {
      int e = dmalloc(c, dst, v.size());
      if (e) return e;
      if (!v.empty()) MHD_HIP(hipMemcpy(*dst, v.data(), sizeof(v[0]) * v.size(), hipMemcpyHostToDevice));
      return 0;
    };
    if ((rc = up(&S->d_psize, psize)) || (rc = up(&S->d_pidx, pidx)) || (rc = up(&S->d_pcptr, pcptr)) ||
        (rc = up(&S->d_pcell, pcell)) || (rc = up(&S->d_ifirst, ifirst)) || (rc = up(&S->d_npat, npat)) ||
        (rc = up(&S->d_elim, elim)) || (rc = up(&S->d_dptr, dptr)) || (rc = up(&S->d_dent, dent)))
      return rc;
  }
  if ((rc = dmalloc(c, &S->d_ppart, (size_t)S->npatch * S->PS))) return rc;
  if ((rc = dmalloc(c, &S->d_pperm, (size_t)S->npatch * 2 * S->PS))) return rc;
  if ((rc = dmalloc(c, &S->d_pstatus, (size_t)S->npatch))) return rc;
  if ((rc = dmalloc(c, &S->d_rt, (size_t)S->n1))) return rc;
  if ((rc = dmalloc(c, &S->d_cflag, 1))) return rc;
  // Krylov workspace
  S->m = krylov_dim(o->restart);
  S->kin = std::max(0, std::min(o->inner_iters, 120));
  const size_t n = (size_t)S->n;
  {
    size_t fr = 0, tot = 0;
    MHD_HIP(hipMemGetInfo(&fr, &tot));
    if ((2 * (size_t)S->m + 1) * n * sizeof(double) > fr / 2) {
      c->err = "FGMRES restart " + std::to_string(S->m) + " needs more than half of the free device memory";
      return -1;
    }
  }
  if ((rc = dmalloc(c, &S->V, (S->m + 1) * n))) return rc;
  if ((rc = dmalloc(c, &S->Z, S->m * n))) return rc;
  if ((rc = dmalloc(c, &S->w, n))) return rc;
  if ((rc = dmalloc(c, &S->b, n))) return rc;
  if ((rc = dmalloc(c, &S->dx, n))) return rc;
  if ((rc = dmalloc(c, &S->t1, n))) return rc;
  S->nb_dot = 512;
  S->ldots = std::max(S->m, S->kin) + 1;
  if ((rc = dmalloc(c, &S->d_part, (size_t)S->nb_dot * S->ldots))) return rc;
  if ((rc = dmalloc(c, &S->d_dots, 3 * (size_t)S->ldots + 1))) return rc;
  if ((rc = dmalloc(c, &S->d_y, (size_t)S->ldots))) return rc;
  MHD_HIP(hipHostMalloc(reinterpret_cast<void **>(&S->h_dots), sizeof(double) * (3 * S->ldots + 1),
                        hipHostMallocDefault));
  MHD_HIP(hipStreamSynchronize(c->stream));
  if (c->coarse) {
    mhd_ctx *cc = c->coarse->ctx;
    mhd_solver_opts oc = *o;
    oc.restart = 2;  // coarse levels only run the inner solve
    oc.inner_iters = cc->coarse ? 0 : c->coarse->coarse_iters;
    if (cc->solver && (cc->solver->kin != std::max(0, std::min(oc.inner_iters, 120)))) mhd_solver_free(cc);
    if ((rc = solver_init(cc, &oc, condense))) {
      c->err = "coarse level: " + cc->err;
      return rc;
    }
  }
  return 0;
}

int inner_alloc(mhd_ctx *c, int prec) {
  Solver *S = c->solver;
  if (S->inner_prec == prec) return 0;
  void *ptrs[] = {S->V1, S->Z1, S->w1, S->x1, S->r1};
  for (void *p : ptrs)
    if (p) MHD_HIP(hipFree(p));
  const size_t es = prec == 0 ? sizeof(double) : sizeof(float);  // inner vectors
  const size_t n1 = (size_t)S->n1;
  MHD_HIP(hipMalloc(&S->V1, es * (S->kin + 1) * n1 + es));
  MHD_HIP(hipMalloc(&S->Z1, es * std::max(S->kin, 1) * n1 + es));
  MHD_HIP(hipMalloc(&S->w1, es * n1 + es));
  MHD_HIP(hipMalloc(&S->x1, es * n1 + es));
  MHD_HIP(hipMalloc(&S->r1, es * n1 + es));
  if (prec >= 1 && !S->matfree && !S->d_val32)
    MHD_HIP(hipMalloc(&S->d_val32, sizeof(float) * std::max<int64_t>(c->nnz, 1)));
  {
    const size_t ms = prec == 0 ? sizeof(double) : prec == 1 ? sizeof(float) : 2;  // bytes of an inverse's entry
    const int vec = 16 / (int)ms;
    S->ld = (S->PS + vec - 1) / vec * vec;
  }
  const size_t pelems = (size_t)S->npatch * S->PS * S->ld;
  if (prec == 0 && !S->d_pA) MHD_HIP(hipMalloc(&S->d_pA, sizeof(double) * pelems));
  if (prec == 1 && !S->d_pA32) MHD_HIP(hipMalloc(&S->d_pA32, sizeof(float) * pelems));
  if (prec == 2 && !S->d_pA16) MHD_HIP(hipMalloc(&S->d_pA16, sizeof(__hip_bfloat16) * pelems));
  if (prec == 3 && !S->d_pAh) {
    MHD_HIP(hipMalloc(&S->d_pAh, sizeof(__half) * pelems));
    MHD_HIP(hipMalloc(&S->d_pscale, sizeof(float) * std::max(S->npatch, 1)));
  }
  const size_t ce = (size_t)std::max(c->ncells, 1) * NB * NI, cg = (size_t)std::max(c->ncells, 1) * NI * NI;
  if (!S->d_cE64) MHD_HIP(hipMalloc(&S->d_cE64, sizeof(double) * ce));
  if (!S->d_cB64) MHD_HIP(hipMalloc(&S->d_cB64, sizeof(double) * ce));
  if (prec == 0 && !S->d_cF64) {
    MHD_HIP(hipMalloc(&S->d_cF64, sizeof(double) * ce));
    MHD_HIP(hipMalloc(&S->d_cG64, sizeof(double) * cg));
  }
  if (prec >= 1 && !S->d_cE32) {
    MHD_HIP(hipMalloc(&S->d_cE32, sizeof(float) * ce));
    MHD_HIP(hipMalloc(&S->d_cF32, sizeof(float) * ce));
    MHD_HIP(hipMalloc(&S->d_cG32, sizeof(float) * cg));
  }
  if (!S->d_pscratch) {
    // the FP64 patch matrices are inverted chunk by chunk (3.3 GB of them at
    // most): only the inverses of the solve's precision are kept for the mesh
    S->pchunk = (int)std::min<int64_t>(S->npatch, (int64_t)8192 * PATCH_MAX * PATCH_MAX / ((int64_t)S->PS * S->PS));
    MHD_HIP(hipMalloc(&S->d_pscratch, sizeof(double) * (size_t)std::max(S->pchunk, 1) * S->PS * S->PS));
  }
  S->inner_prec = prec;
  return 0;
}

// ---- small host helpers around the device reductions ----------------------
template <class T>
int mdot(mhd_ctx *c, const T *V, int64_t ldv, int K, const T *w, int64_t n, double *d_out) {
  Solver *S = c->solver;
  hipLaunchKernelGGL((k_mdot<T>), dim3(S->nb_dot, K), dim3(TB), 0, c->stream, V, ldv, w, n, S->d_part);
  count(c, OP_VEC, (double)(K + 1) * n * sizeof(T));
  hipLaunchKernelGGL(k_mdot_final, dim3(K), dim3(TB), 0, c->stream, S->nb_dot, S->d_part, d_out);
  MHD_HIP(hipGetLastError());
  return 0;
}

// CGS2 Arnoldi step: orthogonalise w against V[0..K), return h (K) and ||w|| (host), w normalised into V[K].
template <class T>
int arnoldi(mhd_ctx *c, T *V, int64_t ldv, int K, T *w, int64_t n, double *h, double *nrm) {
  Solver *S = c->solver;
  int rc;
  const int M = S->ldots;
  double *d1 = S->d_dots, *d2 = S->d_dots + M, *dn = S->d_dots + 2 * M;
  if ((rc = mdot(c, V, ldv, K, w, n, d1))) return rc;
  hipLaunchKernelGGL((k_gs_update<T>), dim3(nblocks(n)), dim3(TB), sizeof(double) * K, c->stream, K, V, ldv, d1, w,
                     n);
  if ((rc = mdot(c, V, ldv, K, w, n, d2))) return rc;
  hipLaunchKernelGGL((k_gs_update<T>), dim3(nblocks(n)), dim3(TB), sizeof(double) * K, c->stream, K, V, ldv, d2, w,
                     n);
  count(c, OP_VEC, 2.0 * (K + 2) * n * sizeof(T) + 2.0 * n * sizeof(T));
  if ((rc = mdot(c, w, 0, 1, w, n, dn))) return rc;
  MHD_HIP(hipMemcpyAsync(S->h_dots, S->d_dots, sizeof(double) * (2 * M + 1), hipMemcpyDeviceToHost, c->stream));
  MHD_HIP(hipStreamSynchronize(c->stream));
  for (int k = 0; k < K; ++k) h[k] = S->h_dots[k] + S->h_dots[M + k];
  *nrm = std::sqrt(std::max(S->h_dots[2 * M], 0.0));
  T *vk = V + (int64_t)K * ldv;
  if (*nrm > 0.0)
    hipLaunchKernelGGL((k_scale_copy<T>), dim3(nblocks(n)), dim3(TB), 0, c->stream, n, 1.0 / *nrm, w, vk);
  MHD_HIP(hipGetLastError());
  return 0;
}

template <class T>
int vnorm(mhd_ctx *c, const T *x, int64_t n, double *out) {
  Solver *S = c->solver;
  const int slot = 3 * S->ldots;
  int rc = mdot(c, x, 0, 1, x, n, S->d_dots + slot);
  if (rc) return rc;
  MHD_HIP(hipMemcpyAsync(S->h_dots + slot, S->d_dots + slot, sizeof(double), hipMemcpyDeviceToHost, c->stream));
  MHD_HIP(hipStreamSynchronize(c->stream));
  *out = std::sqrt(std::max(S->h_dots[slot], 0.0));
  return 0;
}

// Least-squares solve of the (k+1) x k Hessenberg system via Givens rotations.
void hess_solve(int k, const std::vector<double> &H, int ldh, double beta, std::vector<double> &y) {
  std::vector<double> R(H), g(k + 1, 0.0);
  g[0] = beta;
  // Givens rotations column by column
  std::vector<double> cs(k), sn(k);
  for (int j = 0; j < k; ++j) {
    for (int i = 0; i < j; ++i) {
      const double a = R[i * ldh + j], b = R[(i + 1) * ldh + j];
      R[i * ldh + j] = cs[i] * a + sn[i] * b;
      R[(i + 1) * ldh + j] = -sn[i] * a + cs[i] * b;
    }
    const double a = R[j * ldh + j], b = R[(j + 1) * ldh + j];
    const double d = std::hypot(a, b);
    cs[j] = d > 0 ? a / d : 1.0;
    sn[j] = d > 0 ? b / d : 0.0;
    R[j * ldh + j] = d;
    R[(j + 1) * ldh + j] = 0.0;
    g[j + 1] = -sn[j] * g[j];
    g[j] = cs[j] * g[j];
  }
  y.assign(k, 0.0);
  for (int i = k - 1; i >= 0; --i) {
    double s = g[i];
    for (int j = i + 1; j < k; ++j) s -= R[i * ldh + j] * y[j];
    y[i] = R[i * ldh + i] != 0.0 ? s / R[i * ldh + i] : 0.0;
  }
}

// Additive Schwarz over the vertex patches: y = sum_P R_P^T A_P^-1 R_P r
// y (+)= w sum_P R_P^T A_P^-1 R_P r
template <class MP>
void patch_products(const Solver *S, const MP *inv, const float *scale, hipStream_t st) {
  // 256 threads; 512 where a column of FP64 would leave a quarter of them
  // idle (130 rows: 65 lanes a column), or where the patches are fewer than
  // the CUs can hold at once, so that each takes half as many steps
  const int threads = sizeof(MP) == 8 || S->npatch < 2048 ? 512 : 256;
  const size_t lds = sizeof(double) * (size_t)(threads / (S->ld / MatVec<MP>::VEC)) * S->ld;
  hipLaunchKernelGGL((k_patch_apply<MP>), dim3(S->npatch), dim3(threads), lds, st, S->PS, S->ld, S->d_psize,
                     S->d_pidx, S->d_pperm, inv, S->d_rt, S->d_ppart, scale);
}

template <class T>
int patch_as_on(mhd_ctx *c, const T *r, T *y, int prec, double w, bool accumulate, hipStream_t st) {
  Solver *S = c->solver;
  using TE = T;  // the condensation couplings are kept in the precision of the vectors
  const TE *E, *F, *G;
  if constexpr (std::is_same<T, double>::value) {
    E = S->d_cE64;
    F = S->d_cF64;
    G = S->d_cG64;
  } else {
    E = S->d_cE32;
    F = S->d_cF32;
    G = S->d_cG32;
  }
  if (S->npatch == 0) return 0;
  if (S->unheld && !accumulate)  // k_cond_gather goes through the cells
    hipLaunchKernelGGL((k_fill<T>), dim3(nblocks(S->n1)), dim3(TB), 0, st, S->n1, (T)0, y);
  hipLaunchKernelGGL((k_cond_rhs<T, TE>), dim3((unsigned)((4 * S->n1 + 255) / 256)), dim3(256), 0, st, S->n1,
                     c->d_crow, c->d_centry, S->d_elim, S->d_ifirst, F, r, S->d_rt, (const int32_t *)nullptr);
  if (prec == 0) patch_products(S, S->d_pA, (const float *)nullptr, st);
  else if (prec == 1) patch_products(S, S->d_pA32, (const float *)nullptr, st);
  else if (prec == 2) patch_products(S, S->d_pA16, (const float *)nullptr, st);
  else patch_products(S, S->d_pAh, (const float *)S->d_pscale, st);
  count(c, prec == 0 ? OP_PATCH64 : prec == 1 ? OP_PATCH32 : OP_PATCH16, S->pent);
  hipLaunchKernelGGL((k_cond_gather<T, TE>), dim3((unsigned)((c->ncells + CG_CELLS - 1) / CG_CELLS)),
                     dim3(64 * CG_CELLS), 0, st, c->ncells, S->n1, c->d_dofs, S->d_ifirst, c->d_crow, c->d_centry,
                     S->d_dptr, S->d_dent, S->d_ppart, E, G, r, w, y, accumulate ? 1 : 0);
  MHD_HIP(hipGetLastError());
  return 0;
}

template <class T>
int patch_as(mhd_ctx *c, const T *r, T *y, int prec, double w = 1.0, bool accumulate = false) {
  return patch_as_on<T>(c, r, y, prec, w, accumulate, c->stream);
}

// y = A11 x (MODE 1) or y = v - A11 x (MODE 3) on the [u,j] rows.  Without a
// skeleton term the form is applied cell by cell: a product reads 0.15 GB at
// 64 x 64 x 8 where the matrix has 1.7 GB (FP32) or 3.0 GB (FP64).  With one,
// the matrix is streamed through the row groups, FP64 values for precision 0
// and the FP32 copy otherwise (the face matrices of the skeleton term alone are
// as large as the FP32 matrix).
template <class T, int MODE>
int a11_product(mhd_ctx *c, const T *x, const T *v, T *y, int prec) {
  Solver *S = c->solver;
  if (S->matfree) {
    count(c, prec == 0 ? OP_SPMV64 : OP_SPMV32, (double)S->nnz11);
    return mhd_cellop_apply<T>(c, MHD_OP_UJ, S->transposed, op_scale(c), x, MODE == 3 ? v : (const T *)nullptr, y,
                               S->d_prod, c->stream);
  }
  constexpr int LPG = 16;
  const int grid = (int)((S->ngroups11 * LPG + 255) / 256);
  if (prec == 0)
    hipLaunchKernelGGL((k_spmv_grp<double, T, T, LPG, MODE>), dim3(grid), dim3(256), 0, c->stream, S->ngroups11,
                       S->d_grow, S->d_gcp, S->d_gcol, c->d_rowptr, S->d_split, c->d_val, x, v, y);
  else
    hipLaunchKernelGGL((k_spmv_grp<float, T, T, LPG, MODE>), dim3(grid), dim3(256), 0, c->stream, S->ngroups11,
                       S->d_grow, S->d_gcp, S->d_gcol, c->d_rowptr, S->d_split, S->d_val32, x, v, y);
  count(c, prec == 0 ? OP_SPMV64 : OP_SPMV32, (double)S->nnz11);
  MHD_HIP(hipGetLastError());
  return 0;
}

// y = J x with the full FP64 Jacobian of the context, the same two ways
int full_product(mhd_ctx *c, const double *x, double *y) {
  Solver *S = c->solver;
  if (S->matfree) {
    count(c, OP_SPMV64, (double)c->nnz);
    return mhd_cellop_apply<double>(c, MHD_OP_FULL, S->transposed, op_scale(c), x, (const double *)nullptr, y,
                                    S->d_prod, c->stream);
  }
  constexpr int LPG = 16;
  const int grid = (int)((S->ngroups * LPG + 255) / 256);
  hipLaunchKernelGGL((k_spmv_grp<double, double, double, LPG, 0>), dim3(grid), dim3(256), 0, c->stream, S->ngroups,
                     S->d_grow, S->d_gcp, S->d_gcol, c->d_rowptr, S->d_split, c->d_val, x, (const double *)nullptr,
                     y);
  count(c, OP_SPMV64, (double)c->nnz);
  MHD_HIP(hipGetLastError());
  return 0;
}

template <class T>
int spmv_a11(mhd_ctx *c, const T *x, T *y, int prec) {
  return a11_product<T, 1>(c, x, (const T *)nullptr, y, prec);
}

template <class T>
int inner_solve(mhd_ctx *c, int prec);

// ec = A11c^-1 rc on the coarsest level, its cells' interior current dofs
// condensed out (4,144 of 5,680 unknowns on 4 x 4 x 8 cells): the explicit FP64
// inverse of the condensed block, FP64 couplings; FP32 vectors are widened
// inside the products, since the coarsest block is the worst conditioned one
// and its correction reaches every level above.
template <class T>
int coarse_direct(mhd_ctx *c, const T *rc, T *ec) {
  CoarseLink *L = c->coarse;
  mhd_ctx *cc = L->ctx;
  const Solver *S = cc->solver;
  const int64_t n = L->n1c, m = L->nb;
  hipLaunchKernelGGL((k_cond_rhs<T, double>), dim3((unsigned)((4 * n + 255) / 256)), dim3(256), 0, c->stream, n,
                     cc->d_crow, cc->d_centry, S->d_elim, S->d_ifirst, L->d_cF, rc, L->d_rb, L->d_bmap);
  hipLaunchKernelGGL((k_dense_rowdot<T>), dim3((unsigned)m), dim3(TB), 0, c->stream, m, L->d_Ainv,
                     L->d_rb, L->d_bidx, L->d_yb, ec);
  hipLaunchKernelGGL((k_cond_inner<T>), dim3((unsigned)((cc->ncells + 3) / 4)), dim3(256), 0, c->stream, cc->ncells,
                     cc->d_dofs, S->d_ifirst, S->d_cE64, L->d_cG, rc, L->d_yb, ec);
  count(c, OP_DENSE, (double)m * m + (double)cc->ncells * (2 * NB * NI + NI * NI));
  MHD_HIP(hipGetLastError());
  return 0;
}

// One V-cycle on the [u,j] block of level c: y = M^-1 r with damped
// vertex-star Schwarz pre- and post-smoothing around the coarse correction.
// The coarse correction yc = P A11c^-1 P^T (r - A11 y) enters with the full
// step (coarse_step 0) or with a = argmin ||r - A11 (y + a yc)|| (coarse_step
// 1): the coarse levels are rediscretised, not Galerkin products, and where
// they misrepresent the fine operator (thin boundary layers under-resolved at
// high Ha on coarse meshes) the full step can ruin the cycle while the
// minimal-residual step only rescales it.  Where the coarse levels are good
// the full step converges in fewer iterations.  The coarsest
// level is solved exactly (dense inverse) or by coarse_iters steps of
// Schwarz-preconditioned FGMRES.
template <class T>
int vcycle(mhd_ctx *c, const T *r, T *y, int prec) {
  Solver *S = c->solver;
  int rc;
  CoarseLink *L = c->coarse;
  if (!L) return patch_as<T>(c, r, y, prec);
  if ((rc = patch_as<T>(c, r, y, prec, L->omega))) return rc;
  mhd_ctx *cc = L->ctx;
  Solver *SC = cc->solver;
  // lanes per row: a prolongation row has 1 to 9 entries (3.8 on average, 16
  // lanes took 28 us on the finest level of 32 x 32 x 8, 4 take 12), a
  // restriction row 9 to 25
  constexpr int LPR = 16, LPP = 4;
  const int64_t ld = L->n1 + 1;
  T *rr = (T *)L->rr, *wv = rr + ld, *yc = rr + 2 * ld;
  T *rcv = (T *)L->rc, *ec = (T *)L->ec;
  const int gfine = (int)((S->n1 * LPP + 255) / 256), gc = (int)((L->n1c * LPR + 255) / 256);
  // rr = r - A11 y
  if ((rc = a11_product<T, 3>(c, y, r, rr, prec))) return rc;
  // restriction
  if (prec == 0)
    hipLaunchKernelGGL((k_csr<double, T, LPR, false>), dim3(gc), dim3(256), 0, c->stream, L->n1c, L->d_Trow, L->d_Tcol,
                       L->d_Tval, rr, rcv);
  else
    hipLaunchKernelGGL((k_csr<float, T, LPR, false>), dim3(gc), dim3(256), 0, c->stream, L->n1c, L->d_Trow, L->d_Tcol,
                       L->d_Tval32, rr, rcv);
  MHD_HIP(hipGetLastError());
  // restriction and prolongation (the A11 products count themselves)
  count(c, prec == 0 ? OP_SPMV64 : OP_SPMV32, 2.0 * L->nnzP);
  if (cc->coarse) {
    if ((rc = vcycle<T>(cc, rcv, ec, prec))) return rc;
  } else if (L->coarse_iters == 0) {
    if ((rc = coarse_direct<T>(c, rcv, ec))) return rc;
  } else {
    MHD_HIP(hipMemcpyAsync(SC->r1, rcv, sizeof(T) * L->n1c, hipMemcpyDeviceToDevice, c->stream));
    if ((rc = inner_solve<T>(cc, prec))) return rc;
    MHD_HIP(hipMemcpyAsync(ec, SC->x1, sizeof(T) * L->n1c, hipMemcpyDeviceToDevice, c->stream));
  }
  if (L->step_mode == 0) {  // y += P ec, rr = r - A11 y
    if (prec == 0)
      hipLaunchKernelGGL((k_csr<double, T, LPP, true>), dim3(gfine), dim3(256), 0, c->stream, S->n1, L->d_Prow,
                         L->d_Pcol, L->d_Pval, ec, y);
    else
      hipLaunchKernelGGL((k_csr<float, T, LPP, true>), dim3(gfine), dim3(256), 0, c->stream, S->n1, L->d_Prow,
                         L->d_Pcol, L->d_Pval32, ec, y);
    MHD_HIP(hipGetLastError());
    if ((rc = a11_product<T, 3>(c, y, r, rr, prec))) return rc;
    return patch_as<T>(c, rr, y, prec, L->omega, true);
  }
  // yc = P ec, w = A11 yc
  if (prec == 0)
    hipLaunchKernelGGL((k_csr<double, T, LPP, false>), dim3(gfine), dim3(256), 0, c->stream, S->n1, L->d_Prow,
                       L->d_Pcol, L->d_Pval, ec, yc);
  else
    hipLaunchKernelGGL((k_csr<float, T, LPP, false>), dim3(gfine), dim3(256), 0, c->stream, S->n1, L->d_Prow,
                       L->d_Pcol, L->d_Pval32, ec, yc);
  MHD_HIP(hipGetLastError());
  if ((rc = a11_product<T, 1>(c, yc, (const T *)nullptr, wv, prec))) return rc;
  // (rr . w, w . w) on the device; y += a yc, rr -= a w
  if ((rc = mdot(c, rr, ld, 2, wv, S->n1, L->d_ab))) return rc;
  hipLaunchKernelGGL((k_cc_update<T>), dim3(nblocks(S->n1)), dim3(TB), 0, c->stream, S->n1, L->d_ab, yc, wv, y, rr);
  count(c, OP_VEC, 6.0 * S->n1 * sizeof(T));
  MHD_HIP(hipGetLastError());
  // post-smoothing accumulates into y
  if ((rc = patch_as<T>(c, rr, y, prec, L->omega, true))) return rc;
  return 0;
}

template <class T>
int apply_m(mhd_ctx *c, const T *r, T *y, int prec) {
  return c->coarse ? vcycle<T>(c, r, y, prec) : patch_as<T>(c, r, y, prec);
}

// x1 ~ A11^-1 r1 by kin steps of right-preconditioned flexible GMRES from x = 0.
template <class T>
int inner_solve(mhd_ctx *c, int prec) {
  Solver *S = c->solver;
  const int64_t n1 = S->n1;
  T *V1 = (T *)S->V1, *Z1 = (T *)S->Z1, *w1 = (T *)S->w1, *x1 = (T *)S->x1, *r1 = (T *)S->r1;
  int rc;
  if (S->kin == 0) return apply_m<T>(c, r1, x1, prec);
  double beta;
  if ((rc = vnorm(c, r1, n1, &beta))) return rc;
  hipLaunchKernelGGL((k_fill<T>), dim3(nblocks(n1)), dim3(TB), 0, c->stream, n1, (T)0, x1);
  if (beta == 0.0) return 0;
  hipLaunchKernelGGL((k_scale_copy<T>), dim3(nblocks(n1)), dim3(TB), 0, c->stream, n1, 1.0 / beta, r1, V1);
  const int ldh = S->kin;
  std::vector<double> H((S->kin + 1) * ldh, 0.0), h(S->kin + 1), y;
  int k = 0;
  for (int j = 0; j < S->kin; ++j) {
    if ((rc = apply_m<T>(c, V1 + j * n1, Z1 + j * n1, prec))) return rc;
    if ((rc = spmv_a11<T>(c, Z1 + j * n1, w1, prec))) return rc;
    double nrm;
    if ((rc = arnoldi<T>(c, V1, n1, j + 1, w1, n1, h.data(), &nrm))) return rc;
    for (int i = 0; i <= j; ++i) H[i * ldh + j] = h[i];
    H[(j + 1) * ldh + j] = nrm;
    k = j + 1;
    if (nrm <= 1e-300) break;
  }
  hess_solve(k, H, ldh, beta, y);
  MHD_HIP(hipMemcpyAsync(S->d_y, y.data(), sizeof(double) * k, hipMemcpyHostToDevice, c->stream));
  hipLaunchKernelGGL((k_lincomb<T>), dim3(nblocks(n1)), dim3(TB), sizeof(double) * k, c->stream, k, Z1, n1, S->d_y, 0.0,
                     x1, n1);
  count(c, OP_VEC, (k + 1.0) * n1 * sizeof(T));
  MHD_HIP(hipGetLastError());
  MHD_HIP(hipStreamSynchronize(c->stream));  // y is a pageable host buffer
  return 0;
}

// z = P^-1 v (FP64 in/out)
int precond(mhd_ctx *c, const double *v, double *z, int prec) {
  Solver *S = c->solver;
  int rc;
  hipLaunchKernelGGL((k_schur<double>), dim3(nblocks((int64_t)c->ncells * 12)), dim3(TB), 0, c->stream, c->ncells,
                     S->d_pfirst, S->d_phifirst, S->d_Sp, S->d_Sphi, v, z);
  // rhs1 = v1 - A12 z_p - A13 z_phi (FP64)
  double *rhs1 = prec == 0 ? (double *)S->r1 : S->t1;
  count(c, OP_SPMV64, (double)S->nnz1x);
  if (S->matfree) {
    if ((rc = mhd_cellop_apply<double>(c, MHD_OP_PPHI, S->transposed, op_scale(c), z, v, rhs1, S->d_prod,
                                       c->stream))) return rc;
  } else {
    constexpr int LPR = 16;
    hipLaunchKernelGGL((k_spmv_suffix<LPR>), dim3((unsigned)((S->n1 * LPR + 255) / 256)),
                       dim3(256), 0, c->stream, S->n1, c->d_rowptr, S->d_split, c->d_colind, c->d_val, z, v, rhs1);
    MHD_HIP(hipGetLastError());
  }
  if (prec == 0) {
    if ((rc = inner_solve<double>(c, 0))) return rc;
    MHD_HIP(hipMemcpyAsync(z, S->x1, sizeof(double) * S->n1, hipMemcpyDeviceToDevice, c->stream));
  } else {
    hipLaunchKernelGGL((k_convert<double, float>), dim3(nblocks(S->n1)), dim3(TB), 0, c->stream, S->n1, S->t1,
                       (float *)S->r1);
    MHD_HIP(hipGetLastError());
    if ((rc = inner_solve<float>(c, prec))) return rc;
    hipLaunchKernelGGL((k_convert<float, double>), dim3(nblocks(S->n1)), dim3(TB), 0, c->stream, S->n1,
                       (const float *)S->x1, z);
  }
  MHD_HIP(hipGetLastError());
  return 0;
}

int coarse_alloc(mhd_ctx *c, int prec) {
  CoarseLink *L = c->coarse;
  const int tp = prec == 0 ? 0 : 1;
  if (L->tprec == tp) return 0;
  void *ptrs[] = {L->rr, L->rc, L->ec};
  for (void *p : ptrs)
    if (p) MHD_HIP(hipFree(p));
  const size_t es = tp == 0 ? sizeof(double) : sizeof(float);
  MHD_HIP(hipMalloc(&L->rr, es * 3 * (L->n1 + 1)));  // rr, w, yc (stride n1 + 1)
  if (!L->d_ab) MHD_HIP(hipMalloc(&L->d_ab, sizeof(double) * 2));
  MHD_HIP(hipMalloc(&L->rc, es * (L->n1c + 1)));
  MHD_HIP(hipMalloc(&L->ec, es * (L->n1c + 1)));
  L->tprec = tp;
  return 0;
}

template <class OutT>
void launch_gjd(const mhd_ctx *c, int np, const double *mat, OutT *out, int16_t *pp, int32_t *st, float *sc) {
  const Solver *S = c->solver;
  if (S->PS <= GJSmall::NMAX)
    hipLaunchKernelGGL((k_patch_gjd<GJSmall, OutT>), dim3(np), dim3(GJSmall::T), 0, c->stream, S->PS, S->ld,
                       c->pivot_tau, mat, out, pp, st, sc);
  else
    hipLaunchKernelGGL((k_patch_gjd<GJLarge, OutT>), dim3(np), dim3(GJLarge::T), 0, c->stream, S->PS, S->ld,
                       c->pivot_tau, mat, out, pp, st, sc);
}
template <class OutT>
void launch_gj(const mhd_ctx *c, int np, const int32_t *list, const double *mat, OutT *out, int16_t *pp, int32_t *st,
               float *sc) {
  const Solver *S = c->solver;
  if (S->PS <= GJSmall::NMAX)
    hipLaunchKernelGGL((k_patch_gj<GJSmall, OutT>), dim3(np), dim3(GJSmall::T), 0, c->stream, S->PS, S->ld, list, mat,
                       out, pp, st, sc);
  else
    hipLaunchKernelGGL((k_patch_gj<GJLarge, OutT>), dim3(np), dim3(GJLarge::T), 0, c->stream, S->PS, S->ld, list, mat,
                       out, pp, st, sc);
}

// Condensed patch matrices, chunk by chunk (d_pscratch) -> Gauss-Jordan
// inverses in the array `inv` of the set-up's precision: diagonal pivots
// first, partial pivoting for the patches whose diagonal pivots fail the
// threshold test.
template <class OutT>
int invert_patches_to(mhd_ctx *c, OutT *inv, float *scale) {
  Solver *S = c->solver;
  const int64_t po = (int64_t)S->PS * S->ld;
  S->nflagged = 0;
  count(c, OP_SETUP_PATCH3, S->pcube);
  const int dups = c->dup_dofs ? 1 : 0;
  for (int p0 = 0; p0 < S->npatch; p0 += S->pchunk) {
    const int np = std::min(S->pchunk, S->npatch - p0);
    double *mat = S->d_pscratch;
    const bool small = S->PS <= GJSmall::NMAX, scan = S->scan;
    auto build = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(np), dim3(1024), 0, c->stream, S->PS, S->d_psize + p0,
                         S->d_pidx + (int64_t)p0 * S->PS, S->d_pcptr + p0, S->d_pcell, c->d_rowptr, c->d_colind,
                         c->d_rank, c->d_val, c->d_dofs, S->d_ifirst, dups, S->d_cE64, S->d_cB64, mat);
    };
    if (scan) small ? build(k_patch_build<true, true>) : build(k_patch_build<false, true>);
    else small ? build(k_patch_build<true, false>) : build(k_patch_build<false, false>);
    int16_t *pp = S->d_pperm + (int64_t)p0 * 2 * S->PS;
    int32_t *st = S->d_pstatus + p0;
    OutT *out = inv + p0 * po;
    float *sc = scale ? scale + p0 : nullptr;
    launch_gjd(c, np, mat, out, pp, st, sc);
    MHD_HIP(hipGetLastError());
    std::vector<int32_t> status(np), flagged;
    MHD_HIP(hipMemcpyAsync(status.data(), st, sizeof(int32_t) * np, hipMemcpyDeviceToHost, c->stream));
    MHD_HIP(hipStreamSynchronize(c->stream));
    for (int q = 0; q < np; ++q)
      if (status[q] != 0) flagged.push_back(q);
    if (flagged.empty()) continue;
    S->nflagged += (int64_t)flagged.size();
    int32_t *d_list = nullptr;
    MHD_HIP(hipMalloc(&d_list, sizeof(int32_t) * flagged.size()));
    MHD_HIP(hipMemcpyAsync(d_list, flagged.data(), sizeof(int32_t) * flagged.size(), hipMemcpyHostToDevice,
                           c->stream));
    launch_gj(c, (int)flagged.size(), d_list, mat, out, pp, st, sc);
    MHD_HIP(hipGetLastError());
    MHD_HIP(hipMemcpyAsync(status.data(), st, sizeof(int32_t) * np, hipMemcpyDeviceToHost, c->stream));
    MHD_HIP(hipStreamSynchronize(c->stream));
    MHD_HIP(hipFree(d_list));
    for (int q : flagged)
      if (status[q] != 0) {
        c->err = "vertex patch " + std::to_string(p0 + q) + " is singular (zero pivot at step " +
                 std::to_string(status[q] - 1) + ")";
        return -3;
      }
  }
  return 0;
}

int invert_patches(mhd_ctx *c, int prec) {
  Solver *S = c->solver;
  hipLaunchKernelGGL((k_fill<int32_t>), dim3(1), dim3(TB), 0, c->stream, (int64_t)1, (int32_t)0, S->d_cflag);
  const int dups = c->dup_dofs ? 1 : 0;
  if (prec == 0)
    hipLaunchKernelGGL(k_condense<double>, dim3(c->ncells), dim3(CND_T), 0, c->stream, c->ncells, c->d_dofs,
                       S->d_ifirst, S->d_npat, dups, c->d_rowptr, c->d_rank, c->d_val, S->d_cE64, S->d_cB64,
                       (double *)nullptr, S->d_cF64, S->d_cG64, S->d_cflag);
  else
    hipLaunchKernelGGL(k_condense<float>, dim3(c->ncells), dim3(CND_T), 0, c->stream, c->ncells, c->d_dofs,
                       S->d_ifirst, S->d_npat, dups, c->d_rowptr, c->d_rank, c->d_val, S->d_cE64, S->d_cB64, S->d_cE32, S->d_cF32,
                       S->d_cG32, S->d_cflag);
  MHD_HIP(hipGetLastError());
  int rc;
  if (prec == 0) rc = invert_patches_to(c, S->d_pA, nullptr);
  else if (prec == 1) rc = invert_patches_to(c, S->d_pA32, nullptr);
  else if (prec == 2) rc = invert_patches_to(c, S->d_pA16, nullptr);
  else rc = invert_patches_to(c, S->d_pAh, S->d_pscale);
  if (rc) return rc;
  int32_t flag = 0;
  MHD_HIP(hipMemcpyAsync(&flag, S->d_cflag, sizeof(int32_t), hipMemcpyDeviceToHost, c->stream));
  MHD_HIP(hipStreamSynchronize(c->stream));
  if (flag) {
    c->err = "the interior current block of cell " + std::to_string(flag - 1) + " is singular";
    return -3;
  }
  return 0;
}

// the arrays of the exact coarsest solve
void dense_free(CoarseLink *L) {
  auto drop = [](auto *&p) {
    if (p) (void)hipFree(p);
    p = nullptr;
  };
  drop(L->d_bidx), drop(L->d_bmap), drop(L->d_ones), drop(L->d_piv), drop(L->d_info), drop(L->d_gjflag);
  drop(L->d_cF), drop(L->d_cG), drop(L->d_rb), drop(L->d_yb), drop(L->d_Ainv), drop(L->d_LU), drop(L->d_gjw);
}

// Per-Jacobian set-up of one level: Schur scalings, FP32 copy and patch
// factorisation, then the coarser levels: the u state is injected from
// `d_state` and the [u,j] block re-assembled with the same kernels
// (rediscretisation).  Every level runs on the fine level's stream.
int precond_setup(mhd_ctx *c, int prec, const double *d_state) {
  Solver *S = c->solver;
  int rc;
  if ((rc = inner_alloc(c, prec))) return rc;
  if (c->coarse && (rc = coarse_alloc(c, prec))) return rc;
  const double ap = -1.0 / (c->phys.beta + c->phys.zeta_u);
  const double aphi = -1.0 / (1.0 + c->phys.zeta_j);
  if (ap != S->alpha_p || aphi != S->alpha_phi) {
    std::vector<double> sp(S->h_Mp), sf(S->h_Mphi);
    for (auto &v : sp) v /= ap;
    for (auto &v : sf) v /= aphi;
    MHD_HIP(hipMemcpy(S->d_Sp, sp.data(), sizeof(double) * sp.size(), hipMemcpyHostToDevice));
    MHD_HIP(hipMemcpy(S->d_Sphi, sf.data(), sizeof(double) * sf.size(), hipMemcpyHostToDevice));
    S->alpha_p = ap;
    S->alpha_phi = aphi;
  }
  if (S->matfree) {
    if (!S->d_prod && (rc = dmalloc(c, &S->d_prod, (size_t)c->ncells * NDOF))) return rc;
  } else if (prec >= 1)
    hipLaunchKernelGGL((k_convert<double, float>), dim3(nblocks(c->nnz)), dim3(TB), 0, c->stream, c->nnz, c->d_val,
                       S->d_val32);
  if ((rc = invert_patches(c, prec))) return rc;
  MHD_HIP(hipGetLastError());
  if (!c->coarse) return 0;
  CoarseLink *L = c->coarse;
  mhd_ctx *cc = L->ctx;
  hipStream_t cs = cc->stream;
  cc->phys = c->phys;
  hipLaunchKernelGGL(k_state_restrict, dim3(nblocks(cc->n)), dim3(TB), 0, cs, cc->n, L->nuc, L->d_Rrow, L->d_Rcol,
                     L->d_Rval, d_state, cc->d_x);
  MHD_HIP(hipGetLastError());
  if ((rc = mhd_assemble_own(cc, cs))) {
    c->err = "coarse level: " + cc->err;
    return rc;
  }
  count(c, OP_SETUP_CELLS, (double)cc->ncells);
  if (S->transposed) {
    // adjoint: the coarse levels carry A_c^T (same transfers P, P^T); the
    // element buffer, free after the assembly, holds the transposed copy
    if (!cc->d_ebuf) MHD_HIP(hipMalloc(&cc->d_ebuf, sizeof(double) * (size_t)std::max(cc->ncells, 1) * NENT));
    if ((rc = mhd_launch_transpose_values(cc, cc->d_val, cc->d_ebuf, cs))) {
      c->err = "coarse level: " + cc->err;
      return rc;
    }
    MHD_HIP(hipMemcpyAsync(cc->d_val, cc->d_ebuf, sizeof(double) * cc->nnz, hipMemcpyDeviceToDevice, cs));
    hipLaunchKernelGGL(k_adj_scale, dim3(nblocks(cc->n)), dim3(TB), 0, cs, cc->n, cc->d_rowptr, cc->d_colind,
                       cc->d_val, (int64_t)cc->nfree[0], (int64_t)cc->nfree[0] + cc->nfree[2], (int64_t)cc->nfree[1],
                       adjoint_scale(c));
    MHD_HIP(hipGetLastError());
    if (cc->solver) cc->solver->transposed = true;
  }
  if ((rc = precond_setup(cc, prec, cc->d_x))) {
    c->err = "coarse level: " + cc->err;
    return rc;
  }
  if (L->coarse_iters == 0 && !cc->coarse) {
    // exact coarsest solve: the explicit inverse of its condensed [u,j] block,
    // row-major (the layout of the row-dot product).  The row-major copy of the
    // block S is the column-major S^T; block Gauss-Jordan inverts it in place
    // into (S^T)^-1, whose column-major storage is S^-1 row-major.
    Solver *SC = cc->solver;
    if (!L->d_Ainv || L->condensed != SC->condense) {
      dense_free(L);
      L->condensed = SC->condense;
      std::vector<int32_t> bidx, bmap(L->n1c, -1), ones(cc->ncells, 1);
      std::vector<uint8_t> elim(L->n1c);
      MHD_HIP(hipMemcpy(elim.data(), SC->d_elim, (size_t)L->n1c, hipMemcpyDeviceToHost));
      for (int64_t i = 0; i < L->n1c; ++i)
        if (!elim[i]) {
          bmap[i] = (int32_t)bidx.size();
          bidx.push_back((int32_t)i);
        }
      const int64_t m = L->nb = (int64_t)bidx.size();
      const int64_t nw = 2 * m * BGJ_B + 2 * (int64_t)BGJ_B * BGJ_B + 3 * m + 2;
      MHD_HIP(hipMalloc(&L->d_bidx, sizeof(int32_t) * (size_t)std::max<int64_t>(m, 1)));
      MHD_HIP(hipMalloc(&L->d_bmap, sizeof(int32_t) * (size_t)L->n1c));
      MHD_HIP(hipMalloc(&L->d_ones, sizeof(int32_t) * (size_t)cc->ncells));
      MHD_HIP(hipMemcpy(L->d_bidx, bidx.data(), sizeof(int32_t) * (size_t)m, hipMemcpyHostToDevice));
      MHD_HIP(hipMemcpy(L->d_bmap, bmap.data(), sizeof(int32_t) * (size_t)L->n1c, hipMemcpyHostToDevice));
      MHD_HIP(hipMemcpy(L->d_ones, ones.data(), sizeof(int32_t) * (size_t)cc->ncells, hipMemcpyHostToDevice));
      MHD_HIP(hipMalloc(&L->d_cF, sizeof(double) * (size_t)cc->ncells * NB * NI));
      MHD_HIP(hipMalloc(&L->d_cG, sizeof(double) * (size_t)cc->ncells * NI * NI));
      MHD_HIP(hipMalloc(&L->d_rb, sizeof(double) * (size_t)std::max<int64_t>(m, 1)));
      MHD_HIP(hipMalloc(&L->d_yb, sizeof(double) * (size_t)L->n1c));
      MHD_HIP(hipMalloc(&L->d_LU, sizeof(double) * (size_t)(m * m)));
      MHD_HIP(hipMalloc(&L->d_piv, sizeof(int32_t) * (size_t)std::max<int64_t>(m, 1)));
      MHD_HIP(hipMalloc(&L->d_info, sizeof(int32_t)));
      MHD_HIP(hipMalloc(&L->d_gjw, sizeof(double) * (size_t)nw));
      MHD_HIP(hipMalloc(&L->d_gjflag, sizeof(int32_t)));
      MHD_HIP(hipMalloc(&L->d_Ainv, sizeof(double) * (size_t)(m * m)));
    }
    const int64_t m = L->nb;
    const int dups = cc->dup_dofs ? 1 : 0;
    // FP64 couplings of single cells (the level's set-up has left its own for the smoother)
    hipLaunchKernelGGL(k_condense<double>, dim3(cc->ncells), dim3(CND_T), 0, cs, cc->ncells, cc->d_dofs, SC->d_ifirst,
                       L->d_ones, dups, cc->d_rowptr, cc->d_rank, cc->d_val, SC->d_cE64, SC->d_cB64, (double *)nullptr,
                       L->d_cF, L->d_cG, SC->d_cflag);
    hipLaunchKernelGGL(k_dense_cond, dim3((unsigned)m), dim3(256), 0, cs, m, L->d_bidx, L->d_bmap, cc->d_rowptr,
                       SC->d_split, cc->d_colind, cc->d_val, cc->d_crow, cc->d_centry, cc->d_dofs, SC->d_ifirst, dups,
                       SC->d_cE64, SC->d_cB64, L->d_LU);
    MHD_HIP(hipGetLastError());
    MHD_HIP(hipMemcpyAsync(L->d_Ainv, L->d_LU, sizeof(double) * (size_t)(m * m), hipMemcpyDeviceToDevice, cs));
    MHD_HIP(hipMemsetAsync(L->d_gjflag, 0, sizeof(int32_t), cs));
    double *M = L->d_Ainv, *C = L->d_gjw, *R = C + m * BGJ_B, *P = R + m * BGJ_B;
    double *D = P + (int64_t)BGJ_B * BGJ_B;
    double *vb = D + (int64_t)BGJ_B * BGJ_B, *vy = vb + m, *vz = vy + m, *chk = vz + m;
    if (m > 0)
      hipLaunchKernelGGL(k_block_inv, dim3(1), dim3(GJ_T), 0, cs, m, (int)std::min<int64_t>(BGJ_B, m), M, P,
                         L->d_gjflag);
    const unsigned panels = (unsigned)((m + GJ_PC - 1) / GJ_PC);
    const unsigned tiles = (unsigned)(((m + 4 * GJ_W - 1) / (4 * GJ_W)) * ((m + 2 * GJ_W - 1) / (2 * GJ_W)));
    for (int64_t k0 = 0; k0 < m; k0 += BGJ_B) {
      const int kb = (int)std::min<int64_t>(BGJ_B, m - k0);
      const int kd = (int)std::max<int64_t>(0, std::min<int64_t>(BGJ_B, m - k0 - BGJ_B));
      hipLaunchKernelGGL(k_gj_panel, dim3(panels), dim3(GJ_T), 0, cs, m, k0, kb, kd, M, P, C, R, D);
      hipLaunchKernelGGL(k_gj_update, dim3(tiles + 1), dim3(GJ_T), 0, cs, m, k0, kb, kd, C, R, D, P, L->d_gjflag, M);
    }
    MHD_HIP(hipGetLastError());
    // check: z = A (A^-1 b) against b for a fixed b
    hipLaunchKernelGGL(k_check_rhs, dim3(nblocks(m)), dim3(TB), 0, cs, m, vb);
    hipLaunchKernelGGL((k_dense_rowdot<double>), dim3((unsigned)m), dim3(TB), 0, cs, m, M, vb,
                       (const int32_t *)nullptr, vy, (double *)nullptr);
    hipLaunchKernelGGL((k_dense_rowdot<double>), dim3((unsigned)m), dim3(TB), 0, cs, m, L->d_LU, vy,
                       (const int32_t *)nullptr, vz, (double *)nullptr);
    hipLaunchKernelGGL(k_check_residual, dim3(1), dim3(1024), 0, cs, m, vz, vb, chk);
    MHD_HIP(hipGetLastError());
    double hchk[2] = {0.0, 1.0};
    int32_t flag = 0;
    MHD_HIP(hipMemcpyAsync(hchk, chk, sizeof(hchk), hipMemcpyDeviceToHost, cs));
    MHD_HIP(hipMemcpyAsync(&flag, L->d_gjflag, sizeof(int32_t), hipMemcpyDeviceToHost, cs));
    MHD_HIP(hipStreamSynchronize(cs));
    count(c, OP_SETUP_DENSE3, (double)L->n1c * L->n1c * L->n1c);
    if (flag || !(hchk[0] <= 1e-6 * hchk[1])) {
      // redo with the row-pivoted LU: getrf of A^T (the row-major copy), then
      // A^T X = I gives X = A^-T column-major = A^-1 row-major
      ++L->dense_fallbacks;
      count(c, OP_SETUP_DENSE3, (double)L->n1c * L->n1c * L->n1c);  // a second inversion
      MHD_HIP(hipMemsetAsync(M, 0, sizeof(double) * (size_t)(m * m), cs));
      hipLaunchKernelGGL(k_set_diag, dim3(nblocks(m)), dim3(TB), 0, cs, m, 1.0, M);
      MHD_HIP(hipGetLastError());
      if (!SC->rb) {
        if (rocblas_create_handle(&SC->rb) != rocblas_status_success) {
          SC->rb = nullptr;
          c->err = "rocblas_create_handle failed";
          return -2;
        }
        rocblas_set_stream(SC->rb, cs);
        // the same bits in every run: no atomics inside rocSOLVER routines
        rocblas_set_atomics_mode(SC->rb, rocblas_atomics_not_allowed);
      }
      rocblas_handle rb = SC->rb;
      if (rocsolver_dgetrf(rb, (rocblas_int)m, (rocblas_int)m, L->d_LU, (rocblas_int)m, L->d_piv, L->d_info) !=
              rocblas_status_success ||
          rocsolver_dgetrs(rb, rocblas_operation_none, (rocblas_int)m, (rocblas_int)m, L->d_LU, (rocblas_int)m,
                           L->d_piv, M, (rocblas_int)m) != rocblas_status_success) {
        c->err = "rocsolver LU of the coarsest level failed";
        return -2;
      }
      int32_t info = 0;
      MHD_HIP(hipMemcpyAsync(&info, L->d_info, sizeof(int32_t), hipMemcpyDeviceToHost, cs));
      MHD_HIP(hipStreamSynchronize(cs));
      if (info != 0) {
        c->err = "coarsest [u,j] block is singular (getrf info " + std::to_string(info) + ")";
        return -3;
      }
    }
  }
  return 0;
}

// Right-preconditioned restarted FGMRES (FP64) for J dx = b, dx = 0 on entry.
int fgmres(mhd_ctx *c, const double *b, double *x, double tol, int maxit, int prec, int *iters, int verbose,
           double *final_res = nullptr) {
  Solver *S = c->solver;
  const int64_t n = S->n;
  const int m = S->m;
  int rc, it = 0;
  std::vector<double> H((m + 1) * m), h(m + 1), y, cs(m), sn(m), g(m + 1);
  hipLaunchKernelGGL((k_fill<double>), dim3(nblocks(n)), dim3(TB), 0, c->stream, n, 0.0, x);
  // r = b (x = 0)
  MHD_HIP(hipMemcpyAsync(S->w, b, sizeof(double) * n, hipMemcpyDeviceToDevice, c->stream));
  double beta;
  if ((rc = vnorm(c, S->w, n, &beta))) return rc;
  const double b0 = beta;
  while (it < maxit && beta > tol) {
    hipLaunchKernelGGL((k_scale_copy<double>), dim3(nblocks(n)), dim3(TB), 0, c->stream, n, 1.0 / beta, S->w, S->V);
    std::fill(H.begin(), H.end(), 0.0);
    std::fill(g.begin(), g.end(), 0.0);
    g[0] = beta;
    int k = 0;
    double est = beta;
    for (int j = 0; j < m && it < maxit; ++j) {
      if ((rc = precond(c, S->V + j * n, S->Z + j * n, prec))) return rc;
      if ((rc = full_product(c, S->Z + j * n, S->w))) return rc;
      count(c, OP_OUTER, 1.0);
      double nrm;
      if ((rc = arnoldi<double>(c, S->V, n, j + 1, S->w, n, h.data(), &nrm))) return rc;
      for (int i = 0; i <= j; ++i) H[i * m + j] = h[i];
      H[(j + 1) * m + j] = nrm;
      // incremental Givens for the residual estimate
      for (int i = 0; i < j; ++i) {
        const double a = H[i * m + j], bb = H[(i + 1) * m + j];
        H[i * m + j] = cs[i] * a + sn[i] * bb;
        H[(i + 1) * m + j] = -sn[i] * a + cs[i] * bb;
      }
      const double a = H[j * m + j], bb = H[(j + 1) * m + j];
      const double d = std::hypot(a, bb);
      cs[j] = d > 0 ? a / d : 1.0;
      sn[j] = d > 0 ? bb / d : 0.0;
      H[j * m + j] = d;
      H[(j + 1) * m + j] = 0.0;
      g[j + 1] = -sn[j] * g[j];
      g[j] = cs[j] * g[j];
      est = std::fabs(g[j + 1]);
      ++it;
      k = j + 1;
      if (verbose > 1) fprintf(stderr, "    fgmres it %d  est %.3e\n", it, est / b0);
      if (est <= tol || nrm <= 1e-300) break;
    }
    // back substitution on the rotated (upper triangular) H
    y.assign(k, 0.0);
    for (int i = k - 1; i >= 0; --i) {
      double s = g[i];
      for (int j = i + 1; j < k; ++j) s -= H[i * m + j] * y[j];
      y[i] = s / H[i * m + i];
    }
    MHD_HIP(hipMemcpyAsync(S->d_y, y.data(), sizeof(double) * k, hipMemcpyHostToDevice, c->stream));
    hipLaunchKernelGGL((k_lincomb<double>), dim3(nblocks(n)), dim3(TB), sizeof(double) * k, c->stream, k, S->Z, n,
                       S->d_y, 1.0, x, n);
    MHD_HIP(hipGetLastError());
    // true residual for the restart: w = b - J x
    if ((rc = full_product(c, x, S->w))) return rc;
    count(c, OP_VEC, (k + 2.0) * n * sizeof(double));
    hipLaunchKernelGGL((k_scale_copy<double>), dim3(nblocks(n)), dim3(TB), 0, c->stream, n, -1.0, S->w, S->w);
    hipLaunchKernelGGL((k_axpy<double>), dim3(nblocks(n)), dim3(TB), 0, c->stream, n, 1.0, b, S->w);
    MHD_HIP(hipGetLastError());
    if ((rc = vnorm(c, S->w, n, &beta))) return rc;
    if (verbose) fprintf(stderr, "  fgmres restart: it %d  true rel res %.3e\n", it, beta / b0);
    if (k == 0) break;
  }
  *iters = it;
  if (final_res) *final_res = beta;
  return beta <= tol ? 0 : 1;
}

double now() { return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count(); }

}  // namespace

void mhd_solver_free(mhd_ctx *c) {
  if (!c || !c->solver) return;
  Solver *S = c->solver;
  void *ptrs[] = {S->d_split, S->d_pfirst, S->d_phifirst, S->d_Sp, S->d_Sphi, S->d_psize, S->d_pidx, S->d_pA,
                  S->d_pA32, S->d_pA16, S->d_pAh, S->d_pscale, S->d_pperm, S->d_pstatus, S->d_pscratch, S->d_val32, S->V, S->Z, S->w, S->b, S->dx, S->t1,
                  S->V1, S->Z1, S->w1, S->x1, S->r1, S->d_part, S->d_dots, S->d_y, S->d_dptr, S->d_dent,
                  S->d_ppart, S->d_grow, S->d_gcp, S->d_gcol, S->d_pcptr, S->d_pcell, S->d_ifirst, S->d_npat, S->d_elim,
                  S->d_cE64, S->d_cB64, S->d_cF64, S->d_cG64, S->d_cE32, S->d_cF32, S->d_cG32, S->d_cflag, S->d_rt, S->d_prod};
  for (void *p : ptrs)
    if (p) (void)hipFree(p);
  if (S->h_dots) (void)hipHostFree(S->h_dots);
  if (S->rb) rocblas_destroy_handle(S->rb);
  delete S;
  c->solver = nullptr;
}

void mhd_coarse_free(mhd_ctx *c) {
  if (!c || !c->coarse) return;
  CoarseLink *L = c->coarse;
  void *ptrs[] = {L->d_Prow, L->d_Trow, L->d_Pcol, L->d_Tcol, L->d_Pval, L->d_Tval, L->d_Pval32, L->d_Tval32,
                  L->d_Rrow, L->d_Rcol, L->d_Rval, L->rr, L->rc, L->ec, L->d_ab};
  for (void *q : ptrs)
    if (q) (void)hipFree(q);
  dense_free(L);
  if (L->ctx) mhd_destroy(L->ctx);
  delete L;
  c->coarse = nullptr;
}

extern "C" {

int mhd_attach_coarse(mhd_ctx *c, mhd_ctx *coarse, int64_t nrows, int64_t ncols, const int64_t *P_rowptr,
                      const int32_t *P_col, const double *P_val, const int64_t *R_rowptr, const int32_t *R_col,
                      const double *R_val, int32_t coarse_iters, double smoother_weight, int32_t coarse_step) {
  if (coarse_step != 0 && coarse_step != 1) {
    if (c) c->err = "mhd_attach_coarse: coarse_step must be 0 (full) or 1 (minimal residual)";
    return -1;
  }
  if (!(smoother_weight > 0.0 && smoother_weight <= 1.0)) {
    if (c) c->err = "mhd_attach_coarse: smoother_weight must be in (0, 1]";
    return -1;
  }
  if (!c || !coarse || !P_rowptr || !P_col || !P_val || !R_rowptr || !R_col || !R_val) return -1;
  if (c->coarse) {
    c->err = "a coarse level is already attached";
    return -1;
  }
  const int64_t n1 = (int64_t)c->nfree[0] + c->nfree[2];
  const int64_t n1c = (int64_t)coarse->nfree[0] + coarse->nfree[2];
  if (nrows != n1 || ncols != n1c || coarse->device != c->device || coarse->block_style != 1) {
    c->err = "mhd_attach_coarse: P must be (nfree[u]+nfree[j]) fine x coarse, same device, block numbering";
    return -1;
  }
  const int64_t nnzP = P_rowptr[nrows];
  for (int64_t k = 0; k < nnzP; ++k)
    if (P_col[k] < 0 || P_col[k] >= ncols) {
      c->err = "mhd_attach_coarse: P column out of range";
      return -1;
    }
  const int64_t nnzR = R_rowptr[coarse->nfree[0]];
  for (int64_t k = 0; k < nnzR; ++k)
    if (R_col[k] < 0 || R_col[k] >= c->nfree[0]) {
      c->err = "mhd_attach_coarse: state interpolation column out of range";
      return -1;
    }
  MHD_HIP(hipSetDevice(c->device));
  CoarseLink *L = new CoarseLink();
  L->n1 = n1;
  L->n1c = n1c;
  L->nuc = coarse->nfree[0];
  L->nnzP = nnzP;
  L->coarse_iters = coarse_iters <= 0 ? 0 : std::min(coarse_iters, 120);
  if (L->coarse_iters == 0 && !coarse->coarse && n1c > 32768) {
    c->err = "mhd_attach_coarse: coarse_iters = 0 (dense coarsest solve) needs at most 32768 [u,j] dofs there";
    delete L;
    return -1;
  }
  L->omega = smoother_weight;
  L->step_mode = coarse_step;
  // transpose on the host
  std::vector<int64_t> trow(ncols + 1, 0);
  for (int64_t k = 0; k < nnzP; ++k) trow[P_col[k] + 1]++;
  for (int64_t i = 0; i < ncols; ++i) trow[i + 1] += trow[i];
  std::vector<int32_t> tcol(nnzP);
  std::vector<double> tval(nnzP);
  {
    std::vector<int64_t> fill(trow.begin(), trow.end() - 1);
    for (int64_t i = 0; i < nrows; ++i)
      for (int64_t k = P_rowptr[i]; k < P_rowptr[i + 1]; ++k) {
        const int64_t q = fill[P_col[k]]++;
        tcol[q] = (int32_t)i;
        tval[q] = P_val[k];
      }
  }
  std::vector<float> pv32(P_val, P_val + nnzP), tv32(tval.begin(), tval.end());
  auto up = [&](void **dst, const void *src, size_t bytes) -> int {
    MHD_HIP(hipMalloc(dst, std::max<size_t>(bytes, 8)));
    if (bytes) MHD_HIP(hipMemcpy(*dst, src, bytes, hipMemcpyHostToDevice));
    return 0;
  };
  int rc = 0;
  if (!rc) rc = up((void **)&L->d_Prow, P_rowptr, sizeof(int64_t) * (nrows + 1));
  if (!rc) rc = up((void **)&L->d_Pcol, P_col, sizeof(int32_t) * nnzP);
  if (!rc) rc = up((void **)&L->d_Pval, P_val, sizeof(double) * nnzP);
  if (!rc) rc = up((void **)&L->d_Pval32, pv32.data(), sizeof(float) * nnzP);
  if (!rc) rc = up((void **)&L->d_Trow, trow.data(), sizeof(int64_t) * (ncols + 1));
  if (!rc) rc = up((void **)&L->d_Tcol, tcol.data(), sizeof(int32_t) * nnzP);
  if (!rc) rc = up((void **)&L->d_Tval, tval.data(), sizeof(double) * nnzP);
  if (!rc) rc = up((void **)&L->d_Tval32, tv32.data(), sizeof(float) * nnzP);
  if (!rc) rc = up((void **)&L->d_Rrow, R_rowptr, sizeof(int64_t) * (L->nuc + 1));
  if (!rc) rc = up((void **)&L->d_Rcol, R_col, sizeof(int32_t) * nnzR);
  if (!rc) rc = up((void **)&L->d_Rval, R_val, sizeof(double) * nnzR);
  L->ctx = coarse;
  c->coarse = L;
  if (rc) return rc;
  // the coarse level runs on the fine level's stream
  MHD_HIP(hipStreamSynchronize(coarse->stream));
  if (coarse->own_stream) MHD_HIP(hipStreamDestroy(coarse->stream));
  coarse->stream = c->stream;
  coarse->own_stream = false;
  if (coarse->coarse) {  // re-point the whole chain
    for (mhd_ctx *q = coarse->coarse->ctx; q; q = q->coarse ? q->coarse->ctx : nullptr) q->stream = c->stream;
  }
  if (c->solver) mhd_solver_free(c);  // re-initialised with the chain on the next solve
  return 0;
}

int mhd_op_counts(mhd_ctx *c, double *out, int reset) {
  if (!c || !out) return -1;
  for (int k = 0; k < MHD_NOPS; ++k) out[k] = 0.0;
  for (mhd_ctx *q = c; q; q = q->coarse ? q->coarse->ctx : nullptr) {
    if (!q->solver) continue;
    for (int k = 0; k < MHD_NOPS; ++k) {
      out[k] += q->solver->ops[k];
      if (reset) q->solver->ops[k] = 0.0;
    }
  }
  return 0;
}

void mhd_default_solver_opts(mhd_solver_opts *o) {
  std::memset(o, 0, sizeof(*o));
  o->max_newton = 20;
  o->restart = 40;
  o->max_krylov = 400;
  o->precision = 0;
  o->rtol = 1e-6;
  o->atol = 1e-8;
  o->ls_rtol = 1e-7;
  o->inner_iters = 8;
}

int mhd_precond_setup(mhd_ctx *c, const mhd_solver_opts *o) {
  if (!c || !o) return -1;
  if (o->precision < 0 || o->precision > 3) {
    c->err = "precision must be 0, 1, 2 or 3";
    return -1;
  }
  if (!c->jac_valid) {
    c->err = "mhd_precond_setup needs a Jacobian assembled into the context (mhd_jacobian, a solve, or "
             "mhd_jacobian_d with d_nzval_csr = NULL)";
    return -1;
  }
  MHD_HIP(hipSetDevice(c->device));
  int rc;
  if (c->solver && (c->solver->m != krylov_dim(o->restart) ||
                    c->solver->kin != std::max(0, std::min(o->inner_iters, 120))))
    mhd_solver_free(c);
  if ((rc = solver_init(c, o, may_condense(c)))) return rc;
  if ((rc = precond_setup(c, o->precision, c->d_x))) return rc;
  MHD_HIP(hipStreamSynchronize(c->stream));
  return 0;
}

int mhd_smoother_apply_d(mhd_ctx *c, const void *d_r, void *d_y, void *stream) {
  if (!c || !d_r || !d_y) return -1;
  if (!c->solver || c->solver->inner_prec < 0) {
    c->err = "mhd_smoother_apply_d needs mhd_precond_setup first";
    return -1;
  }
  MHD_HIP(hipSetDevice(c->device));
  Solver *S = c->solver;
  hipStream_t s = stream ? (hipStream_t)stream : c->stream;
  if (S->inner_prec == 0) return patch_as_on<double>(c, (const double *)d_r, (double *)d_y, 0, 1.0, true, s);
  return patch_as_on<float>(c, (const float *)d_r, (float *)d_y, S->inner_prec, 1.0, true, s);
}

int mhd_set_pivot_threshold(mhd_ctx *c, double tau) {
  if (!c) return -1;
  if (!(tau >= 0.0 && tau <= 1.0)) {
    c->err = "pivot threshold must lie in [0, 1]";
    return -1;
  }
  c->pivot_tau = tau;
  for (mhd_ctx *q = c->coarse ? c->coarse->ctx : nullptr; q; q = q->coarse ? q->coarse->ctx : nullptr)
    q->pivot_tau = tau;
  return 0;
}

int mhd_smoother_info(mhd_ctx *c, int64_t *npatch, int64_t *patch_dim, int64_t *patch_entries,
                      int64_t *npivoted) {
  if (!c || !c->solver) return -1;
  if (npivoted) *npivoted = c->solver->nflagged;
  if (npatch) *npatch = c->solver->npatch;
  if (patch_dim) *patch_dim = c->solver->PS_all;
  if (patch_entries) *patch_entries = c->solver->pent_all;
  return 0;
}

int mhd_dresidual_dparam(mhd_ctx *c, const double *x_free, int32_t param, double *out) {
  if (!c || !x_free || !out) return -1;
  if (param != 0 && param != 1) {
    c->err = "mhd_dresidual_dparam: param must be 0 (gamma) or 1 (cw)";
    return -1;
  }
  MHD_HIP(hipSetDevice(c->device));
  MHD_HIP(hipMemcpyAsync(c->d_x, x_free, sizeof(double) * c->n, hipMemcpyHostToDevice, c->stream));
  int rc = mhd_launch_residual_mode(c, c->d_x, c->d_r, c->stream, param == 0 ? 1 : 2);
  if (rc) return rc;
  MHD_HIP(hipMemcpyAsync(out, c->d_r, sizeof(double) * c->n, hipMemcpyDeviceToHost, c->stream));
  MHD_HIP(hipStreamSynchronize(c->stream));
  return 0;
}

namespace {

// x = A(x_state)^-1 rhs, or A^-T rhs.  A^T has the saddle-point block
// structure of A (its (uj, p) block is A's (p, uj) block transposed, which is
// A's (uj, p) block again; likewise sigma times the (j, phi) block), so the
// adjoint uses Badia2024's upper block-triangular preconditioner built on A^T
// itself, every level of a V-cycle hierarchy on its transposed Jacobian.  (The
// exact transpose of the forward preconditioner, lower block-triangular,
// stalls with an inexact [u,j] solve on any right-hand side with pressure or
// potential components: measured from 16 x 16 x 8 up.)  Solver workspaces are
// rebuilt by the next solve.
int linear_solve(mhd_ctx *c, const double *x_state, const double *rhs, double *lambda,
                 const mhd_solver_opts *o, mhd_solve_info *info, bool transpose) {
  if (!c || !x_state || !rhs || !lambda || !o || !info) return -1;
  std::memset(info, 0, sizeof(*info));
  if (o->precision < 0 || o->precision > 3) {
    c->err = "precision must be 0, 1, 2 or 3";
    return -1;
  }
  MHD_HIP(hipSetDevice(c->device));
  int rc;
  // every level of an attached V-cycle hierarchy works on its transposed
  // Jacobian for the duration (the transfers P, P^T are unchanged)
  if (c->solver) mhd_solver_free(c);
  rc = solver_init(c, o, may_condense(c));
  if (rc) return rc;
  Solver *S = c->solver;
  const int64_t n = c->n;
  double *d_valT = nullptr;
  auto finish = [&](int code) {
    if (d_valT) {
      std::swap(c->d_val, d_valT);
      (void)hipFree(d_valT);
    }
    // the solvers (and the coarse levels' transposed values) are rebuilt by the next solve
    mhd_solver_free(c);
    for (mhd_ctx *q = c->coarse ? c->coarse->ctx : nullptr; q; q = q->coarse ? q->coarse->ctx : nullptr)
      if (q->solver) q->solver->transposed = false;
    return code;
  };
  MHD_HIP(hipMemcpyAsync(c->d_x, x_state, sizeof(double) * n, hipMemcpyHostToDevice, c->stream));
  double t = now();
  if ((rc = mhd_assemble_own(c, c->stream))) return finish(rc);
  if (transpose && hipMalloc(&d_valT, sizeof(double) * std::max<int64_t>(c->nnz, 1)) != hipSuccess) {
    c->err = "out of device memory for A^T";
    d_valT = nullptr;
    return finish(-2);
  }
  const int64_t nu = c->nfree[0], n1 = (int64_t)c->nfree[0] + c->nfree[2], np = c->nfree[1];
  const double sc = adjoint_scale(c);
  if (transpose) {
    if ((rc = mhd_launch_transpose_values(c, c->d_val, d_valT, c->stream))) return finish(rc);
    std::swap(c->d_val, d_valT);  // the solver now sees A^T; d_valT holds A
    hipLaunchKernelGGL(k_adj_scale, dim3(nblocks(n)), dim3(TB), 0, c->stream, n, c->d_rowptr, c->d_colind, c->d_val,
                       nu, n1, np, sc);
    MHD_HIP(hipGetLastError());
  }
  MHD_HIP(hipStreamSynchronize(c->stream));
  info->t_jacobian = now() - t;
  t = now();
  S->transposed = transpose;
  if ((rc = precond_setup(c, o->precision, c->d_x))) return finish(rc);
  MHD_HIP(hipStreamSynchronize(c->stream));
  info->t_setup = now() - t;
  t = now();
  MHD_HIP(hipMemcpyAsync(S->b, rhs, sizeof(double) * n, hipMemcpyHostToDevice, c->stream));
  if (transpose)  // (D^-1 A^T D) mu = D^-1 rhs, lambda = D mu
    hipLaunchKernelGGL(k_adj_scale_vec, dim3(nblocks(n)), dim3(TB), 0, c->stream, n, nu, n1, np, 1.0 / sc, S->b);
  double bn;
  if ((rc = vnorm(c, S->b, n, &bn))) return finish(rc);
  int kits = 0;
  double rfin = 0.0;
  rc = fgmres(c, S->b, S->dx, o->ls_rtol * bn, o->max_krylov, o->precision, &kits, o->verbose, &rfin);
  if (rc < 0) return finish(rc);
  info->residual = rfin;
  if (transpose)
    hipLaunchKernelGGL(k_adj_scale_vec, dim3(nblocks(n)), dim3(TB), 0, c->stream, n, nu, n1, np, sc, S->dx);
  MHD_HIP(hipGetLastError());
  MHD_HIP(hipMemcpyAsync(lambda, S->dx, sizeof(double) * n, hipMemcpyDeviceToHost, c->stream));
  MHD_HIP(hipStreamSynchronize(c->stream));
  info->t_solve = now() - t;
  info->krylov_iters = kits;
  info->converged = rc == 0;
  info->residual0 = bn;
  return finish(rc);
}

}  // namespace

int mhd_adjoint_solve(mhd_ctx *c, const double *x_state, const double *rhs, double *lambda,
                      const mhd_solver_opts *o, mhd_solve_info *info) {
  return linear_solve(c, x_state, rhs, lambda, o, info, true);
}

int mhd_linear_solve(mhd_ctx *c, const double *x_state, const double *rhs, double *sol, const mhd_solver_opts *o,
                     mhd_solve_info *info) {
  return linear_solve(c, x_state, rhs, sol, o, info, false);
}

int mhd_newton_solve(mhd_ctx *c, double *x_host, const mhd_solver_opts *o, mhd_solve_info *info) {
  if (!c || !x_host || !o || !info) return -1;
  std::memset(info, 0, sizeof(*info));
  if (o->precision < 0 || o->precision > 3) {
    c->err = "precision must be 0 (FP64), 1 (FP32 inner, FP32 patches), 2 (FP32 inner, BF16 patches) or 3 (FP32 "
             "inner, FP16 patches scaled per patch)";
    return -1;
  }
  MHD_HIP(hipSetDevice(c->device));
  int rc;
  double t0 = now();
  if ((rc = solver_init(c, o, may_condense(c)))) return rc;
  Solver *S = c->solver;
  if (S->m != krylov_dim(o->restart) || S->kin != std::max(0, std::min(o->inner_iters, 120))) {
    mhd_solver_free(c);
    if ((rc = solver_init(c, o, may_condense(c)))) return rc;
    S = c->solver;
  }
  info->t_setup += now() - t0;
  const int64_t n = c->n;
  MHD_HIP(hipMemcpyAsync(c->d_x, x_host, sizeof(double) * n, hipMemcpyHostToDevice, c->stream));
  double t = now();
  if ((rc = mhd_launch_residual(c, c->d_x, c->d_r, c->stream))) return rc;
  double r0;
  if ((rc = vnorm(c, c->d_r, n, &r0))) return rc;
  info->t_residual += now() - t;
  info->residual0 = r0;
  info->newton_residuals[0] = r0;
  double rn = r0;
  int it = 0;
  int lin_fail = 0;
  while (it < o->max_newton) {
    if (rn <= std::max(o->atol, o->rtol * r0)) break;
    t = now();
    if ((rc = mhd_assemble_own(c, c->stream))) return rc;
    MHD_HIP(hipStreamSynchronize(c->stream));
    info->t_jacobian += now() - t;
    t = now();
    if ((rc = precond_setup(c, o->precision, c->d_x))) return rc;
    MHD_HIP(hipStreamSynchronize(c->stream));
    info->t_setup += now() - t;
    t = now();
    // b = -r
    hipLaunchKernelGGL((k_scale_copy<double>), dim3(nblocks(n)), dim3(TB), 0, c->stream, n, -1.0, c->d_r, S->b);
    int kits = 0;
    // linear tolerance: ls_rtol relative to this step's residual, but never
    // below half the Newton target (the FP64 residual floor lies near 1e-11
    // relative; solving past the target only stalls there)
    const double lin_tol = std::max(o->ls_rtol * rn, 0.5 * std::max(o->atol, o->rtol * r0));
    rc = fgmres(c, S->b, S->dx, lin_tol, o->max_krylov, o->precision, &kits, o->verbose);
    if (rc < 0) return rc;
    if (rc > 0) lin_fail = 1;
    hipLaunchKernelGGL((k_axpy<double>), dim3(nblocks(n)), dim3(TB), 0, c->stream, n, 1.0, S->dx, c->d_x);
    MHD_HIP(hipStreamSynchronize(c->stream));
    info->t_solve += now() - t;
    if (it < 64) info->krylov_per_step[it] = kits;
    info->krylov_iters += kits;
    ++it;
    t = now();
    if ((rc = mhd_launch_residual(c, c->d_x, c->d_r, c->stream))) return rc;
    if ((rc = vnorm(c, c->d_r, n, &rn))) return rc;
    info->t_residual += now() - t;
    if (it < 64) info->newton_residuals[it] = rn;
    if (o->verbose) fprintf(stderr, "newton %d  |R| = %.6e  krylov %d\n", it, rn, kits);
  }
  MHD_HIP(hipMemcpyAsync(x_host, c->d_x, sizeof(double) * n, hipMemcpyDeviceToHost, c->stream));
  MHD_HIP(hipStreamSynchronize(c->stream));
  info->newton_iters = it;
  info->residual = rn;
  info->converged = rn <= std::max(o->atol, o->rtol * r0);
  info->flags = lin_fail;
  return info->converged ? 0 : 1;
}

}  // extern "C"

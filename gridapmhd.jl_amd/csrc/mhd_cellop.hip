// The weak form applied cell by cell, without the matrix: the residual
// (src/weakforms.jl:255-312 and the thin-wall terms :721-726) and the products
// with the Jacobian, its [u,j] block, its (u,j) x (p,phi) block, and their
// transposes.
//
// Half a wave (32 lanes) per cell, two cells per 64-thread workgroup (one wave:
// its barriers cost nothing).  The cell's 129 input values go to LDS; the
// fields at the 27 quadrature points come from them by sum factorisation, one
// axis per pass: lane (d0, d1, d2) owns row d0 + 3 d1 + 9 d2 of the cell's
// buffer, and its digits turn from node to point indices axis by axis, in
// place.  There the lane is a quadrature point: it maps to physical
// coordinates, forms the fluxes of the weak form and pulls them back to the
// reference cell (17 numbers).  Three passes back contract them with the test
// functions, until the lane is a Q2 node and up to three RT1 dofs and a dQ1
// vertex.  About 550 FMAs and 310 LDS accesses per lane; evaluating every point
// from all nodal values directly took 1,300 and 610.  Element results go to a
// buffer [cell][129] and a second kernel adds them per dof in increasing cell
// order: no atomics, the same bits in every run.
//
// Residual at 64 x 64 x 8 (32,768 cells): 2.31 -> 0.132 ms (cell kernel 0.105,
// sums 0.025), at 8 x 8 x 3: 53 -> 14 us (10 + 4); an A11 product on 8,192 cells:
// 132 us streamed in FP32 -> 22 + 7 us on average over the V-cycle's levels.  Bound by
// latency at two waves per SIMD (200 VGPRs): direct evaluation took 0.136 ms,
// and a register budget for three waves spills and is slower (0.112 ms).
#include <algorithm>

#include "mhd_cell.h"

using namespace mhd;

namespace {

// Slot of local dof l in a cell's 129 element results: the three components of
// a velocity node side by side, as their dofs are, then j, p, phi.
constexpr int SLOT_J = NU, SLOT_P = NU + NJ, SLOT_PHI = NU + NJ + NP;

constexpr int ROW = 18;  // doubles per row of the cell's buffer
struct CellIn {
  double x[NDOF + 1];    // input values, RT1 face dofs times their orientation
  double xyz[24];
  double minv[16];       // inverse dP1 mass matrix (augmented-Lagrangian term)
  double sg[6];
  double dq[4];          // int psi_k div u
  double wd[NQ + 1];     // W div u at the points
  double fl[NQ][ROW];    // pass results; fluxes 3 x (S_k, T_0k, T_1k, T_2k), (v_0, v_1, v_2, c), W div j
};

// factors of the test functions with index i along one axis at the three points
struct TestAxis {
  double b[3], d[3], g[3], l[3];
  __device__ explicit TestAxis(int i) {
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      b[q] = q2_val(i, q);
      d[q] = q2_der(i, q);
      g[q] = g2_val(i, q);
      l[q] = i ? GX[q] : 1.0 - GX[q];
    }
  }
};

// OP_RES: residual at x.  OP_FULL: A dx.  OP_UJ: the [u,j] block.  OP_PPHI: the
// (u,j) rows' products with the p and phi parts.  TRANS: the same of A^T.
enum { OP_RES = 0, OP_FULL = 1, OP_UJ = 2, OP_PPHI = 3 };

struct CellOpArgs {
  int ncells;
  int64_t n, nu, n1, n1p;        // free dofs; ends of the u, [u,j] and p parts of the block numbering (scale)
  const double *xyz, *dir, *minv, *state;
  const int32_t *dofs;
  const int8_t *sign;
  const int32_t *cfptr, *cface;  // thin-wall faces of every cell
  const int8_t *flf;
  const double *fK, *fc;         // [nfaces][4][36] face matrices, [nfaces][4] constant parts
  double *out;                   // [ncells][129]
  double scale;                  // input j and phi dofs times this (adjoint scaling; 1: none)
  int mode;                      // OP_RES: 0 residual, 1 dR/dgamma
};

template <int OP, bool TRANS, class T>
__global__ __launch_bounds__(64) void k_cell_op(CellOpArgs A, MhdPhys ph, const T *__restrict__ x) {
  constexpr bool RES = OP == OP_RES, UJ = OP != OP_PPHI, PPHI = OP != OP_UJ, ROWS2 = OP == OP_RES || OP == OP_FULL;
  __shared__ CellIn sh[2];
  const int half = threadIdx.x >> 5, hl = threadIdx.x & 31;
  const int c = blockIdx.x * 2 + half;
  const bool live = c < A.ncells;
  CellIn &S = sh[half];
  constexpr bool LIN = OP == OP_FULL || OP == OP_UJ;
  double st[12];  // state at the lane's point, on its way during the passes
  int e0 = 0, e1 = 0;
  if (live) {
    if (LIN && ph.convection) {
      const double *sp = A.state + (int64_t)c * 12 * NQ + (hl < NQ ? hl : NQ - 1);
#pragma unroll
      for (int k = 0; k < 12; ++k) st[k] = k < 3 || ph.convection == 2 ? sp[k * NQ] : 0.0;
    }
    if (UJ) {
      e0 = A.cfptr[c];
      e1 = A.cfptr[c + 1];
    }
    const int32_t *cd = A.dofs + (int64_t)c * NDOF;
    if (hl < 24) S.xyz[hl] = A.xyz[(int64_t)c * 24 + hl];
    if (hl < 16) S.minv[hl] = A.minv[(int64_t)c * 16 + hl];
    if (hl < 6) S.sg[hl] = A.sign ? (double)A.sign[(int64_t)c * 6 + hl] : 1.0;
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      const int l = hl + 32 * k;
      if (l >= NDOF) break;
      const bool uj = l < OFF_P || (l >= OFF_J && l < OFF_PHI);
      if (!(uj ? UJ : PPHI)) continue;
      const int32_t g = cd[l];
      double v = 0.0;
      if (g >= 0) {
        v = (double)x[g];
        if (TRANS && l >= OFF_J) v *= A.scale;
      } else if (RES) {
        v = A.dir[-(int64_t)g - 1];
      }
      if (l >= OFF_J && l < OFF_J + 24 && A.sign) v *= (double)A.sign[(int64_t)c * 6 + ((l - OFF_J) >> 2)];
      S.x[l] = v;
    }
  }
  __syncthreads();
  const int q = hl < NQ ? hl : NQ - 1;  // lanes 27..31 repeat the last row and write nothing
  const int d[3] = {q % 3, (q / 3) % 3, q / 9};
  const bool wr = hl < NQ;
  const double px = gauss_x(d[0]), py = gauss_x(d[1]), pz = gauss_x(d[2]);
  double J[9], Ji[9], W = 0.0, id = 0.0;
  double u[3] = {0, 0, 0}, gu[9], j[3] = {0, 0, 0}, dj = 0.0, p = 0.0, phi = 0.0, divu = 0.0;
  double fw[3][4], V[3], dv = 0.0;
  if (UJ)  // every lane takes part (the passes hold barriers); a dead half works on its own unused buffer
    fields_forward<true>(S.x, S.x + OFF_J, &S.fl[0][0], ROW, d, wr, fw, V, dv);
  if (live) {
    tri_jacobian(S.xyz, px, py, pz, J);
    const double det = inv3(J, Ji);
    id = 1.0 / det;
    W = gauss_w(d[0]) * gauss_w(d[1]) * gauss_w(d[2]) * fabs(det);
    if (UJ) {
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        u[k] = fw[k][0];
#pragma unroll
        for (int i = 0; i < 3; ++i) gu[3 * i + k] = Ji[i] * fw[k][1] + Ji[3 + i] * fw[k][2] + Ji[6 + i] * fw[k][3];
        j[k] = (J[3 * k] * V[0] + J[3 * k + 1] * V[1] + J[3 * k + 2] * V[2]) * id;
      }
      divu = gu[0] + gu[4] + gu[8];
      dj = dv * id;
    }
    if (PPHI) {
      const double *xp = S.x + OFF_P, *xf = S.x + OFF_PHI;
      p = xp[0] * (1.0 - px - py - pz) + xp[1] * px + xp[2] * py + xp[3] * pz;
      const double x0 = 1.0 - px, y0 = 1.0 - py;
      phi = (1.0 - pz) * (y0 * (x0 * xf[0] + px * xf[1]) + py * (x0 * xf[2] + px * xf[3])) +
            pz * (y0 * (x0 * xf[4] + px * xf[5]) + py * (x0 * xf[6] + px * xf[7]));
    }
    if (UJ && hl < NQ) S.wd[hl] = W * divu;
  }
  __syncthreads();
  // int psi_k div u, k < 4: lane k + 4 m adds the points m, m + 8, ..., then the
  // eight partial sums are added (the p rows, and the augmented-Lagrangian term)
  if (UJ && (ROWS2 || ph.zeta_u != 0.0)) {
    const int k = hl & 3;
    double s = 0.0;
    if (live)
      for (int m = hl >> 2; m < NQ; m += 8) {
        const double ax = gauss_x(m % 3), ay = gauss_x((m / 3) % 3), az = gauss_x(m / 9);
        s += S.wd[m] * (k == 0 ? 1.0 - ax - ay - az : (k == 1 ? ax : (k == 2 ? ay : az)));
      }
    s += __shfl_xor(s, 4, 32);
    s += __shfl_xor(s, 8, 32);
    s += __shfl_xor(s, 16, 32);
    if (hl < 4) S.dq[hl] = s;
    __syncthreads();
  }
  if (live) {
    const double B0 = ph.B[0], B1 = ph.B[1], B2 = ph.B[2];
    double Sk[3] = {0, 0, 0}, Tk[9], v[3] = {0, 0, 0}, cc = 0.0;
    double pr = PPHI ? -p : 0.0;  // isotropic part of T
    if (UJ && ph.zeta_u != 0.0) {
      double t = 0.0;
      const double ps[4] = {1.0 - px - py - pz, px, py, pz};
#pragma unroll
      for (int k = 0; k < 4; ++k)
        t += ps[k] * (S.minv[4 * k] * S.dq[0] + S.minv[4 * k + 1] * S.dq[1] + S.minv[4 * k + 2] * S.dq[2] +
                      S.minv[4 * k + 3] * S.dq[3]);
      pr += ph.zeta_u * t;
    }
#pragma unroll
    for (int e = 0; e < 9; ++e) Tk[e] = UJ ? ph.beta * gu[e] : 0.0;
    Tk[0] += pr;
    Tk[4] += pr;
    Tk[8] += pr;
    if (UJ) {
      if (ph.convection) {
        if (RES) {
#pragma unroll
          for (int k = 0; k < 3; ++k) Sk[k] = ph.alpha * (gu[k] * u[0] + gu[3 + k] * u[1] + gu[6 + k] * u[2]);
        } else {
          const double *us = st, *gs = st + 3;
          if (!TRANS) {  // alpha ((grad du)^T u0 [+ (grad u0)^T du])
#pragma unroll
            for (int k = 0; k < 3; ++k) {
              double t = gu[k] * us[0] + gu[3 + k] * us[1] + gu[6 + k] * us[2];
              if (ph.convection == 2) t += gs[k] * u[0] + gs[3 + k] * u[1] + gs[6 + k] * u[2];
              Sk[k] = ph.alpha * t;
            }
          } else {
#pragma unroll
            for (int i = 0; i < 3; ++i) {
              if (ph.convection == 2)
                Sk[i] = ph.alpha * (gs[3 * i] * u[0] + gs[3 * i + 1] * u[1] + gs[3 * i + 2] * u[2]);
#pragma unroll
              for (int k = 0; k < 3; ++k) Tk[3 * i + k] += ph.alpha * us[i] * u[k];
            }
          }
        }
      }
      // Lorentz force and u x B; transposed: -sigma B x j and -gamma B x u
      const double cl = TRANS ? -ph.sigma : ph.gamma, cu = TRANS ? -ph.gamma : ph.sigma;
      Sk[0] -= cl * (j[1] * B2 - j[2] * B1);
      Sk[1] -= cl * (j[2] * B0 - j[0] * B2);
      Sk[2] -= cl * (j[0] * B1 - j[1] * B0);
      v[0] = j[0] - cu * (u[1] * B2 - u[2] * B1);
      v[1] = j[1] - cu * (u[2] * B0 - u[0] * B2);
      v[2] = j[2] - cu * (u[0] * B1 - u[1] * B0);
      cc = ph.zeta_j * dj;
    }
    if (PPHI) cc -= TRANS ? phi : ph.sigma * phi;
    if (RES) {  // sources f = f0 + fx X, g = g0 + gx X
      double X[3];
      const double x0 = 1.0 - px, y0 = 1.0 - py;
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const double *Y = S.xyz + k;
        X[k] = (1.0 - pz) * (y0 * (x0 * Y[0] + px * Y[3]) + py * (x0 * Y[6] + px * Y[9])) +
               pz * (y0 * (x0 * Y[12] + px * Y[15]) + py * (x0 * Y[18] + px * Y[21]));
      }
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        Sk[k] -= ph.f0[k] + ph.fx[3 * k] * X[0] + ph.fx[3 * k + 1] * X[1] + ph.fx[3 * k + 2] * X[2];
        v[k] -= ph.g0[k] + ph.gx[3 * k] * X[0] + ph.gx[3 * k + 1] * X[1] + ph.gx[3 * k + 2] * X[2];
      }
      if (A.mode == 1) {  // dR/dgamma = -int (j x B).v
        Sk[0] = -(j[1] * B2 - j[2] * B1);
        Sk[1] = -(j[2] * B0 - j[0] * B2);
        Sk[2] = -(j[0] * B1 - j[1] * B0);
#pragma unroll
        for (int e = 0; e < 9; ++e) Tk[e] = 0.0;
        v[0] = v[1] = v[2] = cc = dj = 0.0;
      }
    }
    if (hl < NQ) {
      double *f = S.fl[hl];
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        f[4 * k] = W * Sk[k];
#pragma unroll
        for (int l = 0; l < 3; ++l)
          f[4 * k + 1 + l] = W * (Ji[3 * l] * Tk[k] + Ji[3 * l + 1] * Tk[3 + k] + Ji[3 * l + 2] * Tk[6 + k]);
      }
      const double wi = W * id;
#pragma unroll
      for (int l = 0; l < 3; ++l) f[12 + l] = wi * (J[l] * v[0] + J[3 + l] * v[1] + J[6 + l] * v[2]);
      f[15] = wi * cc;
      if (ROWS2) f[16] = W * dj;
    }
  }
  __syncthreads();
  // Test functions.  Along x: lane (node / dof index, qy, qz) reads its group's
  // three rows, all before any lane writes (one wave), then writes its own.
  double *fl = &S.fl[0][0], *own = fl + q * ROW;
  {
    const TestAxis tx(d[0]);
    const double *r = fl + (3 * d[1] + 9 * d[2]) * ROW;
    double s[9], w[5];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      s[3 * k] = dot3(tx.b, r + 4 * k, ROW) + dot3(tx.d, r + 4 * k + 1, ROW);
      s[3 * k + 1] = dot3(tx.b, r + 4 * k + 2, ROW);
      s[3 * k + 2] = dot3(tx.b, r + 4 * k + 3, ROW);
    }
    w[0] = dot3(tx.b, r + 12, ROW) + dot3(tx.d, r + 15, ROW);  // RT1 axis x: done with the normal direction
    w[1] = dot3(tx.g, r + 13, ROW);
    w[2] = dot3(tx.g, r + 14, ROW);
    w[3] = dot3(tx.g, r + 15, ROW);
    if (ROWS2) w[4] = dot3(tx.l, r + 16, ROW);
    __syncthreads();
    if (wr) {
#pragma unroll
      for (int k = 0; k < 9; ++k) own[k] = s[k];
#pragma unroll
      for (int k = 0; k < (ROWS2 ? 5 : 4); ++k) own[9 + k] = w[k];
    }
    __syncthreads();
  }
  {
    const TestAxis ty(d[1]);
    const double *r = fl + (d[0] + 9 * d[2]) * ROW;
    double s[6], w[5];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      s[2 * k] = dot3(ty.b, r + 3 * k, 3 * ROW) + dot3(ty.d, r + 3 * k + 1, 3 * ROW);
      s[2 * k + 1] = dot3(ty.b, r + 3 * k + 2, 3 * ROW);
    }
    w[0] = dot3(ty.g, r + 9, 3 * ROW);
    w[1] = dot3(ty.b, r + 10, 3 * ROW) + dot3(ty.d, r + 12, 3 * ROW);
    w[2] = dot3(ty.g, r + 11, 3 * ROW);
    w[3] = dot3(ty.g, r + 12, 3 * ROW);
    if (ROWS2) w[4] = dot3(ty.l, r + 13, 3 * ROW);
    __syncthreads();
    if (wr) {
#pragma unroll
      for (int k = 0; k < 6; ++k) own[k] = s[k];
#pragma unroll
      for (int k = 0; k < (ROWS2 ? 5 : 4); ++k) own[6 + k] = w[k];
    }
    __syncthreads();
  }
  if (!live) return;
  double *out = A.out + (int64_t)c * NDOF;
  if (ROWS2 && hl >= 28) out[SLOT_P + hl - 28] = RES && A.mode == 1 ? 0.0 : -S.dq[hl - 28];  // p rows: -int psi_k div u
  if (!wr) return;
  const TestAxis tz(d[2]);
  const double *r = fl + (d[0] + 3 * d[1]) * ROW;
#pragma unroll
  for (int k = 0; k < 3; ++k) out[3 * q + k] = dot3(tz.b, r + 2 * k, 9 * ROW) + dot3(tz.d, r + 2 * k + 1, 9 * ROW);
  if (ROWS2 && d[0] < 2 && d[1] < 2 && d[2] < 2) {
    const double t = dot3(tz.l, r + 10, 9 * ROW);
    out[SLOT_PHI + d[0] + 2 * d[1] + 4 * d[2]] = TRANS ? -ph.sigma * t : -t;
  }
  double w[3];
  w[0] = dot3(tz.g, r + 6, 9 * ROW);
  w[1] = dot3(tz.g, r + 7, 9 * ROW);
  w[2] = dot3(tz.b, r + 8, 9 * ROW) + dot3(tz.d, r + 9, 9 * ROW);
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const int m = d[a], ga = a == 0 ? d[1] : d[0], gb = a == 2 ? d[1] : d[2];
    if (ga > 1 || gb > 1) continue;  // spare lanes of this axis
    const int face = 2 * (2 - a) + (m >> 1);
    const int row = m == 1 ? 24 + 4 * a + ga + 2 * gb : 4 * face + ga + 2 * gb;
    double t = w[a];
    if (UJ)  // thin-wall faces: their own four rows, every current dof of the cell
      for (int e = e0; e < e1; ++e) {
        const int f = A.cface[e], lf = A.flf[f];
        const double *K = A.fK + (int64_t)f * 4 * NJ;
        if (!TRANS && m != 1 && face == lf && !(RES && A.mode == 1)) {
          if (RES) t += A.fc[4 * f + (row & 3)];
          for (int b = 0; b < NJ; ++b) t += K[(row & 3) * NJ + b] * S.x[OFF_J + b];
        } else if (TRANS) {
          for (int k = 0; k < 4; ++k) t += K[k * NJ + row] * S.x[OFF_J + 4 * lf + k];
        }
      }
    if (m != 1) t *= S.sg[face];
    out[SLOT_J + row] = t;
  }
}

// u0 and grad u0 (grad[3 i + k] = d u_k / d x_i) of a state at the quadrature
// points, [cell][12][27]: what the products need of the linearisation point.
__global__ __launch_bounds__(64) void k_cell_state(int ncells, const double *__restrict__ xyz,
                                                   const int32_t *__restrict__ dofs, const double *__restrict__ dir,
                                                   const double *__restrict__ x, double *__restrict__ state) {
  __shared__ double xs[2][NU], X[2][24], fl[2][NQ * 9];
  const int half = threadIdx.x >> 5, hl = threadIdx.x & 31;
  const int c = blockIdx.x * 2 + half;
  if (c < ncells) {
    for (int l = hl; l < NU; l += 32) {
      const int32_t g = dofs[(int64_t)c * NDOF + l];
      xs[half][l] = g >= 0 ? x[g] : dir[-(int64_t)g - 1];
    }
    if (hl < 24) X[half][hl] = xyz[(int64_t)c * 24 + hl];
  }
  __syncthreads();
  const int q = hl < NQ ? hl : NQ - 1;
  const int d[3] = {q % 3, (q / 3) % 3, q / 9};
  double fw[3][4], V[3], dv;
  fields_forward<false>(xs[half], nullptr, fl[half], 9, d, hl < NQ, fw, V, dv);
  if (c >= ncells || hl >= NQ) return;
  double J[9], Ji[9];
  tri_jacobian(X[half], gauss_x(d[0]), gauss_x(d[1]), gauss_x(d[2]), J);
  inv3(J, Ji);
  double *o = state + (int64_t)c * 12 * NQ + hl;
  for (int k = 0; k < 3; ++k) {
    o[k * NQ] = fw[k][0];
    for (int i = 0; i < 3; ++i)
      o[(3 + 3 * i + k) * NQ] = Ji[i] * fw[k][1] + Ji[3 + i] * fw[k][2] + Ji[6 + i] * fw[k][3];
  }
}

// y_i = sum of the element results of dof i in increasing cell order (MODE 0),
// or v_i - that sum (MODE 1); j and phi rows times `scale` (adjoint scaling).
template <class T, int MODE>
__global__ __launch_bounds__(256) void k_op_gather(int64_t n, const int32_t *__restrict__ crow,
                                                   const int32_t *__restrict__ slot, const double *__restrict__ buf,
                                                   const T *__restrict__ v, T *__restrict__ y, int64_t nu, int64_t n1,
                                                   int64_t n1p, double scale) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int32_t b = crow[i], e = crow[i + 1];
  double s = 0.0;
  for (int32_t h = b; h < e; h += 4) {  // four in flight
    const double p0 = buf[slot[h]], p1 = h + 1 < e ? buf[slot[h + 1]] : 0.0;
    const double p2 = h + 2 < e ? buf[slot[h + 2]] : 0.0, p3 = h + 3 < e ? buf[slot[h + 3]] : 0.0;
    s = (((s + p0) + p1) + p2) + p3;
  }
  if (scale != 1.0 && ((i >= nu && i < n1) || i >= n1p)) s *= scale;
  y[i] = MODE == 1 ? (T)((double)v[i] - s) : (T)s;
}

__global__ void k_gslot(int64_t nh, const int32_t *__restrict__ centry, int32_t *__restrict__ slot) {
  const int64_t h = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (h >= nh) return;
  const int32_t ce = centry[h], c = ce / NDOF, l = ce - c * NDOF;
  const int s = l < OFF_P ? (l % 27) * 3 + l / 27
                          : (l < OFF_J ? SLOT_P + l - OFF_P : (l < OFF_PHI ? SLOT_J + l - OFF_J : l));
  slot[h] = c * NDOF + s;
}

// Inverse dP1 mass matrices (3x3x3 Gauss): one thread per cell, Gauss-Jordan on
// the symmetric positive definite 4 x 4.
__global__ void k_cell_minv(int ncells, const double *__restrict__ xyz, double *__restrict__ minv) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= ncells) return;
  double X[24], M[4][8];
  for (int i = 0; i < 24; ++i) X[i] = xyz[(int64_t)c * 24 + i];
  for (int i = 0; i < 4; ++i)
    for (int j = 0; j < 8; ++j) M[i][j] = j == 4 + i ? 1.0 : 0.0;
  for (int q = 0; q < NQ; ++q) {
    const double px = gauss_x(q % 3), py = gauss_x((q / 3) % 3), pz = gauss_x(q / 9);
    double J[9], Ji[9];
    tri_jacobian(X, px, py, pz, J);
    const double W = gauss_w(q % 3) * gauss_w((q / 3) % 3) * gauss_w(q / 9) * fabs(inv3(J, Ji));
    const double ps[4] = {1.0 - px - py - pz, px, py, pz};
    for (int i = 0; i < 4; ++i)
      for (int j = 0; j < 4; ++j) M[i][j] += W * ps[i] * ps[j];
  }
  for (int k = 0; k < 4; ++k) {
    const double d = 1.0 / M[k][k];
    for (int j = 0; j < 8; ++j) M[k][j] *= d;
    for (int i = 0; i < 4; ++i)
      if (i != k) {
        const double f = M[i][k];
        for (int j = 0; j < 8; ++j) M[i][j] -= f * M[k][j];
      }
  }
  for (int i = 0; i < 4; ++i)
    for (int j = 0; j < 4; ++j) minv[(int64_t)c * 16 + 4 * i + j] = M[i][4 + j];
}

template <int OP, bool TRANS, class T>
int launch_op(mhd_ctx *c, const T *x, const T *v, T *y, int64_t rows, double *buf, int mode, double scale,
              hipStream_t s) {
  CellOpArgs A{};
  A.ncells = c->ncells;
  A.n = c->n;
  A.nu = c->nfree[0];
  A.n1 = (int64_t)c->nfree[0] + c->nfree[2];
  A.n1p = A.n1 + c->nfree[1];
  A.xyz = c->d_xyz;
  A.dir = c->d_dir;
  A.minv = c->d_minv;
  A.state = c->d_state;
  A.dofs = c->d_dofs;
  A.sign = c->d_sign;
  A.cfptr = c->d_cfptr;
  A.cface = c->d_cface;
  A.flf = c->d_flf;
  A.fK = c->d_fK;
  A.fc = c->d_fc;
  A.out = buf;
  A.scale = scale;
  A.mode = mode;
  hipLaunchKernelGGL((k_cell_op<OP, TRANS, T>), dim3((unsigned)((c->ncells + 1) / 2)), dim3(64), 0, s, A,
                     OP == OP_RES ? c->phys : c->jac_phys, x);
  const dim3 g((unsigned)((rows + 255) / 256));
  const double rs = TRANS ? 1.0 / scale : 1.0;
  if (v)
    hipLaunchKernelGGL((k_op_gather<T, 1>), g, dim3(256), 0, s, rows, c->d_crow, c->d_gslot, buf, v, y, A.nu, A.n1,
                       A.n1p, rs);
  else
    hipLaunchKernelGGL((k_op_gather<T, 0>), g, dim3(256), 0, s, rows, c->d_crow, c->d_gslot, buf, v, y, A.nu, A.n1,
                       A.n1p, rs);
  MHD_HIP(hipGetLastError());
  return 0;
}

}  // namespace

// Everything that the products need is allocated with the context: an assembly
// into it may be the first one and under capture, where nothing can be.
int mhd_cellop_build(mhd_ctx *c, bool products) {
  MHD_HIP(hipMalloc(&c->d_gslot, sizeof(int32_t) * (size_t)std::max<int64_t>(c->nhold, 1)));
  MHD_HIP(hipMalloc(&c->d_minv, sizeof(double) * (size_t)c->ncells * 16));
  if (products) {
    MHD_HIP(hipMalloc(&c->d_state, sizeof(double) * (size_t)c->ncells * 12 * NQ));
    if (c->nnz >= APPLY_NNZ &&
        hipMalloc(&c->d_sbuf, sizeof(double) * (size_t)c->ncells * NDOF) != hipSuccess) {
      c->d_sbuf = nullptr;  // mhd_spmv_d streams the matrix
      (void)hipGetLastError();
    }
  }
  if (c->nhold > 0)
    hipLaunchKernelGGL(k_gslot, dim3((unsigned)((c->nhold + 255) / 256)), dim3(256), 0, c->stream, c->nhold,
                       c->d_centry, c->d_gslot);
  hipLaunchKernelGGL(k_cell_minv, dim3((unsigned)((c->ncells + 63) / 64)), dim3(64), 0, c->stream, c->ncells, c->d_xyz,
                     c->d_minv);
  MHD_HIP(hipGetLastError());
  MHD_HIP(hipStreamSynchronize(c->stream));  // used on any stream from here on
  return 0;
}

int mhd_cellop_residual(mhd_ctx *c, const double *d_x, double *d_r, double *buf, int mode, hipStream_t s) {
  return launch_op<OP_RES, false, double>(c, d_x, (const double *)nullptr, d_r, c->n, buf, mode, 1.0, s);
}

int mhd_cellop_state(mhd_ctx *c, const double *d_x, hipStream_t s) {
  if (c->phys.convection == 0) return 0;
  hipLaunchKernelGGL(k_cell_state, dim3((unsigned)((c->ncells + 1) / 2)), dim3(64), 0, s, c->ncells, c->d_xyz,
                     c->d_dofs, c->d_dir, d_x, c->d_state);
  MHD_HIP(hipGetLastError());
  return 0;
}

template <class T>
int mhd_cellop_apply(mhd_ctx *c, int op, bool trans, double scale, const T *x, const T *v, T *y, double *buf,
                     hipStream_t s) {
  const int64_t rows = op == MHD_OP_FULL ? c->n : (int64_t)c->nfree[0] + c->nfree[2];
  if (op == MHD_OP_FULL)
    return trans ? launch_op<OP_FULL, true, T>(c, x, v, y, rows, buf, 0, scale, s)
                 : launch_op<OP_FULL, false, T>(c, x, v, y, rows, buf, 0, 1.0, s);
  if (op == MHD_OP_UJ)
    return trans ? launch_op<OP_UJ, true, T>(c, x, v, y, rows, buf, 0, scale, s)
                 : launch_op<OP_UJ, false, T>(c, x, v, y, rows, buf, 0, 1.0, s);
  return trans ? launch_op<OP_PPHI, true, T>(c, x, v, y, rows, buf, 0, scale, s)
               : launch_op<OP_PPHI, false, T>(c, x, v, y, rows, buf, 0, 1.0, s);
}
template int mhd_cellop_apply<double>(mhd_ctx *, int, bool, double, const double *, const double *, double *, double *,
                                      hipStream_t);
template int mhd_cellop_apply<float>(mhd_ctx *, int, bool, double, const float *, const float *, float *, double *,
                                     hipStream_t);

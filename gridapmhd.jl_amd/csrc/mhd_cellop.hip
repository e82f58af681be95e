// The weak form applied cell by cell, without the matrix: the residual
// (src/weakforms.jl:255-312 and the thin-wall terms :721-726) and the products
// with the Jacobian, its [u,j] block, its (u,j) x (p,phi) block, and their
// transposes.
//
// Half a wave (32 lanes) per cell, two cells per 64-thread workgroup.  A lane
// is first a quadrature point: it evaluates every field of the input there
// from the cell's 129 values in LDS (broadcast reads) with its own 1-D
// factors, maps to physical coordinates, forms the fluxes of the weak form and
// pulls them back to the reference cell (18 numbers per point, LDS).  Then it
// is a test function: a Q2 node with its three components, then an RT1 face
// dof, then an RT1 interior / dP1 / dQ1 dof, and sums the fluxes over the 27
// points, again with 1-D factors.  No basis vector is mapped or stored: a cell
// costs about 1,300 FMAs per lane and 600 LDS reads, where a kernel that works
// in physical space pushes 27 x (27 + 36) basis vectors through LDS per cell.
// Element results go to a buffer [cell][129] and a second kernel adds them per
// dof in increasing cell order: no atomics, the same bits in every run.
//
// Residual at 64 x 64 x 8 (32,768 cells): 2.31 -> 0.158 ms (cell kernel 0.136,
// sums 0.025), at 8 x 8 x 3: 53 -> 17 us (13 + 4, latency of one cell).  The
// cell kernel is bound by LDS reads (0.06 ms of them) and their latency at two
// waves per SIMD.
#include <algorithm>

#include "mhd_internal.h"

using namespace mhd;

namespace {

// Slot of local dof l in a cell's 129 element results: the three components of
// a velocity node side by side, as their dofs are, then j, p, phi.
constexpr int SLOT_J = NU, SLOT_P = NU + NJ, SLOT_PHI = NU + NJ + NP;

// 1-D factors at the 3-point Gauss rule on [0, 1], correctly rounded: points,
// weights, Q2 values and derivatives (also the normal factor of RT1), linear
// factors on the 2-point Gauss nodes (the tangential factor of RT1).  [q][i]
constexpr double GX[3] = {0.11270166537925831148, 0.5, 0.88729833462074168852};
constexpr double GW[3] = {5.0 / 18.0, 8.0 / 18.0, 5.0 / 18.0};
constexpr double QV[3][3] = {{0.68729833462074168852, 0.4, -0.08729833462074168852},
                             {0.0, 1.0, 0.0},
                             {-0.08729833462074168852, 0.4, 0.68729833462074168852}};
constexpr double QD[3][3] = {{-2.54919333848296675407, 3.09838667696593350814, -0.54919333848296675407},
                             {-1.0, 0.0, 1.0},
                             {0.54919333848296675407, -3.09838667696593350814, 2.54919333848296675407}};
constexpr double LG[3][2] = {{1.17082039324993690892, -0.17082039324993690892},
                             {0.5, 0.5},
                             {-0.17082039324993690892, 1.17082039324993690892}};

__device__ inline double pick(int q, double a, double b, double c) { return q == 0 ? a : (q == 1 ? b : c); }
__device__ inline double gauss_x(int q) { return pick(q, GX[0], GX[1], GX[2]); }
__device__ inline double gauss_w(int q) { return pick(q, GW[0], GW[1], GW[2]); }
__device__ inline double q2_val(int i, int q) {
  return pick(q, pick(i, QV[0][0], QV[0][1], QV[0][2]), pick(i, QV[1][0], QV[1][1], QV[1][2]),
              pick(i, QV[2][0], QV[2][1], QV[2][2]));
}
__device__ inline double q2_der(int i, int q) {
  return pick(q, pick(i, QD[0][0], QD[0][1], QD[0][2]), pick(i, QD[1][0], QD[1][1], QD[1][2]),
              pick(i, QD[2][0], QD[2][1], QD[2][2]));
}
__device__ inline double g2_val(int i, int q) {
  return pick(q, i ? LG[0][1] : LG[0][0], i ? LG[1][1] : LG[1][0], i ? LG[2][1] : LG[2][0]);
}

// the factors of one axis at point q
struct Axis {
  double b[3], d[3], g[2];
  __device__ explicit Axis(int q) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      b[i] = q2_val(i, q);
      d[i] = q2_der(i, q);
    }
    g[0] = g2_val(0, q);
    g[1] = g2_val(1, q);
  }
};

struct CellIn {
  double x[NDOF + 1];    // input values, RT1 face dofs times their orientation
  double xyz[24];
  double minv[16];       // inverse dP1 mass matrix (augmented-Lagrangian term)
  double sg[6];
  double dq[4];          // int psi_k div u
  double wd[NQ + 1];     // W div u at the points
  double fl[NQ][18];     // fluxes: 3 x (S_k, T_0k, T_1k, T_2k), (v_0, v_1, v_2, c), W div j, unused
};

// value and reference gradient of one Q2 component from its 27 nodal values
__device__ inline void q2_eval(const double *__restrict__ v, const Axis &ax, const Axis &ay, const Axis &az, double &f,
                               double &f0, double &f1, double &f2) {
  f = f0 = f1 = f2 = 0.0;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    double s = 0.0, s0 = 0.0, s1 = 0.0;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const double *r = v + 3 * j + 9 * k;
      const double a = ax.b[0] * r[0] + ax.b[1] * r[1] + ax.b[2] * r[2];
      const double da = ax.d[0] * r[0] + ax.d[1] * r[1] + ax.d[2] * r[2];
      s += ay.b[j] * a;
      s0 += ay.b[j] * da;
      s1 += ay.d[j] * a;
    }
    f += az.b[k] * s;
    f0 += az.b[k] * s0;
    f1 += az.b[k] * s1;
    f2 += az.d[k] * s;
  }
}

// reference component d of the RT1 field and its derivative along d; the face
// dofs of the lower / upper side at lo / hi, the interior ones at in
__device__ inline void rt_eval(const double *__restrict__ lo, const double *__restrict__ hi,
                               const double *__restrict__ in, const Axis &ad, const Axis &ta, const Axis &tb, double &v,
                               double &dv) {
  double s[3];
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    const double *r = m == 0 ? lo : (m == 1 ? in : hi);
    s[m] = tb.g[0] * (ta.g[0] * r[0] + ta.g[1] * r[1]) + tb.g[1] * (ta.g[0] * r[2] + ta.g[1] * r[3]);
  }
  v = ad.b[0] * s[0] + ad.b[1] * s[1] + ad.b[2] * s[2];
  dv = ad.d[0] * s[0] + ad.d[1] * s[1] + ad.d[2] * s[2];
}

// Jacobian of the trilinear map at a point: J[3 k + l] = d x_k / d xi_l
__device__ inline void tri_jacobian(const double *__restrict__ X, double x, double y, double z, double *J) {
  const double x0 = 1.0 - x, y0 = 1.0 - y, z0 = 1.0 - z;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const double a0 = X[k], a1 = X[3 + k], a2 = X[6 + k], a3 = X[9 + k];
    const double b0 = X[12 + k], b1 = X[15 + k], b2 = X[18 + k], b3 = X[21 + k];
    J[3 * k] = z0 * (y0 * (a1 - a0) + y * (a3 - a2)) + z * (y0 * (b1 - b0) + y * (b3 - b2));
    J[3 * k + 1] = z0 * (x0 * (a2 - a0) + x * (a3 - a1)) + z * (x0 * (b2 - b0) + x * (b3 - b1));
    J[3 * k + 2] = y0 * (x0 * (b0 - a0) + x * (b1 - a1)) + y * (x0 * (b2 - a2) + x * (b3 - a3));
  }
}

// inverse (Ji[3 l + i] = d xi_l / d x_i) and determinant
__device__ inline double inv3(const double *J, double *Ji) {
  const double c00 = J[4] * J[8] - J[5] * J[7], c01 = J[5] * J[6] - J[3] * J[8], c02 = J[3] * J[7] - J[4] * J[6];
  const double det = J[0] * c00 + J[1] * c01 + J[2] * c02, id = 1.0 / det;
  Ji[0] = c00 * id;
  Ji[3] = c01 * id;
  Ji[6] = c02 * id;
  Ji[1] = (J[2] * J[7] - J[1] * J[8]) * id;
  Ji[4] = (J[0] * J[8] - J[2] * J[6]) * id;
  Ji[7] = (J[1] * J[6] - J[0] * J[7]) * id;
  Ji[2] = (J[1] * J[5] - J[2] * J[4]) * id;
  Ji[5] = (J[2] * J[3] - J[0] * J[5]) * id;
  Ji[8] = (J[0] * J[4] - J[1] * J[3]) * id;
  return det;
}

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
  if (live) {
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
  const int q = hl < NQ ? hl : NQ - 1;  // lanes 27..31 repeat the last point and write nothing
  const int qx = q % 3, qy = (q / 3) % 3, qz = q / 9;
  const double px = gauss_x(qx), py = gauss_x(qy), pz = gauss_x(qz);
  double J[9], Ji[9], W, id;
  double u[3] = {0, 0, 0}, gu[9], j[3] = {0, 0, 0}, dj = 0.0, p = 0.0, phi = 0.0, divu = 0.0;
  if (live) {
    const Axis ax(qx), ay(qy), az(qz);
    tri_jacobian(S.xyz, px, py, pz, J);
    const double det = inv3(J, Ji);
    id = 1.0 / det;
    W = gauss_w(qx) * gauss_w(qy) * gauss_w(qz) * fabs(det);
    if (UJ) {
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        double r0, r1, r2;
        q2_eval(S.x + 27 * k, ax, ay, az, u[k], r0, r1, r2);
#pragma unroll
        for (int i = 0; i < 3; ++i) gu[3 * i + k] = Ji[i] * r0 + Ji[3 + i] * r1 + Ji[6 + i] * r2;
      }
      divu = gu[0] + gu[4] + gu[8];
      const double *xj = S.x + OFF_J;
      double r0, r1, r2, d0, d1, d2;
      rt_eval(xj + 16, xj + 20, xj + 24, ax, ay, az, r0, d0);
      rt_eval(xj + 8, xj + 12, xj + 28, ay, ax, az, r1, d1);
      rt_eval(xj, xj + 4, xj + 32, az, ax, ay, r2, d2);
#pragma unroll
      for (int k = 0; k < 3; ++k) j[k] = (J[3 * k] * r0 + J[3 * k + 1] * r1 + J[3 * k + 2] * r2) * id;
      dj = (d0 + d1 + d2) * id;
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
        double us[3], gs[9];
        if (RES) {
#pragma unroll
          for (int k = 0; k < 3; ++k) Sk[k] = ph.alpha * (gu[k] * u[0] + gu[3 + k] * u[1] + gu[6 + k] * u[2]);
        } else {
          const double *st = A.state + (int64_t)c * 12 * NQ + q;
#pragma unroll
          for (int k = 0; k < 3; ++k) us[k] = st[k * NQ];
          if (ph.convection == 2)
#pragma unroll
            for (int e = 0; e < 9; ++e) gs[e] = st[(3 + e) * NQ];
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
  if (!live) return;
  double *out = A.out + (int64_t)c * NDOF;
  // Q2 node hl: three components
  if (hl < 27) {
    const int i = hl % 3, jj = (hl / 3) % 3, k = hl / 9;
    double bx[3], dx[3], by[3], dy[3], bz[3], dz[3];
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      bx[m] = q2_val(i, m);
      dx[m] = q2_der(i, m);
      by[m] = q2_val(jj, m);
      dy[m] = q2_der(jj, m);
      bz[m] = q2_val(k, m);
      dz[m] = q2_der(k, m);
    }
#pragma unroll
    for (int comp = 0; comp < 3; ++comp) {
      double r = 0.0;
#pragma unroll
      for (int c2 = 0; c2 < 3; ++c2) {
        double t0 = 0.0, t2 = 0.0;
#pragma unroll
        for (int c1 = 0; c1 < 3; ++c1) {
          double s0 = 0.0, s1 = 0.0, s2 = 0.0;
#pragma unroll
          for (int c0 = 0; c0 < 3; ++c0) {
            const double *f = &S.fl[c0 + 3 * c1 + 9 * c2][4 * comp];
            s0 += bx[c0] * f[0] + dx[c0] * f[1];
            s1 += bx[c0] * f[2];
            s2 += bx[c0] * f[3];
          }
          t0 += by[c1] * s0 + dy[c1] * s1;
          t2 += by[c1] * s2;
        }
        r += bz[c2] * t0 + dz[c2] * t2;
      }
      out[3 * hl + comp] = r;
    }
  }
  // 24 face dofs of RT1, then its 12 interior dofs with the dP1 and dQ1 rows:
  // sum_q f_x f_y f_z V + g_x g_y g_z C with the lane's own factors
#pragma unroll 1
  for (int pass = 0; pass < 2; ++pass) {
    if (hl >= 24 || (pass && !ROWS2 && hl >= 12)) continue;
    int d, m, ga, gb, vi;
    bool rt = true;
    if (pass == 0) {
      d = 2 - (hl >> 3);
      m = (hl >> 2 & 1) ? 2 : 0;
    } else {
      d = hl >> 2;
      m = 1;
      rt = hl < 12;
    }
    ga = hl & 1;
    gb = (hl & 3) >> 1;
    vi = 12 + d;
    if (pass && !rt) {
      if (hl < 16) {  // p row: -int psi_k div u
        out[SLOT_P + hl - 12] = RES && A.mode == 1 ? 0.0 : -S.dq[hl - 12];
        continue;
      }
      vi = 16;
    }
    double F[3][3], G[3][3];
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int t = 0; t < 3; ++t) {
        const double xt = gauss_x(t);
        if (!rt) {  // dQ1 vertex hl - 16
          F[a][t] = ((hl - 16) >> a & 1) ? xt : 1.0 - xt;
          G[a][t] = 0.0;
        } else if (a == d) {
          F[a][t] = q2_val(m, t);
          G[a][t] = q2_der(m, t);
        } else {
          const bool low = a == (d == 0 ? 1 : 0);  // the lower of the two tangential axes
          F[a][t] = G[a][t] = g2_val(low ? ga : gb, t);
        }
      }
    double r = 0.0;
#pragma unroll
    for (int c2 = 0; c2 < 3; ++c2) {
      double t0 = 0.0, t1 = 0.0;
#pragma unroll
      for (int c1 = 0; c1 < 3; ++c1) {
        double s0 = 0.0, s1 = 0.0;
#pragma unroll
        for (int c0 = 0; c0 < 3; ++c0) {
          const double *f = S.fl[c0 + 3 * c1 + 9 * c2];
          s0 += F[0][c0] * f[vi];
          s1 += G[0][c0] * f[15];
        }
        t0 += F[1][c1] * s0;
        t1 += G[1][c1] * s1;
      }
      r += F[2][c2] * t0 + G[2][c2] * t1;
    }
    if (!rt) {
      out[SLOT_PHI + hl - 16] = TRANS ? -ph.sigma * r : -r;
      continue;
    }
    const int row = pass == 0 ? hl : 24 + hl;
    if (UJ) {  // thin-wall faces: their own four rows, every current dof of the cell
      for (int e = A.cfptr[c]; e < A.cfptr[c + 1]; ++e) {
        const int f = A.cface[e], lf = A.flf[f];
        const double *K = A.fK + (int64_t)f * 4 * NJ;
        if (!TRANS && (row >> 2) == lf && !(RES && A.mode == 1)) {
          double t = RES ? A.fc[4 * f + (row & 3)] : 0.0;
          for (int b = 0; b < NJ; ++b) t += K[(row & 3) * NJ + b] * S.x[OFF_J + b];
          r += t;
        } else if (TRANS) {
          for (int a = 0; a < 4; ++a) r += K[a * NJ + row] * S.x[OFF_J + 4 * lf + a];
        }
      }
    }
    if (pass == 0) r *= S.sg[hl >> 2];
    out[SLOT_J + row] = r;
  }
}

// u0 and grad u0 (grad[3 i + k] = d u_k / d x_i) of a state at the quadrature
// points, [cell][12][27]: what the products need of the linearisation point.
__global__ __launch_bounds__(64) void k_cell_state(int ncells, const double *__restrict__ xyz,
                                                   const int32_t *__restrict__ dofs, const double *__restrict__ dir,
                                                   const double *__restrict__ x, double *__restrict__ state) {
  __shared__ double xs[2][NU], X[2][24];
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
  if (c >= ncells || hl >= NQ) return;
  const double px = gauss_x(hl % 3), py = gauss_x((hl / 3) % 3), pz = gauss_x(hl / 9);
  const Axis ax(hl % 3), ay((hl / 3) % 3), az(hl / 9);
  double J[9], Ji[9];
  tri_jacobian(X[half], px, py, pz, J);
  inv3(J, Ji);
  double *o = state + (int64_t)c * 12 * NQ + hl;
  for (int k = 0; k < 3; ++k) {
    double f, r0, r1, r2;
    q2_eval(xs[half] + 27 * k, ax, ay, az, f, r0, r1, r2);
    o[k * NQ] = f;
    for (int i = 0; i < 3; ++i) o[(3 + 3 * i + k) * NQ] = Ji[i] * r0 + Ji[3 + i] * r1 + Ji[6 + i] * r2;
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
  hipLaunchKernelGGL((k_cell_op<OP, TRANS, T>), dim3((unsigned)((c->ncells + 1) / 2)), dim3(64), 0, s, A, c->phys, x);
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

int mhd_cellop_build(mhd_ctx *c) {
  MHD_HIP(hipMalloc(&c->d_gslot, sizeof(int32_t) * (size_t)std::max<int64_t>(c->nhold, 1)));
  MHD_HIP(hipMalloc(&c->d_minv, sizeof(double) * (size_t)c->ncells * 16));
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
  if (!c->d_state) MHD_HIP(hipMalloc(&c->d_state, sizeof(double) * (size_t)c->ncells * 12 * NQ));
  hipLaunchKernelGGL(k_cell_state, dim3((unsigned)((c->ncells + 1) / 2)), dim3(64), 0, s, c->ncells, c->d_xyz,
                     c->d_dofs, c->d_dir, d_x, c->d_state);
  MHD_HIP(hipGetLastError());
  return 0;
}

template <class T>
int mhd_cellop_apply(mhd_ctx *c, int op, bool trans, double scale, const T *x, const T *v, T *y, hipStream_t s) {
  const int64_t rows = op == MHD_OP_FULL ? c->n : (int64_t)c->nfree[0] + c->nfree[2];
  if (!c->d_rbuf) MHD_HIP(hipMalloc(&c->d_rbuf, sizeof(double) * (size_t)c->ncells * NDOF));
  if (op == MHD_OP_FULL)
    return trans ? launch_op<OP_FULL, true, T>(c, x, v, y, rows, c->d_rbuf, 0, scale, s)
                 : launch_op<OP_FULL, false, T>(c, x, v, y, rows, c->d_rbuf, 0, 1.0, s);
  if (op == MHD_OP_UJ)
    return trans ? launch_op<OP_UJ, true, T>(c, x, v, y, rows, c->d_rbuf, 0, scale, s)
                 : launch_op<OP_UJ, false, T>(c, x, v, y, rows, c->d_rbuf, 0, 1.0, s);
  return trans ? launch_op<OP_PPHI, true, T>(c, x, v, y, rows, c->d_rbuf, 0, scale, s)
               : launch_op<OP_PPHI, false, T>(c, x, v, y, rows, c->d_rbuf, 0, 1.0, s);
}
template int mhd_cellop_apply<double>(mhd_ctx *, int, bool, double, const double *, const double *, double *,
                                      hipStream_t);
template int mhd_cellop_apply<float>(mhd_ctx *, int, bool, double, const float *, const float *, float *, hipStream_t);

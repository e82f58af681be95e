// Device functions of the cell kernels: 1-D factors at the quadrature points,
// the fields of a cell by sum factorisation, the trilinear map.
#pragma once

#include "mhd_internal.h"

namespace mhd {

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

// The cell's rows are exchanged between the lanes of one wave, whose LDS
// accesses the hardware keeps in program order: this keeps the compiler's.
__device__ inline void wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

__device__ inline double dot3(const double *__restrict__ f, const double *__restrict__ v, int stride) {
  return f[0] * v[0] + f[1] * v[stride] + f[2] * v[2 * stride];
}

// Values and reference gradients out[c] = (f, d0 f, d1 f, d2 f) of the three
// velocity components from node values v[27 c + node], and with RT the
// reference components V of the RT1 field and its reference divergence from
// the 36 dofs xj: three passes through rows of `st` doubles (9, or 14 with RT)
// for lane digits d.  wr: the lane owns its row.
template <bool RT>
__device__ inline void fields_forward(const double *__restrict__ v, const double *__restrict__ xj,
                                      double *__restrict__ fl, int st, const int *d, bool wr, double (*out)[4],
                                      double *V, double &div) {
  double *own = fl + (d[0] + 3 * d[1] + 9 * d[2]) * st;
  const int t1 = d[1] ? 1 : 0, t2 = d[2] ? 1 : 0;  // tangential index of the RT1 dofs (digit 2: a spare lane)
  {
    const Axis a(d[0]);
    if (wr) {
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const double *r = v + 27 * c + 3 * d[1] + 9 * d[2];
        own[2 * c] = dot3(a.b, r, 1);
        own[2 * c + 1] = dot3(a.d, r, 1);
      }
      if (RT) {
        const double *r = xj + t1 + 2 * t2;  // axis x: (normal; y, z), normal dofs at 16, 24, 20
        own[6] = a.b[0] * r[16] + a.b[1] * r[24] + a.b[2] * r[20];
        own[7] = a.d[0] * r[16] + a.d[1] * r[24] + a.d[2] * r[20];
        const double *ry = xj + (d[1] == 0 ? 8 : (d[1] == 1 ? 28 : 12)) + 2 * t2;  // axis y: (x, z)
        own[8] = a.g[0] * ry[0] + a.g[1] * ry[1];
        const double *rz = xj + (d[2] == 0 ? 0 : (d[2] == 1 ? 32 : 4)) + 2 * t1;   // axis z: (x, y)
        own[9] = a.g[0] * rz[0] + a.g[1] * rz[1];
      }
    }
  }
  wave_order();
  {
    const Axis a(d[1]);
    const double *r = fl + (d[0] + 9 * d[2]) * st;
    double y[14];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      y[3 * c] = dot3(a.b, r + 2 * c, 3 * st);
      y[3 * c + 1] = dot3(a.b, r + 2 * c + 1, 3 * st);
      y[3 * c + 2] = dot3(a.d, r + 2 * c, 3 * st);
    }
    if (RT) {
      y[9] = a.g[0] * r[6] + a.g[1] * r[3 * st + 6];
      y[10] = a.g[0] * r[7] + a.g[1] * r[3 * st + 7];
      y[11] = dot3(a.b, r + 8, 3 * st);
      y[12] = dot3(a.d, r + 8, 3 * st);
      y[13] = a.g[0] * r[9] + a.g[1] * r[3 * st + 9];
    }
    wave_order();
    if (wr)
#pragma unroll
      for (int k = 0; k < (RT ? 14 : 9); ++k) own[k] = y[k];
  }
  wave_order();
  const Axis a(d[2]);
  const double *r = fl + (d[0] + 3 * d[1]) * st;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    out[c][0] = dot3(a.b, r + 3 * c, 9 * st);
    out[c][1] = dot3(a.b, r + 3 * c + 1, 9 * st);
    out[c][2] = dot3(a.b, r + 3 * c + 2, 9 * st);
    out[c][3] = dot3(a.d, r + 3 * c, 9 * st);
  }
  if (RT) {
    V[0] = a.g[0] * r[9] + a.g[1] * r[9 * st + 9];
    V[1] = a.g[0] * r[11] + a.g[1] * r[9 * st + 11];
    V[2] = dot3(a.b, r + 13, 9 * st);
    div = (a.g[0] * r[10] + a.g[1] * r[9 * st + 10]) + (a.g[0] * r[12] + a.g[1] * r[9 * st + 12]) +
          dot3(a.d, r + 13, 9 * st);
  }
  wave_order();
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

}  // namespace mhd

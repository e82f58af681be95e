// Cell-wise assembly of the H1-HDiv residual and Newton Jacobian on CDNA4.
//
// Weak form (src/weakforms.jl:255-312, conv at :670):
//   R(x)(y) = int  beta grad u : grad v + alpha v.((grad u)^T u) - p div v - gamma (j x B).v
//                 - div u q + j.s - sigma phi div s - sigma (u x B).s - div j phi_t
//                 - f.v - g.s  [+ zeta_u Pi_p(div u) div v + zeta_j div j div s]
//   J(x)(dx,y) = its derivative (Picard keeps only (grad du)^T u).
// Thin-wall faces (src/weakforms.jl:721-733, residual evaluated at x):
//   R += int_G tau (s.n)(j.n - jw + cw n.(grad j).n),  J += int_G tau (s.n)(dj.n + cw n.(grad dj).n)
//
// This file: the Jacobian assembly, the thin-wall and skeleton faces, the
// post-processing integrals; the residual and the matrix-free products are in
// mhd_cellop.hip.
#include <algorithm>
#include <mutex>

#include "mhd_cell.h"

using namespace mhd;

namespace {

constexpr int WG = 256;

// Decode canonical entry e -> (local row a, local column b).
__device__ inline void decode_entry(int e, int &a, int &b) {
  if (e < E_P) {
    a = e / ROWS_U_LEN;
    b = e % ROWS_U_LEN;
  } else if (e < E_J) {
    const int t = e - E_P;
    a = OFF_P + t / ROWS_P_LEN;
    b = t % ROWS_P_LEN;
  } else if (e < E_PHI) {
    const int t = e - E_J;
    a = OFF_J + t / ROWS_J_LEN;
    const int k = t % ROWS_J_LEN;
    b = k < NU ? k : (k < NU + NJ ? OFF_J + (k - NU) : OFF_PHI + (k - NU - NJ));
  } else {
    const int t = e - E_PHI;
    a = OFF_PHI + t / ROWS_PHI_LEN;
    b = OFF_J + t % ROWS_PHI_LEN;
  }
}

typedef double d4_t __attribute__((ext_vector_type(4)));

// How a cell's Jacobian entries leave the kernel:
//   SCATTER_ATOMIC  FP64 atomic add into the CSR values;
//   SCATTER_COLOUR  plain read-modify-write (the launch covers one colour class:
//                   no two of its cells share a dof);
//   SCATTER_EBUF    plain store of every canonical entry into the cell's slot of
//                   the element buffer (summed into CSR rows by k_row_assemble).
enum { SCATTER_ATOMIC = 0, SCATTER_COLOUR = 1, SCATTER_EBUF = 2 };

// Reference values at the quadrature points, the same for every cell: loaded
// into LDS once per workgroup.  Point 27 is all zeros (the padding of K = 27 to
// 28), and a tile's padding rows and columns read whatever follows.
struct JacTab {
  double t4[NQ + 1][4][27];      // d_0, d_1, d_2 and value of the Q2 functions
  double rv[NQ + 1][NJ];         // RT1: the component along axis d of its dofs, [12 d + i]
  double rd[NQ + 1][NJ];         // ... their divergence
  double q1[NQ + 1][8];
  double p1[NQ + 1][4];
  double slack[16];
};

// Weights of one cell at the quadrature points, and what its stores need.
struct JacCell {
  double mq[NQ + 1][12];         // W beta G (3 x 3, G = J^-1 J^-T), then W alpha u . J^-T (row 3)
  double wN[NQ + 1][9];          // W alpha d_d u_c at [3 c + d] (Newton)
  double wd[NQ + 1][6];          // W / det^2 (J^T J)_{dd'}, d <= d'
  double wx[NQ + 1][9];          // W / det (J_{:,d} x B)_c at [3 c + d]
  double wj[NQ + 1][9];          // W J^-1[l][c] at [3 l + c]
  double wv[NQ + 1];             // W zeta_j / det^2
  double ws[NQ + 1];             // W / det
  union {
    struct {
      double x[NU], xyz[24], fl[NQ * 9];
    };
    struct {
      double D[4][NU];           // int psi_k div v_b
      double MD[4][NU];          // zeta_u M^-1 D
    };
  };
  double minv[16];
  double sg[NJ + 12];            // orientation signs at [12 d + i]
  int64_t rp[NDOF];
  int32_t g[NDOF];
};

// local RT1 dof i of axis d: its two faces' four dofs, then the interior ones
__device__ inline int rt_local(int d, int i) { return i < 8 ? 8 * (2 - d) + i : 24 + 4 * d + i - 8; }

// Entry e (canonical index) of local row lr / local column lc with value v.
template <int MODE>
__device__ inline void emit(const JacCell &S, const uint16_t *__restrict__ rk, double *__restrict__ out, int e, int lr,
                            int lc, double v) {
  if (MODE == SCATTER_EBUF) {
    out[e] = v;
    return;
  }
  if (S.g[lr] < 0 || S.g[lc] < 0) return;
  double *p = &out[S.rp[lr] + rk[e]];
  if (MODE == SCATTER_ATOMIC) atomicAdd(p, v);
  else *p += v;
}

__device__ inline d4_t mfma16(double a, double b, d4_t c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// One 16x16 MFMA result tile times `scale`.  Lane l holds rows l/16 + 4 r
// (r = 0..3), column l%16 (v_mfma_f64_16x16x4f64 output layout); `place(i, j, e,
// lr, lc)` gives the canonical entry and local dofs of tile-local (i, j).
template <int MODE, class Place>
__device__ inline void store_tile(const JacCell &S, const d4_t &acc, double scale, int nrow, int ncol,
                                  const uint16_t *__restrict__ rk, double *__restrict__ out, Place place) {
  const int lane = threadIdx.x & 63;
  const int j = lane & 15;
  if (j >= ncol) return;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int i = (lane >> 4) + 4 * r;
    if (i >= nrow) continue;
    int e, lr, lc;
    place(i, j, e, lr, lc);
    emit<MODE>(S, rk, out, e, lr, lc, scale * acc[r]);
  }
}

// Jacobian of one cell per workgroup and turn, on FP64 MFMA tiles (16x16x4) in
// reference space: every factor that is the same for all cells (reference
// values and gradients) sits in LDS tables loaded once per workgroup, and a
// cell brings 47 weights per quadrature point.  With a, b Q2 nodes, r, s RT1
// dofs of the axes d, d' (one nonzero reference component each):
//   uu(c,d) = delta_cd S + N^{cd} + zeta_u D_c^T M^-1 D_d
//     S   = sum_q [d_0 a, d_1 a, d_2 a, a] . mq [d_l b]                    (K = 27 x 4)
//     N   = sum_q wN_cd a b                                              (K = 27)
//   up / pu = -D, D = sum_q d_l a (W J^-1_lc) psi_k                        (K = 27 x 3)
//   X_c[a][r] = sum_q wx_cd a r -> uj = -gamma X, ju = +sigma X^T          (K = 27)
//   jj  = sum_q wd_dd' r s + wv div r div s                              (K = 2 x 27)
//   jphi / phij = sum_q ws q1 div r                                      (K = 27)
// The first version mapped the 27 + 36 basis functions to physical space at
// every point: half of a cell's 124 K cycles went into that staging and jj took
// K = 27 x 4.  At 64 x 64 x 8 the kernel went from 3.34 to 1.73 ms (33.7 TFLOP/s
// of matrix instructions, the matrix unit 45 % busy), at 8 x 8 x 3 from 52 to 34
// us, one cell's serial chain.  Up to 2,048 cells every workgroup takes one cell
// and loads the tables for it alone.  It is bound by latency at two waves a SIMD (225
// VGPRs): two accumulator chains in flight in the uu job instead of three cost
// 6 %.  Writing the rows of one cell's own dofs straight into the CSR values
// was tried, on a version of 1.93 ms: 2.74 ms with a look-up for every row (2.34 for the p, phi
// and interior j rows alone), more than the sums save (2.20 -> 1.65, 1.76 ms).
template <int MODE>
__global__ __launch_bounds__(WG, 2) void k_cell_jacobian(int ncells, const int32_t *__restrict__ cells,
                                                      const double *__restrict__ xyz,
                                                      const int32_t *__restrict__ dofs,
                                                      const int8_t *__restrict__ sign,
                                                      const double *__restrict__ dir, const double *__restrict__ x,
                                                      const double *__restrict__ minv,
                                                      const RefTables *__restrict__ T,
                                                      const int64_t *__restrict__ rowptr,
                                                      const uint16_t *__restrict__ rank, double *__restrict__ val,
                                                      MhdPhys ph) {
  __shared__ JacTab R;
  __shared__ JacCell S;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, li = lane & 15, lk = lane >> 4;
  const d4_t zero = {0.0, 0.0, 0.0, 0.0};
  for (int e = tid; e < (NQ + 1) * 108; e += WG) {
    const int q = e / 108, l = e / 27 % 4, a = e % 27;
    R.t4[q][l][a] = q == NQ ? 0.0 : (l < 3 ? T->dq2[q][a][l] : T->q2[q][a]);
  }
  for (int e = tid; e < (NQ + 1) * NJ; e += WG) {
    const int q = e / NJ, d = e % NJ / 12, r = rt_local(d, e % 12);
    R.rv[q][e % NJ] = q == NQ ? 0.0 : T->rt[q][r][d];
    R.rd[q][e % NJ] = q == NQ ? 0.0 : T->rtdiv[q][r];
  }
  for (int e = tid; e < (NQ + 1) * 8; e += WG) R.q1[e / 8][e % 8] = e < NQ * 8 ? T->q1[e / 8][e % 8] : 0.0;
  for (int e = tid; e < (NQ + 1) * 4; e += WG) R.p1[e / 4][e % 4] = e < NQ * 4 ? T->p1[e / 4][e % 4] : 0.0;
  if (tid < 16) R.slack[tid] = 0.0;
  if (tid < 12) S.mq[NQ][tid] = S.sg[NJ + tid] = 0.0;
  if (tid < 9) S.wN[NQ][tid] = S.wx[NQ][tid] = S.wj[NQ][tid] = 0.0;
  if (tid < 6) S.wd[NQ][tid] = 0.0;
  if (tid == 0) S.wv[NQ] = S.ws[NQ] = 0.0;
  // this thread's share of a cell's data
  auto fetch = [&](int cell) {
    const int c = cells ? cells[cell] : cell;
    if (tid < NU) {
      const int32_t g = dofs[(int64_t)c * NDOF + tid];
      return g >= 0 ? x[g] : dir[-(int64_t)g - 1];
    }
    if (tid >= 96 && tid < 120) return xyz[(int64_t)c * 24 + tid - 96];
    if (tid >= 128 && tid < 128 + NJ) {
      const int i = tid - 128;
      return sign && i % 12 < 8 ? (double)sign[(int64_t)c * 6 + (rt_local(i / 12, i % 12) >> 2)] : 1.0;
    }
    if (tid >= 192 && tid < 208) return minv[(int64_t)c * 16 + tid - 192];
    return 0.0;
  };
  double pre = blockIdx.x < ncells ? fetch(blockIdx.x) : 0.0;
  for (int cell = blockIdx.x; cell < ncells; cell += gridDim.x) {
    const int c = cells ? cells[cell] : cell;
    const uint16_t *rk = rank + (int64_t)c * NENT;
    double *out = MODE == SCATTER_EBUF ? val + (int64_t)c * NENT : val;
    // ---- the cell's data, loaded during the previous cell (whose tiles are done)
    if (tid < NU) S.x[tid] = pre;
    else if (tid >= 96 && tid < 120) S.xyz[tid - 96] = pre;
    else if (tid >= 128 && tid < 128 + NJ) S.sg[tid - 128] = pre;
    else if (tid >= 192 && tid < 208) S.minv[tid - 192] = pre;
    if (MODE != SCATTER_EBUF && tid < NDOF) {
      const int32_t g = dofs[(int64_t)c * NDOF + tid];
      S.g[tid] = g;
      S.rp[tid] = g >= 0 ? rowptr[g] : -1;
    }
    __syncthreads();
    // ---- weights at the points: wave 0, one lane per point
    if (wave == 0) {
      const int q = lane < NQ ? lane : NQ - 1;
      const int d[3] = {q % 3, (q / 3) % 3, q / 9};
      double fw[3][4], V[3], dv, J[9], Ji[9];
      if (ph.convection) fields_forward<false>(S.x, nullptr, S.fl, 9, d, lane < NQ, fw, V, dv);
      tri_jacobian(S.xyz, gauss_x(d[0]), gauss_x(d[1]), gauss_x(d[2]), J);
      const double det = inv3(J, Ji);
      const double W = gauss_w(d[0]) * gauss_w(d[1]) * gauss_w(d[2]) * fabs(det), id = 1.0 / det;
      if (lane < NQ) {
        const double wb = W * ph.beta, wi = W * id, wii = wi * id;
#pragma unroll
        for (int l = 0; l < 3; ++l)
#pragma unroll
          for (int m = 0; m < 3; ++m) {
            S.mq[q][3 * l + m] = wb * (Ji[3 * l] * Ji[3 * m] + Ji[3 * l + 1] * Ji[3 * m + 1] + Ji[3 * l + 2] * Ji[3 * m + 2]);
            S.wj[q][3 * l + m] = W * Ji[3 * l + m];
          }
#pragma unroll
        for (int m = 0; m < 3; ++m)
          S.mq[q][9 + m] = ph.convection ? W * ph.alpha * (fw[0][0] * Ji[3 * m] + fw[1][0] * Ji[3 * m + 1] + fw[2][0] * Ji[3 * m + 2])
                                         : 0.0;
        if (ph.convection == 2)
#pragma unroll
          for (int k = 0; k < 3; ++k)
#pragma unroll
            for (int i = 0; i < 3; ++i)  // d u_k / d x_i
              S.wN[q][3 * k + i] = W * ph.alpha * (Ji[i] * fw[k][1] + Ji[3 + i] * fw[k][2] + Ji[6 + i] * fw[k][3]);
        int e = 0;
#pragma unroll
        for (int l = 0; l < 3; ++l)
#pragma unroll
          for (int m = l; m < 3; ++m) S.wd[q][e++] = wii * (J[l] * J[m] + J[3 + l] * J[3 + m] + J[6 + l] * J[6 + m]);
#pragma unroll
        for (int l = 0; l < 3; ++l) {
          S.wx[q][l] = wi * (J[3 + l] * ph.B[2] - J[6 + l] * ph.B[1]);
          S.wx[q][3 + l] = wi * (J[6 + l] * ph.B[0] - J[l] * ph.B[2]);
          S.wx[q][6 + l] = wi * (J[l] * ph.B[1] - J[3 + l] * ph.B[0]);
        }
        S.wv[q] = wii * ph.zeta_j;
        S.ws[q] = wi;
      }
    }
    __syncthreads();
    if (cell + (int)gridDim.x < ncells) pre = fetch(cell + gridDim.x);
    // ---- S tile of the wave; the waves of the first column tile also form D
    const int ti = wave >> 1, tj = wave & 1;
    const int a = 16 * ti + li, b = 16 * tj + li;
    d4_t Sacc = zero, Dacc = zero;
    {
      const int cc = min(li >> 2, 2), kk = li & 3;
#pragma unroll 3
      for (int q = 0; q < NQ; ++q) {
        const double A = (&R.t4[q][lk][0])[a];
        const double *m = &S.mq[q][3 * lk];
        const double *t = &R.t4[q][0][0] + b;
        Sacc = mfma16(A, m[0] * t[0] + m[1] * t[27] + m[2] * t[54], Sacc);
        if (tj == 0) Dacc = mfma16(A, lk < 3 ? S.wj[q][3 * lk + cc] * R.p1[q][kk] : 0.0, Dacc);
      }
    }
    if (tj == 0 && li < 12) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 16 * ti + lk + 4 * r;
        if (row < 27) S.D[li & 3][(li >> 2) * 27 + row] = Dacc[r];
      }
    }
    __syncthreads();
    for (int e = tid; e < 4 * NU; e += WG) {
      const int k = e / NU, row = e % NU;
      const double dk = S.D[k][row];
      if (ph.zeta_u != 0.0)
        S.MD[k][row] = ph.zeta_u * (S.minv[4 * k] * S.D[0][row] + S.minv[4 * k + 1] * S.D[1][row] +
                                    S.minv[4 * k + 2] * S.D[2][row] + S.minv[4 * k + 3] * S.D[3][row]);
      emit<MODE>(S, rk, out, row * ROWS_U_LEN + OFF_P + k, row, OFF_P + k, -dk);  // - dp div v
      emit<MODE>(S, rk, out, E_P + k * ROWS_P_LEN + row, OFF_P + k, row, -dk);    // - div du q
    }
    // ---- 18 cross, 9 jj and 3 jphi jobs of 14 MFMAs each
    for (int job = wave; job < 30; job += WG / 64) {
      if (job < 18) {
        const int at = job / 9, d = job / 3 % 3, cc = job % 3;
        const double sgr = S.sg[12 * d + li];
        d4_t acc = zero, accT = zero;
#pragma unroll
        for (int st = 0; st < 7; ++st) {
          const int q = 4 * st + lk;
          const double A = (&R.t4[q][3][0])[16 * at + li];
          const double Bv = S.wx[q][3 * cc + d] * sgr * (&R.rv[q][12 * d])[li];
          acc = mfma16(A, Bv, acc);
          accT = mfma16(Bv, A, accT);  // A and B share the lane layout: swapped, they give X^T
        }
        const int a0 = cc * 27 + 16 * at, na = at ? 11 : 16;
        store_tile<MODE>(S, acc, -ph.gamma, na, 12, rk, out, [&](int i, int j, int &e, int &lr, int &lc) {
          lr = a0 + i;
          lc = OFF_J + rt_local(d, j);
          e = lr * ROWS_U_LEN + lc;
        });
        store_tile<MODE>(S, accT, ph.sigma, 12, na, rk, out, [&](int i, int j, int &e, int &lr, int &lc) {
          const int r = rt_local(d, i);
          lr = OFF_J + r;
          lc = a0 + j;
          e = E_J + r * ROWS_J_LEN + lc;
        });
      } else if (job < 27) {
        const int d = (job - 18) / 3, d2 = (job - 18) % 3;
        const int lo = min(d, d2), hi = max(d, d2), wk = lo == 0 ? hi : lo + hi + 1;  // place of (lo, hi) in wd
        const double sr = S.sg[12 * d + li], ss = S.sg[12 * d2 + li];
        d4_t acc = zero, acc2 = zero;
#pragma unroll
        for (int st = 0; st < 7; ++st) {
          const int q = 4 * st + lk;
          acc = mfma16(sr * (&R.rv[q][12 * d])[li], S.wd[q][wk] * ss * (&R.rv[q][12 * d2])[li], acc);
          acc2 = mfma16(sr * (&R.rd[q][12 * d])[li], S.wv[q] * ss * (&R.rd[q][12 * d2])[li], acc2);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] += acc2[r];
        store_tile<MODE>(S, acc, 1.0, 12, 12, rk, out, [&](int i, int j, int &e, int &lr, int &lc) {
          const int r = rt_local(d, i), s2 = rt_local(d2, j);
          lr = OFF_J + r;
          lc = OFF_J + s2;
          e = E_J + r * ROWS_J_LEN + NU + s2;
        });
      } else {
        const int d = job - 27;
        const double sr = S.sg[12 * d + li];
        d4_t acc = zero, accT = zero;
#pragma unroll
        for (int st = 0; st < 7; ++st) {
          const int q = 4 * st + lk;
          const double A = sr * (&R.rd[q][12 * d])[li], Bv = S.ws[q] * (&R.q1[q][0])[li & 7];
          acc = mfma16(A, Bv, acc);
          accT = mfma16(Bv, A, accT);
        }
        store_tile<MODE>(S, acc, -ph.sigma, 12, 8, rk, out, [&](int i, int j, int &e, int &lr, int &lc) {
          const int r = rt_local(d, i);
          lr = OFF_J + r;
          lc = OFF_PHI + j;
          e = E_J + r * ROWS_J_LEN + NU + NJ + j;  // - sigma dphi div s
        });
        store_tile<MODE>(S, accT, -1.0, 8, 12, rk, out, [&](int i, int j, int &e, int &lr, int &lc) {
          const int r = rt_local(d, j);
          lr = OFF_PHI + i;
          lc = OFF_J + r;
          e = E_PHI + i * ROWS_PHI_LEN + r;  // - div dj phi_t
        });
      }
    }
    __syncthreads();
    // ---- the nine (c, d) blocks of the wave's uu tile
    double qa[7], qb[7];
#pragma unroll
    for (int st = 0; st < 7; ++st) {
      qa[st] = (&R.t4[4 * st + lk][3][0])[a];
      qb[st] = (&R.t4[4 * st + lk][3][0])[b];
    }
    const int na = ti ? 11 : 16, nb = tj ? 11 : 16;
#pragma unroll 1
    for (int cc = 0; cc < 3; ++cc) {  // three independent MFMA chains
      d4_t acc[3];
#pragma unroll
      for (int dd = 0; dd < 3; ++dd) acc[dd] = cc == dd ? Sacc : zero;
      if (ph.convection == 2)
#pragma unroll
        for (int st = 0; st < 7; ++st) {
          const double *w = &S.wN[4 * st + lk][3 * cc];
#pragma unroll
          for (int dd = 0; dd < 3; ++dd) acc[dd] = mfma16(qa[st], w[dd] * qb[st], acc[dd]);
        }
      if (ph.zeta_u != 0.0) {
        const double A = a < 27 ? S.D[lk][cc * 27 + a] : 0.0;
#pragma unroll
        for (int dd = 0; dd < 3; ++dd) acc[dd] = mfma16(A, b < 27 ? S.MD[lk][dd * 27 + b] : 0.0, acc[dd]);
      }
#pragma unroll
      for (int dd = 0; dd < 3; ++dd) {
        const int r0 = cc * 27 + 16 * ti, c0 = dd * 27 + 16 * tj;
        store_tile<MODE>(S, acc[dd], 1.0, na, nb, rk, out, [&](int i, int j, int &e, int &lr, int &lc) {
          lr = r0 + i;
          lc = c0 + j;
          e = lr * ROWS_U_LEN + lc;
        });
      }
    }
    __syncthreads();
  }
}

// Per-cell integrals of the state (post-processing, src/Applications/hunt.jl:247-260):
// out[c] = (int u.u, int grad u : grad u, int j.j, int (div j)^2, int p, |K|).  The 3x3x3
// Gauss rule integrates these polynomial quantities exactly on affine cells.  Half a
// wave per cell, one lane per point (see mhd_cellop.hip).
__global__ __launch_bounds__(64) void k_cell_integrals(int ncells, const double *__restrict__ xyz,
                                                       const int32_t *__restrict__ dofs,
                                                       const int8_t *__restrict__ sign,
                                                       const double *__restrict__ dir, const double *__restrict__ x,
                                                       double *__restrict__ out) {
  __shared__ double xs[2][NDOF + 1], X[2][24], fl[2][NQ * 14];
  const int half = threadIdx.x >> 5, hl = threadIdx.x & 31;
  const int c = blockIdx.x * 2 + half;
  if (c < ncells) {
    for (int l = hl; l < NDOF; l += 32) {
      const int32_t g = dofs[(int64_t)c * NDOF + l];
      double v = g >= 0 ? x[g] : dir[-(int64_t)g - 1];
      if (l >= OFF_J && l < OFF_J + 24 && sign) v *= (double)sign[(int64_t)c * 6 + ((l - OFF_J) >> 2)];
      xs[half][l] = v;
    }
    if (hl < 24) X[half][hl] = xyz[(int64_t)c * 24 + hl];
  }
  __syncthreads();
  const int q = hl < NQ ? hl : NQ - 1;
  const int d[3] = {q % 3, (q / 3) % 3, q / 9};
  double fw[3][4], V[3], dv, J[9], Ji[9];
  fields_forward<true>(xs[half], xs[half] + OFF_J, fl[half], 14, d, hl < NQ, fw, V, dv);
  const double px = gauss_x(d[0]), py = gauss_x(d[1]), pz = gauss_x(d[2]);
  tri_jacobian(X[half], px, py, pz, J);
  const double det = inv3(J, Ji), id = 1.0 / det;
  const double W = hl < NQ && c < ncells ? gauss_w(d[0]) * gauss_w(d[1]) * gauss_w(d[2]) * fabs(det) : 0.0;
  double v[6] = {0.0, 0.0, 0.0, dv * id * dv * id, 0.0, 1.0};
  for (int k = 0; k < 3; ++k) {
    v[0] += fw[k][0] * fw[k][0];
    for (int i = 0; i < 3; ++i) {
      const double g = Ji[i] * fw[k][1] + Ji[3 + i] * fw[k][2] + Ji[6 + i] * fw[k][3];
      v[1] += g * g;
    }
    const double jk = (J[3 * k] * V[0] + J[3 * k + 1] * V[1] + J[3 * k + 2] * V[2]) * id;
    v[2] += jk * jk;
  }
  const double *xp = xs[half] + OFF_P;
  v[4] = xp[0] * (1.0 - px - py - pz) + xp[1] * px + xp[2] * py + xp[3] * pz;
  for (int k = 0; k < 6; ++k) {
    double s = W != 0.0 ? W * v[k] : 0.0;
    for (int off = 16; off > 0; off >>= 1) s += __shfl_xor(s, off, 32);
    if (hl == 0 && c < ncells) out[(int64_t)c * 6 + k] = s;
  }
}

// Thin-wall face terms: one 64-wide workgroup per boundary face.
//
// Only the face's own four RT dofs (local 4 lf .. 4 lf + 3) have a nonzero
// normal flux on it: every other reference field is either tangential to the
// face or carries a 1-D Lagrange factor that vanishes there.  The normal flux
// s.n is taken from the reference field, s.n = sgn rt_d (+-1) / (det J |J^-T n^|)
// (the contravariant Piola identity), which is exactly zero for the other 32
// dofs, so a face adds to the rows of its own dofs only.  A boundary face dof
// belongs to one face, so every residual and Jacobian entry receives at most
// one face contribution: the sums do not depend on the launch order, on
// non-affine cells too.
struct FaceLDS {
  double W[NQF];
  double ndn[NQF];           // +-1 / (det J |J^-T n^|): s.n = sgn * rt_d * ndn
  double n[NQF][3];
  double gpsi[NQF][36][9];   // [i][k] = d psi_k / d x_i
  double jnn[NQF];           // n.(grad j).n of the state
  double xl[NJ];
  double xyz[24];
  int32_t g[NJ];
};

// geometry of a face and, with a state x, the current on it
__device__ void stage_face(FaceLDS &S, int f, const double *__restrict__ xyz, const int32_t *__restrict__ dofs,
                           const int8_t *__restrict__ sign, const double *__restrict__ dir,
                           const double *__restrict__ x, const FaceTables *__restrict__ F,
                           const int32_t *__restrict__ fcell, const int8_t *__restrict__ flf, int &cell, int &lf) {
  const int tid = threadIdx.x, nt = blockDim.x;
  cell = fcell[f];
  lf = flf[f];
  if (tid < 24) S.xyz[tid] = xyz[(int64_t)cell * 24 + tid];
  if (x && tid < NJ) {
    const int32_t g = dofs[(int64_t)cell * NDOF + OFF_J + tid];
    S.g[tid] = g;
    S.xl[tid] = g >= 0 ? x[g] : dir[-(int64_t)g - 1];
  }
  __syncthreads();
  __shared__ double Jq[NQF][9], Jiq[NQF][9], detq[NQF];
  if (tid < NQF) {
    const int q = tid;
    double J[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
    for (int v = 0; v < 8; ++v)
      for (int i = 0; i < 3; ++i)
        for (int l = 0; l < 3; ++l) J[i][l] += S.xyz[3 * v + i] * F->dq1[lf][q][v][l];
    const double c00 = J[1][1] * J[2][2] - J[1][2] * J[2][1];
    const double c01 = J[1][2] * J[2][0] - J[1][0] * J[2][2];
    const double c02 = J[1][0] * J[2][1] - J[1][1] * J[2][0];
    const double det = J[0][0] * c00 + J[0][1] * c01 + J[0][2] * c02;
    const double id = 1.0 / det;
    double Ji[3][3];
    Ji[0][0] = c00 * id;
    Ji[1][0] = c01 * id;
    Ji[2][0] = c02 * id;
    Ji[0][1] = (J[0][2] * J[2][1] - J[0][1] * J[2][2]) * id;
    Ji[1][1] = (J[0][0] * J[2][2] - J[0][2] * J[2][0]) * id;
    Ji[2][1] = (J[0][1] * J[2][0] - J[0][0] * J[2][1]) * id;
    Ji[0][2] = (J[0][1] * J[1][2] - J[0][2] * J[1][1]) * id;
    Ji[1][2] = (J[0][2] * J[1][0] - J[0][0] * J[1][2]) * id;
    Ji[2][2] = (J[0][0] * J[1][1] - J[0][1] * J[1][0]) * id;
    const int d = 2 - lf / 2;
    const double nh = (lf & 1) ? 1.0 : -1.0;
    double n[3], nn = 0.0;
    for (int i = 0; i < 3; ++i) {
      n[i] = Ji[d][i] * nh;
      nn += n[i] * n[i];
    }
    nn = sqrt(nn);
    for (int i = 0; i < 3; ++i) S.n[q][i] = n[i] / nn;
    S.W[q] = F->w[q] * fabs(det) * nn;
    S.ndn[q] = nh / (det * nn);
    for (int i = 0; i < 3; ++i)
      for (int l = 0; l < 3; ++l) {
        Jq[q][3 * i + l] = J[i][l];
        Jiq[q][3 * i + l] = Ji[i][l];
      }
    detq[q] = det;
  }
  __syncthreads();
  for (int idx = tid; idx < NQF * 36; idx += nt) {
    const int q = idx / 36, r = idx % 36;
    const double sgn = r < 24 ? (sign ? (double)sign[(int64_t)cell * 6 + (r >> 2)] : 1.0) : 1.0;
    const double id = sgn / detq[q];
    const double *J = Jq[q], *Ji = Jiq[q];
    // grad psi [i][k] = id * sum_l J[k][l] sum_m drt[l][m] Ji[m][i]  (affine push-forward)
    for (int i = 0; i < 3; ++i)
      for (int k = 0; k < 3; ++k) {
        double acc = 0.0;
        for (int l = 0; l < 3; ++l) {
          double dl = 0.0;
          for (int m = 0; m < 3; ++m) dl += F->drt[lf][q][r][l][m] * Ji[3 * m + i];
          acc += J[3 * k + l] * dl;
        }
        S.gpsi[q][r][3 * i + k] = id * acc;
      }
  }
  __syncthreads();
  if (x && tid < NQF) {
    const int q = tid;
    const double *n = S.n[q];
    double jnn = 0.0;
    for (int r = 0; r < 36; ++r) {
      const double *gs = S.gpsi[q][r];
      double t = 0.0;
      for (int i = 0; i < 3; ++i) t += n[i] * (gs[3 * i + 0] * n[0] + gs[3 * i + 1] * n[1] + gs[3 * i + 2] * n[2]);
      jnn += S.xl[r] * t;
    }
    S.jnn[q] = jnn;
  }
  __syncthreads();
}

// dR/dcw of a face: sum_q W tau (s.n) n.(grad j).n
__global__ __launch_bounds__(64) void k_face_dcw(int nfaces, const double *__restrict__ xyz,
                                                 const int32_t *__restrict__ dofs, const int8_t *__restrict__ sign,
                                                 const double *__restrict__ dir, const double *__restrict__ x,
                                                 const FaceTables *__restrict__ F, const int32_t *__restrict__ fcell,
                                                 const int8_t *__restrict__ flf, const double *__restrict__ ftau,
                                                 double *__restrict__ r) {
  __shared__ FaceLDS S;
  for (int f = blockIdx.x; f < nfaces; f += gridDim.x) {
    int cell, lf;
    stage_face(S, f, xyz, dofs, sign, dir, x, F, fcell, flf, cell, lf);
    const int a = 4 * lf + threadIdx.x;
    if (threadIdx.x < 4 && S.g[a] >= 0) {
      const double tau = ftau[f];
      const int d = 2 - lf / 2;
      const double sgn = sign ? (double)sign[(int64_t)cell * 6 + lf] : 1.0;
      double acc = 0.0;
      for (int q = 0; q < NQF; ++q) acc += S.W[q] * tau * (sgn * F->rt[lf][q][a][d] * S.ndn[q]) * S.jnn[q];
      atomicAdd(&r[S.g[a]], acc);
    }
    __syncthreads();
  }
}

// Face matrices K[a][b] = sum_q W tau (s_a.n)(s_b.n + cw n.(grad s_b).n) of the
// face's four own test functions and the cell's 36 current dofs, and constant
// parts -jw sum_q W tau (s_a.n), without the orientation signs: the term is
// linear and depends on the geometry and the face's parameters only, so they
// are computed once per context (1.2 KB per face).
__global__ __launch_bounds__(64) void k_face_matrix(int nfaces, const double *__restrict__ xyz,
                                                    const FaceTables *__restrict__ F,
                                                    const int32_t *__restrict__ fcell, const int8_t *__restrict__ flf,
                                                    const double *__restrict__ ftau, const double *__restrict__ fcw,
                                                    const double *__restrict__ fjw, double *__restrict__ K,
                                                    double *__restrict__ cst) {
  __shared__ FaceLDS S;
  for (int f = blockIdx.x; f < nfaces; f += gridDim.x) {
    int cell, lf;
    stage_face(S, f, xyz, nullptr, nullptr, nullptr, nullptr, F, fcell, flf, cell, lf);
    const double tau = ftau[f], cw = fcw[f], jw = fjw[f];
    const int dax = 2 - lf / 2;
    for (int idx = threadIdx.x; idx < 4 * NJ; idx += blockDim.x) {
      const int a = 4 * lf + idx / NJ, b = idx % NJ;
      const bool bface = (b >> 2) == lf;
      double acc = 0.0, one = 0.0;
      for (int q = 0; q < NQF; ++q) {
        const double *n = S.n[q], *gd = S.gpsi[q][b];
        const double sn = F->rt[lf][q][a][dax] * S.ndn[q];
        const double dn = bface ? F->rt[lf][q][b][dax] * S.ndn[q] : 0.0;
        double dnn = 0.0;
        for (int i = 0; i < 3; ++i) dnn += n[i] * (gd[3 * i + 0] * n[0] + gd[3 * i + 1] * n[1] + gd[3 * i + 2] * n[2]);
        acc += S.W[q] * tau * sn * (dn + cw * dnn);
        one += S.W[q] * tau * sn;
      }
      K[(int64_t)f * 4 * NJ + idx] = acc;
      if (b == 0) cst[4 * (int64_t)f + idx / NJ] = -jw * one;
    }
    __syncthreads();
  }
}

// The faces' Jacobian entries, added to the assembled values: one thread per
// entry of the face matrix.  (Recomputing the matrices at every Jacobian took
// 20 us on 96 faces and 46 us on 2,048, all latency; this takes 3 to 4 us.)
__global__ __launch_bounds__(256) void k_face_jacobian(int nfaces, const int32_t *__restrict__ dofs,
                                                       const int8_t *__restrict__ sign,
                                                       const int32_t *__restrict__ fcell,
                                                       const int8_t *__restrict__ flf, const double *__restrict__ K,
                                                       const int64_t *__restrict__ rowptr,
                                                       const uint16_t *__restrict__ rank, double *__restrict__ val) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t >= (int64_t)nfaces * 4 * NJ) return;
  const int f = (int)(t / (4 * NJ)), idx = (int)(t % (4 * NJ));
  const int cell = fcell[f], lf = flf[f], a = 4 * lf + idx / NJ, b = idx % NJ;
  const int32_t ga = dofs[(int64_t)cell * NDOF + OFF_J + a], gb = dofs[(int64_t)cell * NDOF + OFF_J + b];
  if (ga < 0 || gb < 0) return;
  double v = K[t];
  if (sign) {
    v *= (double)sign[(int64_t)cell * 6 + lf];
    if (b < 24) v *= (double)sign[(int64_t)cell * 6 + (b >> 2)];
  }
  // jj block entry of j row a, j column b inside the cell's rank map
  atomicAdd(&val[rowptr[ga] + rank[(int64_t)cell * NENT + E_J + a * ROWS_J_LEN + NU + b]], v);
}

// Canonical entry range [start, start + len) of local row a of a cell.
__device__ inline void row_segment(int a, int &start, int &len) {
  if (a < OFF_P) {
    start = a * ROWS_U_LEN;
    len = ROWS_U_LEN;
  } else if (a < OFF_J) {
    start = E_P + (a - OFF_P) * ROWS_P_LEN;
    len = ROWS_P_LEN;
  } else if (a < OFF_PHI) {
    start = E_J + (a - OFF_J) * ROWS_J_LEN;
    len = ROWS_J_LEN;
  } else {
    start = E_PHI + (a - OFF_PHI) * ROWS_PHI_LEN;
    len = ROWS_PHI_LEN;
  }
}

// Row assembly from the element buffer: one 64-lane wave per CSR row at a time.
// The row is accumulated in LDS -- every (cell, local row) holding the row's dof
// adds its contiguous element-buffer segment at the entries' ranks, in
// increasing cell order -- and then written once, coalesced.  Every entry of
// the row is written, so val needs no clearing.  A cell holds a dof at most
// once, so the ranks of one segment are distinct and its lanes never collide in
// LDS.  All holders of a dof hold it as the same field, so the segments of a
// row share one length (<= 125 = 2 x 64 lanes).  In a context with a skeleton
// term (sptr not null) the row's skeleton entries are added last.
//
// It streams 10 bytes for an element entry and 8 for a CSR entry.  Four of five
// rows have one or two holders, too little to keep in flight for a wave that
// ends each row before it loads the next, so a wave runs through rows with the
// next row's first RA_BATCH segments already loading, and a row of one holder,
// which has no sums, goes to its place without the LDS.  That pays where the
// skeleton entries lengthen a row's work, 186 -> 148 us at 21 x 17 x 5; at 64 x
// 64 x 8 without them it makes no difference to a wave per row and turn: 2.10 ->
// 2.09 ms (8.2 GB, 3.9 TB/s; 4.3 with the parts of cache lines beside the
// segments, against 4.9 of a copy).  Of the 2,048 workgroups 1,792 are resident
// at once there (7 fit a CU by the LDS of their rows).
constexpr int RA_WAVES = 4;
constexpr int RA_BATCH = 4;
constexpr int RA_BLOCKS = 256 * 8;
struct RowMeta {
  int64_t b;
  int len, p0, p1;
};
struct RowSegs {
  double v0[RA_BATCH], v1[RA_BATCH];
  int k0[RA_BATCH], k1[RA_BATCH];
};
__device__ inline RowMeta row_meta(int64_t row, int64_t n, const int64_t *__restrict__ rowptr,
                                   const int32_t *__restrict__ crow) {
  if (row >= n) return RowMeta{0, 0, 0, 0};
  return RowMeta{rowptr[row], (int)(rowptr[row + 1] - rowptr[row]), crow[row], crow[row + 1]};
}
__device__ inline void row_load(RowSegs &S, int pb, int p1, int lane, const int32_t *__restrict__ centry,
                                const double *__restrict__ ebuf, const uint16_t *__restrict__ rank) {
#pragma unroll
  for (int u = 0; u < RA_BATCH; ++u) {
    S.k0[u] = S.k1[u] = RANK_NONE;
    S.v0[u] = S.v1[u] = 0.0;
    if (pb + u < p1) {
      const int32_t ce = centry[pb + u];
      const int cell = ce / NDOF, a = ce - cell * NDOF;
      int start, slen;
      row_segment(a, start, slen);
      const int64_t base = (int64_t)cell * NENT + start;
      if (lane < slen) {
        S.k0[u] = rank[base + lane];
        S.v0[u] = ebuf[base + lane];
      }
      if (lane + 64 < slen) {
        S.k1[u] = rank[base + lane + 64];
        S.v1[u] = ebuf[base + lane + 64];
      }
    }
  }
}
__global__ __launch_bounds__(64 * RA_WAVES) void k_row_assemble(int64_t n, const int64_t *__restrict__ rowptr,
                                                                const int32_t *__restrict__ crow,
                                                                const int32_t *__restrict__ centry,
                                                                const double *__restrict__ ebuf,
                                                                const uint16_t *__restrict__ rank,
                                                                const int64_t *__restrict__ sptr,
                                                                const uint16_t *__restrict__ srank,
                                                                const double *__restrict__ sval,
                                                                double *__restrict__ val, int maxrow) {
  extern __shared__ double ra_lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  double *buf = ra_lds + (size_t)wave * maxrow;
  auto finish = [&](int64_t row, const RowMeta &m, RowSegs &S) {
    if (row >= n) return;
    if (m.p1 - m.p0 == 1 && !sptr) {
      if (S.k0[0] != RANK_NONE) val[m.b + S.k0[0]] = S.v0[0];
      if (S.k1[0] != RANK_NONE) val[m.b + S.k1[0]] = S.v1[0];
      return;
    }
    for (int t = lane; t < m.len; t += 64) buf[t] = 0.0;
    __builtin_amdgcn_wave_barrier();
    for (int pb = m.p0;;) {
#pragma unroll
      for (int u = 0; u < RA_BATCH; ++u) {
        if (pb + u >= m.p1) break;
        if (S.k0[u] != RANK_NONE) buf[S.k0[u]] += S.v0[u];
        if (S.k1[u] != RANK_NONE) buf[S.k1[u]] += S.v1[u];
        __builtin_amdgcn_wave_barrier();
      }
      pb += RA_BATCH;
      if (pb >= m.p1) break;
      row_load(S, pb, m.p1, lane, centry, ebuf, rank);
    }
    if (sptr) {
      const int64_t s1 = sptr[row + 1];
      for (int64_t p = sptr[row] + lane; p < s1; p += 64) buf[srank[p]] += sval[p];
      __builtin_amdgcn_wave_barrier();
    }
    for (int t = lane; t < m.len; t += 64) val[m.b + t] = buf[t];
    __builtin_amdgcn_wave_barrier();
  };
  const int64_t step = (int64_t)gridDim.x * RA_WAVES;
  int64_t row = (int64_t)blockIdx.x * RA_WAVES + wave;
  RowSegs A, B;
  RowMeta ma = row_meta(row, n, rowptr, crow), mb = row_meta(row + step, n, rowptr, crow);
  row_load(A, ma.p0, ma.p1, lane, centry, ebuf, rank);
  while (row < n) {
    row_load(B, mb.p0, mb.p1, lane, centry, ebuf, rank);
    RowMeta next = row_meta(row + 2 * step, n, rowptr, crow);
    finish(row, ma, A);
    ma = next;
    row_load(A, ma.p0, ma.p1, lane, centry, ebuf, rank);
    next = row_meta(row + 3 * step, n, rowptr, crow);
    finish(row + step, mb, B);
    mb = next;
    row += 2 * step;
  }
}

// Rank of every touched cell entry inside its CSR row (binary search).
__global__ void k_rank_map(int ncells, const int32_t *__restrict__ dofs, const int64_t *__restrict__ rowptr,
                           const int32_t *__restrict__ colind, uint16_t *__restrict__ rank, int *__restrict__ bad) {
  const int64_t total = (int64_t)ncells * NENT;
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x) {
    const int c = (int)(t / NENT), e = (int)(t % NENT);
    int a, b;
    decode_entry(e, a, b);
    const int32_t ga = dofs[(int64_t)c * NDOF + a], gb = dofs[(int64_t)c * NDOF + b];
    uint16_t out = RANK_NONE;
    if (ga >= 0 && gb >= 0) {
      int64_t lo = rowptr[ga], hi = rowptr[ga + 1];
      const int64_t base = lo;
      while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (colind[mid] < gb) lo = mid + 1;
        else hi = mid;
      }
      if (lo < rowptr[ga + 1] && colind[lo] == gb && lo - base < RANK_NONE) out = (uint16_t)(lo - base);
      else atomicAdd(bad, 1);
    }
    rank[t] = out;
  }
}

// tperm[p] = CSR position of the transposed entry of p.
__global__ void k_tperm(int64_t n, const int64_t *__restrict__ rowptr, const int32_t *__restrict__ colind,
                        int64_t *__restrict__ tperm, int *__restrict__ bad) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    for (int64_t p = rowptr[i]; p < rowptr[i + 1]; ++p) {
      const int32_t j = colind[p];
      int64_t lo = rowptr[j], hi = rowptr[j + 1];
      while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (colind[mid] < i) lo = mid + 1;
        else hi = mid;
      }
      if (lo < rowptr[j + 1] && colind[lo] == i) tperm[p] = lo;
      else {
        tperm[p] = -1;
        atomicAdd(bad, 1);
      }
    }
  }
}

// CSR SpMV, one 64-lane wavefront per group of rows, `LPR` lanes per row.
template <int LPR>
__global__ __launch_bounds__(256) void k_spmv(int64_t n, const int64_t *__restrict__ rowptr,
                                              const int32_t *__restrict__ colind, const double *__restrict__ val,
                                              const double *__restrict__ x, double *__restrict__ y) {
  const int64_t gid = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  const int64_t row = gid / LPR;
  const int lane = threadIdx.x % LPR;
  double acc = 0.0;
  if (row < n) {
    // four independent accumulators: four loads in flight per lane
    const int64_t e = rowptr[row + 1];
    double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
    int64_t p = rowptr[row] + lane;
    for (; p + 3 * LPR < e; p += 4 * LPR) {
      a0 += val[p] * x[colind[p]];
      a1 += val[p + LPR] * x[colind[p + LPR]];
      a2 += val[p + 2 * LPR] * x[colind[p + 2 * LPR]];
      a3 += val[p + 3 * LPR] * x[colind[p + 3 * LPR]];
    }
    for (; p < e; p += LPR) a0 += val[p] * x[colind[p]];
    acc = (a0 + a1) + (a2 + a3);
  }
  for (int off = LPR / 2; off > 0; off >>= 1) acc += __shfl_down(acc, off, LPR);
  if (row < n && lane == 0) y[row] = acc;
}

// Skeleton stabilisation (src/weakforms.jl:685-688):
//   a_Lambda(u, v) = int_Lambda (1/2) mu h^2 [grad u] : [grad v],  h^2 = |face|.
// [grad u] : [grad v] = sum_c sum_i [d_i u_c][d_i v_c]: the three velocity
// components share one scalar face matrix over the face's 54 node slots,
//   K_f[a][b] = (mu/2) |f| sum_q W_q G_q[a] . G_q[b],
// G_q[a] the jump of the physical gradient of node a's Q2 function at face
// point q (first cell's minus the second cell's, at the coinciding points),
// W_q = w_q |det J| |J^-T n^| on the first cell.  a_Lambda is linear and
// depends on the geometry only, so K_f is computed once per context.
__global__ __launch_bounds__(64) void k_skel_matrix(int nf, const double *__restrict__ xyz,
                                                    const int32_t *__restrict__ fcell,
                                                    const int8_t *__restrict__ flf, const int8_t *__restrict__ fperm,
                                                    const uint8_t *__restrict__ mslot, const double *__restrict__ mu,
                                                    const FaceTables *__restrict__ F, double *__restrict__ K) {
  __shared__ double X[2][24];
  __shared__ double Jis[2][NQF][9];      // (J^-1)[l][i] of each side at the first side's point q
  __shared__ double W[NQF];
  __shared__ double G[NQF][SKEL_SLOTS][3];
  const int tid = threadIdx.x;
  for (int f = blockIdx.x; f < nf; f += gridDim.x) {
    const int c0 = fcell[2 * f], c1 = fcell[2 * f + 1];
    const int lf0 = flf[2 * f], lf1 = flf[2 * f + 1];
    if (tid < 48) X[tid / 24][tid % 24] = xyz[(int64_t)(tid < 24 ? c0 : c1) * 24 + tid % 24];
    for (int e = tid; e < NQF * SKEL_SLOTS * 3; e += 64) (&G[0][0][0])[e] = 0.0;
    __syncthreads();
    if (tid < 2 * NQF) {
      const int s = tid / NQF, q = tid % NQF;
      const int lf = s ? lf1 : lf0, qs = s ? fperm[(int64_t)NQF * f + q] : q;
      double J[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
      for (int v = 0; v < 8; ++v)
        for (int i = 0; i < 3; ++i)
          for (int l = 0; l < 3; ++l) J[i][l] += X[s][3 * v + i] * F->dq1[lf][qs][v][l];
      const double c00 = J[1][1] * J[2][2] - J[1][2] * J[2][1];
      const double c01 = J[1][2] * J[2][0] - J[1][0] * J[2][2];
      const double c02 = J[1][0] * J[2][1] - J[1][1] * J[2][0];
      const double det = J[0][0] * c00 + J[0][1] * c01 + J[0][2] * c02;
      const double id = 1.0 / det;
      double *Ji = Jis[s][q];
      Ji[0] = c00 * id;
      Ji[3] = c01 * id;
      Ji[6] = c02 * id;
      Ji[1] = (J[0][2] * J[2][1] - J[0][1] * J[2][2]) * id;
      Ji[4] = (J[0][0] * J[2][2] - J[0][2] * J[2][0]) * id;
      Ji[7] = (J[0][1] * J[2][0] - J[0][0] * J[2][1]) * id;
      Ji[2] = (J[0][1] * J[1][2] - J[0][2] * J[1][1]) * id;
      Ji[5] = (J[0][2] * J[1][0] - J[0][0] * J[1][2]) * id;
      Ji[8] = (J[0][0] * J[1][1] - J[0][1] * J[1][0]) * id;
      if (s == 0) {
        const int d = 2 - lf / 2;
        const double nn = sqrt(Ji[3 * d] * Ji[3 * d] + Ji[3 * d + 1] * Ji[3 * d + 1] + Ji[3 * d + 2] * Ji[3 * d + 2]);
        W[q] = F->w[q] * fabs(det) * nn;
      }
    }
    __syncthreads();
    // first cell: slots 0..26 (distinct); then the second cell subtracts its
    // gradients at the slots mslot (distinct among themselves)
    for (int s = 0; s < 2; ++s) {
      for (int e = tid; e < NQF * 27; e += 64) {
        const int q = e / 27, a = e % 27;
        const int lf = s ? lf1 : lf0, qs = s ? fperm[(int64_t)NQF * f + q] : q;
        const int slot = s ? mslot[(int64_t)27 * f + a] : a;
        const double *g = F->dq2[lf][qs][a];
        const double *Ji = Jis[s][q];
        const double sg = s ? -1.0 : 1.0;
        for (int i = 0; i < 3; ++i) G[q][slot][i] += sg * (Ji[i] * g[0] + Ji[3 + i] * g[1] + Ji[6 + i] * g[2]);
      }
      __syncthreads();
    }
    double area = 0.0;
    for (int q = 0; q < NQF; ++q) area += W[q];
    const double coef = 0.5 * mu[f] * area;
    double *Kf = K + (int64_t)f * SKEL_SLOTS * SKEL_SLOTS;
    for (int e = tid; e < SKEL_SLOTS * SKEL_SLOTS; e += 64) {
      const int a = e / SKEL_SLOTS, b = e % SKEL_SLOTS;
      double acc = 0.0;
      for (int q = 0; q < NQF; ++q)
        acc += W[q] * (G[q][a][0] * G[q][b][0] + G[q][a][1] * G[q][b][1] + G[q][a][2] * G[q][b][2]);
      Kf[e] = coef * acc;
    }
    __syncthreads();
  }
}

// Skeleton residual, in two steps.  k_skel_face_product: one wave per face,
// lane a < 54 forms (K_f x_c)[a] for the three components c from the slot
// values x_c (Dirichlet values for non-free slots, 0 for unused ones), reading
// K_f by rows b (K_f is symmetric bit for bit: its entries are sums of the
// same products in the same order), so the loads are coalesced.
// k_skel_res_gather: one thread per row adds the face products of the row's
// (face, component, slot) entries, whose index is the product's own index, in
// increasing face order: the sums do not depend on the launch.  Up to 36 faces
// a row, one load after another 24 us at 21 x 17 x 5, eight at a time 16.
__global__ __launch_bounds__(64) void k_skel_face_product(int nf, const int32_t *__restrict__ sdofs,
                                                          const double *__restrict__ K, const double *__restrict__ x,
                                                          const double *__restrict__ dir, double *__restrict__ fres) {
  __shared__ double xs[SKEL_DOFS];
  const int lane = threadIdx.x;
  for (int f = blockIdx.x; f < nf; f += gridDim.x) {
    for (int e = lane; e < SKEL_DOFS; e += 64) {
      const int32_t g = sdofs[(int64_t)f * SKEL_DOFS + e];
      xs[e] = g == SKEL_NONE ? 0.0 : (g >= 0 ? x[g] : dir[-(int64_t)g - 1]);
    }
    __syncthreads();
    if (lane < SKEL_SLOTS) {
      const double *Kf = K + (int64_t)f * SKEL_SLOTS * SKEL_SLOTS;
      double a0 = 0.0, a1 = 0.0, a2 = 0.0;
      for (int b = 0; b < SKEL_SLOTS; ++b) {
        const double k = Kf[b * SKEL_SLOTS + lane];
        a0 += k * xs[b];
        a1 += k * xs[SKEL_SLOTS + b];
        a2 += k * xs[2 * SKEL_SLOTS + b];
      }
      double *o = fres + (int64_t)f * SKEL_DOFS;
      o[lane] = a0;
      o[SKEL_SLOTS + lane] = a1;
      o[2 * SKEL_SLOTS + lane] = a2;
    }
    __syncthreads();
  }
}

__global__ void k_skel_res_gather(int64_t n, const int32_t *__restrict__ srow, const int32_t *__restrict__ sentry,
                                  const double *__restrict__ fres, double *__restrict__ r) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int p0 = srow[i], p1 = srow[i + 1];
    if (p0 == p1) continue;
    double acc = 0.0;
    int p = p0;
    for (; p + 8 <= p1; p += 8) {  // eight products in flight, added in order
      int32_t e[8];
      double v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) e[u] = sentry[p + u];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = fres[e[u]];
#pragma unroll
      for (int u = 0; u < 8; ++u) acc += v[u];
    }
    for (; p < p1; ++p) acc += fres[sentry[p]];
    r[i] += acc;
  }
}

// Skeleton part of the matrix, constant for a context: every row's entries
// (rank in the CSR row, sum of K_f[slot][b] over the row's skeleton entries in
// increasing face order) are summed once at creation, and the Jacobian adds
// them to the assembled rows.  Summing them from the face matrices in every
// assembly read 420 MB at 21 x 17 x 5 (each K_f three times, a rank for each
// entry) in chains of dependent loads: 212 us, against 85 MB for the sums, which
// cost the row assembly 29 us.
// One wave per row; the slot dofs of one entry are distinct, so lanes never
// collide.  The first pass (srank null) counts a row's entries into cnt, the
// second writes them at sptr.  flag and buf share the LDS: max_row doubles.
__device__ inline int skel_rank(const int32_t *colind, int64_t rb, int len, int32_t g) {
  int lo = 0, hi = len;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (colind[rb + mid] < g) lo = mid + 1;
    else hi = mid;
  }
  return lo < len && colind[rb + lo] == g ? lo : -1;
}

__global__ __launch_bounds__(64) void k_skel_rows(int64_t n, const int64_t *__restrict__ rowptr,
                                                  const int32_t *__restrict__ colind, const int32_t *__restrict__ srow,
                                                  const int32_t *__restrict__ sentry,
                                                  const int32_t *__restrict__ sdofs, const double *__restrict__ K,
                                                  int32_t *__restrict__ cnt, const int64_t *__restrict__ sptr,
                                                  uint16_t *srank, double *__restrict__ sval) {
  extern __shared__ double sk_lds[];
  uint8_t *flag = reinterpret_cast<uint8_t *>(sk_lds);
  const int lane = threadIdx.x;
  for (int64_t i = blockIdx.x; i < n; i += gridDim.x) {
    const int p0 = srow[i], p1 = srow[i + 1];
    if (p0 == p1) {
      if (!srank && lane == 0) cnt[i] = 0;
      continue;
    }
    const int64_t rb = rowptr[i];
    const int len = (int)(rowptr[i + 1] - rb);
    auto each = [&](auto &&visit) {
      for (int p = p0; p < p1; ++p) {
        const int32_t e = sentry[p];
        const int f = e / SKEL_DOFS, comp = (e % SKEL_DOFS) / SKEL_SLOTS, a = e % SKEL_SLOTS;
        const int32_t g = lane < SKEL_SLOTS ? sdofs[(int64_t)f * SKEL_DOFS + comp * SKEL_SLOTS + lane] : -1;
        const int rk = g >= 0 ? skel_rank(colind, rb, len, g) : -1;
        if (rk >= 0) visit(rk, ((int64_t)f * SKEL_SLOTS + a) * SKEL_SLOTS + lane);
        __syncthreads();
      }
    };
    for (int t = lane; t < len; t += 64) flag[t] = 0;
    __syncthreads();
    each([&](int rk, int64_t) { flag[rk] = 1; });
    int m = 0;
    for (int t0 = 0; t0 < len; t0 += 64) {
      const bool on = t0 + lane < len && flag[t0 + lane];
      const uint64_t mask = __ballot(on);
      if (srank && on) srank[sptr[i] + m + __popcll(mask & ((1ull << lane) - 1))] = (uint16_t)(t0 + lane);
      m += __popcll(mask);
    }
    __syncthreads();
    if (!srank) {
      if (lane == 0) cnt[i] = m;
      continue;
    }
    for (int t = lane; t < len; t += 64) sk_lds[t] = 0.0;
    __syncthreads();
    each([&](int rk, int64_t k) { sk_lds[rk] += K[k]; });
    __threadfence_block();
    for (int t = lane; t < m; t += 64) sval[sptr[i] + t] = sk_lds[srank[sptr[i] + t]];
    __syncthreads();
  }
}

// The skeleton rows added to CSR values that other kernels wrote (k_row_assemble
// adds them itself): one wave per row.
__global__ __launch_bounds__(256) void k_skel_add(int64_t n, const int64_t *__restrict__ rowptr,
                                                  const int64_t *__restrict__ sptr,
                                                  const uint16_t *__restrict__ srank,
                                                  const double *__restrict__ sval, double *__restrict__ val) {
  const int lane = threadIdx.x & 63;
  for (int64_t i = blockIdx.x * (int64_t)4 + (threadIdx.x >> 6); i < n; i += (int64_t)gridDim.x * 4) {
    const int64_t p1 = sptr[i + 1], rb = rowptr[i];
    for (int64_t p = sptr[i] + lane; p < p1; p += 64) val[rb + srank[p]] += sval[p];
  }
}

}  // namespace

// Workgroups of the cell kernel: it loads 43 KB of tables, so a workgroup takes
// several cells.  Two fit a CU (256 CUs); four times that many keep the last
// round short (tables are then under a tenth of a workgroup's 16 cells).
static unsigned jacobian_blocks(int ncells) { return (unsigned)std::min(ncells, 2048); }

int mhd_launch_jacobian(mhd_ctx *c, const double *d_x, double *d_val, hipStream_t s) {
  if (c->nskel > 0 && c->max_row > SKEL_MAX_ROW) {
    c->err = "skeleton Jacobian: a CSR row longer than 8192 entries";
    return -1;
  }
  // a cell holding one dof twice (a periodic direction one cell thick) needs
  // the atomic scatter: its own entries may coincide
  int mode = c->dup_dofs ? 0 : c->assembly_mode;
  if (mode == 2 && sizeof(double) * (size_t)RA_WAVES * c->max_row > 65536) mode = 1;  // row too long for LDS
  if (mode == 2 && c->ncells > 0) {
    if (!c->d_ebuf) MHD_HIP(hipMalloc(&c->d_ebuf, sizeof(double) * (size_t)c->ncells * NENT));
    hipLaunchKernelGGL((k_cell_jacobian<SCATTER_EBUF>), dim3(jacobian_blocks(c->ncells)), dim3(WG), 0, s, c->ncells,
                       (const int32_t *)nullptr, c->d_xyz, c->d_dofs, c->d_sign, c->d_dir, d_x, c->d_minv, c->d_ref,
                       c->d_rowptr, c->d_rank, c->d_ebuf, c->phys);
    MHD_HIP(hipGetLastError());
    if (c->n > 0) {
      const int64_t blocks = std::min<int64_t>((c->n + RA_WAVES - 1) / RA_WAVES, RA_BLOCKS);
      const size_t lds = sizeof(double) * (size_t)RA_WAVES * c->max_row;
      hipLaunchKernelGGL(k_row_assemble, dim3((unsigned)blocks), dim3(64 * RA_WAVES), lds, s, c->n, c->d_rowptr,
                         c->d_crow, c->d_centry, c->d_ebuf, c->d_rank, c->d_skel_ptr, c->d_skel_rank, c->d_skel_val,
                         d_val, c->max_row);
      MHD_HIP(hipGetLastError());
    }
  } else {
    MHD_HIP(hipMemsetAsync(d_val, 0, sizeof(double) * c->nnz, s));
  }
  if (mode == 2 || c->ncells == 0) {
  } else if (mode == 0 || c->color_ptr.size() < 2) {
    hipLaunchKernelGGL((k_cell_jacobian<SCATTER_ATOMIC>), dim3(jacobian_blocks(c->ncells)), dim3(WG), 0, s, c->ncells,
                       (const int32_t *)nullptr, c->d_xyz, c->d_dofs, c->d_sign, c->d_dir, d_x, c->d_minv, c->d_ref,
                       c->d_rowptr, c->d_rank, d_val, c->phys);
    MHD_HIP(hipGetLastError());
  } else {
    for (size_t k = 0; k + 1 < c->color_ptr.size(); ++k) {
      const int n = c->color_ptr[k + 1] - c->color_ptr[k];
      if (n == 0) continue;
      hipLaunchKernelGGL((k_cell_jacobian<SCATTER_COLOUR>), dim3(jacobian_blocks(n)), dim3(WG), 0, s, n,
                         c->d_color_cells + c->color_ptr[k], c->d_xyz, c->d_dofs, c->d_sign, c->d_dir, d_x, c->d_minv,
                         c->d_ref, c->d_rowptr, c->d_rank, d_val, c->phys);
      MHD_HIP(hipGetLastError());
    }
  }
  if (c->nfaces > 0) {
    const int64_t ne = (int64_t)c->nfaces * 4 * NJ;
    hipLaunchKernelGGL(k_face_jacobian, dim3((unsigned)((ne + 255) / 256)), dim3(256), 0, s, c->nfaces, c->d_dofs,
                       c->d_sign, c->d_fcell, c->d_flf, c->d_fK, c->d_rowptr, c->d_rank, d_val);
    MHD_HIP(hipGetLastError());
  }
  if (mode != 2 && c->nskel > 0 && c->n > 0) {
    const int64_t blocks = std::min<int64_t>((c->n + 3) / 4, 1 << 20);
    hipLaunchKernelGGL(k_skel_add, dim3((unsigned)blocks), dim3(256), 0, s, c->n, c->d_rowptr, c->d_skel_ptr,
                       c->d_skel_rank, c->d_skel_val, d_val);
    MHD_HIP(hipGetLastError());
  }
  return 0;
}

// Whether s records its work into a graph (an error counts as yes: the stream
// of a capture elsewhere that cannot be asked).
static bool capturing(hipStream_t s) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &st) == hipSuccess) return st != hipStreamCaptureStatusNone;
  (void)hipGetLastError();
  return true;
}

int mhd_assemble_own(mhd_ctx *c, hipStream_t s) {
  c->jac_valid = false;
  // a replay changes d_val and the state later, with the parameters of now
  if (c->d_sbuf && capturing(s)) c->jac_replayed = true;
  int rc = mhd_launch_jacobian(c, c->d_x, c->d_val, s);
  if (!rc && c->nskel == 0) rc = mhd_cellop_state(c, c->d_x, s);
  if (rc) return rc;
  c->jac_phys = c->phys;
  c->jac_valid = true;
  return 0;
}

int mhd_build_skeleton(mhd_ctx *c, const int32_t *d_fcell, const int8_t *d_flf, const int8_t *d_fperm,
                       const uint8_t *d_mslot, const double *d_mu) {
  if (c->nskel <= 0) return 0;
  MHD_HIP(hipMalloc(&c->d_skel_K, sizeof(double) * (size_t)c->nskel * SKEL_SLOTS * SKEL_SLOTS));
  MHD_HIP(hipMalloc(&c->d_skel_res, sizeof(double) * (size_t)c->nskel * SKEL_DOFS));
  const int blocks = std::min(c->nskel, 1 << 20);
  hipLaunchKernelGGL(k_skel_matrix, dim3(blocks), dim3(64), 0, c->stream, c->nskel, c->d_xyz, d_fcell, d_flf,
                     d_fperm, d_mslot, d_mu, c->d_fref, c->d_skel_K);
  MHD_HIP(hipGetLastError());
  if (c->n <= 0 || c->max_row > SKEL_MAX_ROW) return 0;  // the Jacobian refuses longer rows
  int32_t *d_cnt = nullptr;
  MHD_HIP(hipMalloc(&d_cnt, sizeof(int32_t) * (size_t)c->n));
  std::vector<int32_t> cnt((size_t)c->n);
  std::vector<int64_t> ptr((size_t)c->n + 1, 0);
  const dim3 grid((unsigned)std::min<int64_t>(c->n, 1 << 20));
  const size_t lds = sizeof(double) * (size_t)c->max_row;
  hipLaunchKernelGGL(k_skel_rows, grid, dim3(64), lds, c->stream, c->n, c->d_rowptr, c->d_colind, c->d_srow,
                     c->d_sentry, c->d_skel_dofs, c->d_skel_K, d_cnt, (const int64_t *)nullptr, (uint16_t *)nullptr,
                     (double *)nullptr);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess)
    e = hipMemcpyAsync(cnt.data(), d_cnt, sizeof(int32_t) * (size_t)c->n, hipMemcpyDeviceToHost, c->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
  (void)hipFree(d_cnt);
  MHD_HIP(e);
  for (int64_t i = 0; i < c->n; ++i) ptr[i + 1] = ptr[i] + cnt[i];
  const size_t m = (size_t)std::max<int64_t>(ptr[c->n], 1);
  MHD_HIP(hipMalloc(&c->d_skel_ptr, sizeof(int64_t) * ptr.size()));
  MHD_HIP(hipMalloc(&c->d_skel_rank, sizeof(uint16_t) * m));
  MHD_HIP(hipMalloc(&c->d_skel_val, sizeof(double) * m));
  MHD_HIP(hipMemcpyAsync(c->d_skel_ptr, ptr.data(), sizeof(int64_t) * ptr.size(), hipMemcpyHostToDevice, c->stream));
  hipLaunchKernelGGL(k_skel_rows, grid, dim3(64), lds, c->stream, c->n, c->d_rowptr, c->d_colind, c->d_srow,
                     c->d_sentry, c->d_skel_dofs, c->d_skel_K, (int32_t *)nullptr, c->d_skel_ptr, c->d_skel_rank,
                     c->d_skel_val);
  MHD_HIP(hipGetLastError());
  MHD_HIP(hipStreamSynchronize(c->stream));
  return 0;
}

int mhd_launch_skeleton_residual(mhd_ctx *c, const double *d_x, double *d_r, hipStream_t s) {
  if (c->nskel <= 0 || c->n <= 0) return 0;
  hipLaunchKernelGGL(k_skel_face_product, dim3((unsigned)std::min(c->nskel, 1 << 20)), dim3(64), 0, s, c->nskel,
                     c->d_skel_dofs, c->d_skel_K, d_x, c->d_dir, c->d_skel_res);
  const int64_t blocks = std::min<int64_t>((c->n + 255) / 256, 65536);
  hipLaunchKernelGGL(k_skel_res_gather, dim3((unsigned)blocks), dim3(256), 0, s, c->n, c->d_srow, c->d_sentry,
                     c->d_skel_res, d_r);
  MHD_HIP(hipGetLastError());
  return 0;
}

int mhd_build_face_matrices(mhd_ctx *c) {
  const size_t nf = (size_t)std::max(c->nfaces, 1);
  MHD_HIP(hipMalloc(&c->d_fK, sizeof(double) * nf * 4 * NJ));
  MHD_HIP(hipMalloc(&c->d_fc, sizeof(double) * nf * 4));
  if (c->nfaces <= 0) return 0;
  hipLaunchKernelGGL(k_face_matrix, dim3((unsigned)std::min(c->nfaces, 1 << 20)), dim3(64), 0, c->stream, c->nfaces,
                     c->d_xyz, c->d_fref, c->d_fcell, c->d_flf, c->d_ftau, c->d_fcw, c->d_fjw, c->d_fK, c->d_fc);
  MHD_HIP(hipGetLastError());
  return 0;
}

// mode 0: residual; 1: dR/dgamma; 2: dR/dcw
int mhd_launch_residual_mode(mhd_ctx *c, const double *d_x, double *d_r, hipStream_t s, int mode) {
  if (mode == 2) {
    MHD_HIP(hipMemsetAsync(d_r, 0, sizeof(double) * c->n, s));
    if (c->nfaces > 0)
      hipLaunchKernelGGL(k_face_dcw, dim3(c->nfaces), dim3(64), 0, s, c->nfaces, c->d_xyz, c->d_dofs, c->d_sign,
                         c->d_dir, d_x, c->d_fref, c->d_fcell, c->d_flf, c->d_ftau, d_r);
    MHD_HIP(hipGetLastError());
    return 0;
  }
  if (!c->d_rbuf) MHD_HIP(hipMalloc(&c->d_rbuf, sizeof(double) * (size_t)c->ncells * NDOF));
  int rc = mhd_cellop_residual(c, d_x, d_r, c->d_rbuf, mode, s);
  if (rc) return rc;
  // the skeleton term depends on neither gamma nor cw (modes 1, 2: dR/dtheta)
  return mode == 0 ? mhd_launch_skeleton_residual(c, d_x, d_r, s) : 0;
}

int mhd_launch_residual(mhd_ctx *c, const double *d_x, double *d_r, hipStream_t s) {
  return mhd_launch_residual_mode(c, d_x, d_r, s, 0);
}

// ---------------------------------------------------------------------------
// Allocation-free residual.  Its element residuals live in `scratch`, device
// memory of the code object: every GPU the library runs on holds its own
// copy (NOALLOC_DOUBLES doubles = 128 MiB) until the process ends.  Host code
// never passes `scratch` itself to a kernel (on the host it only names the
// symbol): the device address of each GPU's copy is looked up once per device
// with hipGetSymbolAddress while that device is current, and that pointer is
// what the launches take.  Every call on one GPU shares that GPU's copy, so
// calls that overlap on one GPU race.  The cell kernel writes every element
// residual that the gather reads, so nothing is cleared between calls.

namespace {
constexpr int64_t NOALLOC_DOUBLES = int64_t(1) << 24;
constexpr int NOALLOC_MAX_DEVICES = 64;
static __device__ __align__(256) double scratch[NOALLOC_DOUBLES];
std::mutex g_scratch_mu;
double *g_scratch_ptr[NOALLOC_MAX_DEVICES] = {};
}  // namespace

int mhd_noalloc_init(mhd_ctx *c) {
  if (c->device < 0 || c->device >= NOALLOC_MAX_DEVICES) {
    c->err = "device index beyond the allocation-free workspace table";
    return -1;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[c->device]) {
    void *p = nullptr;
    MHD_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_scratch_ptr[c->device] = static_cast<double *>(p);
  }
  c->d_scratch = g_scratch_ptr[c->device];
  return 0;
}

int mhd_launch_residual_noalloc(mhd_ctx *c, const double *d_x, double *d_r, hipStream_t s) {
  if ((int64_t)c->ncells * NDOF > NOALLOC_DOUBLES) {
    c->err = "mhd_residual_d_noalloc: " + std::to_string(c->ncells) + " cells exceed the allocation-free workspace (" +
             std::to_string(NOALLOC_DOUBLES / NDOF) + " cells at most)";
    return -1;
  }
  if (!c->d_scratch) {
    c->err = "mhd_residual_d_noalloc: workspace address not set up for this device";
    return -2;
  }
  int rc = mhd_cellop_residual(c, d_x, d_r, c->d_scratch, 0, s);
  if (rc) return rc;
  // the skeleton face matrices and face products are context memory made at creation
  return mhd_launch_skeleton_residual(c, d_x, d_r, s);
}

// val_t[p] = val[tperm[p]]: the CSR values of A^T on the (symmetric) pattern
__global__ void k_gather_t(int64_t nnz, const int64_t *__restrict__ tperm, const double *__restrict__ val,
                           double *__restrict__ val_t) {
  for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < nnz; p += (int64_t)gridDim.x * blockDim.x)
    val_t[p] = val[tperm[p]];
}

int mhd_launch_transpose_values(mhd_ctx *c, const double *d_val, double *d_val_t, hipStream_t s) {
  int rc;
  if (!c->d_tperm) {
    MHD_HIP(hipMalloc(&c->d_tperm, sizeof(int64_t) * std::max<int64_t>(c->nnz, 1)));
    if ((rc = mhd_build_tperm(c))) return rc;
  }
  const int grid = (int)std::min<int64_t>((c->nnz + 255) / 256, 1 << 20);
  hipLaunchKernelGGL(k_gather_t, dim3(grid), dim3(256), 0, s, c->nnz, c->d_tperm, d_val, d_val_t);
  MHD_HIP(hipGetLastError());
  return 0;
}

int mhd_launch_cell_integrals(mhd_ctx *c, const double *d_x, double *d_out, hipStream_t s) {
  hipLaunchKernelGGL(k_cell_integrals, dim3((unsigned)((c->ncells + 1) / 2)), dim3(64), 0, s, c->ncells, c->d_xyz,
                     c->d_dofs, c->d_sign, c->d_dir, d_x, d_out);
  MHD_HIP(hipGetLastError());
  return 0;
}

int mhd_build_rank_map(mhd_ctx *c) {
  int *d_bad = nullptr;
  MHD_HIP(hipMalloc(&d_bad, sizeof(int)));
  MHD_HIP(hipMemsetAsync(d_bad, 0, sizeof(int), c->stream));
  const int64_t total = (int64_t)c->ncells * NENT;
  const int grid = (int)std::min<int64_t>((total + 255) / 256, 65536);
  hipLaunchKernelGGL(k_rank_map, dim3(grid), dim3(256), 0, c->stream, c->ncells, c->d_dofs, c->d_rowptr, c->d_colind,
                     c->d_rank, d_bad);
  MHD_HIP(hipGetLastError());
  int bad = 0;
  MHD_HIP(hipMemcpyAsync(&bad, d_bad, sizeof(int), hipMemcpyDeviceToHost, c->stream));
  MHD_HIP(hipStreamSynchronize(c->stream));
  MHD_HIP(hipFree(d_bad));
  if (bad) {
    c->err = "rank map: " + std::to_string(bad) + " entries missing from the pattern";
    return -3;
  }
  return 0;
}

int mhd_build_tperm(mhd_ctx *c) {
  int *d_bad = nullptr;
  MHD_HIP(hipMalloc(&d_bad, sizeof(int)));
  MHD_HIP(hipMemsetAsync(d_bad, 0, sizeof(int), c->stream));
  const int grid = (int)std::min<int64_t>((c->n + 255) / 256, 65536);
  hipLaunchKernelGGL(k_tperm, dim3(grid), dim3(256), 0, c->stream, c->n, c->d_rowptr, c->d_colind, c->d_tperm, d_bad);
  MHD_HIP(hipGetLastError());
  int bad = 0;
  MHD_HIP(hipMemcpyAsync(&bad, d_bad, sizeof(int), hipMemcpyDeviceToHost, c->stream));
  MHD_HIP(hipStreamSynchronize(c->stream));
  MHD_HIP(hipFree(d_bad));
  if (bad) {
    c->err = "pattern is not structurally symmetric (" + std::to_string(bad) + " entries)";
    return -3;
  }
  return 0;
}

// y = A x with the Jacobian in d_val.  Without a skeleton term, and from
// APPLY_NNZ nonzeros on, the form is applied cell by cell.
// That needs a buffer of element results, so it belongs to the first stream
// that calls; calls on any other stream, which may overlap it, stream the
// matrix as before, and so does a context whose buffer could not be allocated.
// The matrix is streamed as well where the host does not know when the product
// runs or what it is a product with: a captured call (its graph may run beside
// other calls, and after another assembly), the per-thread stream (one handle
// for many streams), and every call once an assembly was captured.
int mhd_launch_spmv(mhd_ctx *c, const double *d_x, double *d_y, hipStream_t s) {
  if (c->jac_valid && c->d_sbuf && c->own_stream &&  // coarse levels make no products for callers
      !c->jac_replayed && s != hipStreamPerThread && !capturing(s)) {
    if (!c->sbuf_bound) {
      c->sbuf_bound = true;
      c->sbuf_stream = s;
    }
    if (c->sbuf_stream == s)
      return mhd_cellop_apply<double>(c, MHD_OP_FULL, false, 1.0, d_x, (const double *)nullptr, d_y, c->d_sbuf, s);
  }
  constexpr int LPR = 16;
  const int64_t threads = c->n * LPR;
  const int grid = (int)((threads + 255) / 256);
  hipLaunchKernelGGL(k_spmv<LPR>, dim3(grid), dim3(256), 0, s, c->n, c->d_rowptr, c->d_colind, c->d_val, d_x, d_y);
  MHD_HIP(hipGetLastError());
  return 0;
}

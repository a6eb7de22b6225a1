// Stage adjoint in the q1-line layout [q2][p][q1] for WENO5 (FP64), with every
// WENO5 indicator and face evaluated once per cell and axis (reverse mode),
// instead of once per cell of each face's stencil as in adj_stage_kernel.
//
// For one axis with upwind face states s_k (the lower face of cell k, built
// from the window of cells b..b+4, b = k-3 for C > 0 and k-2 otherwise, and
// the indicators beta of cells b+1..b+3; weno5.py:57-98), the adjoint of the
// advective term of L seen through mu is
//   sum_k g_k ds_k/du,   g_k = (C/dq) (mu_k - mu_{k-1})
// (df_dt_fvm.py:56-85).  With weights W_m = c_m / (16 beta_m^2) (c = (1, 10,
// 5) for a right face, (5, 10, 1) for a left one), D = sum W_m, substencil
// values u_m and s = sum W_m u_m / D:
//   A_m = g W_m / D                      (adjoint of u_m)
//   h_m = -2 A_m (u_m - s) / beta_m      (adjoint of beta_m)
// and cell j collects sum_m A_m coef(m, j - b) over the five faces whose
// window holds it, plus H_c dbeta_c/du_j for the indicators c = j-1, j, j+1,
// H_c being the sum of the h that name c.
//
// adj_line_kernel: a wave owns one p-cell and the whole q1 line (NR adjacent
// cells per lane, n1 = 64 NR) and marches along q2 over a segment of rows, as
// qline_kernel does forward:
//  * q2: at step t row t is in the window (loaded one step ahead); the march
//    forms the indicator of cell t-1 and the face whose window is rows t-4..t,
//    adds that face's A into the pending adjoints of rows t-4..t and its h into
//    the indicator adjoints of cells t-3..t-1; the indicator adjoint of cell t-3
//    is then complete and goes into rows t-4..t-2, and row t-4 is complete;
//  * q1: the completed row's adjoint.  Each cell's lower face is formed where the
//    cell is, its adjoints are collected by shifting running sums one cell per
//    step along the wave (DPP rotates, q1 is periodic), so nothing goes through
//    LDS.
// Register roles rotate over six unrolled steps instead of sliding.
#pragma once
#include "adjoint.h"
#include "qline.h"

namespace bx {

// Substencil values of a right (or left) face window y[0..4].
template <bool RIGHT>
__device__ __forceinline__ void al_substencils(const double* y, double u[3]) {
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    double acc = 0.0;
#pragma unroll
    for (int e = 0; e < 5; ++e)
      if (weno_sub_coef<RIGHT>(m + 1, e) != 0.0) acc += weno_sub_coef<RIGHT>(m + 1, e) * y[e];
    u[m] = acc;
  }
}

// Reverse mode of one face: A (adjoints of the substencil values) and h
// (adjoints of the three indicators) from g, the window y[0..4] and IB = 1/beta
// of cells b+1..b+3.  (Neither depends on the scale of the weights, so they are
// 1/beta^2 times c.)
template <bool RIGHT>
__device__ __forceinline__ void al_face(const double* y, const double* IB, double g, double A[3],
                                        double h[3]) {
  double u[3];
  al_substencils<RIGHT>(y, u);
  const double r1 = IB[0] * IB[0], r2 = IB[1] * IB[1], r3 = IB[2] * IB[2];
  const double W1 = RIGHT ? r1 : 5.0 * r1, W2 = 10.0 * r2, W3 = RIGHT ? 5.0 * r3 : r3;
  const double rD = fast_rcp(W1 + W2 + W3);
  const double sv = (W1 * u[0] + W2 * u[1] + W3 * u[2]) * rD;
  const double gr = g * rD;
  A[0] = gr * W1;
  A[1] = gr * W2;
  A[2] = gr * W3;
#pragma unroll
  for (int m = 0; m < 3; ++m) h[m] = -2.0 * A[m] * (u[m] - sv) * IB[m];
}

// Add a face's A into the adjoints of its window cells aw[0..4].
template <bool RIGHT>
__device__ __forceinline__ void al_scatter(const double A[3], double* aw) {
#pragma unroll
  for (int e = 0; e < 5; ++e) {
    double x = 0.0;
#pragma unroll
    for (int m = 0; m < 3; ++m)
      if (weno_sub_coef<RIGHT>(m + 1, e) != 0.0) x += A[m] * weno_sub_coef<RIGHT>(m + 1, e);
    aw[e] += x;
  }
}

// x(c) becomes x(c + 1) (UP) or x(c - 1) over the periodic line.
template <bool UP, int NR>
__device__ __forceinline__ void al_shift(double (&x)[NR]) {
  if constexpr (UP) {
    const double in = ql_rot<true>(x[0]);
#pragma unroll
    for (int k = 0; k + 1 < NR; ++k) x[k] = x[k + 1];
    x[NR - 1] = in;
  } else {
    const double in = ql_rot<false>(x[NR - 1]);
#pragma unroll
    for (int k = NR - 1; k > 0; --k) x[k] = x[k - 1];
    x[0] = in;
  }
}

// Adjoint of the q1 advection for one completed row: u and mu of the row
// (the lane's NR adjacent cells) in, the q1 part of J^T mu for them out.
template <int NR, bool P1>
__device__ __forceinline__ void al_q1_row(const double* ur, const double* mr, double cdq1,
                                          double* out) {
  // window b..b+4 of the lower face of cell c: b = c - 3 (P1) or c - 2
  constexpr int LO = P1 ? 3 : 2, HI = P1 ? 1 : 2;
  double x[LO + NR + HI], mx[1 + NR];
#pragma unroll
  for (int k = 0; k < NR; ++k) {
    x[LO + k] = ur[k];
    mx[1 + k] = mr[k];
  }
  ql_neighbours<NR, LO, HI>(x);
  ql_neighbours<NR, 1, 0>(mx);
  constexpr int KLO = P1 ? 2 : 1, KHI = P1 ? 0 : 1;
  double ib[KLO + NR + KHI];
#pragma unroll
  for (int k = 0; k < NR; ++k)
    ib[KLO + k] = fast_rcp(weno_beta<double>(x[LO + k - 1], x[LO + k], x[LO + k + 1]));
  ql_neighbours<NR, KLO, KHI>(ib);
  // y[e][k]: what the lower face of cell k gives to entry e of its window
  double y[5][NR], h[3][NR];
#pragma unroll
  for (int k = 0; k < NR; ++k) {
    double A[3], hk[3], a[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    al_face<P1>(x + k, ib + k, cdq1 * (mx[k + 1] - mx[k]), A, hk);
    al_scatter<P1>(A, a);
#pragma unroll
    for (int e = 0; e < 5; ++e) y[e][k] = a[e];
#pragma unroll
    for (int m = 0; m < 3; ++m) h[m][k] = hk[m];
  }
  // H(c): indicator m of the face of cell k is that of cell k - 2 + m (P1) or
  // k - 1 + m
  double H[NR], t[NR];
#pragma unroll
  for (int k = 0; k < NR; ++k) H[k] = h[0][k];
  al_shift<true, NR>(H);
#pragma unroll
  for (int k = 0; k < NR; ++k) H[k] += h[1][k];
  if constexpr (P1) al_shift<true, NR>(H);
#pragma unroll
  for (int k = 0; k < NR; ++k) t[k] = h[2][k];
  if constexpr (!P1) al_shift<false, NR>(t);
#pragma unroll
  for (int k = 0; k < NR; ++k) H[k] += t[k];
  // what reaches cell c from cells above it, then from itself and below: entry
  // e of the face of cell k is cell k - LO + e, an indicator adjoint H(c) goes
  // to c - 1, c and c + 1
  double up[NR], dn[NR];
#pragma unroll
  for (int k = 0; k < NR; ++k) up[k] = y[0][k];
#pragma unroll
  for (int e = 1; e < LO; ++e) {
    al_shift<true, NR>(up);
#pragma unroll
    for (int k = 0; k < NR; ++k) up[k] += y[e][k];
  }
#pragma unroll
  for (int k = 0; k < NR; ++k)
    up[k] += H[k] * beta_da(x[LO + k - 1], x[LO + k], x[LO + k + 1]);
  al_shift<true, NR>(up);
#pragma unroll
  for (int k = 0; k < NR; ++k) {
    out[k] = up[k] + y[LO][k] + H[k] * beta_db(x[LO + k - 1], x[LO + k], x[LO + k + 1]);
    dn[k] = HI == 2 ? y[4][k] : 0.0;
  }
  if constexpr (HI == 2) al_shift<false, NR>(dn);
#pragma unroll
  for (int k = 0; k < NR; ++k)
    dn[k] += y[LO + 1][k] + H[k] * beta_dc(x[LO + k - 1], x[LO + k], x[LO + k + 1]);
  al_shift<false, NR>(dn);
#pragma unroll
  for (int k = 0; k < NR; ++k) out[k] += dn[k];
}

// One wave's march over the q2 segment ``seg`` of p-cell p (P1: C_q1 > 0,
// P2: C_q2 > 0, wave-uniform).
template <int NR, bool P1, bool P2>
__device__ __forceinline__ void al_march(const AdjParams& ap, int p, int seg, int nseg, int lane) {
  const int n1 = ap.n1, n2 = ap.n2, P = ap.P;
  const int S = (n2 + nseg - 1) / nseg;
  const int r0 = seg * S, r1 = min(n2, r0 + S);
  if (r0 >= n2) return;
  int j1, j2;
  const int j23 = fdivmod(p, ap.n_p1, 1.0f / float(ap.n_p1), j1);
  const int j3 = fdivmod(j23, ap.n_p2, 1.0f / float(ap.n_p2), j2);
  const double v1 = centre(ap.p1s, j1, ap.dp1), v2 = centre(ap.p2s, j2, ap.dp2);
  const double v3 = centre(ap.p3s, j3, ap.dp3);
  const double e3 = 0.5 * ((v1 * v1 + v2 * v2) + v3 * v3);
  const double cdq1 = v1 * ap.inv_dq1;
  const double cdq2 = n2 > 1 ? v2 * ap.inv_dq2 : 0.0;
  const long rs = (long)n1 * P, col = (long)p * n1 + lane * NR;
  const long Qn = (long)n1 * n2;
  // rings over the rows: u and mu of rows t-4..t and the row loaded ahead, the
  // pending adjoints of rows t-4..t, 1/beta of cells t-3..t-1 and their adjoints
  double uw[6][NR], mw[6][NR], aw[6][NR], IBw[3][NR], Hw[3][NR];
#pragma unroll
  for (int k = 0; k < NR; ++k) {
#pragma unroll
    for (int r = 0; r < 6; ++r) uw[r][k] = mw[r][k] = aw[r][k] = 0.0;
#pragma unroll
    for (int r = 0; r < 3; ++r) IBw[r][k] = Hw[r][k] = 0.0;
  }
  int t = r0 - 4;
  int row = t % n2;
  if (row < 0) row += n2;
#pragma unroll
  for (int k = 0; k < NR; ++k) {
    uw[4][k] = ap.u[row * rs + col + k];
    mw[4][k] = ap.lam[row * rs + col + k];
  }
  auto step = [&](auto rot) {
    constexpr int Z = decltype(rot)::value;
    constexpr int s0 = Z % 6, s1 = (Z + 1) % 6, s2 = (Z + 2) % 6, s3 = (Z + 3) % 6,
                  s4 = (Z + 4) % 6, s5 = (Z + 5) % 6;
    constexpr int b0 = Z % 3, b1 = (Z + 1) % 3, b2 = (Z + 2) % 3;
    const int j = t - 4;  // the row that this step completes
    const bool done = j >= r0;
    row = row + 1 == n2 ? 0 : row + 1;
    // the next row, and the completed row's pointwise inputs
    double gq[5][NR], ba[NR], ba2[NR];
#pragma unroll
    for (int k = 0; k < NR; ++k) {
      uw[s5][k] = ap.u[row * rs + col + k];
      mw[s5][k] = ap.lam[row * rs + col + k];
    }
    const long base = j * rs + col;
    if (done) {
      if (ap.source) {
        const double* g = ap.gq + (long)j * n1 + lane * NR;
#pragma unroll
        for (int i = 0; i < 5; ++i)
#pragma unroll
          for (int k = 0; k < NR; ++k) gq[i][k] = g[i * Qn + k];
      }
#pragma unroll
      for (int k = 0; k < NR; ++k) {
        if (ap.base) ba[k] = ap.base[base + k];
        if (ap.base2) ba2[k] = ap.base2[base + k];
      }
    }
#pragma unroll
    for (int k = 0; k < NR; ++k) {
      aw[s4][k] = 0.0;
      // indicator of cell t-1
      IBw[b2][k] = fast_rcp(weno_beta<double>(uw[s2][k], uw[s3][k], uw[s4][k]));
      Hw[b2][k] = 0.0;
    }
    if (t >= r0) {
      // the face with window rows t-4..t: the lower face of row t-1 (C > 0)
      // or of row t-2
#pragma unroll
      for (int k = 0; k < NR; ++k) {
        const double g = P2 ? cdq2 * (mw[s3][k] - mw[s2][k]) : cdq2 * (mw[s2][k] - mw[s1][k]);
        const double y[5] = {uw[s0][k], uw[s1][k], uw[s2][k], uw[s3][k], uw[s4][k]};
        const double IB[3] = {IBw[b0][k], IBw[b1][k], IBw[b2][k]};
        double A[3], h[3], a[5] = {aw[s0][k], aw[s1][k], aw[s2][k], aw[s3][k], aw[s4][k]};
        al_face<P2>(y, IB, g, A, h);
        al_scatter<P2>(A, a);
        aw[s0][k] = a[0];
        aw[s1][k] = a[1];
        aw[s2][k] = a[2];
        aw[s3][k] = a[3];
        aw[s4][k] = a[4];
        Hw[b0][k] += h[0];
        Hw[b1][k] += h[1];
        Hw[b2][k] += h[2];
      }
    }
    if (t >= r0 + 2) {
      // the indicator adjoint of cell t-3 is complete: rows t-4, t-3, t-2
#pragma unroll
      for (int k = 0; k < NR; ++k) {
        const double H = Hw[b0][k];
        aw[s0][k] += H * beta_da(uw[s0][k], uw[s1][k], uw[s2][k]);
        aw[s1][k] += H * beta_db(uw[s0][k], uw[s1][k], uw[s2][k]);
        aw[s2][k] += H * beta_dc(uw[s0][k], uw[s1][k], uw[s2][k]);
      }
    }
    if (done) {
      double q1[NR];
      al_q1_row<NR, P1>(uw[s0], mw[s0], cdq1, q1);
#pragma unroll
      for (int k = 0; k < NR; ++k) {
        const double mu = mw[s0][k];
        double acc = q1[k] + aw[s0][k];
        if (ap.source)
          acc += ap.inv_tau * (ap.measure * (gq[0][k] + gq[1][k] * v1 + gq[2][k] * v2 +
                                             gq[3][k] * v3 + gq[4][k] * e3) - mu);
        double x = ap.b * mu + ap.c * acc;
        if (ap.base) x += ap.a * ba[k];
        if (ap.base2) x += ap.a2 * ba2[k];
        ap.out[base + k] = x;
      }
    }
  };
  using std::integral_constant;
  for (;;) {
    step(integral_constant<int, 0>());
    if (++t > r1 + 3) break;
    step(integral_constant<int, 1>());
    if (++t > r1 + 3) break;
    step(integral_constant<int, 2>());
    if (++t > r1 + 3) break;
    step(integral_constant<int, 3>());
    if (++t > r1 + 3) break;
    step(integral_constant<int, 4>());
    if (++t > r1 + 3) break;
    step(integral_constant<int, 5>());
    if (++t > r1 + 3) break;
  }
}

#ifndef BX_NO_KERNELS
// Blocks are numbered segment-major and spread over the eight XCDs in
// contiguous ranges (as for qline_kernel); wave w of a block takes p-cell
// 4 * (block's p-group) + w.
// Waves per SIMD: 3 with one cell per lane (149 VGPRs; at 4 it spills 106 of
// them), 2 with two (256 VGPRs).  Without LDS in the chain and with the rows
// loaded ahead that is enough: at 64^2 q x 32^2 p 67.7 us a launch with LDS
// lines and 4 waves, 54 us now, bound by FP64 issue.
constexpr int al_waves(int nr) { return nr == 1 ? 3 : 2; }

template <int NR>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(al_waves(NR)))) void adj_line_kernel(AdjParams ap, int nseg) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int nb = gridDim.x;
  const int t = (nb % 8 == 0) ? (blockIdx.x % 8) * (nb / 8) + blockIdx.x / 8 : blockIdx.x;
  const int npg = (ap.P + 3) / 4;
  const int seg = t / npg;
  const int p = (t % npg) * 4 + wave;
  if (p >= ap.P) return;  // no workgroup barriers below
  int j1, j2;
  fdivmod(p, ap.n_p1, 1.0f / float(ap.n_p1), j1);
  const int j23 = p / ap.n_p1;
  j2 = j23 % ap.n_p2;
  const bool pos1 = centre(ap.p1s, j1, ap.dp1) > 0.0;
  const bool pos2 = centre(ap.p2s, j2, ap.dp2) > 0.0;
  if (pos1) {
    if (pos2) al_march<NR, true, true>(ap, p, seg, nseg, lane);
    else al_march<NR, true, false>(ap, p, seg, nseg, lane);
  } else {
    if (pos2) al_march<NR, false, true>(ap, p, seg, nseg, lane);
    else al_march<NR, false, false>(ap, p, seg, nseg, lane);
  }
}
#endif

}  // namespace bx

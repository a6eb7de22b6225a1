// RK stage with p-advection (fields on) as two kernels over a chunk of q2
// rows, reference layout [q2][q1][P]:
//
//  * qdiff_kernel: D = -dF_1/dq1 - dF_2/dq2, the q-part of L.  A lane owns one
//    p-cell (64 consecutive p per wave: every access is one contiguous run)
//    and N neighbouring q1 cells, and marches along q2 with the window of its
//    cells in registers: each cell's aux quantity and state (dir_recon.h) are
//    formed once along q2 and shared by the tile along q1, instead of twice
//    per axis from a seven-cell gather.  On request it also sums the currents
//    of u (charge * mom_v1(f_left), mom_v2(f_bot), mom_v3(f)) over its 64 p
//    into partials.
//  * pplane_kernel: the rest of the stage.  A workgroup owns a q-cell, a thread
//    one (p1, p2) column, and marches along p3.  The p3 window lives in
//    registers; of p only the current plane is in LDS, where the p1 and p2
//    neighbours' values, aux quantities and states are shared, so each is
//    formed once per cell and axis.  A p-block in LDS as a whole (110 KB in
//    FP64 at 24^3) leaves one workgroup per CU; five planes (23 KB) leave
//    room for several, which cover each other's barriers.
//
// Measured at 64^2 x 24^3 (56.6 M cells, PPM in q, WENO5 in p) per stage:
// FP64 2470 us as one kernel (110 KB p-block, 1150 VALU per cell), 304 + 795 us
// as two; FP32 1010 us, 151 + 402 us.  qdiff_kernel issues on 73 % of the cycles
// (FP64, 139 VALU per cell, three waves per SIMD); pplane_kernel (212 VALU per
// cell) waits half of its time on its two barriers per plane with nine waves
// per CU.  D costs one more pass each way.
//
// The lanes of a wave have both upwind directions (natural p order), which
// dir_recon.h makes one instruction stream.
//
// Reference: df_dt_fvm.py:56-97, 214-224, 251-323; riemann.py:46-49;
// collision_operator.py:52-65, 102-128; moments.py:5-22.
#pragma once
#include <type_traits>
#include "dir_recon.h"
#include "qsweep.h"

namespace bx {

struct QDiffParams {
  StageParams sp;
  int r0, r1;                // q2 rows of the chunk
  int nslab, ntile, nseg;    // 64-wide p slabs, groups of 4 q1 tiles, q2 segments of the chunk
  void* D;                   // [r1 - r0][n_q1][P] (QK_DIV)
  double* part;              // [nslab][3 or 5][(r1 - r0) * n_q1] partial currents or moments
  const void* tab;           // [r1 - r0][n_q1][n_p1 + n_p2 + n_p3] Maxwellian factors (QK_STAGE)
};

// What qdiff_kernel produces: currents of u and / or the q-part of L, or the
// whole stage of a problem without p-advection, with the partial moments of
// its output (as a separate pass they would read it again).  The last is the
// slab kernel's work at 2-V sizes: 100 x 75 q x 30 x 28 p, PPM, FP64: 141 us per
// stage there; here 76 us, 6 for the Maxwellian factors and 5 for the moments.
// It is bound by its own latency (three waves per SIMD, 2900 waves) and, with
// scalar registers spilled to vector lanes, by about 190 VALU per cell; reading
// the stage's arguments again in every row instead made it slower (270 -> 284 us
// per step).  Two q1 cells per lane in FP64 (270 us per step; four: 316), four in
// FP32 (206; two: 221).
enum QDiffKind : int { QK_CUR = 1, QK_DIV = 2, QK_DIV_CUR = 3, QK_STAGE = 4 };

// Sums of x[0..M-1] (M at most 16) over the 64 lanes through the wave's LDS
// area of M rows: the sum of value lane / 4 is returned in every lane of the
// four (lanes 4 M and beyond: meaningless).  A butterfly of each value would
// cost six exchanges a value; here a lane sums 16 entries of one row.
constexpr int LS_PITCH = 65;
template <int M>
__device__ __forceinline__ double lane_sums(const double (&x)[M], double* area, int lane) {
#pragma unroll
  for (int i = 0; i < M; ++i) area[i * LS_PITCH + lane] = x[i];
  __builtin_amdgcn_wave_barrier();
  const double* r = area + (lane / 4 < M ? lane / 4 : 0) * LS_PITCH + (lane & 3) * 16;
  double s = 0.0;
#pragma unroll
  for (int e = 0; e < 16; ++e) s += r[e];
  __builtin_amdgcn_wave_barrier();
  s += __shfl_xor(s, 1, 64);
  return s + __shfl_xor(s, 2, 64);
}

// Consecutive values as a raw buffer: a lane offset and a uniform offset (both
// in bytes) address it without any vector arithmetic.
template <typename T>
struct Block {
  __amdgpu_buffer_rsrc_t r;
  __device__ __forceinline__ Block(const T* p, long n)
      : r(__builtin_amdgcn_make_buffer_rsrc((void*)p, 0, (int)(n * sizeof(T)), 0x00027000)) {}
  __device__ __forceinline__ T load(unsigned lane, unsigned off) const {
    if constexpr (sizeof(T) == 8)
      return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, lane, off, 0));
    else
      return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, lane, off, 0));
  }
  __device__ __forceinline__ void store(T x, unsigned lane, unsigned off) const {
    typedef unsigned V2 __attribute__((ext_vector_type(2)));
    if constexpr (sizeof(T) == 8)
      __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(V2, x), r, lane, off, 0);
    else
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, x), r, lane, off, 0);
  }
};

// GH: one of the q axes has ghost rows (plain addressing of whole rows).
template <typename T, int R, int N, bool GH, int KIND>
__global__ __launch_bounds__(256, (KIND == QK_STAGE ? 3 : 1)) void qdiff_kernel(QDiffParams q) {
  constexpr bool DIV = (KIND & QK_DIV) != 0, CUR = (KIND & QK_CUR) != 0, STAGE = KIND == QK_STAGE;
  constexpr int NS = CUR ? 3 : STAGE ? 4 : 0;  // sums per cell taken together
  __shared__ double area[NS ? 4 : 1][NS ? NS * N * LS_PITCH : 1];
  const StageParams& sp = q.sp;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int nb = gridDim.x;
  int b = (nb % 8 == 0) ? (blockIdx.x % 8) * (nb / 8) + blockIdx.x / 8 : blockIdx.x;
  const int slab = b % q.nslab;
  b /= q.nslab;
  const int c0 = ((b % q.ntile) * 4 + wave) * N;  // first q1 cell of the tile
  const int seg = b / q.ntile;
  const int n1 = sp.n_q1, n2 = sp.n_q2;
  if (c0 >= n1) return;  // no workgroup barriers below
  const long P = sp.P;
  const bool valid = slab * 64 + lane < sp.P;
  const unsigned p = valid ? slab * 64 + lane : sp.P - 1;
  const unsigned pb = p * (unsigned)sizeof(T);
  const int rows = q.r1 - q.r0;
  const int ra = q.r0 + (int)((long)seg * rows / q.nseg);
  const int rb = q.r0 + (int)((long)(seg + 1) * rows / q.nseg);

  int j1, j2;
  const int j23 = fdivmod((int)p, sp.n_p1, 1.0f / float(sp.n_p1), j1);
  const int j3 = fdivmod(j23, sp.n_p2, 1.0f / float(sp.n_p2), j2);
  const double v1 = centre(sp.p1s, j1, sp.dp1), v2 = centre(sp.p2s, j2, sp.dp2);
  const double v3 = CUR || STAGE ? centre(sp.p3s, j3, sp.dp3) : 0.0;
  const T C1 = T(v1), C2 = T(v2);
  // QK_STAGE: energy weight, RK coefficients and the offsets of the lane's
  // Maxwellian factors in a q-cell's row of the table
  const double ev = 0.5 * ((v1 * v1 + v2 * v2) + v3 * v3);
  const T ta = T(sp.a), tb = T(sp.b), tcdt = T(sp.cdt), ttau = T(sp.inv_tau);
  const bool use_un = sp.a != 0.0, w_is_u = sp.w == sp.u, b_one = sp.b == 1.0;
  const int TS = sp.n_p1 + sp.n_p2 + sp.n_p3;
  const unsigned x1 = j1 * (unsigned)sizeof(T), x2 = (sp.n_p1 + j2) * (unsigned)sizeof(T),
                 x3 = (sp.n_p1 + sp.n_p2 + j3) * (unsigned)sizeof(T);
  const bool pos1 = C1 > T(0), pos2 = C2 > T(0);
  const DirCoef<T> k1 = dir_coef<R, T>(pos1), k2 = dir_coef<R, T>(pos2);
  const T tinv1 = T(sp.inv_dq1), tinv2 = T(sp.inv_dq2);
  const bool do2 = n2 > 1;
  const T* u = (const T*)sp.u;

  // Columns c0-3 .. c0+N+2 of the tile: cell m is column c0 - 3 + m, a
  // periodic image or (GH) a ghost column beyond the domain.  A cell of the
  // tile past the last column is a neighbour of the cells before it; its own
  // q2 neighbours, never used, repeat the nearest interior row of a ghost
  // column.  Periodic q: the byte offset of the column in its row of q-cells.
  constexpr int RE = recon_reach(R) + 1;  // halo cells read on each side
  constexpr int M = N + 6;
  int col[M];
#pragma unroll
  for (int m = 0; m < M; ++m) {
    const int c = q_row_1(sp, c0 - 3 + m, 0);
    col[m] = GH ? c : c * (int)(P * (long)sizeof(T));
  }
  // row of q-cells i2 (interior) / of the window index i2 (any)
  auto buffer = [&](int i2) { return Block<T>(u + (long)i2 * n1 * P, n1 * P); };
  auto load_halo = [&](int i2, int m) -> T {
    if constexpr (GH) {
      const int row = col[m] < sp.Q ? col[m] + n1 * i2 : col[m] + i2;
      return u[(long)row * P + p];
    } else {
      return buffer(i2).load(pb, col[m]);
    }
  };
  auto load_own = [&](int i2, int k) -> T {
    if constexpr (GH) {
      const int near = i2 < 0 ? 0 : (i2 < n2 ? i2 : n2 - 1);
      const int row = col[k + 3] < sp.Q ? col[k + 3] + q_row_2(sp, 0, i2) : col[k + 3] + near;
      return u[(long)row * P + p];
    } else {
      return buffer(i2).load(pb, col[k + 3]);
    }
  };
  auto image = [&](int i2) { return GH ? i2 : qm_mod(i2, n2); };

  // Y: window rows r-1 .. r+3 and the row on its way; st: state of row r; bs:
  // upwind state of its lower face; PPM: A[0] slope of row r+1, A[1] value at
  // the face between rows r and r+1; else aux quantities, rotating
  T Y[6][N], A[3][N], st[N], H[2][6], bs[N];
#pragma unroll
  for (int k = 0; k < N; ++k) {
    st[k] = bs[k] = T(0);
    A[0][k] = A[1][k] = A[2][k] = T(0);
  }
  if (do2) {
    T z[2][N];
#pragma unroll
    for (int j = 0; j < 7; ++j) {
      const int i2 = image(ra - 3 + j);
#pragma unroll
      for (int k = 0; k < N; ++k) (j < 2 ? z[j < 2 ? j : 0][k] : Y[j < 2 ? 0 : j - 2][k]) = load_own(i2, k);
    }
#pragma unroll
    for (int k = 0; k < N; ++k) {
      const T am2 = dir_aux<R, T>(z[0][k], z[1][k], Y[0][k]);
      const T am1 = dir_aux<R, T>(z[1][k], Y[0][k], Y[1][k]);
      const T a0 = dir_aux<R, T>(Y[0][k], Y[1][k], Y[2][k]);
      const T a1 = dir_aux<R, T>(Y[1][k], Y[2][k], Y[3][k]);
      const T sm = dir_state<R, T>(z[0][k], z[1][k], Y[0][k], Y[1][k], Y[2][k], am2, am1, a0, pos2,
                                   k2);
      st[k] = dir_state<R, T>(z[1][k], Y[0][k], Y[1][k], Y[2][k], Y[3][k], am1, a0, a1, pos2, k2);
      bs[k] = pos2 ? sm : st[k];
      if constexpr (R == RC_PPM) {
        A[0][k] = a1;
        A[1][k] = dir_ppm_face(Y[1][k], Y[2][k], a0, a1);
      } else {
        A[0][k] = a0;
        A[1][k] = a1;
      }
    }
  } else {
#pragma unroll
    for (int k = 0; k < N; ++k) Y[1][k] = load_own(ra, k);
  }
#pragma unroll
  for (int m = 0; m < 6; ++m)
    if (m >= 3 - RE && m < 3 + RE) H[0][m] = load_halo(ra, m < 3 ? m : m + N);

  T* Dp = DIV ? (T*)q.D : nullptr;
  int r = ra, next = image(ra + 4);  // the window row loaded next
  auto row = [&](auto rot) {
#pragma clang fp contract(off)
    constexpr int S = decltype(rot)::value;
    constexpr int y0 = S % 6, y1 = (S + 1) % 6, y2 = (S + 2) % 6, y3 = (S + 3) % 6,
                  y4 = (S + 4) % 6, yl = (S + 5) % 6;
    constexpr int ka = S % 3, kb = (S + 1) % 3, kc = (S + 2) % 3;
    constexpr int cu = S % 2, nx = (S + 1) % 2;
    // the next row's loads, in flight across this row's work (a segment's
    // last row loads what it does not use)
    if (do2) {
#pragma unroll
      for (int k = 0; k < N; ++k) Y[yl][k] = load_own(next, k);
      next = !GH && next + 1 == n2 ? 0 : next + 1;
    }
    {
      const int rn = r + 1 < n2 ? r + 1 : r;
#pragma unroll
      for (int m = 3 - RE; m < 3 + RE; ++m) H[nx][m] = load_halo(rn, m < 3 ? m : m + N);
    }
    // flux differences and lower-face states along q1 and q2
    T f[N], t1[N], t2[N], b1[N], b2[N];
#pragma unroll
    for (int k = 0; k < N; ++k) {
      f[k] = Y[y1][k];
      t2[k] = T(0);
      b2[k] = f[k];
    }
    {
      // cells -3 .. N+2 of the row
      T v[M], a[N + 4], s[N + 2];
#pragma unroll
      for (int m = 0; m < M; ++m)
        v[m] = m < 3 ? (m >= 3 - RE ? H[cu][m] : T(0))
               : m < N + 3 ? f[m - 3 < N ? m - 3 : 0]
                           : (m - N < 3 + RE ? H[cu][m - N < 6 ? m - N : 0] : T(0));
#pragma unroll
      for (int m = 0; m < N + 4; ++m) a[m] = dir_aux<R, T>(v[m], v[m + 1], v[m + 2]);
#pragma unroll
      for (int m = 0; m < N + 2; ++m)
        s[m] = dir_state<R, T>(v[m], v[m + 1], v[m + 2], v[m + 3], v[m + 4], a[m], a[m + 1],
                               a[m + 2], pos1, k1);
      T F[N + 1];  // upwind states of the faces
#pragma unroll
      for (int m = 0; m <= N; ++m) F[m] = pos1 ? s[m] : s[m + 1];
#pragma unroll
      for (int k = 0; k < N; ++k) {
        t1[k] = ql_fma(C1, F[k + 1], -(C1 * F[k]));
        b1[k] = F[k];
      }
    }
    if (do2) {
#pragma unroll
      for (int k = 0; k < N; ++k) {
        T sn;
        if constexpr (R == RC_PPM) {
          const T ap = dir_aux<R, T>(Y[y2][k], Y[y3][k], Y[y4][k]);
          const T fp = dir_ppm_face(Y[y2][k], Y[y3][k], A[0][k], ap);
          sn = dir_ppm_state(Y[y2][k], A[1][k], fp, pos2);
          A[0][k] = ap;
          A[1][k] = fp;
        } else {
          A[kc][k] = dir_aux<R, T>(Y[y2][k], Y[y3][k], Y[y4][k]);
          sn = dir_state<R, T>(Y[y0][k], Y[y1][k], Y[y2][k], Y[y3][k], Y[y4][k], A[ka][k],
                               A[kb][k], A[kc][k], pos2, k2);
        }
        const T fs = pos2 ? st[k] : sn;  // upwind state of the row's upper face
        t2[k] = ql_fma(C2, fs, -(C2 * bs[k]));
        b2[k] = bs[k];
        bs[k] = fs;
        st[k] = sn;
      }
    }
    if constexpr (DIV) {
      const Block<T> Dr(Dp + (long)(r - q.r0) * n1 * P, n1 * P);
      if (valid) {
#pragma unroll
        for (int k = 0; k < N; ++k)
          if (c0 + k < n1)
            Dr.store(ql_fma(-t1[k], tinv1, -(t2[k] * tinv2)), pb,
                     (c0 + k) * (int)(P * (long)sizeof(T)));
      }
    }
    if constexpr (STAGE) {
      const long at = (long)r * n1 * P;
      const Block<T> wr((const T*)sp.w + at, n1 * P), unr((const T*)sp.un + at, n1 * P),
          outr((const T*)sp.out + at, n1 * P),
          tr((const T*)q.tab + (long)(r - q.r0) * n1 * TS, (long)n1 * TS);
      T wv[N], uv[N], fmb[N];
#pragma unroll
      for (int k = 0; k < N; ++k) {
        const int c = c0 + k < n1 ? c0 + k : n1 - 1;
        const int o = c * (int)(P * (long)sizeof(T)), to = c * TS * (int)sizeof(T);
        wv[k] = w_is_u ? f[k] : wr.load(pb, o);
        uv[k] = use_un ? unr.load(pb, o) : T(0);
        fmb[k] = T(0);
        if (sp.source) {
          fmb[k] = tr.load(x1, to);
          if (sp.p_dim >= 2) fmb[k] = fmb[k] * tr.load(x2, to);
          if (sp.p_dim >= 3) fmb[k] = fmb[k] * tr.load(x3, to);
        }
      }
      double x[4 * N], m3[N];
#pragma unroll
      for (int k = 0; k < N; ++k) {
        T d = ql_fma(-t1[k], tinv1, -(t2[k] * tinv2));
        if (sp.source) d = ql_fma(fmb[k] - f[k], ttau, d);
        const T tv = ql_fma(d, tcdt, wv[k]);
        const T o = use_un ? ql_fma(tb, tv, ta * uv[k]) : (b_one ? tv : tb * tv);
        if (valid && c0 + k < n1) outr.store(o, pb, (c0 + k) * (int)(P * (long)sizeof(T)));
        const double od = valid ? double(o) : 0.0;
        x[4 * k] = od;
        x[4 * k + 1] = od * v1;
        x[4 * k + 2] = od * v2;
        x[4 * k + 3] = od * ev;
        m3[k] = od * v3;
      }
      const int idx = lane / 4, k = idx / 4, comp = idx - 4 * k;
      const long nq = (long)rows * n1, cell = (long)(r - q.r0) * n1 + c0 + k;
      const double sum = lane_sums<4 * N>(x, area[wave], lane);
      if ((lane & 3) == 0 && k < N && c0 + k < n1)
        q.part[((long)slab * 5 + (comp < 3 ? comp : 4)) * nq + cell] = sum;
      // mom_v3: of one p3 cell it is the density's multiple
      if (sp.n_p3 > 1) {
        const double s3 = lane_sums<N>(m3, area[wave], lane);
        if ((lane & 3) == 0 && idx < N && c0 + idx < n1)
          q.part[((long)slab * 5 + 3) * nq + (long)(r - q.r0) * n1 + c0 + idx] = s3;
      }
    }
    if constexpr (CUR) {
      double x[3 * N];
#pragma unroll
      for (int k = 0; k < N; ++k) {
        x[3 * k] = valid ? double(b1[k]) * v1 : 0.0;
        x[3 * k + 1] = valid ? double(b2[k]) * v2 : 0.0;
        x[3 * k + 2] = valid ? double(f[k]) * v3 : 0.0;
      }
      const double sum = lane_sums<3 * N>(x, area[wave], lane);
      const int idx = lane / 4, k = idx / 3, comp = idx - 3 * k;
      if ((lane & 3) == 0 && k < N && c0 + k < n1)
        q.part[((long)slab * 3 + comp) * ((long)rows * n1) + (long)(r - q.r0) * n1 + c0 + k] = sum;
    }
  };
  using std::integral_constant;
  // six rows per pass, so the register roles are back in place on the back edge
  while (r < rb) {
    row(integral_constant<int, 0>());
    if (++r == rb) break;
    row(integral_constant<int, 1>());
    if (++r == rb) break;
    row(integral_constant<int, 2>());
    if (++r == rb) break;
    row(integral_constant<int, 3>());
    if (++r == rb) break;
    row(integral_constant<int, 4>());
    if (++r == rb) break;
    row(integral_constant<int, 5>());
    ++r;
  }
}

// J of the chunk from the partials: 16 threads per q-cell take interleaved
// slabs, and the 16 sums are added in order.
constexpr int QCUR_SUBS = 16;
static __global__ __launch_bounds__(256) void qcur_reduce_kernel(const double* part, int nslab, int nq,
                                                          int q0, int Q, double charge,
                                                          double measure, double* J) {
  __shared__ double red[QCUR_SUBS][16];
  const int ci = threadIdx.x & 15, sub = threadIdx.x >> 4;
  const int i = blockIdx.x * 16 + ci, comp = blockIdx.y;
  double a = 0.0;
  if (i < nq)
    for (int s = sub; s < nslab; s += QCUR_SUBS) a += part[((long)s * 3 + comp) * nq + i];
  red[sub][ci] = a;
  __syncthreads();
  if (sub == 0 && i < nq) {
    double x = 0.0;
#pragma unroll
    for (int s = 0; s < QCUR_SUBS; ++s) x += red[s][ci];
    J[(long)comp * Q + q0 + i] = charge * (x * measure);
  }
}

// Maxwellian factors of the chunk's q-cells from the raw moments
// (collision_operator.py:52-65, 102-116): per q-cell prefactor * e1 (rounded as
// the other stage kernels round it), e2, e3; a wave per q-cell.
template <typename T>
__global__ __launch_bounds__(256) void qtab_kernel(StageParams sp, int q0, int nq, T* tab) {
  const int i = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (i >= nq) return;
  const BgkCell b = qcell_bgk(sp, q0 + i);
  const T pref = T(maxwell_prefactor(b, sp.mass, sp.kB, sp.p_dim));
  const int TS = sp.n_p1 + sp.n_p2 + sp.n_p3;
  T* row = tab + (long)i * TS;
  for (int j = lane; j < TS; j += 64) {
    const int ax = j < sp.n_p1 ? 0 : j < sp.n_p1 + sp.n_p2 ? 1 : 2;
    const double v = ax == 0 ? centre(sp.p1s, j, sp.dp1)
                     : ax == 1 ? centre(sp.p2s, j - sp.n_p1, sp.dp2)
                               : centre(sp.p3s, j - sp.n_p1 - sp.n_p2, sp.dp3);
    const T e = T(maxwell_factor(v, ax == 0 ? b.u1 : ax == 1 ? b.u2 : b.u3, b.T, sp.mass, sp.kB));
    row[j] = ax == 0 ? pref * e : e;
  }
}

// Moment blocks of the chunk from the partial moments: 16 threads per q-cell
// take interleaved slabs, and the 16 sums are added in order.
static __global__ __launch_bounds__(256) void qmom_reduce_kernel(StageParams sp, const double* part,
                                                                 int nslab, int nq, int q0) {
  __shared__ double red[5][QCUR_SUBS][16];
  const int ci = threadIdx.x & 15, sub = threadIdx.x >> 4;
  const int i = blockIdx.x * 16 + ci;
  double a[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
  if (i < nq)
    for (int s = sub; s < nslab; s += QCUR_SUBS)
#pragma unroll
      for (int k = 0; k < 5; ++k)
        if (k != 3 || sp.n_p3 > 1) a[k] += part[((long)s * 5 + k) * nq + i];
#pragma unroll
  for (int k = 0; k < 5; ++k) red[k][sub][ci] = a[k];
  __syncthreads();
  if (sub == 0 && i < nq) {
    double m[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      double x = 0.0;
#pragma unroll
      for (int s = 0; s < QCUR_SUBS; ++s) x += red[k][s][ci];
      m[k] = x * sp.measure;
    }
    if (sp.n_p3 == 1) m[3] = m[0] * centre(sp.p3s, 0, sp.dp3);
    finish_moments(sp, q0 + i, m);
  }
}

// Stage forms pplane_kernel is specialised for (out = a*un + b*(w + cdt*L)).
enum PlaneMode : int {
  PM_FIRST = 0,    // w == u, a == 0, b == 1: the first stage of either stepper
  PM_COMBINE = 1,  // w == u, a != 0: SSP-RK3 stages 2 and 3
  PM_MIDPOINT = 2, // w != u, a == 0, b == 1: the second stage of the RK2 midpoint
  PM_GENERAL = 3   // decided at run time
};

// State of the centre cell f of y[0], y[1], f, y[2], y[3] along a p axis (the
// face on its downwind side) with its aux quantity k and its neighbours' km
// (of y[1]) and kp (of y[2]).  FP32 WENO5 takes the right-face form on the
// window in upwind order, the rounding the FP32-bulk results have always had.
template <int R, typename T>
__device__ __forceinline__ T p_state(const T* y, T f, T km, T k, T kp, bool pos) {
#pragma clang fp contract(off)
  if constexpr (R == RC_WENO5 && sizeof(T) == 4) {
    const T y0 = pos ? y[0] : y[3], y1 = pos ? y[1] : y[2], y3 = pos ? y[2] : y[1],
            y4 = pos ? y[3] : y[0];
    return qs_face(y0, y1, f, y3, y4, pos ? km : kp, k, pos ? kp : km);
  } else {
    return dir_state<R, T>(y[0], y[1], f, y[2], y[3], km, k, kp, pos, dir_coef<R, T>(pos));
  }
}

// Flux difference of a cell from its state s and the state sn of its
// neighbour on the upwind side: C*s - C*sn (C > 0) or C*sn - C*s.
template <int R, typename T>
__device__ __forceinline__ T p_diff(T C, bool pos, T s, T sn) {
#pragma clang fp contract(off)
  if constexpr (R != RC_WENO5 && sizeof(T) == 4) {
    const T hi = pos ? s : sn, lo = pos ? sn : s;
    return ql_fma(C, hi, -(C * lo));
  } else {
    return ql_fma(aabs(C), s, -(aabs(C) * sn));
  }
}

#define PP_SCHED() do { if constexpr (sizeof(T) == 8) __builtin_amdgcn_sched_barrier(0); } while (0)

// The stage value of the chunk's q-cells from D (see the head of the file).
// All three p axes have more than one cell.
template <typename T, int RP, int MODE, int NT, int WAVES>
__global__ __launch_bounds__(NT, WAVES) void pplane_kernel(StageParams sp, const T* D, int q0) {
  extern __shared__ __align__(16) unsigned char smem[];
  // the plane's aux quantities and states, and the window of planes: FP32
  // keeps its column's window in registers and shares this plane and the next;
  // FP64 keeps it in LDS (six planes), so that the march fits in the 96
  // registers that leave two workgroups per CU
  constexpr bool WL = sizeof(T) == 8;
  __shared__ T U[WL ? 6 : 2][NT], K3[WL ? 3 : 1][WL ? NT : 1], K1[NT], K2[NT], S1[NT], S2[NT];
  __shared__ double red[5][NT / 64];
  __shared__ double bgk[5];
  const int t = threadIdx.x, NB = blockDim.x;
  T* e1 = reinterpret_cast<T*>(smem);
  T* e2 = e1 + sp.n_p1;
  T* e3 = e2 + sp.n_p2;
  const int n1 = sp.n_p1, n2 = sp.n_p2, n3 = sp.n_p3, ncol = n1 * n2;
  const int q = q0 + blockIdx.x;
  const bool live = t < ncol;
  const int c = live ? t : 0;
  int j1;
  const int j2 = fdivmod(c, n1, 1.0f / float(n1), j1);
  // LDS slots of the p1 and p2 neighbours (periodic)
  int m1[4], m2[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int o = k < 2 ? k - 2 : k - 1;
    m1[k] = c - j1 + wrap_once(j1 + o, n1);
    m2[k] = j1 + n1 * wrap_once(j2 + o, n2);
  }
  const double v1 = centre(sp.p1s, j1, sp.dp1), v2 = centre(sp.p2s, j2, sp.dp2);
  const long base = (long)q * sp.P;
  const Block<T> u((const T*)sp.u + base, sp.P), wv((const T*)sp.w + base, sp.P),
      unv((const T*)sp.un + base, sp.P), outv((const T*)sp.out + base, sp.P),
      Dv(D + (long)blockIdx.x * sp.P, sp.P);
  const unsigned cb = t * (unsigned)sizeof(T), row = ncol * (unsigned)sizeof(T);
  const bool use_un = MODE == PM_GENERAL ? sp.a != 0.0 : MODE == PM_COMBINE;
  const bool w_is_u = MODE == PM_GENERAL ? sp.w == sp.u : MODE != PM_MIDPOINT;
  const bool b_one = MODE == PM_GENERAL ? sp.b == 1.0 : MODE != PM_COMBINE;
  const T ta = T(sp.a), tb = T(sp.b), tcdt = T(sp.cdt), ttau = T(sp.inv_tau);
  const T ti1 = T(sp.inv_dp1), ti2 = T(sp.inv_dp2), ti3 = T(sp.inv_dp3);
  auto load = [&](int j) { return u.load(cb, qm_mod(j, n3) * row); };

  // Loads run a plane ahead of their use: the row that enters the p3 window
  // next (L) and the row's pointwise inputs.  (Past the last plane the buffers'
  // bounds return 0.)
  T L, DC, WC, UC;
  auto load_pointwise = [&](unsigned o) {
    DC = Dv.load(cb, o);
    WC = w_is_u ? T(0) : wv.load(cb, o);
    UC = use_un ? unv.load(cb, o) : T(0);
  };
  // p3: window rows -1 .. 3 in Y[0..4] (and two rows before it)
  T Y[6], A[3];
  const T z0 = load(-3), z1 = load(-2);
#pragma unroll
  for (int j = 0; j < 5; ++j) Y[j] = load(j - 1);
  L = load(4);
  load_pointwise(0);

  // the q-cell's Maxwellian: one lane derives it from the raw moments, all
  // threads fill the factor tables (1 along the axes that have no factor)
  if (sp.source && t == 0) {
    const BgkCell bc = qcell_bgk(sp, q);
    bgk[0] = maxwell_prefactor(bc, sp.mass, sp.kB, sp.p_dim);
    bgk[1] = bc.u1;
    bgk[2] = bc.u2;
    bgk[3] = bc.u3;
    bgk[4] = bc.T;
  }
  if constexpr (WL) {
#pragma unroll
    for (int j = 0; j < 5; ++j) U[j][t] = Y[j];
  } else {
    U[0][t] = Y[1];
  }
  __syncthreads();
  T c12 = T(0);
  if (sp.source) {
    for (int i = t; i < n1 + n2 + n3; i += NB) {
      const int ax = i < n1 ? 0 : i < n1 + n2 ? 1 : 2;
      const double v = ax == 0 ? centre(sp.p1s, i, sp.dp1)
                       : ax == 1 ? centre(sp.p2s, i - n1, sp.dp2)
                                 : centre(sp.p3s, i - n1 - n2, sp.dp3);
      e1[i] = ax < sp.p_dim ? T(maxwell_factor(v, bgk[1 + ax], bgk[4], sp.mass, sp.kB)) : T(1);
    }
    __syncthreads();
    c12 = (T(bgk[0]) * e1[j1]) * e2[j2];
  }
  // fields of the q-cell (advection_terms.py:179-186)
  const double em = sp.charge / sp.mass;
  const int Q = sp.Q;
  const double E1 = sp.fp1[q], E2 = sp.fp2[Q + q], E3 = sp.fp3[2 * Q + q];
  const double B12 = sp.fp1[4 * Q + q], B13 = sp.fp1[5 * Q + q];
  const double B21 = sp.fp2[3 * Q + q], B23 = sp.fp2[5 * Q + q];
  const double B31 = sp.fp3[3 * Q + q], B32 = sp.fp3[4 * Q + q];
  const double C1u = ql_fma(v2, B13, E1), C2u = v1 * B23;  // the parts of C_p1, C_p2 fixed in p3
  const T C3 = T(em * (E3 + v1 * B32 - v2 * B31));
  int up3 = C3 > T(0);
  // p3 states of the previous row and of this one
  T sp3, st;
  {
    const T am2 = dir_aux<RP, T>(z0, z1, Y[0]);
    const T am1 = dir_aux<RP, T>(z1, Y[0], Y[1]);
    A[0] = dir_aux<RP, T>(Y[0], Y[1], Y[2]);
    A[1] = dir_aux<RP, T>(Y[1], Y[2], Y[3]);
    const T ym[4] = {z0, z1, Y[1], Y[2]}, yc[4] = {z1, Y[0], Y[2], Y[3]};
    sp3 = p_state<RP, T>(ym, Y[0], am2, am1, A[0], up3 != 0);
    st = p_state<RP, T>(yc, Y[1], am1, A[0], A[1], up3 != 0);
    if constexpr (WL) {
      K3[0][t] = A[0];
      K3[1][t] = A[1];
    }
  }
  double s0 = 0.0, s3 = 0.0, s33 = 0.0;  // sums over p3 of x, x v3, x v3^2
  int j = 0;
  unsigned off = 0, ahead = qm_mod(5, n3) * row;  // ahead: the row loaded next
  auto plane = [&](auto rot) {
#pragma clang fp contract(off)
    constexpr int S = decltype(rot)::value;
    constexpr int y1 = (S + 1) % 6, yl = (S + 5) % 6;
    constexpr int ka = S % 3, kb = (S + 1) % 3, kc = (S + 2) % 3;
    constexpr int hf = WL ? y1 : S % 2, nx = (S + 1) % 2;
    // window row j - 1 + k
    auto win = [&](int k) -> T { return WL ? U[(S + k) % 6][t] : Y[(S + k) % 6]; };
    if constexpr (WL) U[yl][t] = L;
    else Y[yl] = L;
    L = u.load(cb, ahead);
    ahead = ahead + row == n3 * row ? 0 : ahead + row;
    const T f = win(1);
    const double v3 = centre(sp.p3s, j, sp.dp3);
    // what a thread shares goes through LDS for itself as well, and (FP64) the
    // axes' work is not interleaved: fewer registers live across the plane
    // aux quantities of the plane's cells along p1 and p2
    K1[t] = dir_aux<RP, T>(U[hf][m1[1]], f, U[hf][m1[2]]);
    PP_SCHED();
    K2[t] = dir_aux<RP, T>(U[hf][m2[1]], f, U[hf][m2[2]]);
    __syncthreads();
    // states; FP32: the next plane goes into the other half of U
    {
      const T a[4] = {U[hf][m1[0]], U[hf][m1[1]], U[hf][m1[2]], U[hf][m1[3]]};
      const T C1 = T(em * ql_fma(-v3, B12, C1u));
      S1[t] = p_state<RP, T>(a, f, K1[m1[1]], K1[t], K1[m1[2]], C1 > T(0));
    }
    PP_SCHED();
    {
      const T b[4] = {U[hf][m2[0]], U[hf][m2[1]], U[hf][m2[2]], U[hf][m2[3]]};
      const T C2 = T(em * (ql_fma(v3, B21, E2) - C2u));
      S2[t] = p_state<RP, T>(b, f, K2[m2[1]], K2[t], K2[m2[2]], C2 > T(0));
    }
    PP_SCHED();
    // pos3 is formed anew in each plane, so what is selected by it does not
    // stay in registers across the march
    asm volatile("" : "+v"(up3));
    const bool pos3 = up3 != 0;
    T d3;
    {
      const T yn[4] = {win(0), win(1), win(3), win(4)}, y = win(2);
      if constexpr (!WL) U[nx][t] = y;
      const T an = dir_aux<RP, T>(y, yn[2], yn[3]);
      const T sn = p_state<RP, T>(yn, y, WL ? K3[ka][t] : A[ka], WL ? K3[kb][t] : A[kb], an, pos3);
      if constexpr (WL) K3[kc][t] = an;
      else A[kc] = an;
      d3 = p_diff<RP, T>(C3, pos3, st, pos3 ? sp3 : sn);
      sp3 = st;
      st = sn;
    }
    __syncthreads();
    const T C1 = T(em * ql_fma(-v3, B12, C1u)), C2 = T(em * (ql_fma(v3, B21, E2) - C2u));
    const bool pos1 = C1 > T(0), pos2 = C2 > T(0);
    // flux differences: along p1 and p2 from the neighbour on the upwind side
    T dp = p_diff<RP, T>(C1, pos1, S1[t], S1[pos1 ? m1[1] : m1[2]]) * ti1;
    dp = ql_fma(p_diff<RP, T>(C2, pos2, S2[t], S2[pos2 ? m2[1] : m2[2]]), ti2, dp);
    dp = ql_fma(d3, ti3, dp);
    T d = DC;
    if (sp.source) d = ql_fma(c12 * e3[j] - f, ttau, d);
    d = d - dp;
    const T tv = ql_fma(d, tcdt, w_is_u ? f : WC);
    const T x = use_un ? ql_fma(tb, tv, ta * UC) : (b_one ? tv : tb * tv);
    if (live) outv.store(x, cb, off);
    load_pointwise(off + row);
    const double xd = double(x), xv = xd * v3;
    s0 += xd;
    s3 += xv;
    s33 = ql_fma(xv, v3, s33);
    off += row;
  };
  using std::integral_constant;
  while (j < n3) {
    plane(integral_constant<int, 0>());
    if (++j == n3) break;
    plane(integral_constant<int, 1>());
    if (++j == n3) break;
    plane(integral_constant<int, 2>());
    if (++j == n3) break;
    plane(integral_constant<int, 3>());
    if (++j == n3) break;
    plane(integral_constant<int, 4>());
    if (++j == n3) break;
    plane(integral_constant<int, 5>());
    ++j;
  }
  if (!sp.mom_out) return;
  // the column's velocities again (not kept across the march)
  int ce = c;
  asm volatile("" : "+v"(ce));
  int i1;
  const int i2 = fdivmod(ce, n1, 1.0f / float(n1), i1);
  const double w1 = centre(sp.p1s, i1, sp.dp1), w2 = centre(sp.p2s, i2, sp.dp2);
  double m[5] = {s0, s0 * w1, s0 * w2, s3, 0.5 * (s0 * (w1 * w1 + w2 * w2) + s33)};
  const int wave = t >> 6, lane = t & 63;
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    double x = live ? m[k] : 0.0;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
    if (lane == 0) red[k][wave] = x;
  }
  __syncthreads();
  if (t == 0) {
    for (int k = 0; k < 5; ++k) {
      double x = red[k][0];
      for (int w = 1; w < NB / 64; ++w) x += red[k][w];
      m[k] = x * sp.measure;
    }
    finish_moments(sp, q, m);
  }
}

}  // namespace bx

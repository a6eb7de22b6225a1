// Electrostatic fields of a charge density on the periodic q grid
// (electrostatic/fft.py:9-78): phi_hat = rho_hat / (4 pi^2 |k|^2) with
// phi_hat(0, 0) = 0, E = -grad phi / eps.
//
// Grids of one axis: E is the convolution of rho with a fixed odd kernel, one
// launch.  Grids of two: Fourier sums along q1 (real input, half the
// wavenumbers), along q2 there and back around the division, and back along
// q1, one launch each.  The sums are written out, O(N) per value: at the sizes
// the electrostatic problems have, the arithmetic (9216 cells: 4 MFMA) costs
// less than the launches of a fast transform and of the elementwise operations
// around it (35 launches a solve).  Whole electrostatic RK2 steps, which solve
// twice, with the transforms / with these kernels: 96 q-cells x 64 p 481 / 65 us,
// 1024 x 64 489 / 85, 32^2 x 24^2 505 / 101, 200^2 x 8^2 1584 / 1286 (the stage kernel
// is most of the last).  At 512^2 the sums lose (7965 / 8404): grids beyond 2^25
// terms per sum and axis pair go through the transforms.
//
// A Nyquist wavenumber contributes nothing to the field along its own axis:
// its derivative is purely imaginary on the grid.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstring>

#include "../../include/boltx.h"
#include "bx_status.h"

namespace bx {
namespace {

constexpr int POI_MAX_1D = 4096;  // r and the kernel in LDS: 64 KB
constexpr int POI_MAX_2D = 512;        // per axis (columns and twiddles in LDS)
constexpr long POI_MAX_WORK = 1L << 25;  // n1 n2 (n1 + n2)
constexpr int POI_SPECIES = 8;
constexpr int POI_THREADS = 256;

struct PoiDensity {
  int ns;
  const double* n[POI_SPECIES];
  double charge[POI_SPECIES];
  __device__ double at(int q) const {
    double r = charge[0] * n[0][q];
    for (int s = 1; s < ns; ++s) r = r + charge[s] * n[s][q];
    return r;
  }
};

// Workspace of a two-axis grid, doubles: twiddles cos, sin (2 pi m / N) of both axes,
// then the half-spectra R, G1, G2 as [n2][h] complex.
struct PoiMap {
  int n1, n2, h;
  long tw1, tw2, R, G1, G2, total;
};
PoiMap poi_map(int n1, int n2) {
  PoiMap m;
  m.n1 = n1;
  m.n2 = n2;
  m.h = n1 / 2 + 1;
  const long c = 2L * n2 * m.h;
  m.tw1 = 0;
  m.tw2 = 2L * n1;
  m.R = m.tw2 + 2L * n2;
  m.G1 = m.R + c;
  m.G2 = m.G1 + c;
  m.total = m.G2 + c;
  return m;
}

// ws[d] = (dq / pi) sum_{0 < k < n/2} sin(2 pi k d / n) / k: the field of a unit
// charge per cell at distance d.
__global__ void poi_kernel_1d(int n, double dq, double* ws) {
  const int d = blockIdx.x * blockDim.x + threadIdx.x;
  if (d >= n) return;
  double s = 0.0;
  for (int k = 1; 2 * k < n; ++k) s += sinpi(2.0 * double((long)k * d % n) / n) / k;
  ws[d] = s * dq / 3.141592653589793;
}

__global__ void poi_twiddles(int n, double* tw) {
  const int m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= n) return;
  double s, c;
  sincospi(2.0 * m / n, &s, &c);
  tw[2 * m] = c;
  tw[2 * m + 1] = s;
}

// Grids of one axis.  64 outputs per workgroup, four threads each.
__global__ __launch_bounds__(POI_THREADS) void poi_conv(int n, const double* g, PoiDensity rho,
                                                        double eps, double* E, double* other) {
  extern __shared__ double lds[];
  double* r = lds;
  double* gl = lds + n;
  // the mean drops out (the kernel is odd); without the bulk of it the sums
  // keep the perturbation's digits
  const double r0 = rho.at(0);
  for (int j = threadIdx.x; j < n; j += POI_THREADS) {
    r[j] = rho.at(j) - r0;
    gl[j] = g[j];
  }
  __syncthreads();
  const int sub = threadIdx.x & 3, i = blockIdx.x * 64 + (threadIdx.x >> 2);
  double s = 0.0;
  if (i < n) {
    int d = i - sub;
    if (d < 0) d += n;
    for (int j = sub; j < n; j += 4) {
      s += gl[d] * r[j];
      d -= 4;
      if (d < 0) d += n;
    }
  }
  s += __shfl_xor(s, 1, 64);
  s += __shfl_xor(s, 2, 64);
  if (sub == 0 && i < n) {
    E[i] = s / eps;
    other[i] = 0.0;
  }
}

// Threads per output of n outputs in a workgroup: a power of two that keeps
// the workgroup busy and inside a wave.
__device__ inline int poi_subs(int n) {
  int s = 1;
  while (s < 16 && 2 * s * n <= POI_THREADS) s *= 2;
  return s;
}
__device__ inline double poi_sum(double x, int subs) {
  for (int o = 1; o < subs; o *= 2) x += __shfl_xor(x, o, 64);
  return x;
}

// R(i2, k1) = sum_i1 (rho(i1, i2) - rho(0, 0)) exp(-2 pi i k1 i1 / n1); one
// workgroup per row.
__global__ __launch_bounds__(POI_THREADS) void poi_rows(PoiMap m, double* ws, PoiDensity rho) {
  __shared__ double r[POI_MAX_2D], tc[POI_MAX_2D], ts[POI_MAX_2D];
  const int i2 = blockIdx.x, n = m.n1;
  const double r0 = rho.at(0);
  for (int i = threadIdx.x; i < n; i += POI_THREADS) {
    r[i] = rho.at(i2 * n + i) - r0;
    tc[i] = ws[m.tw1 + 2 * i];
    ts[i] = ws[m.tw1 + 2 * i + 1];
  }
  __syncthreads();
  const int subs = poi_subs(m.h), sub = threadIdx.x % subs;
  for (int k = threadIdx.x / subs; k < m.h; k += POI_THREADS / subs) {
    int id = (k * sub) % n;
    const int step = (k * subs) % n;
    double a = 0.0, b = 0.0;
    for (int i = sub; i < n; i += subs) {
      a += r[i] * tc[id];
      b -= r[i] * ts[id];
      id += step;
      if (id >= n) id -= n;
    }
    a = poi_sum(a, subs);
    b = poi_sum(b, subs);
    if (sub == 0) {
      ws[m.R + 2 * ((long)i2 * m.h + k)] = a;
      ws[m.R + 2 * ((long)i2 * m.h + k) + 1] = b;
    }
  }
}

// Column k1: the sums along q2, the division by 4 pi^2 |k|^2, and the sums
// back, of phi for E1 (times -2 pi i k1 in the caller of G1) and of k2 phi for
// E2; one workgroup per column.
__global__ __launch_bounds__(POI_THREADS) void poi_columns(PoiMap m, double* ws, double l1,
                                                           double l2) {
  __shared__ double2 c[POI_MAX_2D], f[POI_MAX_2D];
  __shared__ double tc[POI_MAX_2D], ts[POI_MAX_2D];
  const int k1 = blockIdx.x, n = m.n2, h = m.h;
  for (int i = threadIdx.x; i < n; i += POI_THREADS) {
    const double* R = ws + m.R + 2 * ((long)i * h + k1);
    c[i] = make_double2(R[0], R[1]);
    tc[i] = ws[m.tw2 + 2 * i];
    ts[i] = ws[m.tw2 + 2 * i + 1];
  }
  __syncthreads();
  const int subs = poi_subs(n), sub = threadIdx.x % subs;
  const double w1 = k1 / l1;
  const double tp = 2.0 * 3.141592653589793;
  for (int k = threadIdx.x / subs; k < n; k += POI_THREADS / subs) {
    int id = (k * sub) % n;
    const int step = (k * subs) % n;
    double a = 0.0, b = 0.0;
    for (int i = sub; i < n; i += subs) {
      a += c[i].x * tc[id] + c[i].y * ts[id];
      b += c[i].y * tc[id] - c[i].x * ts[id];
      id += step;
      if (id >= n) id -= n;
    }
    a = poi_sum(a, subs);
    b = poi_sum(b, subs);
    if (sub == 0) {
      const double w2 = (2 * k < n ? k : k - n) / l2;
      const double d = (tp * tp) * (w1 * w1 + w2 * w2);
      f[k] = k1 == 0 && k == 0 ? make_double2(0.0, 0.0) : make_double2(a / d, b / d);
    }
  }
  __syncthreads();
  for (int i = threadIdx.x / subs; i < n; i += POI_THREADS / subs) {
    int id = (i * sub) % n;
    const int step = (i * subs) % n;
    double a = 0.0, b = 0.0, p = 0.0, q = 0.0;
    for (int k = sub; k < n; k += subs) {
      // f exp(+2 pi i k i / n); its k2 multiple without the Nyquist wavenumber
      const double x = f[k].x * tc[id] - f[k].y * ts[id];
      const double y = f[k].y * tc[id] + f[k].x * ts[id];
      const double w2 = (2 * k < n ? k : 2 * k == n ? 0 : k - n) / l2;
      a += x;
      b += y;
      p += w2 * x;
      q += w2 * y;
      id += step;
      if (id >= n) id -= n;
    }
    a = poi_sum(a, subs);
    b = poi_sum(b, subs);
    p = poi_sum(p, subs);
    q = poi_sum(q, subs);
    if (sub == 0) {
      // times -2 pi i k1 and -2 pi i, the mean over n2
      const double w = (2 * k1 == m.n1 ? 0.0 : w1) * (tp / n), v = tp / n;
      double* G1 = ws + m.G1 + 2 * ((long)i * h + k1);
      double* G2 = ws + m.G2 + 2 * ((long)i * h + k1);
      G1[0] = w * b;
      G1[1] = -w * a;
      G2[0] = v * q;
      G2[1] = -v * p;
    }
  }
}

// E(i1, i2) = 1/n1 Re sum_k1 G(i2, k1) exp(+2 pi i k1 i1 / n1) over both halves of
// the spectrum; one workgroup per row.
__global__ __launch_bounds__(POI_THREADS) void poi_back(PoiMap m, const double* ws, double eps,
                                                        double* E1, double* E2) {
  __shared__ double2 a[POI_MAX_2D / 2 + 1], b[POI_MAX_2D / 2 + 1];
  __shared__ double tc[POI_MAX_2D], ts[POI_MAX_2D];
  const int i2 = blockIdx.x, n = m.n1;
  for (int k = threadIdx.x; k < m.h; k += POI_THREADS) {
    const double w = (k == 0 || 2 * k == n ? 1.0 : 2.0) / n;
    const double* G1 = ws + m.G1 + 2 * ((long)i2 * m.h + k);
    const double* G2 = ws + m.G2 + 2 * ((long)i2 * m.h + k);
    a[k] = make_double2(w * G1[0], w * G1[1]);
    b[k] = make_double2(w * G2[0], w * G2[1]);
  }
  for (int i = threadIdx.x; i < n; i += POI_THREADS) {
    tc[i] = ws[m.tw1 + 2 * i];
    ts[i] = ws[m.tw1 + 2 * i + 1];
  }
  __syncthreads();
  const int subs = poi_subs(n), sub = threadIdx.x % subs;
  for (int i = threadIdx.x / subs; i < n; i += POI_THREADS / subs) {
    int id = (i * sub) % n;
    const int step = (i * subs) % n;
    double x = 0.0, y = 0.0;
    for (int k = sub; k < m.h; k += subs) {
      x += a[k].x * tc[id] - a[k].y * ts[id];
      y += b[k].x * tc[id] - b[k].y * ts[id];
      id += step;
      if (id >= n) id -= n;
    }
    x = poi_sum(x, subs);
    y = poi_sum(y, subs);
    if (sub == 0) {
      E1[(long)i2 * n + i] = x / eps;
      E2[(long)i2 * n + i] = y / eps;
    }
  }
}

bool one_axis(const boltx_grid* g) { return g->n_q1 == 1 || g->n_q2 == 1; }

}  // namespace
}  // namespace bx

using namespace bx;

extern "C" size_t boltx_poisson_workspace_size(const boltx_grid* grid) {
  if (check_grid(grid)) return 0;
  if (one_axis(grid)) {
    const int n = grid->n_q1 * grid->n_q2;
    return n <= POI_MAX_1D ? (size_t)n * sizeof(double) : 0;
  }
  const long n1 = grid->n_q1, n2 = grid->n_q2;
  if (n1 > POI_MAX_2D || n2 > POI_MAX_2D || n1 * n2 * (n1 + n2) > POI_MAX_WORK) return 0;
  return (size_t)poi_map(grid->n_q1, grid->n_q2).total * sizeof(double);
}

extern "C" int boltx_poisson_init(const boltx_grid* grid, void* workspace, void* stream) {
  if (boltx_poisson_workspace_size(grid) == 0)
    return fail(BOLTX_EUNSUPPORTED, "poisson: the grid is too large");
  if (!workspace) return fail(BOLTX_EINVAL, "poisson: workspace is NULL");
  double* ws = (double*)workspace;
  hipStream_t s = (hipStream_t)stream;
  if (one_axis(grid)) {
    const int n = grid->n_q1 * grid->n_q2;
    const double dq = grid->n_q1 > 1 ? grid->dq1 : grid->dq2;
    hipLaunchKernelGGL(poi_kernel_1d, dim3((n + 63) / 64), dim3(64), 0, s, n, dq, ws);
    return launch_status("poi_kernel_1d");
  }
  const PoiMap m = poi_map(grid->n_q1, grid->n_q2);
  hipLaunchKernelGGL(poi_twiddles, dim3((m.n1 + 63) / 64), dim3(64), 0, s, m.n1, ws + m.tw1);
  hipLaunchKernelGGL(poi_twiddles, dim3((m.n2 + 63) / 64), dim3(64), 0, s, m.n2, ws + m.tw2);
  return launch_status("poi_twiddles");
}

extern "C" int boltx_poisson(const boltx_grid* grid, int n_species, const double* const* density,
                             const double* charge, double eps, double* cc, void* workspace,
                             void* stream) {
  if (boltx_poisson_workspace_size(grid) == 0)
    return fail(BOLTX_EUNSUPPORTED, "poisson: the grid is too large");
  if (n_species < 1 || n_species > POI_SPECIES)
    return fail(BOLTX_EUNSUPPORTED, "poisson: %d species (1..%d)", n_species, POI_SPECIES);
  if (!density || !charge || !cc || !workspace)
    return fail(BOLTX_EINVAL, "poisson pointers missing");
  PoiDensity rho;
  memset(&rho, 0, sizeof(rho));
  rho.ns = n_species;
  for (int k = 0; k < n_species; ++k) {
    if (!density[k]) return fail(BOLTX_EINVAL, "poisson: density of species %d is NULL", k);
    rho.n[k] = density[k];
    rho.charge[k] = charge[k];
  }
  double* ws = (double*)workspace;
  hipStream_t s = (hipStream_t)stream;
  const int Q = grid->n_q1 * grid->n_q2;
  if (one_axis(grid)) {
    const int axis = grid->n_q1 > 1 ? 0 : 1;
    hipLaunchKernelGGL(poi_conv, dim3((Q + 63) / 64), dim3(POI_THREADS),
                       2 * (size_t)Q * sizeof(double), s, Q, (const double*)ws, rho, eps,
                       cc + (long)axis * Q, cc + (long)(1 - axis) * Q);
    return launch_status("poi_conv");
  }
  const PoiMap m = poi_map(grid->n_q1, grid->n_q2);
  hipLaunchKernelGGL(poi_rows, dim3(m.n2), dim3(POI_THREADS), 0, s, m, ws, rho);
  int rc = launch_status("poi_rows");
  if (rc) return rc;
  hipLaunchKernelGGL(poi_columns, dim3(m.h), dim3(POI_THREADS), 0, s, m, ws,
                     m.n1 * grid->dq1, m.n2 * grid->dq2);
  if ((rc = launch_status("poi_columns"))) return rc;
  hipLaunchKernelGGL(poi_back, dim3(m.n2), dim3(POI_THREADS), 0, s, m, (const double*)ws, eps, cc,
                     cc + Q);
  return launch_status("poi_back");
}

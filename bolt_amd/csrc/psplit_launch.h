// Launches of the two-kernel stage with p-advection (psplit.h), compiled once
// per storage type in its own translation unit.
#pragma once
#include "fvm_stage.h"
#ifdef BX_PSPLIT_INSTANTIATE
#include "bx_status.h"
#include "psplit.h"
#endif

namespace bx {

// One stage (sp complete, mom and fields set) over all q2 rows, ``rows`` of
// them at a time, with D (rows * n_q1 * P values) and, when J is wanted, the
// partial currents ``part`` (psplit_part_bytes).  have_D: D holds the q-part
// of sp.u already (rows = n_q2).
template <typename T>
int psplit_stage(const StageParams& sp, int recon_q, int recon_p, int rows, void* D, double* part,
                 double* J, bool have_D, hipStream_t s);

// The currents of sp.u; with rows = n_q2 the q-part of sp.u is left in D for
// the stage that follows.
template <typename T>
int psplit_currents(const StageParams& sp, int recon_q, int rows, void* D, double* part, double* J,
                    hipStream_t s);

// One stage of a problem without p-advection, ``rows`` q2 rows at a time, with
// the Maxwellian factors ``tab`` (rows * n_q1 * (n_p1 + n_p2 + n_p3) values)
// and the partial moments ``part``.
template <typename T>
int qmarch_stage(const StageParams& sp, int recon_q, int rows, void* tab, double* part,
                 hipStream_t s);

inline size_t psplit_part_bytes(const StageParams& sp, int rows) {
  return (size_t)((sp.P + 63) / 64) * 3 * (size_t)rows * sp.n_q1 * sizeof(double);
}

#ifdef BX_PSPLIT_INSTANTIATE

template <typename T, int R, int KIND>
static int qdiff_launch(const StageParams& sp, int r0, int r1, void* D, double* part,
                        const void* tab, hipStream_t s) {
  constexpr int N = KIND == QK_STAGE && sizeof(T) == 8 ? 2 : 4;
  QDiffParams q;
  q.sp = sp;
  q.r0 = r0;
  q.r1 = r1;
  q.nslab = (sp.P + 63) / 64;
  q.ntile = (sp.n_q1 + 4 * N - 1) / (4 * N);
  const int rows = r1 - r0;
  // segments of about 16 rows, halved while they would not fill the chip
  int nseg = rows / 16 > 1 ? rows / 16 : 1;
  while ((long)q.nslab * q.ntile * nseg < 768 && rows / (2 * nseg) >= 2) nseg *= 2;
  q.nseg = nseg;
  q.D = D;
  q.part = part;
  q.tab = tab;
  const unsigned nb = (unsigned)(q.nslab * q.ntile * nseg);
  if (sp.gh1 || sp.gh2) {
    // (ghost rows occur with electrostatic fields only: no currents)
    if constexpr ((KIND & QK_CUR) == 0)
      hipLaunchKernelGGL((qdiff_kernel<T, R, N, true, KIND>), dim3(nb), dim3(256), 0, s, q);
    else
      return fail(BOLTX_EUNSUPPORTED, "currents of a grid with ghost rows");
  } else {
    hipLaunchKernelGGL((qdiff_kernel<T, R, N, false, KIND>), dim3(nb), dim3(256), 0, s, q);
  }
  return launch_status("qdiff_kernel");
}

template <typename T, int KIND>
static int qdiff_recon(const StageParams& sp, int rq, int r0, int r1, void* D, double* part,
                       const void* tab, hipStream_t s) {
  switch (rq) {
    case RC_PC: return qdiff_launch<T, RC_PC, KIND>(sp, r0, r1, D, part, tab, s);
    case RC_MINMOD: return qdiff_launch<T, RC_MINMOD, KIND>(sp, r0, r1, D, part, tab, s);
    case RC_PPM: return qdiff_launch<T, RC_PPM, KIND>(sp, r0, r1, D, part, tab, s);
    default: return qdiff_launch<T, RC_WENO5, KIND>(sp, r0, r1, D, part, tab, s);
  }
}

static int qcur_reduce(const StageParams& sp, int r0, int r1, const double* part, double* J,
                       hipStream_t s) {
  const int nq = (r1 - r0) * sp.n_q1;
  hipLaunchKernelGGL(qcur_reduce_kernel, dim3((unsigned)((nq + 15) / 16), 3), dim3(256), 0, s, part,
                     (sp.P + 63) / 64, nq, r0 * sp.n_q1, sp.Q, sp.charge, sp.measure, J);
  return launch_status("qcur_reduce_kernel");
}

template <typename T, int RP, int MODE>
static int pplane_launch(const StageParams& sp, int r0, int r1, const void* D, hipStream_t s) {
  const int nt = (sp.n_p1 * sp.n_p2 + 63) / 64 * 64;
  const size_t lds = sizeof(T) * (size_t)(sp.n_p1 + sp.n_p2 + sp.n_p3);
  const dim3 grid((unsigned)((r1 - r0) * sp.n_q1)), block(nt);
  const int q0 = r0 * sp.n_q1;
  // waves per SIMD asked for: see pplane_kernel
  constexpr int W = sizeof(T) == 8 ? 5 : 6;
  auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, block, lds, s, sp, (const T*)D, q0); };
  if (nt <= 256) go(pplane_kernel<T, RP, MODE, 256, W>);
  else if (nt <= 576) go(pplane_kernel<T, RP, MODE, 576, W>);
  else go(pplane_kernel<T, RP, MODE, 1024, 4>);
  return launch_status("pplane_kernel");
}

template <typename T, int RP>
static int pplane_mode(const StageParams& sp, int r0, int r1, const void* D, hipStream_t s) {
  if (sp.a == 0.0 && sp.b == 1.0)
    return sp.w == sp.u ? pplane_launch<T, RP, PM_FIRST>(sp, r0, r1, D, s)
                        : pplane_launch<T, RP, PM_MIDPOINT>(sp, r0, r1, D, s);
  if (sp.w == sp.u && sp.a != 0.0) return pplane_launch<T, RP, PM_COMBINE>(sp, r0, r1, D, s);
  return pplane_launch<T, RP, PM_GENERAL>(sp, r0, r1, D, s);
}

template <typename T>
static int pplane_recon(const StageParams& sp, int rp, int r0, int r1, const void* D,
                        hipStream_t s) {
  switch (rp) {
    case RC_PC: return pplane_mode<T, RC_PC>(sp, r0, r1, D, s);
    case RC_MINMOD: return pplane_mode<T, RC_MINMOD>(sp, r0, r1, D, s);
    case RC_PPM: return pplane_mode<T, RC_PPM>(sp, r0, r1, D, s);
    default: return pplane_mode<T, RC_WENO5>(sp, r0, r1, D, s);
  }
}

template <typename T>
int psplit_stage(const StageParams& sp, int rq, int rp, int rows, void* D, double* part, double* J,
                 bool have_D, hipStream_t s) {
  if (have_D && !J && rows >= sp.n_q2) return pplane_recon<T>(sp, rp, 0, sp.n_q2, D, s);
  for (int r0 = 0; r0 < sp.n_q2; r0 += rows) {
    const int r1 = r0 + rows < sp.n_q2 ? r0 + rows : sp.n_q2;
    int rc = J ? qdiff_recon<T, QK_DIV_CUR>(sp, rq, r0, r1, D, part, nullptr, s)
               : qdiff_recon<T, QK_DIV>(sp, rq, r0, r1, D, nullptr, nullptr, s);
    if (rc) return rc;
    if (J && (rc = qcur_reduce(sp, r0, r1, part, J, s))) return rc;
    if ((rc = pplane_recon<T>(sp, rp, r0, r1, D, s))) return rc;
  }
  return 0;
}

template <typename T>
int psplit_currents(const StageParams& sp, int rq, int rows, void* D, double* part, double* J,
                    hipStream_t s) {
  for (int r0 = 0; r0 < sp.n_q2; r0 += rows) {
    const int r1 = r0 + rows < sp.n_q2 ? r0 + rows : sp.n_q2;
    int rc = rows >= sp.n_q2 ? qdiff_recon<T, QK_DIV_CUR>(sp, rq, r0, r1, D, part, nullptr, s)
                             : qdiff_recon<T, QK_CUR>(sp, rq, r0, r1, nullptr, part, nullptr, s);
    if (rc) return rc;
    if ((rc = qcur_reduce(sp, r0, r1, part, J, s))) return rc;
  }
  return 0;
}

template <typename T>
int qmarch_stage(const StageParams& sp, int rq, int rows, void* tab, double* part,
                 hipStream_t s) {
  for (int r0 = 0; r0 < sp.n_q2; r0 += rows) {
    const int r1 = r0 + rows < sp.n_q2 ? r0 + rows : sp.n_q2;
    const int q0 = r0 * sp.n_q1, nq = (r1 - r0) * sp.n_q1;
    int rc;
    if (sp.source) {
      hipLaunchKernelGGL(qtab_kernel<T>, dim3((unsigned)((nq + 3) / 4)), dim3(256), 0, s, sp, q0,
                         nq, (T*)tab);
      if ((rc = launch_status("qtab_kernel"))) return rc;
    }
    if ((rc = qdiff_recon<T, QK_STAGE>(sp, rq, r0, r1, nullptr, part, tab, s))) return rc;
    if (!sp.mom_out) continue;
    hipLaunchKernelGGL(qmom_reduce_kernel, dim3((unsigned)((nq + 15) / 16)), dim3(256), 0, s, sp,
                       (const double*)part, (sp.P + 63) / 64, nq, q0);
    if ((rc = launch_status("qmom_reduce_kernel"))) return rc;
  }
  return 0;
}
#endif

}  // namespace bx

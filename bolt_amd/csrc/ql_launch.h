// Launch of the q1-line stage kernel, compiled once per storage type in its
// own translation unit (ql_f64.hip, ql_f32.hip) so the many specialisations
// of qline_kernel build in parallel.
#pragma once
#include "qline.h"

namespace bx {

// Launches qline_kernel over nb workgroups for reconstruction ``recon``,
// stage form ``mode`` (enum QlMode), by DPP rotates if ``rot`` (ql_rot_applies), and ``pd`` Maxwellian factors per cell
// (0 = no source).  WENO5 has a kernel per (mode, pd); the other
// reconstructions use the run-time form.
template <typename T>
void ql_launch(const QLParams& q, bool rot, int recon, int nb, int mode, int pd, hipStream_t s);

// Whether neighbours come by DPP rotates: a line fills the wave's lanes with 1,
// 2 or 4 cells each, and every array is aligned to a lane's cells.  FP32 takes
// them for 4 cells only, where the LDS form spills: a step at 256 x 128 q,
// 40^2 p 968 -> 553 us; with 1 and 2 cells its LDS traffic is half of FP64's and
// hidden, and the rotates are instructions more (64^2 q, 48^2 p graph replay
// 75.7 -> 78.5 us, 128^2 q, 48^2 p 408 -> 412 us).  FP64: 756 -> 686 us at
// 128^2 q, 48^2 p; 4630 -> 1090 us at 256 x 128 q, 40^2 p.
template <typename T>
inline bool ql_rot_applies(const QLParams& q) {
  if (q.n1 != 256 && (sizeof(T) != 8 || (q.n1 != 64 && q.n1 != 128))) return false;
  const uintptr_t all = (uintptr_t)q.u | (uintptr_t)q.w | (uintptr_t)q.un | (uintptr_t)q.out |
                        (uintptr_t)q.tab;
  return all % (q.n1 / 64 * sizeof(T)) == 0;
}

// Resident workgroups per CU of the kernel ql_launch picks for these
// arguments (0 if the runtime cannot say).
template <typename T>
int ql_blocks_per_cu(int n1, bool rot, int recon, int mode, int pd);

#ifdef BX_QL_INSTANTIATE
using QlKernel = void (*)(QLParams);

template <typename T, int NR, bool ROT, int M>
static QlKernel ql_weno_pd(int pd) {
  switch (pd) {
    case 0: return qline_kernel<T, RC_WENO5, NR, ROT, M, 0>;
    case 1: return qline_kernel<T, RC_WENO5, NR, ROT, M, 1>;
    case 2: return qline_kernel<T, RC_WENO5, NR, ROT, M, 2>;
    default: return qline_kernel<T, RC_WENO5, NR, ROT, M, 3>;
  }
}

template <typename T, int NR, bool ROT>
static QlKernel ql_nr(int recon, int mode, int pd) {
  switch (recon) {
    case RC_PC: return qline_kernel<T, RC_PC, NR, ROT, QL_GENERAL, -1>;
    case RC_MINMOD: return qline_kernel<T, RC_MINMOD, NR, ROT, QL_GENERAL, -1>;
    case RC_PPM: return qline_kernel<T, RC_PPM, NR, ROT, QL_GENERAL, -1>;
    default: break;
  }
  switch (mode) {
    case QL_WU_PLAIN: return ql_weno_pd<T, NR, ROT, QL_WU_PLAIN>(pd);
    case QL_WU_COMB: return ql_weno_pd<T, NR, ROT, QL_WU_COMB>(pd);
    case QL_W_PLAIN: return ql_weno_pd<T, NR, ROT, QL_W_PLAIN>(pd);
    default: return qline_kernel<T, RC_WENO5, NR, ROT, QL_GENERAL, -1>;
  }
}

template <typename T>
static QlKernel ql_pick(int n1, bool rot, int recon, int mode, int pd) {
  if (rot) {
    if constexpr (sizeof(T) == 8) {
      if (n1 == 64) return ql_nr<T, 1, true>(recon, mode, pd);
      if (n1 == 128) return ql_nr<T, 2, true>(recon, mode, pd);
    }
    return ql_nr<T, 4, true>(recon, mode, pd);
  }
  if (n1 <= 64) return ql_nr<T, 1, false>(recon, mode, pd);
  if (n1 <= 128) return ql_nr<T, 2, false>(recon, mode, pd);
  return ql_nr<T, 4, false>(recon, mode, pd);
}

template <typename T>
void ql_launch(const QLParams& q, bool rot, int recon, int nb, int mode, int pd, hipStream_t s) {
  hipLaunchKernelGGL(ql_pick<T>(q.n1, rot, recon, mode, pd), dim3(nb), dim3(256), 0, s, q);
}

template <typename T>
int ql_blocks_per_cu(int n1, bool rot, int recon, int mode, int pd) {
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, ql_pick<T>(n1, rot, recon, mode, pd), 256, 0) !=
      hipSuccess)
    return 0;
  return n;
}
#endif

}  // namespace bx

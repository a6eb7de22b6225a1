// Reconstruction for lanes whose upwind directions differ.
//
// The upwind state of a face is always a face state of the cell on its upwind
// side (riemann.py:46-49): the right face of cell j when C > 0, the left face
// of cell j + 1 otherwise.  So every cell is given ONE state, the one of the
// face on its downwind side,
//   s_j = right face of cell j (C > 0)  or  left face of cell j (C <= 0),
// reconstructed from the same five cells j-2 .. j+2 either way, and the flux
// through face j+1/2 is C * (C > 0 ? s_j : s_{j+1}).  A wave whose lanes have
// both signs then runs one instruction stream: the direction enters through a
// few per-lane coefficients (WENO5) or one select (PPM, minmod).
//
// What a cell's state needs besides the values is one quantity per cell (aux),
// computed once and shared by the three states that use it: the WENO5
// indicator (weno5.py:58-71), PPM's limited slope (ppm.py:58-80), minmod's
// slope (minmod.py:4-62).
//
// Everything here evaluates without contraction and fuses explicitly, so a
// cell rounds alike in every copy of an unrolled march.
#pragma once
#include "qline.h"

namespace bx {

// Per-lane coefficients of the WENO5 state (the scaled substencils of
// ql_face: all exact in binary).
template <typename T>
struct DirCoef {
  T g0, a1, b3, c4, d1, d3;
};

template <int R, typename T>
__host__ __device__ __forceinline__ DirCoef<T> dir_coef(bool pos) {
  DirCoef<T> c;
  if constexpr (R == RC_WENO5) {
    c.g0 = pos ? T(0.375) : T(-0.625);
    c.a1 = pos ? T(-1.25) : T(3.75);
    c.b3 = pos ? T(3.75) : T(-1.25);
    c.c4 = pos ? T(-0.625) : T(0.375);
    c.d1 = pos ? T(1) : T(5);
    c.d3 = pos ? T(5) : T(1);
  } else {
    c.g0 = pos ? T(1) : T(-1);
    c.a1 = c.b3 = c.c4 = c.d1 = c.d3 = T(0);
  }
  return c;
}

__host__ __device__ __forceinline__ double dir_min(double a, double b) { return __builtin_fmin(a, b); }
__host__ __device__ __forceinline__ float dir_min(float a, float b) { return __builtin_fminf(a, b); }
__host__ __device__ __forceinline__ double dir_sign(double a, double b) { return __builtin_copysign(a, b); }
__host__ __device__ __forceinline__ float dir_sign(float a, float b) { return __builtin_copysignf(a, b); }

// ppm_dq (ppm.py:58-80) in fewer instructions: the same value for finite
// cells (powers of two taken out of the minimum are exact; a zero may differ
// in sign).
template <typename T>
__host__ __device__ __forceinline__ T dir_ppm_slope(T ym, T y, T yp) {
#pragma clang fp contract(off)
  const T dm = y - ym, dp = yp - y;
  const T D = T(0.5) * (yp - ym);
  const T m = dir_min(aabs(D), T(2) * dir_min(aabs(dm), aabs(dp)));
  return dp * dm <= T(0) ? T(0) : dir_sign(m, D);
}

// PPM's uncorrected value at the face between cells y and yp with slopes k and
// kp (ppm.py:82-83): the right value of the one and the left value of the
// other, so both share it.
template <typename T>
__host__ __device__ __forceinline__ T dir_ppm_face(T y, T yp, T k, T kp) {
#pragma clang fp contract(off)
  return T(0.5) * (yp + y) - (kp - k) * T(1.0 / 6.0);
}

// The corrected state (ppm.py:85-98) of cell y with uncorrected left and
// right values l and r on its downwind side: of the two corrections that
// follow one another there, only what reaches that side.
template <typename T>
__host__ __device__ __forceinline__ T dir_ppm_state(T y, T l, T r, bool pos) {
#pragma clang fp contract(off)
  const bool flat = (r - y) * (y - l) <= T(0);
  const T qd = r - l;
  const T qe = T(6) * (y - T(0.5) * (r + l));
  const bool c2 = qd * (qd - qe) < T(0);
  const bool c3 = qd * (qd + qe) < T(0);
  const T near = flat ? y : (pos ? r : l);
  const T far = flat ? y : (pos ? l : r);
  return (pos ? (c3 && !c2) : c2) ? T(3) * y - T(2) * far : near;
}

// The aux quantity of the centre cell b of a, b, c.
template <int R, typename T>
__host__ __device__ __forceinline__ T dir_aux(T a, T b, T c) {
#pragma clang fp contract(off)
  if constexpr (R == RC_WENO5) return ql_kappa<R, T>(a, b, c);
  else if constexpr (R == RC_PPM) return dir_ppm_slope(a, b, c);
  else if constexpr (R == RC_MINMOD) return mc_slope(a, b, c);
  else return T(0);
}

// The state of the centre cell y2 of y0 .. y4 with the aux quantities of y1,
// y2, y3.
template <int R, typename T>
__host__ __device__ __forceinline__ T dir_state(T y0, T y1, T y2, T y3, T y4, T k1, T k2, T k3,
                                                bool pos, const DirCoef<T>& c) {
#pragma clang fp contract(off)
  if constexpr (R == RC_PC) {
    return y2;
  } else if constexpr (R == RC_MINMOD) {
    return y2 + c.g0 * (T(0.5) * k2);
  } else if constexpr (R == RC_PPM) {
    return dir_ppm_state(y2, dir_ppm_face(y1, y2, k1, k2), dir_ppm_face(y2, y3, k2, k3), pos);
  } else {
    const T u1 = ql_fma(T(1.875), y2, ql_fma(c.a1, y1, c.g0 * y0));
    const T u2 = ql_fma(c.b3, y3, ql_fma(T(7.5), y2, c.a1 * y1));
    const T u3 = ql_fma(c.c4, y4, ql_fma(c.b3, y3, T(1.875) * y2));
    T w1, w2, w3;
    if constexpr (sizeof(T) == 8) {
      w1 = k2 * k3;
      w2 = k1 * k3;
      w3 = k1 * k2;
    } else {
      w1 = k1;
      w2 = k2;
      w3 = k3;
    }
    const T num = ql_fma(w3, u3, ql_fma(w2, u2, w1 * u1));
    const T den = ql_fma(c.d3, w3, ql_fma(T(10), w2, c.d1 * w1));
    return num * fast_rcp(den);
  }
}

}  // namespace bx

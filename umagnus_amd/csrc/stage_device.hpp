// A solver stage inside the X forward pass of the demag convolution: m is
// formed, stored and transformed by one kernel.
#pragma once
#include "fft_device.hpp"
#include "vec.hpp"

namespace um {

// Component c of the stage at cells i and i + 1.  All
// three components are summed, since the norm needs them; up to 18 loads are
// in flight.  Every product and fused multiply-add is written out: they are
// those of k_stage (vec.hip), which runs the stages of the same grids where
// this form does not apply (time functions, the tape), so m has the same bits
// whichever kernel forms it.
template <typename T, int NS>
__device__ __forceinline__ void stage_pair_n(const StageArgs<T> &s, int c, long i) {
#pragma clang fp contract(off)
  const T h = s.dev_dt ? (T)(s.dev_dt[0] * s.gam) : T(1);
  C2<T> x[3][NS], vv{T(1), T(1)};
#pragma unroll
  for (int e = 0; e < 3; e++)
#pragma unroll
    for (int k = 0; k < NS; k++) x[e][k] = *(const C2<T> *)(s.src[k][e] + i);
  if (s.vol) vv = *(const C2<T> *)(s.vol + i);
  T f[NS], r[2][3];
#pragma unroll
  for (int k = 0; k < NS; k++) f[k] = s.dev_dt && k > 0 ? s.fac[k] * h : s.fac[k];
#pragma unroll
  for (int w = 0; w < 2; w++) {
#pragma unroll
    for (int e = 0; e < 3; e++) {
      T u[NS];
#pragma unroll
      for (int k = 0; k < NS; k++) u[k] = w ? x[e][k].y : x[e][k].x;
      T acc = f[0] * u[0];
      if constexpr (NS == 3) {   // both orders: a branch for each component would wait for its loads
        const T g = acc + fma(f[1], u[1], f[2] * u[2]), q = fma(f[2], u[2], fma(f[1], u[1], acc));
        acc = s.group3 ? g : q;
      } else {
#pragma unroll
        for (int k = 1; k < NS; k++) acc = fma(f[k], u[k], acc);
      }
      r[w][e] = acc;
    }
    if (s.normalize) {   // normalize2.cl:8-23
      const T v = w ? vv.y : vv.x;
      const T X = v * r[w][0], Y = v * r[w][1], Z = v * r[w][2];
      const T l = sqrt(fma(Z, Z, fma(X, X, Y * Y)));
      const T inv = (l != T(0)) ? T(1) / l : T(0);
      r[w][0] = v == T(0) ? T(0) : X * inv;
      r[w][1] = v == T(0) ? T(0) : Y * inv;
      r[w][2] = v == T(0) ? T(0) : Z * inv;
    }
  }
  T *const d0 = s.dst[0], *const d1 = s.dst[1], *const d2 = s.dst[2];
  T *dst = c == 0 ? d0 : c == 1 ? d1 : d2;
  *(C2<T> *)(dst + i) = C2<T>{c == 0 ? r[0][0] : c == 1 ? r[0][1] : r[0][2], c == 0 ? r[1][0] : c == 1 ? r[1][1] : r[1][2]};
}
template <typename T>
__device__ __forceinline__ void stage_pair(const StageArgs<T> &s, int c, long i) {
  switch (s.nsrc) {   // uniform
    case 2: stage_pair_n<T, 2>(s, c, i); break;
    case 3: stage_pair_n<T, 3>(s, c, i); break;
    case 4: stage_pair_n<T, 4>(s, c, i); break;
    case 5: stage_pair_n<T, 5>(s, c, i); break;
    default: stage_pair_n<T, 6>(s, c, i); break;
  }
}
// what stage_pair takes: three components, no norms kept, every array aligned
// to pairs, and no source that a work-group of another component overwrites
template <typename T>
inline bool stage_pair_ok(const StageArgs<T> &s, int Nx) {
  if (s.ncomp != 3 || s.nrm || s.nsrc < 2 || s.nsrc > 6 || Nx % 2) return false;
  uintptr_t bits = (uintptr_t)s.vol;
  for (int c = 0; c < 3; c++) {
    bits |= (uintptr_t)s.dst[c];
    for (int k = 0; k < s.nsrc; k++) {
      bits |= (uintptr_t)s.src[k][c];
      for (int e = 0; e < 3; e++)
        if (s.src[k][c] < s.dst[e] + s.N && s.dst[e] < s.src[k][c] + s.N) return false;
    }
  }
  return (bits & (2 * sizeof(T) - 1)) == 0;
}

}  // namespace um

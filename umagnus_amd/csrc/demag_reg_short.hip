// Register z columns of the demag convolution (demag_reg.hpp), both precisions.
#include <cmath>

#include "demag_reg_kernels.hpp"

namespace um {

// ---- short z columns ---------------------------------------------------------------
// One thread per (kx, ky) column, the three components in registers, no LDS.
// Pz = 2 Nz: the even and odd frequencies are two Nz-point transforms
//   X[2m] = DFT(x)[m], X[2m+1] = DFT(x W_Pz^n)[m],
// multiplied and transformed back one after the other; Pz = 2 Nz - 1 (Nz <= 5)
// and Pz = Nz (periodic z): one Pz-point transform.  160 x 160 x 10 FP32: 93.8 -> 11.8 us (32 MB),
// 320 x 200 x 6: 166 -> 11.6, against the generic convolution kernel.
// Periodic z in FP32, a whole convolution with k_rconv -> with this: 128 x 128
// x 3 26.3 -> 21.5 us, x 7 38.4 -> 28.0, 512 x 512 x 7 272 -> 121, x 16 336 ->
// 268; 16 points need many columns to hide a thread's chain (128 x 96 x 16,
// 24768 columns, 40.5 -> 40.1; 96 x 96 x 16, 18624, 33.8 -> 38.6).
// A wave holds 32 kx of ky (lanes 0-31) and of its
// mirror Py - ky (lanes 32-63), which read the same tensor lines.
template <typename T, int NZ, int PZ>
struct BRShort {
  using Args = RShortArgs<T>;
  static constexpr int NT = 256, MINB = 1;
  static __device__ __forceinline__ void run(const RShortArgs<T> &a, uint3 blockIdx, uint3) {
    const int lane = threadIdx.x & 63, half = lane >> 5;
    const int kx = blockIdx.x * 32 + (lane & 31);
    const int kyt = blockIdx.y * 4 + (threadIdx.x >> 6);   // tensor row
    if (kyt >= a.KHy || kx >= a.H) return;
    if (half && (kyt == 0 || 2 * kyt == a.Py)) return;     // no mirror row
    const int ky = half ? a.Py - kyt : kyt;
    const T sy = half ? T(-1) : T(1);
    const long o = (long)ky * a.ystride + kx;
    C2<T> x[3][NZ];
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
      for (int z = 0; z < NZ; z++) x[c][z] = a.buf[c][o + z * a.zstride];
    const long kzs = (long)a.KHy * a.Hk, ko = (long)kyt * a.Hk + kx;
    // tensor times the spectrum at frequency k (kt and PZ - kt share |K|)
    auto mul = [&](C2<T> &M0, C2<T> &M1, C2<T> &M2, int k) {
      const bool zm = 2 * k > PZ;
      const long I = ko + (zm ? PZ - k : k) * kzs;
      const T sz = zm ? T(-1) : T(1);
      sym_mul(M0, M1, M2, a.K[0][I], a.K[1][I], a.K[2][I], sy * sz * a.K[3][I], sz * a.K[4][I], sy * a.K[5][I]);
    };
    if constexpr (PZ == 2 * NZ) {
      C2<T> e[3][NZ];
#pragma unroll
      for (int c = 0; c < 3; c++) {
#pragma unroll
        for (int z = 0; z < NZ; z++) e[c][z] = x[c][z];
        dft<NZ, -1>(e[c]);
      }
#pragma unroll
      for (int m = 0; m < NZ; m++) mul(e[0][m], e[1][m], e[2][m], 2 * m);
#pragma unroll
      for (int c = 0; c < 3; c++) {
        dft<NZ, +1>(e[c]);
#pragma unroll
        for (int z = 1; z < NZ; z++) x[c][z] = cmul(x[c][z], cexpi<T>(z, PZ, -1));
        dft<NZ, -1>(x[c]);
      }
#pragma unroll
      for (int m = 0; m < NZ; m++) mul(x[0][m], x[1][m], x[2][m], 2 * m + 1);
#pragma unroll
      for (int c = 0; c < 3; c++) {
        dft<NZ, +1>(x[c]);
#pragma unroll
        for (int z = 0; z < NZ; z++)
          a.buf[c][o + z * a.zstride] = cadd(e[c][z], z == 0 ? x[c][0] : cmul(x[c][z], cexpi<T>(z, PZ, +1)));
      }
    } else {
      C2<T> e[3][PZ];
#pragma unroll
      for (int c = 0; c < 3; c++) {
#pragma unroll
        for (int z = 0; z < PZ; z++) e[c][z] = z < NZ ? x[c][z] : C2<T>{T(0), T(0)};
        dft<PZ, -1>(e[c]);
      }
#pragma unroll
      for (int k = 0; k < PZ; k++) mul(e[0][k], e[1][k], e[2][k], k);
#pragma unroll
      for (int c = 0; c < 3; c++) {
        dft<PZ, +1>(e[c]);
#pragma unroll
        for (int z = 0; z < NZ; z++) a.buf[c][o + z * a.zstride] = e[c][z];
      }
    }
  }
};
template <typename T, int NZ, int PZ>
__global__ __launch_bounds__(256) void k_rshort(RShortArgs<T> a) { BRShort<T, NZ, PZ>::run(a, hw_bid(), hw_grid()); }

template <typename T>
void launch_rshort(const RShortArgs<T> &a, int Nz, int Pz, hipStream_t s) {
  const dim3 grid((a.H + 31) / 32, (a.KHy + 3) / 4);
#define UM_RSHORT(NZ, PZ) \
  case NZ: launch_b<BRShort<T, NZ, PZ>>(k_rshort<T, NZ, PZ>, grid, dim3(256), 0, s, a); break;
  if (Pz == Nz) {
    if constexpr (sizeof(T) == 4) {
      switch (Nz) {
        UM_RSHORT(2, 2) UM_RSHORT(3, 3) UM_RSHORT(4, 4) UM_RSHORT(5, 5) UM_RSHORT(6, 6) UM_RSHORT(7, 7)
        UM_RSHORT(8, 8) UM_RSHORT(16, 16)
        default: throw Error(UM_EUNSUP, "register z columns: unsupported Nz");
      }
      UM_HIP(hipGetLastError());
      return;
    }
    throw Error(UM_EUNSUP, "register z columns: unsupported Nz");
  }
  switch (Nz) {
    UM_RSHORT(2, 3) UM_RSHORT(3, 5) UM_RSHORT(4, 7) UM_RSHORT(5, 9) UM_RSHORT(6, 12) UM_RSHORT(7, 14)
    default:
      if constexpr (sizeof(T) == 4) {
        switch (Nz) {
          UM_RSHORT(9, 18) UM_RSHORT(10, 20) UM_RSHORT(12, 24)
          default: throw Error(UM_EUNSUP, "register z columns: unsupported Nz");
        }
        break;
      }
      throw Error(UM_EUNSUP, "register z columns: unsupported Nz");
  }
#undef UM_RSHORT
  UM_HIP(hipGetLastError());
}
template <typename T>
bool short_ok(int Nz, int Pz, long columns) {
  if (Pz == Nz) return sizeof(T) == 4 && Nz >= 2 && (Nz <= 8 || (Nz == 16 && columns >= 24576));
  if (Nz >= 2 && Nz <= 5) return Pz == 2 * Nz - 1;
  if (Pz != 2 * Nz) return false;
  return Nz == 6 || Nz == 7 || (sizeof(T) == 4 && (Nz == 9 || Nz == 10 || Nz == 12));
}

template void launch_rshort<float>(const RShortArgs<float> &, int, int, hipStream_t);
template void launch_rshort<double>(const RShortArgs<double> &, int, int, hipStream_t);
template bool short_ok<float>(int, int, long);
template bool short_ok<double>(int, int, long);

}  // namespace um

// Pieces shared by the four-step X kernels: argument blocks, the twiddle table
// in LDS and the radix split of each length.
#pragma once
#include "batch.hpp"
#include "fft_device.hpp"
#include "field.hpp"

namespace um {

template <typename T>
struct XArgs {
  FftLen f;               // complex length n = Px/2
  const C2<T> *tw2;       // exp(-2 pi i k / Px), k in [0, Px)
  int mode;               // 0: mu0*Ms*vol*m rows of Nx valid reals; 1: raw real rows of Px
  int nl;                 // lines per work-group
  FastDiv fhalf;          // n/2 + 1
  int Nx;                 // valid reals per input row
  int rows;               // input rows per component
  FastDiv fRy;            // input rows per z-plane (Ny, or Py for mode 1)
  int Py;                 // spectrum rows per z-plane
  int Hp;                 // spectrum row pitch
  long in_pitch;          // input row pitch (reals)
  const T *src[3];
  Par<T> Ms;
  const T *vol;
  C2<T> *out[3];
};

template <typename T>
struct XiArgs {
  FftLen f;
  const C2<T> *tw2;
  int nl, Nx, rows, Py, Hp;
  FastDiv fhalf, fRy;
  const C2<T> *in[3];
  T *dst[3];
};

// Twiddle table of the step between the two register transforms of a
// four-step pass: W_n^(r k2) (r < R, k2 < K) at [r][k2], rows padded by one
// entry.  Loading and storing are split so that a kernel issues the table's
// global loads after its data loads and writes the table once both arrived:
// no memory round trip of its own ahead of the data.
template <typename T, int R, int K, int NT>
struct TwStage {
  static constexpr int Q = (R * K + NT - 1) / NT;
  C2<T> v[Q];
  __device__ __forceinline__ void load(const C2<T> *tw, int step) {   // tw[step r k2] = W_n^(r k2)
  #pragma unroll
    for (int q = 0; q < Q; q++) {
      const int i = (int)threadIdx.x + q * NT;
      if ((R * K) % NT == 0 || i < R * K) {
        const int r = i / K, k2 = i - r * K;
        v[q] = tw[step * r * k2];
      }
    }
  }
  __device__ __forceinline__ void store(C2<T> *lds) const {
  #pragma unroll
    for (int q = 0; q < Q; q++) {
      const int i = (int)threadIdx.x + q * NT;
      if ((R * K) % NT == 0 || i < R * K) {
        const int r = i / K, k2 = i - r * K;
        lds[r * (K + 1) + k2] = v[q];
      }
    }
  }
};

template <int N> struct X4Shape;
template <> struct X4Shape<64> { static constexpr int A = 8, B = 8; };
template <> struct X4Shape<128> { static constexpr int A = 8, B = 16; };
template <> struct X4Shape<256> { static constexpr int A = 16, B = 16; };
template <> struct X4Shape<512> { static constexpr int A = 16, B = 32; };
template <> struct X4Shape<1024> { static constexpr int A = 32, B = 32; };

// X inverse fused with the four-cell field and torque kernel (demag_xfield.hip)
template <typename T> bool xi4_field_ok(const FieldArgs<T> &a, int n);
template <typename T> void launch_xi4_field(const XiArgs<T> &a, const FieldArgs<T> &f, int n, hipStream_t s);

}  // namespace um

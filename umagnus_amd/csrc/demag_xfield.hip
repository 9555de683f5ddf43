// X inverse of the demag convolution fused with the effective field and torque.
#include <type_traits>

#include "demag_x4.hpp"

namespace um {

template <typename B> struct BTag { using type = B; };

// ---------------------------------------------------------------------------
// X inverse fused with the four-cell effective field + torque (FP32).  A
// work-group of XF_NT threads inverts R rows (y0 .. y0+R-1 of one z plane) of
// all three components with the register four-step of k_xi4 (3R lines, G per
// 32-lane group), leaves the real B_demag lines in LDS, then evaluates the
// effective field and torque of those R x Nx cells: B_demag never touches HBM.
// Work-groups run z fastest (tile w -> y block w / Nz, plane w % Nz), so the
// z +- 1 rows of m that the stencil reads were just read by the neighbouring
// work-groups of the same XCD and are still in its L2.
// ---------------------------------------------------------------------------
constexpr int XF_NT = 192;

template <int N> struct XFShape {
  static constexpr int A = X4Shape<N>::A, B = X4Shape<N>::B, G = B / A;
  static constexpr int R = 64 * G / B;    // rows per work-group
  static constexpr int L = 3 * R;         // lines (component-major: line = c R + j)
  static_assert(L / G * B == XF_NT, "the lines of R rows fill the work-group");
};

template <typename T>
struct XiFieldArgs {
  XiArgs<T> x;
  FieldArgs<T> f;
};
// TH = false (no thermal term, checked on the host) at N = 512: at most 128
// VGPRs without spills (the launch bound's second argument is the minimum
// number of waves per SIMD with hipcc), so five work-groups share a CU
// instead of four; the other lengths would spill under that bound
template <typename T, int N, bool REG, int EX, bool UNI, bool TH>
struct BXi4Field {
  using Args = XiFieldArgs<T>;
  static constexpr int NT = XF_NT, MINB = (!TH && N == 512) ? 4 : 1;
  static __device__ __forceinline__ void run(const XiFieldArgs<T> &a, uint3 blockIdx, uint3 gridDim) {
    const XiArgs<T> &x = a.x;
    const FieldArgs<T> &f = a.f;
    using S = XFShape<N>;
    constexpr int A = S::A, B = S::B, G = S::G, R = S::R, TS = B * (A + 1), HB = B / 2;
    static_assert(S::L * N <= S::L * TS, "B_demag lines fit the transpose space");
    // the transpose moves the real, then the imaginary parts (half the LDS of
    // complex entries: more work-groups per CU); afterwards line (c, j) holds
    // B_demag_c of row j, x < N
    __shared__ __align__(16) T ldr[S::L * TS];
    // twiddles of the step between the two transforms, W_N^(n1 k2) at
    // [n1][k2] (rows padded by one entry: the A rows fall on distinct banks);
    // read from LDS instead of global memory, their latency stays out of the
    // transform
    __shared__ C2<T> twb[A * (B + 1)];
    for (int i = threadIdx.x; i < A * B; i += XF_NT) {
      const int r = i / B, k2 = i - r * B;
      twb[r * (B + 1) + k2] = x.tw2[2 * r * k2];
    }
    const int Ny = (int)x.fRy.d, Nz = x.rows / Ny;
    const int w = xcd_tile(blockIdx.x, gridDim.x);
    const int yb = w / Nz, z = w - yb * Nz, y0 = yb * R;
    const int grp = threadIdx.x / B, l = threadIdx.x % B;
    C2<T> v[B];
    const int h1 = l / A, n1 = l % A, line1 = grp * G + h1;
    {
      const int c = line1 / R, y = y0 + (line1 - c * R);
  #pragma unroll
      for (int n2 = 0; n2 < B; n2++) v[n2] = C2<T>{T(0), T(0)};
      if (y < Ny) {
        // component base selected from the uniform arguments (an indexed read
        // of x.in would be a per-lane load ahead of every spectrum load)
        const C2<T> *inc = c == 0 ? x.in[0] : c == 1 ? x.in[1] : x.in[2];
        const C2<T> *irow = inc + ((long)z * x.Py + y) * x.Hp;
        // two halves of loads: half the staging registers live at a time
  #pragma unroll
        for (int hb = 0; hb < 2; hb++) {
          C2<T> xk[HB], xn[HB];
  #pragma unroll
          for (int q = 0; q < HB; q++) {
            const int k = n1 + A * (hb * HB + q);
            xk[q] = irow[k];
            xn[q] = irow[N - k];
          }
  #pragma unroll
          for (int q = 0; q < HB; q++) {
            const int n2 = hb * HB + q, k = n1 + A * n2;
            const C2<T> sm = cadd(xk[q], cconj(xn[q])), d = csub(xk[q], cconj(xn[q]));
            const C2<T> t = cmul(cconj(x.tw2[k]), d);
            v[n2] = C2<T>{sm.x - t.y, sm.y + t.x};
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      dft<B, +1>(v);
      __syncthreads();   // the twiddle table is complete
  #pragma unroll
      for (int k2 = 1; k2 < B; k2++) v[k2] = cmul(v[k2], cconj(twb[n1 * (B + 1) + k2]));   // W_n^-(n1 k2)
    }
    C2<T> u[G][A];
    T *tw = ldr + line1 * TS + n1;
  #pragma unroll
    for (int k2 = 0; k2 < B; k2++) tw[k2 * (A + 1)] = v[k2].x;
    __syncthreads();
  #pragma unroll
    for (int h = 0; h < G; h++) {
      const T *t = ldr + (grp * G + h) * TS + l * (A + 1);
  #pragma unroll
      for (int q = 0; q < A; q++) u[h][q].x = t[q];
    }
    __syncthreads();
  #pragma unroll
    for (int k2 = 0; k2 < B; k2++) tw[k2 * (A + 1)] = v[k2].y;
    __syncthreads();
  #pragma unroll
    for (int h = 0; h < G; h++) {
      const T *t = ldr + (grp * G + h) * TS + l * (A + 1);
  #pragma unroll
      for (int q = 0; q < A; q++) u[h][q].y = t[q];
    }
    T *bl = ldr;
    __syncthreads();   // every transpose read is done: the space now takes the real lines
  #pragma unroll
    for (int h = 0; h < G; h++) {
      dft<A, +1>(u[h]);
      T *o = bl + (grp * G + h) * N;
  #pragma unroll
      for (int k1 = 0; k1 < A / 2; k1++) *(float2 *)(o + 2 * (l + B * k1)) = float2{u[h][k1].x, u[h][k1].y};
    }
    __syncthreads();
    constexpr int NGX = N / 4, NG = R * NGX;
    for (int g = threadIdx.x; g < NG; g += XF_NT) {
      const int j = g / NGX, gx = g - j * NGX, y = y0 + j;
      if (y >= Ny) continue;
      T bdv[3][4];
  #pragma unroll
      for (int c = 0; c < 3; c++) {
        const float4 b = *(const float4 *)(bl + (c * R + j) * N + 4 * gx);
        bdv[c][0] = b.x; bdv[c][1] = b.y; bdv[c][2] = b.z; bdv[c][3] = b.w;
      }
      field_group4<T, REG, EX, false, UNI, false, TH>(f, 4 * gx, y, z, bdv);   // registers over instructions
    }
  }
};
template <typename T, int N, bool REG, int EX, bool UNI, bool TH>
__global__ __launch_bounds__(XF_NT, (BXi4Field<T, N, REG, EX, UNI, TH>::MINB)) void k_xi4_field(XiFieldArgs<T> a) {
  BXi4Field<T, N, REG, EX, UNI, TH>::run(a, hw_bid(), hw_grid());
}

// whether the fused kernel covers these field terms and buffers: the
// four-cell kernel's terms without spin-transfer torques or bulk DMI, every
// per-cell array aligned to four cells
template <typename T>
bool xi4_field_ok(const FieldArgs<T> &a, int n) {
  if (!std::is_same<T, float>::value || a.g.Nx != n || a.g.Nx % 4) return false;
  if (n != 64 && n != 128 && n != 256 && n != 512 && n != 1024) return false;
  if (a.exch_mode == 3 || a.has_zl || a.has_sl) return false;
  auto al = [](const void *p) { return ((uintptr_t)p & (4 * sizeof(T) - 1)) == 0; };
  for (int c = 0; c < 3; c++) {
    if (!al(a.m[c])) return false;
    if (a.tau[0] && !al(a.tau[c])) return false;
    if (a.beff[0] && !al(a.beff[c])) return false;
  }
  return !a.regions || ((uintptr_t)a.regions & 3) == 0;
}

template <typename T>
void launch_xi4_field(const XiArgs<T> &a, const FieldArgs<T> &f, int n, hipStream_t s) {
  if constexpr (std::is_same<T, float>::value) {
    const int Ny = a.fRy.d, Nz = a.rows / Ny;
    const bool reg = f.regions != nullptr, uni = field_uniform(f), th = f.has_therm != 0;
    auto go = [&](auto tag, auto kern, int R) {
      using K = typename decltype(tag)::type;
      const dim3 grid((unsigned)(((Ny + R - 1) / R) * Nz));
      launch_b<K>(kern, grid, dim3(XF_NT), 0, s, XiFieldArgs<T>{a, f});
      UM_HIP(hipGetLastError());
    };
// the thermal-free variants only for uniform parameters (the hot case);
// per-cell parameters without a thermal term take the TH = true kernel
#define UM_XF2(CN, RG, E)                                                                                      \
  { if (uni && !th) go(BTag<BXi4Field<T, CN, RG, E, true, false>>{}, k_xi4_field<T, CN, RG, E, true, false>,    \
                       XFShape<CN>::R);                                                                          \
    else if (uni) go(BTag<BXi4Field<T, CN, RG, E, true, true>>{}, k_xi4_field<T, CN, RG, E, true, true>,         \
                     XFShape<CN>::R);                                                                            \
    else go(BTag<BXi4Field<T, CN, RG, E, false, true>>{}, k_xi4_field<T, CN, RG, E, false, true>, XFShape<CN>::R); }
#define UM_XF(CN)                                                                                    \
  if (n == CN) {                                                                                     \
    if (f.exch_mode == 0) { if (reg) UM_XF2(CN, true, 0) else UM_XF2(CN, false, 0) }                 \
    else if (f.exch_mode == 1) { if (reg) UM_XF2(CN, true, 1) else UM_XF2(CN, false, 1) }            \
    else { if (reg) UM_XF2(CN, true, 2) else UM_XF2(CN, false, 2) }                                  \
    return;                                                                                          \
  }
    UM_XF(64) UM_XF(128) UM_XF(256) UM_XF(512) UM_XF(1024)
#undef UM_XF
#undef UM_XF2
  }
  throw Error(UM_EUNSUP, "fused X inverse: unsupported length");
}

template bool xi4_field_ok<float>(const FieldArgs<float> &, int);
template void launch_xi4_field<float>(const XiArgs<float> &, const FieldArgs<float> &, int, hipStream_t);

}  // namespace um

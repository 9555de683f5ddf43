// Kernels of demag_reg.hpp; included once per precision.
#pragma once
#include "demag_reg.hpp"
#include "fft_device.hpp"
#include "stage_device.hpp"

namespace um {

// a stage body called out of line would keep its captures in scratch memory
#define UM_INLINE __attribute__((always_inline))
template <int R> struct RadixTag { static constexpr int value = R; };
// f(RadixTag<r>) for a run-time radix r <= MAX
template <int MAX, typename F>
__device__ __forceinline__ void with_radix(int r, F &&f) {
  switch (r) {
    case 1: f(RadixTag<1>{}); break;
    case 2: f(RadixTag<2>{}); break;
    case 3: f(RadixTag<3>{}); break;
    case 4: f(RadixTag<4>{}); break;
    case 5: f(RadixTag<5>{}); break;
    case 6: f(RadixTag<6>{}); break;
    case 7: f(RadixTag<7>{}); break;
    case 8: f(RadixTag<8>{}); break;
    case 9: f(RadixTag<9>{}); break;
    case 10: f(RadixTag<10>{}); break;
    case 12: if constexpr (MAX >= 12) f(RadixTag<12>{}); break;
    case 14: if constexpr (MAX >= 14) f(RadixTag<14>{}); break;
    case 15: if constexpr (MAX >= 15) f(RadixTag<15>{}); break;
    case 16: if constexpr (MAX >= 16) f(RadixTag<16>{}); break;
    case 20: if constexpr (MAX >= 20) f(RadixTag<20>{}); break;
    default: break;
  }
}

// value at a wave-uniform base plus a 32-bit byte offset of the lane
template <typename C, typename B>
__device__ __forceinline__ C ldg(const B *base, uint32_t off) {
  return *(const C *)((const char *)base + off);
}
template <typename C>
__device__ __forceinline__ void stg(C *base, uint32_t off, C v) {
  *(C *)((char *)base + off) = v;
}
// v[k] *= W^(i k) from a [k][i] table with rows of `row` entries (conjugated for the inverse)
template <int R, int DIR, typename C>
__device__ __forceinline__ void twiddle(C (&v)[R], const C *tw, int row, int i) {
#pragma unroll
  for (int k = 1; k < R; k++) {
    // long transforms: a bounded number of factors in flight
    if (R > 10 && (k == 1 || k % 6 == 0)) pin(v);
    C w = ldg<C>(tw + (long)k * row, (uint32_t)(i * sizeof(C)));
    if (DIR > 0) w.y = -w.y;
    v[k] = cmul(v[k], w);
  }
}

// LDS layout of a tile: element `slot` of line l at l*ls + slot*es.  LF: lines
// are interleaved (es = lines, adjacent lanes take adjacent lines), else each
// line is contiguous (adjacent lanes take adjacent butterflies).
template <bool LF>
struct Tile {
  int nl, lsh, ls, es;
  __device__ __forceinline__ Tile(int nl_, int lsh_, int line) : nl(nl_), lsh(lsh_), ls(LF ? 1 : line), es(LF ? nl_ : 1) {}
  // work item g -> line l, butterfly q of `nb` per line
  __device__ __forceinline__ void split(int g, const FastDiv &fb, int &l, int &q) const {
    if (LF) { l = g & (nl - 1); q = g >> lsh; }
    else { l = (int)fb.div(g); q = g - l * (int)fb.d; }
  }
};

// middle stage (r1) of nl lines (x comps), in place; ends with a barrier.
// Forward stages transform, then twiddle; inverse ones (INV) untwiddle first.
template <typename T, int DIR, bool INV, int MAX, bool LF>
__device__ __forceinline__ void reg_stage1(C2<T> *lds, const RegLen &f, const Tile<LF> &t, int nl) {
  if (f.r[1] == 1) return;
  with_radix<MAX>(f.r[1], [&](auto tag) UM_INLINE {
    constexpr int R = decltype(tag)::value;
    const int step = f.n2 * t.es;
    for (int g = threadIdx.x; g < nl * (int)f.fb1.d; g += blockDim.x) {
      int l, q;
      t.split(g, f.fb1, l, q);
      const int k0 = (int)f.f2.div(q), i = q - k0 * f.n2;
      C2<T> *p = lds + l * t.ls + (k0 * f.pitch + i) * t.es;
      C2<T> v[R];
#pragma unroll
      for (int j = 0; j < R; j++) v[j] = p[j * step];
      if (INV) twiddle<R, DIR>(v, (const C2<T> *)f.tw1, f.n2, i);
      dft<R, DIR>(v);
      if (!INV) twiddle<R, DIR>(v, (const C2<T> *)f.tw1, f.n2, i);
#pragma unroll
      for (int j = 0; j < R; j++) p[j * step] = v[j];
    }
  });
  __syncthreads();
}

// pointer c of three, by selects of values: an indexed or conditional read of
// the argument block or of captured variables would put them in scratch memory
template <typename P>
__device__ __forceinline__ P sel3(int c, P p0, P p1, P p2) {
  P r = p0;
  if (c == 1) r = p1;
  if (c == 2) r = p2;
  return r;
}
template <typename P>
__device__ __forceinline__ P pick(P const (&p)[3], int c) { return sel3<P>(c, p[0], p[1], p[2]); }

// ---- X forward -----------------------------------------------------------------
// Lanes run along a row: real loads, LDS and the unpacked spectrum stores are
// all unit-stride.  Bound by its LDS round trips and barriers (three stages
// plus the unpacking).  Against the generic Stockham kernel: 1000 x 1000 FP32
// 31.8 -> 17.6 us (36 MB), 160 x 160 x 10 18.7 -> 10.1, 70^3 FP64 13.8 -> 13.0.
template <typename T>
struct BRXfwd {
  using Args = RXArgs<T>;
  static constexpr int NT = 512, MINB = sizeof(T) == 4 ? 4 : 1;
  static __device__ __forceinline__ void run(const RXArgs<T> &a, uint3 blockIdx, uint3) {
    extern __shared__ __align__(16) unsigned char smem_[];
    C2<T> *lds = (C2<T> *)smem_;
    const RegLen &f = a.f;
    const int c = blockIdx.y, row0 = blockIdx.x * a.nl, nl = min(a.nl, a.rows - row0);
    const int n = f.n, Nx = a.Nx, line = f.r[0] * f.pitch;
    const Tile<false> t(nl, 0, line);
    const T *src = pick(a.src, c);
    C2<T> *out = pick(a.spec, c);
    const T *const msa = a.Ms.arr, *const vol = a.vol;
    const T mul = a.Ms.mul, fac = T(MU0) * mul;
    with_radix<RegMax<T>::X>(f.r[0], [&](auto tag) UM_INLINE {
      constexpr int R = decltype(tag)::value;
      for (int g = threadIdx.x; g < nl * f.n1; g += blockDim.x) {
        int l, i;
        t.split(g, f.f1, l, i);
        // reals 2e, 2e+1 of the row for e = i + j n1 (zero beyond Nx)
        const uint32_t o = (uint32_t)((l * a.in_pitch + 2 * i) * sizeof(T));
        const int left = Nx - 2 * i;
        auto row = [&](const T *p, C2<T>(&v)[R]) UM_INLINE {
          const T *b = p + (long)row0 * a.in_pitch;
#pragma unroll
          for (int j = 0; j < R; j++) {
            const int e = 2 * j * f.n1;   // uniform
            v[j] = C2<T>{T(0), T(0)};
            if (a.pairs) {
              if (e < left) v[j] = ldg<C2<T>>(b + e, o);
            } else {
              if (e < left) v[j].x = ldg<T>(b + e, o);
              if (e + 1 < left) v[j].y = ldg<T>(b + e + 1, o);
            }
          }
        };
        C2<T> v[R];
        row(src, v);
        if (!msa && !vol) {
#pragma unroll
          for (int j = 0; j < R; j++) v[j] = C2<T>{fac * v[j].x, fac * v[j].y};
        } else {   // ((mu0 Ms) vol) m, as copypadmul2.cl
          C2<T> w[R];
          if (msa) {
            row(msa, w);
#pragma unroll
            for (int j = 0; j < R; j++) w[j] = C2<T>{T(MU0) * (mul * w[j].x), T(MU0) * (mul * w[j].y)};
          } else {
#pragma unroll
            for (int j = 0; j < R; j++) w[j] = C2<T>{fac, fac};
          }
          if (vol) {
            C2<T> u[R];
            row(vol, u);
#pragma unroll
            for (int j = 0; j < R; j++) w[j] = C2<T>{w[j].x * u[j].x, w[j].y * u[j].y};
          }
#pragma unroll
          for (int j = 0; j < R; j++) v[j] = C2<T>{w[j].x * v[j].x, w[j].y * v[j].y};
        }
        dft<R, -1>(v);
        twiddle<R, -1>(v, (const C2<T> *)f.tw0, f.n1, i);
        C2<T> *p = lds + l * line + i;
#pragma unroll
        for (int k = 0; k < R; k++) p[k * f.pitch] = v[k];
      }
    });
    __syncthreads();
    reg_stage1<T, -1, false, RegMax<T>::X>(lds, f, t, nl);
    with_radix<RegMax<T>::X>(f.r[2], [&](auto tag) UM_INLINE {
      constexpr int R = decltype(tag)::value;
      for (int g = threadIdx.x; g < nl * (int)f.fb2.d; g += blockDim.x) {
        int l, q;
        t.split(g, f.fb2, l, q);
        const int k1 = (int)f.fr0.div(q), k0 = q - k1 * f.r[0];
        C2<T> *p = lds + l * line + k0 * f.pitch + k1 * f.n2;
        C2<T> v[R];
#pragma unroll
        for (int j = 0; j < R; j++) v[j] = p[j];
        dft<R, -1>(v);
#pragma unroll
        for (int j = 0; j < R; j++) p[j] = v[j];
      }
    });
    __syncthreads();
    // two-for-one: X[k] = E[k] + W^k O[k], X[n-k] = conj(E[k] - W^k O[k])
    auto slot = [&](int k) UM_INLINE {
      const int u = (int)f.fr0.div(k), w = (int)f.fr1.div(u);
      return (k - u * f.r[0]) * f.pitch + (u - w * f.r[1]) * f.n2 + w;
    };
    const int half = n / 2 + 1;
    for (int g = threadIdx.x; g < nl * half; g += blockDim.x) {
      const int l = (int)a.fhalf.div(g), k = g - l * half, r = row0 + l;
      const C2<T> A = lds[l * line + slot(k)];
      const C2<T> Bc = cconj(lds[l * line + slot(k == 0 ? 0 : n - k)]);
      const C2<T> E = C2<T>{T(0.5) * (A.x + Bc.x), T(0.5) * (A.y + Bc.y)};
      const C2<T> O = C2<T>{T(0.5) * (A.y - Bc.y), T(-0.5) * (A.x - Bc.x)};
      const C2<T> w = cmul(a.tw2[k], O);
      const int z = (int)a.fRy.div(r), y = r - z * (int)a.fRy.d;
      C2<T> *orow = out + ((long)z * a.Py + y) * a.Hp;
      orow[k] = cadd(E, w);
      if (n - k != k) orow[n - k] = cconj(csub(E, w));
    }
  }
};
template <typename T>
__global__ __launch_bounds__(512, sizeof(T) == 4 ? 4 : 1) void k_rxfwd(RXArgs<T> a) { BRXfwd<T>::run(a, hw_bid(), hw_grid()); }

// X forward of rows that a solver stage forms first: the work-group stores its
// rows of one component, then transforms what it stored.
template <typename T>
struct BRXStage {
  using Args = RXStageArgs<T>;
  static constexpr int NT = 512, MINB = sizeof(T) == 4 ? 4 : 1;
  static __device__ __forceinline__ void run(const RXStageArgs<T> &as, uint3 blockIdx, uint3 gridDim) {
    const RXArgs<T> &a = as.x;
    const int row0 = blockIdx.x * a.nl, pairs = min(a.nl, a.rows - row0) * (a.Nx / 2);
    if (!(as.st.skip && *as.st.skip))
      for (int g = threadIdx.x; g < pairs; g += blockDim.x) stage_pair(as.st, blockIdx.y, (long)row0 * a.Nx + 2 * g);
    __syncthreads();
    BRXfwd<T>::run(a, blockIdx, gridDim);
  }
};
template <typename T>
__global__ __launch_bounds__(512, sizeof(T) == 4 ? 4 : 1) void k_rxstage(RXStageArgs<T> a) { BRXStage<T>::run(a, hw_bid(), hw_grid()); }

// ---- X inverse -----------------------------------------------------------------
// One LDS round trip less than the forward pass: the last stage's lanes hold
// neighbouring outputs of a row and store them directly.  1000 x 1000 FP32
// 33.6 -> 15.5 us, 160 x 160 x 10 19.3 -> 7.0, 70^3 FP64 20.6 -> 9.5.
template <typename T>
struct BRXinv {
  using Args = RXArgs<T>;
  static constexpr int NT = 512, MINB = sizeof(T) == 4 ? 4 : 1;
  static __device__ __forceinline__ void run(const RXArgs<T> &a, uint3 blockIdx, uint3) {
    extern __shared__ __align__(16) unsigned char smem_[];
    C2<T> *lds = (C2<T> *)smem_;
    const RegLen &f = a.f;
    const int c = blockIdx.y, row0 = blockIdx.x * a.nl, nl = min(a.nl, a.rows - row0);
    const int n = f.n, Nx = a.Nx, line = f.r[0] * f.pitch;
    const Tile<false> t(nl, 0, line);
    const int z0 = (int)a.fRy.div(row0);
    const C2<T> *in = pick(a.spec, c) + (long)z0 * a.Py * a.Hp;
    T *dst = pick(a.dst, c);
    // Z'[k] = (X[k] + conj X[n-k]) + i W^-k (X[k] - conj X[n-k]), transformed over its first radix
    with_radix<RegMax<T>::X>(f.r[0], [&](auto tag) UM_INLINE {
      constexpr int R = decltype(tag)::value;
      for (int g = threadIdx.x; g < nl * f.n1; g += blockDim.x) {
        int l, i;
        t.split(g, f.f1, l, i);
        const int r = row0 + l, z = (int)a.fRy.div(r), y = r - z * (int)a.fRy.d;
        // row offset in bytes from the work-group's first row (its z plane at least)
        const uint32_t o = (uint32_t)((((long)(z - z0) * a.Py + y) * a.Hp + i) * sizeof(C2<T>));
        const uint32_t on = (uint32_t)((((long)(z - z0) * a.Py + y) * a.Hp + f.n1 - i) * sizeof(C2<T>));
        // batches of at most 8 loads of each kind in flight: bounded staging registers
        constexpr int LB = sizeof(T) == 4 ? 8 : 4;
        C2<T> v[R];
#pragma unroll
        for (int j0 = 0; j0 < R; j0 += LB) {
          C2<T> xn[LB];
#pragma unroll
          for (int j = j0; j < R && j < j0 + LB; j++) {
            v[j] = ldg<C2<T>>(in + j * f.n1, o);
            xn[j - j0] = ldg<C2<T>>(in + (R - 1 - j) * f.n1, on);   // n - k
          }
#pragma unroll
          for (int j = j0; j < R && j < j0 + LB; j++) {
            const C2<T> x = cconj(xn[j - j0]);
            const C2<T> sm = cadd(v[j], x), d = csub(v[j], x);
            const C2<T> w = cmul(cconj(ldg<C2<T>>(a.tw2 + j * f.n1, (uint32_t)(i * sizeof(C2<T>)))), d);
            v[j] = C2<T>{sm.x - w.y, sm.y + w.x};
          }
          if (R > LB) __builtin_amdgcn_sched_barrier(0);
        }
        dft<R, +1>(v);
        twiddle<R, +1>(v, (const C2<T> *)f.tw0, f.n1, i);
        C2<T> *p = lds + l * line + i;
#pragma unroll
        for (int k = 0; k < R; k++) p[k * f.pitch] = v[k];
      }
    });
    __syncthreads();
    reg_stage1<T, +1, false, RegMax<T>::X>(lds, f, t, nl);
    // outputs m = q + r0 r1 j in natural order along the lanes: x[2m], x[2m+1]
    const int nb = (int)f.fb2.d;
    with_radix<RegMax<T>::X>(f.r[2], [&](auto tag) UM_INLINE {
      constexpr int R = decltype(tag)::value;
      for (int g = threadIdx.x; g < nl * nb; g += blockDim.x) {
        int l, q;
        t.split(g, f.fb2, l, q);
        const int k1 = (int)f.fr0.div(q), k0 = q - k1 * f.r[0];
        const C2<T> *p = lds + l * line + k0 * f.pitch + k1 * f.n2;
        C2<T> v[R];
#pragma unroll
        for (int j = 0; j < R; j++) v[j] = p[j];
        dft<R, +1>(v);
        T *b = dst + (long)row0 * Nx;
        const uint32_t o = (uint32_t)((l * Nx + 2 * q) * sizeof(T));
        const int left = Nx - 2 * q;
#pragma unroll
        for (int j = 0; j < R; j++) {
          const int e = 2 * nb * j;   // uniform
          if (a.pairs) {
            if (e < left) stg((C2<T> *)(b + e), o, v[j]);
          } else {
            if (e < left) stg<T>(b + e, o, v[j].x);
            if (e + 1 < left) stg<T>(b + e + 1, o, v[j].y);
          }
        }
      }
    });
  }
};
template <typename T>
__global__ __launch_bounds__(512, sizeof(T) == 4 ? 4 : 1) void k_rxinv(RXArgs<T> a) { BRXinv<T>::run(a, hw_bid(), hw_grid()); }

// ---- column pass ---------------------------------------------------------------
// Adjacent lanes take adjacent kx, so every global row segment has the tile's
// width; the tiles one XCD runs are adjacent (xcd_tile), so segments shorter
// than a line meet in its L2.  160 x 160 x 10 FP32 27.8 -> 9.9 us (19 MB),
// 320 x 200 x 6 50.9 -> 11.0, 1024 x 1024 x 8 292 -> 200 forward and 222
// inverse (605 MB, 3.0 and 2.7 TB/s; four columns a tile, 64 KB of LDS).
template <typename T, int DIR>
struct BRCol {
  using Args = RColArgs<T>;
  static constexpr int NT = 512, MINB = sizeof(T) == 4 ? 4 : 1;
  static __device__ __forceinline__ void run(const RColArgs<T> &a, uint3 blockIdx, uint3 gridDim) {
    extern __shared__ __align__(16) unsigned char smem_[];
    C2<T> *lds = (C2<T> *)smem_;
    const RegLen &f = a.f;
    const int nl = 1 << a.lsh;
    const Tile<true> t(nl, a.lsh, 0);
    const int ngx = gridDim.x, ngy = gridDim.y;
    const int w = xcd_tile(blockIdx.x + ngx * (blockIdx.y + ngy * blockIdx.z), ngx * ngy * gridDim.z);
    const int gx = w % ngx, gyz = w / ngx, gy = gyz % ngy, gz = gyz / ngy;
    const int kx0 = gx << a.lsh;
    C2<T> *base = pick(a.buf, gz) + (long)gy * a.pstride + kx0;
    with_radix<RegMax<T>::COL>(f.r[0], [&](auto tag) UM_INLINE {
      constexpr int R = decltype(tag)::value;
      for (int g = threadIdx.x; g < nl * f.n1; g += blockDim.x) {
        int l, i;
        t.split(g, f.f1, l, i);
        const int left = kx0 + l < a.H ? a.nvalid - i : 0;
        const uint32_t o = (uint32_t)((i * a.estride + l) * sizeof(C2<T>));
        C2<T> v[R];
#pragma unroll
        for (int j = 0; j < R; j++) {
          v[j] = C2<T>{T(0), T(0)};
          if (j * f.n1 < left) v[j] = ldg<C2<T>>(base + j * f.n1 * a.estride, o);
        }
        dft<R, DIR>(v);
        twiddle<R, DIR>(v, (const C2<T> *)f.tw0, f.n1, i);
        C2<T> *p = lds + l + i * nl;
#pragma unroll
        for (int k = 0; k < R; k++) p[k * f.pitch * nl] = v[k];
      }
    });
    __syncthreads();
    reg_stage1<T, DIR, false, RegMax<T>::COL>(lds, f, t, nl);
    const int nb = (int)f.fb2.d;
    with_radix<RegMax<T>::COL>(f.r[2], [&](auto tag) UM_INLINE {
      constexpr int R = decltype(tag)::value;
      for (int g = threadIdx.x; g < nl * nb; g += blockDim.x) {
        int l, q;
        t.split(g, f.fb2, l, q);
        const int k1 = (int)f.fr0.div(q), k0 = q - k1 * f.r[0];
        const C2<T> *p = lds + l + (k0 * f.pitch + k1 * f.n2) * nl;
        C2<T> v[R];
#pragma unroll
        for (int j = 0; j < R; j++) v[j] = p[j * nl];
        dft<R, DIR>(v);
        const int left = kx0 + l < a.H ? a.nout - q : 0;
        const uint32_t o = (uint32_t)((q * a.estride + l) * sizeof(C2<T>));
#pragma unroll
        for (int j = 0; j < R; j++)
          if (j * nb < left) stg(base + j * nb * a.estride, o, v[j]);
      }
    });
  }
};
template <typename T, int DIR>
__global__ __launch_bounds__(512, sizeof(T) == 4 ? 4 : 1) void k_rcol(RColArgs<T> a) { BRCol<T, DIR>::run(a, hw_bid(), hw_grid()); }

// one symmetric tensor times (M0, M1, M2): xx yy zz yz xz xy = k0..k5
template <typename T>
__device__ __forceinline__ void sym_mul(C2<T> &M0, C2<T> &M1, C2<T> &M2, T xx, T yy, T zz, T yz, T xz, T xy) {
  const C2<T> a = M0, b = M1, c = M2;
  M0 = C2<T>{a.x * xx + b.x * xy + c.x * xz, a.y * xx + b.y * xy + c.y * xz};
  M1 = C2<T>{a.x * xy + b.x * yy + c.x * yz, a.y * xy + b.y * yy + c.y * yz};
  M2 = C2<T>{a.x * xz + b.x * yz + c.x * zz, a.y * xz + b.y * yz + c.y * zz};
}

// ---- convolution pass ------------------------------------------------------------
// The thread that ends the forward transform of a butterfly holds the same
// frequencies of all three components, multiplies them by the tensor in
// registers and starts their inverse transforms (the first inverse stage reads
// exactly the slots the last forward stage left), so a line crosses LDS
// 2 (stages - 1) times and the spectrum is never reordered.  The generic kernel
// it replaces ran every radix pass through LDS with scratch spills.
// 1000 x 1000 FP32 225 -> 66 us, 250 x 250 24.3 -> 14.7, 70^3 FP64 134 -> 44
// (84 MB).  Bound by the round trips of a work-group: 2000-point films hold
// 96 KB of LDS, one work-group a CU.
// ky of grid row w: 0, Py-1, 1, Py-2, ... so that the mirror rows, which read
// the same tensor rows, run next to each other
__device__ __forceinline__ int mirror_order(int w, int Py) { return (w & 1) ? Py - (w + 1) / 2 : w / 2; }

template <typename T>
struct BRConv {
  using Args = RConvArgs<T>;
  static constexpr int NT = 512, MINB = sizeof(T) == 4 ? 4 : 1;
  static __device__ __forceinline__ void run(const RConvArgs<T> &a, uint3 blockIdx, uint3 gridDim) {
    extern __shared__ __align__(16) unsigned char smem_[];
    C2<T> *lds = (C2<T> *)smem_;
    const RegLen &f = a.f;
    const int n = f.n, nl = 1 << a.lsh;
    const Tile<true> t(nl, a.lsh, 0);
    const int cs = (f.r[0] * f.pitch) << a.lsh;   // LDS elements per component
    const int w = xcd_tile(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x * gridDim.y);
    const int kx0 = (w % (int)gridDim.x) << a.lsh, kyw = w / (int)gridDim.x;
    C2<T> *const b0 = a.buf[0], *const b1 = a.buf[1], *const b2 = a.buf[2];
    const T *const K0 = a.K[0], *const K1 = a.K[1], *const K2 = a.K[2], *const K3 = a.K[3], *const K4 = a.K[4],
            *const K5 = a.K[5];
    const int ky = a.is2d ? 0 : mirror_order(kyw, a.Py);
    const bool ym = 2 * ky > a.Py;                 // mirror half: yz and xy change sign
    const int kyt = ym ? a.Py - ky : ky;
    const long off = (long)ky * a.pstride + kx0;
    with_radix<RegMax<T>::CONV>(f.r[0], [&](auto tag) UM_INLINE {
      constexpr int R = decltype(tag)::value;
      for (int g = threadIdx.x; g < 3 * nl * f.n1; g += blockDim.x) {
        const int l = g & (nl - 1), h = g >> a.lsh, c = (int)f.f1.div(h), i = h - c * f.n1;
        const int left = kx0 + l < a.H ? a.nvalid - i : 0;
        const C2<T> *base = sel3(c, b0, b1, b2) + off + i * a.estride + l;   // per lane: c varies
        C2<T> v[R];
#pragma unroll
        for (int j = 0; j < R; j++) {
          v[j] = C2<T>{T(0), T(0)};
          if (j * f.n1 < left) v[j] = base[j * f.n1 * a.estride];
        }
        dft<R, -1>(v);
        twiddle<R, -1>(v, (const C2<T> *)f.tw0, f.n1, i);
        C2<T> *p = lds + c * cs + l + i * nl;
#pragma unroll
        for (int k = 0; k < R; k++) p[k * f.pitch * nl] = v[k];
      }
    });
    __syncthreads();
    for (int c = 0; c < 3 && f.r[1] > 1; c++) reg_stage1<T, -1, false, RegMax<T>::CONV>(lds + c * cs, f, t, nl);
    const int nb = (int)f.fb2.d;
    with_radix<RegMax<T>::MID>(f.r[2], [&](auto tag) UM_INLINE {
      constexpr int R = decltype(tag)::value;
      for (int g = threadIdx.x; g < nl * nb; g += blockDim.x) {
        int l, q;
        t.split(g, f.fb2, l, q);
        const int k1 = (int)f.fr0.div(q), k0 = q - k1 * f.r[0];
        C2<T> *p = lds + l + (k0 * f.pitch + k1 * f.n2) * nl;
        const int kx = min(kx0 + l, a.H - 1);
        C2<T> v[3][R];
#pragma unroll
        for (int c = 0; c < 3; c++) {
#pragma unroll
          for (int j = 0; j < R; j++) v[c][j] = p[c * cs + j * nl];
          dft<R, -1>(v[c]);
          pin(v[c]);   // one transform at a time
        }
#pragma unroll
        for (int j = 0; j < R; j++) {
          if (j % 2 == 0) __builtin_amdgcn_sched_barrier(0);   // tensor values of two frequencies live
          const int k = q + nb * j;
          const bool zm = 2 * k > n;
          const int kt = zm ? n - k : k;
          if (a.is2d) {   // yz = xz = 0; the mirror flips xy
            const long I = (long)kt * a.Hk + kx;
            const T xy = zm ? -K5[I] : K5[I];
            const C2<T> M0 = v[0][j], M1 = v[1][j];
            const T xx = K0[I], yy = K1[I], zz = K2[I];
            v[0][j] = C2<T>{M0.x * xx + M1.x * xy, M0.y * xx + M1.y * xy};
            v[1][j] = C2<T>{M0.x * xy + M1.x * yy, M0.y * xy + M1.y * yy};
            v[2][j] = C2<T>{v[2][j].x * zz, v[2][j].y * zz};
          } else {        // the ky mirror flips yz and xy, the kz mirror yz and xz
            const long I = ((long)kt * a.KHy + kyt) * a.Hk + kx;
            const T yz = K3[I], xz = K4[I], xy = K5[I];
            sym_mul(v[0][j], v[1][j], v[2][j], K0[I], K1[I], K2[I], ym != zm ? -yz : yz, zm ? -xz : xz,
                    ym ? -xy : xy);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < 3; c++) {
          dft<R, +1>(v[c]);
#pragma unroll
          for (int j = 0; j < R; j++) p[c * cs + j * nl] = v[c][j];
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    });
    __syncthreads();
    for (int c = 0; c < 3 && f.r[1] > 1; c++) reg_stage1<T, +1, true, RegMax<T>::CONV>(lds + c * cs, f, t, nl);
    with_radix<RegMax<T>::CONV>(f.r[0], [&](auto tag) UM_INLINE {
      constexpr int R = decltype(tag)::value;
      for (int g = threadIdx.x; g < 3 * nl * f.n1; g += blockDim.x) {
        const int l = g & (nl - 1), h = g >> a.lsh, c = (int)f.f1.div(h), i = h - c * f.n1;
        C2<T> *base = sel3(c, b0, b1, b2) + off + i * a.estride + l;
        const int left = kx0 + l < a.H ? a.nvalid - i : 0;
        const C2<T> *p = lds + c * cs + l + i * nl;
        C2<T> v[R];
#pragma unroll
        for (int k = 0; k < R; k++) v[k] = p[k * f.pitch * nl];
        twiddle<R, +1>(v, (const C2<T> *)f.tw0, f.n1, i);
        dft<R, +1>(v);
#pragma unroll
        for (int j = 0; j < R; j++)
          if (j * f.n1 < left) base[j * f.n1 * a.estride] = v[j];
      }
    });
  }
};
template <typename T>
__global__ __launch_bounds__(512, sizeof(T) == 4 ? 4 : 1) void k_rconv(RConvArgs<T> a) { BRConv<T>::run(a, hw_bid(), hw_grid()); }

// ---- launches ------------------------------------------------------------------------
template <typename K>
static void reg_lds(K kern, size_t bytes) {
  if (bytes > 65536)
    UM_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
}
template <typename T>
void launch_rxfwd(const RXArgs<T> &a, int nt, hipStream_t s) {
  const size_t lds = sizeof(C2<T>) * (size_t)a.nl * a.f.line();
  reg_lds(k_rxfwd<T>, lds);
  launch_b<BRXfwd<T>>(k_rxfwd<T>, dim3((a.rows + a.nl - 1) / a.nl, 3), dim3(nt), lds, s, a);
  UM_HIP(hipGetLastError());
}
template <typename T>
void launch_rxinv(const RXArgs<T> &a, int nt, hipStream_t s) {
  const size_t lds = sizeof(C2<T>) * (size_t)a.nl * a.f.line();
  reg_lds(k_rxinv<T>, lds);
  launch_b<BRXinv<T>>(k_rxinv<T>, dim3((a.rows + a.nl - 1) / a.nl, 3), dim3(nt), lds, s, a);
  UM_HIP(hipGetLastError());
}
template <typename T>
void launch_rxstage(const RXStageArgs<T> &a, int nt, hipStream_t s) {
  const size_t lds = sizeof(C2<T>) * (size_t)a.x.nl * a.x.f.line();
  reg_lds(k_rxstage<T>, lds);
  launch_b<BRXStage<T>>(k_rxstage<T>, dim3((a.x.rows + a.x.nl - 1) / a.x.nl, 3), dim3(nt), lds, s, a);
  UM_HIP(hipGetLastError());
}
template <typename T>
void launch_rcol(const RColArgs<T> &a, int dir, int planes, int nt, hipStream_t s) {
  const size_t lds = sizeof(C2<T>) * ((size_t)a.f.line() << a.lsh);
  const dim3 grid((a.H + (1 << a.lsh) - 1) >> a.lsh, planes, 3);
  if (dir < 0) {
    reg_lds(k_rcol<T, -1>, lds);
    launch_b<BRCol<T, -1>>(k_rcol<T, -1>, grid, dim3(nt), lds, s, a);
  } else {
    reg_lds(k_rcol<T, +1>, lds);
    launch_b<BRCol<T, +1>>(k_rcol<T, +1>, grid, dim3(nt), lds, s, a);
  }
  UM_HIP(hipGetLastError());
}
template <typename T>
void launch_rconv(const RConvArgs<T> &a, int nt, hipStream_t s) {
  const size_t lds = sizeof(C2<T>) * 3 * ((size_t)a.f.line() << a.lsh);
  reg_lds(k_rconv<T>, lds);
  launch_b<BRConv<T>>(k_rconv<T>, dim3((a.H + (1 << a.lsh) - 1) >> a.lsh, a.is2d ? 1 : a.Py), dim3(nt), lds, s, a);
  UM_HIP(hipGetLastError());
}
template <typename T>
void RegTab<T>::append(RegKind kind, int n, long units, long mult, UnitRoots &roots, std::vector<C2<T>> &host) {
  const RegPlan p = reg_plan(kind, sizeof(T) == 8, n, units, mult);
  len = p.f;
  nl = p.nl;
  nt = p.nt;
  if (!len.n) return;
  off = host.size();
  const auto &w = roots.get(n);
  auto put = [&](long m) { host.push_back(C2<T>{(T)w[m % n].x, (T)w[m % n].y}); };
  for (int k = 0; k < len.r[0]; k++)
    for (int i = 0; i < len.n1; i++) put((long)i * k);
  for (int k = 0; k < len.r[1]; k++)
    for (int i = 0; i < len.n2; i++) put((long)i * k * len.r[0]);
}
template <typename T>
void RegTab<T>::bind(const C2<T> *dev) {
  len.tw0 = dev + off;
  len.tw1 = dev + off + (size_t)len.r[0] * len.n1;
}

#define UM_REG_INSTANTIATE(T)                                              \
  template void launch_rxfwd<T>(const RXArgs<T> &, int, hipStream_t);      \
  template void launch_rxinv<T>(const RXArgs<T> &, int, hipStream_t);      \
  template void launch_rxstage<T>(const RXStageArgs<T> &, int, hipStream_t); \
  template void launch_rcol<T>(const RColArgs<T> &, int, int, int, hipStream_t); \
  template void launch_rconv<T>(const RConvArgs<T> &, int, hipStream_t);   \
  template struct RegTab<T>;

}  // namespace um

// Register-stage FFT passes of the demag convolution for any length that
// splits into at most three radices of RegRadix (7-smooth lengths up to a few
// thousand).  A work-group holds its lines in LDS once, in place: stage s
// transforms strided elements in registers (decimation in frequency), so the
// first stage reads global memory directly, the last one writes it directly,
// and a line crosses LDS once per stage boundary.  The frequency of slot
// (k0, k1, j) is k0 + r0 k1 + r0 r1 j; nothing is reordered in memory.
//
// Host side: reg_plan() picks the radices, launch_r*() run a pass.
#pragma once
#include <map>
#include <vector>

#include "batch.hpp"
#include "fft.hpp"
#include "vec.hpp"

namespace um {

struct RegLen {
  int n;                 // length; 0: not available
  int r[3];              // radices in stage order (1 = stage skipped)
  int n1, n2;            // n / r0, n / (r0 r1) = r2
  int pitch;             // LDS pitch of the r0 blocks (odd: the strided stages fall on distinct banks)
  FastDiv f1, f2, fr0, fr1, fb1, fb2;   // n1, n2, r0, r1, n / r1, r0 r1
  const void *tw0;       // [k][i] = W_n^(i k),  k < r0, i < n1
  const void *tw1;       // [k][i] = W_n1^(i k), k < r1, i < n2
  int line() const { return r[0] * pitch; }   // LDS elements of a line
};

// Largest radices of each pass: what the kernels hold in registers without
// spilling (an X row needs its Ms values beside it, the last convolution stage
// the three components), and FP64 values take two registers.
template <typename T> struct RegMax;
template <> struct RegMax<float> { static constexpr int X = 16, COL = 20, CONV = 20, MID = 10; };
template <> struct RegMax<double> { static constexpr int X = 10, COL = 16, CONV = 16, MID = 10; };
// Radices, lines and threads per work-group of a pass of `units` lines (times
// `mult`) of length n; f.n = 0 where n has no split.
struct RegPlan {
  RegLen f{};
  int nl = 1, nt = 64;
};
enum RegKind { REG_X, REG_COL, REG_CONV };
RegPlan reg_plan(RegKind kind, bool f64, int n, long units, long mult);

// exp(-2 pi i m / n), m < n, in long double; a length is evaluated once, or
// read out of a multiple's table
struct UnitRoots {
  struct Z { long double x, y; };
  std::map<int, std::vector<Z>> tab;
  const std::vector<Z> &get(int n);
};

// plan of a pass; its twiddle tables lie in a device buffer shared by the
// passes of a convolution (append, then bind to the uploaded copy)
template <typename T>
struct RegTab {
  RegLen len{};
  int nl = 1, nt = 64;
  size_t off = 0;
  void append(RegKind kind, int n, long units, long mult, UnitRoots &roots, std::vector<C2<T>> &host);
  void bind(const C2<T> *dev);
};

// X passes: rows of Nx reals <-> H = n + 1 complex (two-for-one)
template <typename T>
struct RXArgs {
  RegLen f;
  const C2<T> *tw2;       // exp(-2 pi i k / 2n)
  int nl, Nx, rows, Py, Hp;
  int pairs;              // Nx even and every real row aligned to two values: pairwise access
  FastDiv fhalf, fRy;     // n/2 + 1; rows per z plane
  long in_pitch;
  const T *src[3];        // forward: real rows; inverse: unused
  Par<T> Ms;
  const T *vol;
  C2<T> *spec[3];
  T *dst[3];              // inverse: real rows of Nx
};
template <typename T>
struct RXStageArgs {
  RXArgs<T> x;
  StageArgs<T> st;        // the solver stage that forms the input rows
};
// column pass along y
template <typename T>
struct RColArgs {
  RegLen f;
  int lsh;                // log2(columns per work-group)
  int H, nvalid, nout;
  long estride, pstride;
  C2<T> *buf[3];
};
// forward, tensor multiply, inverse along the last axis
template <typename T>
struct RConvArgs {
  RegLen f;
  int lsh;
  int H, nvalid;
  long estride, pstride;
  int is2d, Py, KHy, Hk;
  const T *K[6];
  C2<T> *buf[3];
};
// the same for short z columns held in registers (one thread per column)
template <typename T>
struct RShortArgs {
  int H, Py, KHy, Hk;
  long zstride, ystride;
  const T *K[6];
  C2<T> *buf[3];
};

template <typename T> void launch_rxfwd(const RXArgs<T> &a, int nt, hipStream_t s);
template <typename T> void launch_rxinv(const RXArgs<T> &a, int nt, hipStream_t s);
template <typename T> void launch_rxstage(const RXStageArgs<T> &a, int nt, hipStream_t s);
template <typename T> void launch_rcol(const RColArgs<T> &a, int dir, int planes, int nt, hipStream_t s);
template <typename T> void launch_rconv(const RConvArgs<T> &a, int nt, hipStream_t s);
// register z columns: columns = kx columns times ky rows
template <typename T> bool short_ok(int Nz, int Pz, long columns);
template <typename T> void launch_rshort(const RShortArgs<T> &a, int Nz, int Pz, hipStream_t s);

}  // namespace um

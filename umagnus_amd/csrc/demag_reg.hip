// Plan of a register-stage FFT pass: radices, lines and threads, and the roots
// of unity of its twiddle tables.
#include <algorithm>
#include <cmath>

#include "demag_reg.hpp"

namespace um {

const std::vector<UnitRoots::Z> &UnitRoots::get(int n) {
  auto it = tab.find(n);
  if (it != tab.end()) return it->second;
  std::vector<Z> v(n);
  for (auto &t : tab)
    if (t.first % n == 0) {
      for (int m = 0; m < n; m++) v[m] = t.second[(size_t)m * (t.first / n)];
      return tab.emplace(n, std::move(v)).first->second;
    }
  for (int m = 0; m < n; m++) {
    const long double ang = -2.0L * 3.14159265358979323846264338327950288L * (long double)m / (long double)n;
    v[m] = Z{cosl(ang), sinl(ang)};
  }
  return tab.emplace(n, std::move(v)).first->second;
}

static RegLen reg_split(int n, int r0, int r1, int r2) {
  RegLen f{};
  f.n = n;
  f.r[0] = r0; f.r[1] = r1; f.r[2] = r2;
  f.n1 = n / r0;
  f.n2 = r2;
  f.pitch = f.n1 | 1;
  f.f1.init(f.n1); f.f2.init(f.n2); f.fr0.init(r0); f.fr1.init(r1);
  f.fb1.init(n / r1); f.fb2.init(r0 * r1);
  return f;
}

// The split with the smallest radix sum: a thread's chain of loads, transform,
// twiddles and LDS accesses grows with its radix, and these passes wait on
// that chain more than on bandwidth (160-point X rows at 160x160x10, FP32:
// 4 8 5 takes 2.5 us less than 10 16; 320-point columns: 8 4 10 3.3 us less
// than 16 20).  A further stage costs a barrier and an LDS round trip, 4 in
// the units of the sum, or 9 in the convolution, where it comes six times
// (140 points in FP64: 14 10 takes 7.5 us less than 7 4 5).
//
// Lines: X rows until a stage has about 384 work items, columns until a row
// segment has 64 bytes or more (LDS allowing), halved while the pass would
// launch fewer than two work-groups a CU.  Threads: one per item of the widest
// stage on small grids, where a second round would add its latency; half as
// many where work-groups queue for the CUs and the other work-groups of a CU
// cover it.
RegPlan reg_plan(RegKind kind, bool f64, int n, long units, long mult) {
  static const int R[] = {1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 12, 14, 15, 16, 20};
  const int es = f64 ? 16 : 8, comps = kind == REG_CONV ? 3 : 1;
  int rmax, rlast;
  auto lim = [&](auto t) {
    using M = RegMax<decltype(t)>;
    rmax = kind == REG_X ? M::X : kind == REG_COL ? M::COL : M::CONV;
    rlast = kind == REG_CONV ? M::MID : rmax;
  };
  if (f64) lim(double()); else lim(float());
  RegPlan p;
  double least = 1e300;
  for (int r0 : R)
    for (int r1 : R) {
      if (r0 > rmax || r1 > rmax || n % (r0 * r1) || (r1 > 1 && r0 == 1)) continue;
      const int r2 = n / (r0 * r1);
      bool ok = false;
      for (int r : R) ok = ok || r == r2;
      if (!ok || r2 > rlast) continue;
      // ties: the convolution runs r1 three times per direction (small r1);
      // an X row's first stage meets the padded zeros (small r0)
      double cost = r0 + r1 + r2 + (kind == REG_CONV ? 9 : 4) * ((r0 > 1) + (r1 > 1) - 1);
      cost += kind == REG_CONV ? 0.1 * r1 - 0.01 * r0 : 0.1 * r0;
      if (cost < least) { least = cost; p.f = reg_split(n, r0, r1, r2); }
    }
  if (!p.f.n) return p;
  const RegLen &f = p.f;
  auto lds = [&](int nl) { return (size_t)es * comps * f.line() * nl; };
  auto wgs = [&](int nl) { return (units + nl - 1) / nl * mult; };
  const long widest = std::max({n / f.r[0], f.r[1] > 1 ? n / f.r[1] : 0, n / f.r[2]});
  long items;
  if (kind == REG_X) {
    p.nl = (int)std::max(1L, std::min(64L, 384 / widest));
    while (p.nl > 1 && (lds(p.nl) > 49152 || wgs(p.nl) < 512)) p.nl--;
    items = p.nl * widest;
  } else if (kind == REG_COL) {
    p.nl = 8;
    while (p.nl > 4 && lds(p.nl) > 49152) p.nl /= 2;
    while (p.nl > 1 && (lds(p.nl) > 81920 || (p.nl > 2 && wgs(p.nl) < 512))) p.nl /= 2;
    items = p.nl * widest;
  } else {
    p.nl = mult == 1 ? 2 : 64 / es;
    while (p.nl > 1 && (lds(p.nl) > 106496 || wgs(p.nl) < 256)) p.nl /= 2;
    items = 3L * p.nl * f.n1;
  }
  if (lds(p.nl) > 163840) { p.f.n = 0; return p; }
  const long per = wgs(p.nl) > 1024 ? 2 : 1, cap = kind == REG_CONV || items >= 1024 ? 512 : 256;
  p.nt = (int)std::max(64L, std::min(cap, (items / per + 63) / 64 * 64));
  return p;
}

}  // namespace um

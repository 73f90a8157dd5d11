// The turbulence line solves in parts against 113-bit solutions, beside the
// one-sided recurrence of the reference (lsolvej / lsolvek), compiled and run
// by tests/test_plain_cpu.py.
//
// Lines of the shape the convection and diffusion of the turbulence models
// give, a(i) = -(u(i) > 0) u(i-1) - nu, c(i) = (u(i) < 0) u(i+1) - nu,
// b(i) = 1/dt + |u(i)| + |v(i)| + 2 nu, times dt: an off-diagonal carries the
// neighbour's speed, so a row need not be dominant.  Speeds change sign along
// the line, smoothly or from cell to cell; dt and nu span their decades.
// Bound: both solvers are off by a few rounding errors of the line's largest
// value, so over the lines of a kind their medians lie within a quarter of each
// other; the 99th percentile of the parts is held to twice the recurrence's.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <random>
#include <vector>

#include "ot2d_plain.h"

using namespace ot2d;
typedef std::vector<double> Vec;

namespace {
// the parts of a line one after another, as the lanes do them side by side
template <int M>
Vec solve_parts(Vec a, Vec b, Vec c, Vec s) {
  const int n = (int)a.size(), P = (n + M - 1) / M;
  a[0] = 0.;
  c[n - 1] = 0.;
  a.resize(P * M, 0.);
  b.resize(P * M, 1.);
  c.resize(P * M, 0.);
  s.resize(P * M, 0.);
  typedef double Part[M];
  auto at = [](Vec& x, int p) -> Part& { return *reinterpret_cast<Part*>(&x[(size_t)p * M]); };
  for (int p = 0; p < P; ++p) part_eliminate<M>(at(a, p), at(b, p), at(c, p), at(s, p));
  std::vector<SepRow> w(P);
  for (int p = 0; p < P; ++p) {
    const bool next = p + 1 < P;
    w[p] = part_separator<M>(at(a, p), at(b, p), at(c, p), at(s, p), next ? s[(p + 1) * M] : 0.,
                             next ? a[(p + 1) * M] : 0., next ? c[(p + 1) * M] : 0.);
  }
  for (int d = 1; d < P; d <<= 1) {
    const std::vector<SepRow> o = w;
    const SepRow none = {0., 0., 0.};
    for (int p = 0; p < P; ++p) w[p] = sep_reduce(o[p], p >= d ? o[p - d] : none, p + d < P ? o[p + d] : none);
  }
  for (int p = 0; p < P; ++p) part_expand<M>(at(a, p), at(c, p), at(s, p), p ? w[p - 1].D : 0., w[p].D);
  s.resize(n);
  return s;
}

Vec solve(const Vec& a, const Vec& b, const Vec& c, const Vec& s) {
  switch (part_cells((int)a.size())) {
    case 8: return solve_parts<8>(a, b, c, s);
    case 12: return solve_parts<12>(a, b, c, s);
    default: return solve_parts<16>(a, b, c, s);
  }
}

template <typename T>
std::vector<T> recurrence(const Vec& a, const Vec& b, const Vec& c, const Vec& s) {
  const int n = (int)a.size();
  std::vector<T> x(n), cp(n);
  T bb = T(1) / b[0];
  x[0] = s[0] * bb;
  cp[0] = c[0] * bb;
  for (int i = 1; i < n; ++i) {
    bb = T(1) / (b[i] - a[i] * cp[i - 1]);
    x[i] = (s[i] - a[i] * x[i - 1]) * bb;
    cp[i] = c[i] * bb;
  }
  for (int i = n - 2; i >= 0; --i) x[i] = x[i] - cp[i] * x[i + 1];
  return x;
}

double quantile(Vec v, double f) {
  std::sort(v.begin(), v.end());
  return v[(size_t)(f * (v.size() - 1))];
}
}  // namespace

int main() {
  enum Kind { MIXED, CONVECTION, DIFFUSION, NO_CROSS, ROUGH, ROUGH_NO_CROSS, ONE_WAY, SMOOTH_NO_CROSS, KINDS };
  std::mt19937_64 g(7);
  std::normal_distribution<double> N(0, 1);
  std::uniform_real_distribution<double> U(0, 1);
  int failed = 0;
  double dom = 1e300, med_lo = 1, med_hi = 0, rec_lo = 1, rec_hi = 0, p99 = 0;
  for (int kind = 0; kind < KINDS; ++kind) {
    Vec er, ep;
    for (int n : {24, 64, 100, 200, 384, 512, 768, 1000})
      for (int it = 0; it < 400; ++it) {
        const double dt = std::pow(10., -1 + 4 * U(g));
        double nu = std::pow(10., -4 + 3 * U(g));
        if (kind == CONVECTION) nu = 0;
        if (kind == DIFFUSION) nu = std::pow(10., -1 + 2 * U(g));
        const bool rough = kind == ROUGH || kind == ROUGH_NO_CROSS;
        const bool cross = kind != NO_CROSS && kind != ROUGH_NO_CROSS && kind != SMOOTH_NO_CROSS;
        const double k1 = 25 * U(g) / n, p1 = 6.28 * U(g), k2 = 126 * U(g) / n, p2 = 6.28 * U(g);
        Vec u(n + 2), v(n + 2, 0.), a(n), b(n), c(n), s(n);
        for (int i = 0; i < n + 2; ++i) {
          u[i] = rough ? N(g) : std::sin(k1 * i + p1) + 0.3 * std::sin(k2 * i + p2);
          if (kind == ONE_WAY) u[i] = std::fabs(u[i]) + 1e-3;
          if (cross) v[i] = 0.2 * N(g);
        }
        for (int i = 0; i < n; ++i) {
          const double uc = u[i + 1], d = dt * (0.5 + U(g));
          a[i] = d * (-(uc > 1e-12 ? u[i] : 0.) - nu);
          c[i] = d * ((uc < -1e-12 ? u[i + 2] : 0.) - nu);
          b[i] = 1 + d * (std::fabs(uc) + std::fabs(v[i + 1]) + 2 * nu);
          s[i] = d * N(g);
          if (i > 0 && i < n - 1) dom = std::min(dom, b[i] / (std::fabs(a[i]) + std::fabs(c[i]) + 1e-300));
        }
        a[0] = 0;
        c[n - 1] = 0;
        const std::vector<__float128> x = recurrence<__float128>(a, b, c, s);
        const Vec r = recurrence<double>(a, b, c, s), p = solve(a, b, c, s);
        double top = 0, dr = 0, dp = 0;
        for (int i = 0; i < n; ++i) {
          top = std::max(top, std::fabs((double)x[i]));
          dr = std::max(dr, std::fabs((double)(x[i] - (__float128)r[i])));
          dp = std::max(dp, std::fabs((double)(x[i] - (__float128)p[i])));
        }
        er.push_back(dr / top);
        ep.push_back(dp / top);
      }
    const double mr = quantile(er, .5), mp = quantile(ep, .5), qr = quantile(er, .99), qp = quantile(ep, .99);
    std::printf("kind %d: recurrence median %.2e p99 %.2e, parts %.2e %.2e\n", kind, mr, qr, mp, qp);
    if (!(mp <= 1.25 * mr && qp <= 2 * qr)) {
      std::printf("failed\n");
      failed = 1;
    }
    med_lo = std::min(med_lo, mp);
    med_hi = std::max(med_hi, mp);
    rec_lo = std::min(rec_lo, mr);
    rec_hi = std::max(rec_hi, mr);
    p99 = std::max(p99, qp / qr);
  }
  std::printf("least dominance %.1e; medians: parts %.2e to %.2e, recurrence %.2e to %.2e; p99 ratio %.2f\n", dom, med_lo,
              med_hi, rec_lo, rec_hi, p99);
  return failed || dom > 0.01;
}

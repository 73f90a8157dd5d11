// Rules and arithmetic on plain values, shared by the kernels and the CPU
// tests (which include this file alone, with the host compiler).
#pragma once
#if defined(__HIP__)
#define OT2D_PLAIN __host__ __device__ __forceinline__
#else
#define OT2D_PLAIN inline
#endif

namespace ot2d {

// Limit of a wait between the workgroups of one sweep launch, or between the
// waves of one of its workgroups: it is given up after POLLS polls that found
// nothing.  A normal wait is a few microseconds.  Polls and not time, for a
// clock runs on while the queue's waves are put aside for other processes'
// work, all of a launch together, and would end a sweep whose neighbour had
// no chance to run.  A poll of LDS takes upwards of 0.08 us of the wave's
// running time and one of memory about 1 us, so 2^22 of them are 0.3 to 5 s.
struct BoundedWait {
  static constexpr unsigned POLLS = 1u << 22;
  unsigned polls;
  OT2D_PLAIN void start() { polls = 0u; }
  // one more poll has found nothing: give up?
  OT2D_PLAIN bool over() { return ++polls > POLLS; }
};

// Tiles over the chip.  Workgroups go to the 8 XCDs in turn, so in a launch of
// (G, records) workgroups those of one record whose x agrees modulo 8 share
// an XCD.  Each of these 8 classes takes a run of neighbouring tiles, whose
// shared halos then come out of that XCD's L2: tile of workgroup x of a record
// of n <= G tiles, or -1.  A class of workgroups has as many members below n as
// its run has tiles, so G need not be a multiple of 8.  Filled up to one, 1000
// cases of 33x17 (2 tiles each) launched 6 empty workgroups in 8: viscous
// terms 114 us, 39 without them, SA right-hand side 88 and 35; 60 cases 1975
// and 1952 us a step.
OT2D_PLAIN int xcd_deal(int x, int n) {
  const int c = x & 7, len = n >> 3, more = n & 7;
  return x < n ? c * len + (c < more ? c : more) + (x >> 3) : -1;
}

// The launch choice a search keeps: n candidates timed in `rounds` rounds,
// candidate k's times at ms[k * rounds].  The fastest (by its best round) is
// taken over candidate `def` only if it wins by more than the rounds of
// both differ among themselves, and by more than 1 %: the choices of a
// class often lie closer than that (513x129 SA FP32: 263.3, 264.4, 264.8,
// 265.6, 268.6, 270.0 us a step), and by the best time alone a search took
// one that is slower than the default.
inline int pick_launch(const float* ms, int n, int rounds, int def) {
  auto low = [&](int k) {
    float v = ms[k * rounds];
    for (int r = 1; r < rounds; ++r) v = ms[k * rounds + r] < v ? ms[k * rounds + r] : v;
    return v;
  };
  auto spread = [&](int k) {
    float v = ms[k * rounds];
    for (int r = 1; r < rounds; ++r) v = ms[k * rounds + r] > v ? ms[k * rounds + r] : v;
    return v - low(k);
  };
  int best = def;
  for (int k = 0; k < n; ++k)
    if (low(k) < low(best)) best = k;
  const float both = spread(def) + spread(best), least = 0.01f * low(def), need = both > least ? both : least;
  return low(def) - low(best) > need ? best : def;
}

// ------------------------------------------------- turbulence line solves
// Tridiagonal line of n cells, a x(i-1) + b x(i) + c x(i+1) = s, solved in
// parts of M cells, one lane per part (the turbulence models' line solves:
// lsolvej / lsolvek and their two-equation forms).  The last cell of every
// part is its separator.  Each lane eliminates its inner cells against the
// separators on both sides, x(i) = S(i) + L(i) XL + R(i) XR; the separators'
// own tridiagonal system (one row per part) is solved by parallel cyclic
// reduction across the parts; the inner cells follow in parallel.  The
// dependent chain is 2 M + log2(n / M) steps instead of n / 2 for an
// elimination from both ends by two lanes, which bound these solves.
// Parts depend on n alone, so every mapping of lines to workgroups gives the
// same bits.  Quotients are corrected by one residual step (num - den q)
// and sums use fused operations.  Rows need not be dominant (an upwind row's
// off-diagonals carry the neighbours' speeds): of 25600 lines of 24 to 1000
// cells, convective, diffusive and mixed, with speeds that change sign and
// rows down to a dominance of 1e-3, the median errors relative to the line's
// largest value are 1.1-3.9e-16 by kind (the one-sided recurrence 1.2-5.1e-16)
// and the 99th percentiles no larger than the recurrence's
// (tests/line_parts_check.cpp, against 113-bit solutions).
// Cells past the line's end are identity rows; a of the first cell and c of
// the last are zero.
OT2D_PLAIN int part_cells(int n) { return n <= 512 ? 8 : (n <= 768 ? 12 : 16); }   // at most 64 parts

OT2D_PLAIN double quot(double num, double den, double r) {   // num / den, r = 1 / den
  const double q = num * r;
  return __builtin_fma(__builtin_fma(-den, q, num), r, q);
}

// inner cells 0 .. M-2: s, a, c become S, L, R
template <int M>
OT2D_PLAIN void part_eliminate(double (&a)[M], const double (&b)[M], double (&c)[M], double (&s)[M]) {
  {
    const double r = 1. / b[0];
    s[0] = quot(s[0], b[0], r);
    a[0] = -quot(a[0], b[0], r);
    c[0] = quot(c[0], b[0], r);
  }
#pragma unroll
  for (int i = 1; i < M - 1; ++i) {
    const double ai = a[i], den = __builtin_fma(-ai, c[i - 1], b[i]);
    const double r = 1. / den;
    c[i] = quot(c[i], den, r);
    s[i] = quot(__builtin_fma(-ai, s[i - 1], s[i]), den, r);
    a[i] = -quot(ai * a[i - 1], den, r);
  }
  c[M - 2] = -c[M - 2];
#pragma unroll
  for (int i = M - 3; i >= 0; --i) {
    const double ci = c[i];
    s[i] = __builtin_fma(-ci, s[i + 1], s[i]);
    a[i] = __builtin_fma(-ci, a[i + 1], a[i]);
    c[i] = -ci * c[i + 1];
  }
}

// the separator's row A X(p-1) + X(p) + C X(p+1) = D from the part's inner
// cells and the next part's first cell (S, L, R)
struct SepRow { double A, C, D; };
template <int M>
OT2D_PLAIN SepRow part_separator(const double (&a)[M], const double (&b)[M], const double (&c)[M],
                                 const double (&s)[M], double Sn, double Ln, double Rn) {
  const double am = a[M - 1], cm = c[M - 1];
  const double den = __builtin_fma(am, c[M - 2], __builtin_fma(cm, Ln, b[M - 1]));
  const double r = 1. / den;
  SepRow o;
  o.A = quot(am * a[M - 2], den, r);
  o.C = quot(cm * Rn, den, r);
  o.D = quot(__builtin_fma(-am, s[M - 2], __builtin_fma(-cm, Sn, s[M - 1])), den, r);
  return o;
}

// one step of the cyclic reduction from the rows at distance d on both sides
// (zero rows past the ends)
OT2D_PLAIN SepRow sep_reduce(const SepRow& x, const SepRow& m, const SepRow& p) {
  const double den = __builtin_fma(-x.C, p.A, __builtin_fma(-x.A, m.C, 1.));
  const double r = 1. / den;
  SepRow o;
  o.A = -quot(x.A * m.A, den, r);
  o.C = -quot(x.C * p.C, den, r);
  o.D = quot(__builtin_fma(-x.C, p.D, __builtin_fma(-x.A, m.D, x.D)), den, r);
  return o;
}

// x of the part's cells from its separators
template <int M>
OT2D_PLAIN void part_expand(const double (&a)[M], const double (&c)[M], double (&s)[M], double XL, double XR) {
#pragma unroll
  for (int i = 0; i < M - 1; ++i) s[i] = __builtin_fma(c[i], XR, __builtin_fma(a[i], XL, s[i]));
  s[M - 1] = XR;
}

}  // namespace ot2d

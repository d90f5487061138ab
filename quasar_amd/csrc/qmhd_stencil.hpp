// Per-face and per-cell stencil code of the MHD step, shared by the gfx950
// kernels and by host builds of the same code (compiled with hipcc as host
// functions) that check the kernel logic on the CPU.
//
// Storage: every plane is a padded row-major array, index (i+ng) + pitch*(j+ng),
// pitch = nx + 2 ng (the reference's Grid2D, include/quasar/core/grid.hpp:84-200).
#pragma once

#include <cstddef>
#include <cstdint>

#include "qmhd_kernels.hpp"

namespace qmhd {

__host__ __device__ __forceinline__ std::size_t idx(const GridD& g, int i, int j) {
  return static_cast<std::size_t>(i + g.ng) + static_cast<std::size_t>(g.pitch) * static_cast<std::size_t>(j + g.ng);
}

// Periodic wrap or clamp of a face/cell coordinate (mode 4 keeps exchanged guards).
__host__ __device__ __forceinline__ int face_index(int q, int n, int lo_mode, int hi_mode) {
  if (lo_mode == 0 && hi_mode == 0) {
    int w = q % n;
    return w < 0 ? w + n : w;
  }
  if (q < 0) return lo_mode == 4 ? q : 0;
  if (q > n) return hi_mode == 4 ? q : n;
  return q;
}

// ---------------------------------------------------------------------------
// Face -> cell collocation of the staggered normal field.

__host__ __device__ __forceinline__ int colloc_width(int extent, int ng) {
  const int req = ng >= 4 ? 8 : ng >= 3 ? 6 : ng >= 2 ? 4 : 2;
  if (req >= 8 && extent >= 8) return 8;
  if (req >= 6 && extent >= 6) return 6;
  if (req >= 4 && extent >= 4) return 4;
  return extent >= 2 ? 2 : 1;
}

// Sample of the face array along `axis` at coordinate q on line `fixed`.
__host__ __device__ __forceinline__ double axis_face(const GridD& g, const double* f, int axis, int q, int fixed) {
  return axis == 0 ? f[idx(g, q, fixed)] : f[idx(g, fixed, q)];
}

// Correctly rounded (half-even) sum of up to N binary64 terms; zero terms are
// skipped and an exactly cancelling sum is +0.  The terms are accumulated into
// a non-overlapping expansion of increasing magnitude (Shewchuk's
// grow-expansion with the swap-ordered fast two-sum), kept in registers by full
// unrolling, and rounded from the top with the half-even correction of the
// published fsum finalisation.  This is the value the reference's exact
// expansion arithmetic returns (include/quasar/numerics/scaled_arithmetic.hpp:
// 121-208).  Callers pass finite terms.
template <int N>
__host__ __device__ __forceinline__ double cr_sum(const double* t) {
#pragma clang fp contract(off)
  double p[N];
#pragma unroll
  for (int k = 0; k < N; ++k) p[k] = 0.0;
#pragma unroll
  for (int k = 0; k < N; ++k) {
    double x = t[k];
    if (x != 0.0) {
#pragma unroll
      for (int q = 0; q < k; ++q) {
        const double y = p[q];
        const bool sw = __builtin_fabs(x) < __builtin_fabs(y);
        const double big = sw ? y : x, small = sw ? x : y;
        const double hi = big + small;
        p[q] = small - (hi - big);
        x = hi;
      }
      p[k] = x;
    }
  }
  double hi = 0.0, lo = 0.0, next = 0.0;
  bool broke = false, have_next = false;
#pragma unroll
  for (int q = N - 1; q >= 0; --q) {
    const double y = p[q];
    if (!broke) {
      const double x = hi;
      hi = x + y;
      lo = y - (hi - x);
      broke = lo != 0.0;
    } else if (!have_next && y != 0.0) {
      next = y;
      have_next = true;
    }
  }
  if (broke && have_next && ((lo < 0.0 && next < 0.0) || (lo > 0.0 && next > 0.0))) {
    const double y = lo * 2.0;
    const double x = hi + y;
    if (y == x - hi) hi = x;
  }
  return hi == 0.0 ? 0.0 : hi;
}

// s + e = a + b exactly (Knuth's two-sum).
__host__ __device__ __forceinline__ void two_sum(double a, double b, double& s, double& e) {
#pragma clang fp contract(off)
  s = a + b;
  const double bv = s - a;
  e = (a - (s - bv)) + (b - bv);
}

// A zero that the compiler does not know: what is computed from it in a loop
// stays in the loop (all terms hoisted out of cr_sum_each's take 20 registers of
// the preparation kernel, past three waves per SIMD).
__host__ __device__ __forceinline__ double opaque_zero() {
  double z = 0.0;
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+v"(z));
#endif
  return z;
}

// Rounds the sum of four accumulators, each under the rounding of the one before
// it or not, with cr_sum's half-even correction.
__host__ __device__ __forceinline__ double rounded_chain(double* c) {
#pragma clang fp contract(off)
#pragma unroll
  for (int pass = 0; pass < 3; ++pass)
#pragma unroll
    for (int q = 2; q >= 0; --q) two_sum(c[q], c[q + 1], c[q], c[q + 1]);
  const double t[4] = {c[3], c[2], c[1], c[0]};
  return cr_sum<4>(t);
}

// Correctly rounded sum of the terms that each(f) hands to f (at most 32; NaN
// where one or the sum is not finite, as the expansion arithmetic gives).  The
// rare path behind certified_sum (a one-sided closure in a thousand is a tie);
// the terms are formed again, so its registers do not grow with their number
// (cr_sum<16> keeps 16 partials).  First in four chained accumulators: every
// two-sum error moves one accumulator down, and the sum is exact while the last
// one does not round.  Where it does (terms that cancel over more than 159
// bits), by error-free extraction (Rump, Ogita and Oishi 2008): against a power
// of two above all partial sums every term splits into a multiple of that
// power's last bit, which add exactly, and a rest for the next, 2^46 smaller
// power; the accumulators take the slices from the top, and what they lose lies
// 159 bits and more under a leading part that no later slice reaches.
template <class E>
__host__ __device__ __forceinline__ double cr_sum_each(E each) {
#pragma clang fp contract(off)
  double c[4] = {0.0, 0.0, 0.0, 0.0};
  bool exact = true;
  each([&](double t) {
    two_sum(c[0], t, c[0], t);
    two_sum(c[1], t, c[1], t);
    two_sum(c[2], t, c[2], t);
    two_sum(c[3], t, c[3], t);
    exact = exact && t == 0.0;
  });
  if (exact) return rounded_chain(c);
  double top = 0.0, bad = 0.0;
  each([&](double t) {
    bad = bad + (t - t);
    top = __builtin_fmax(top, __builtin_fabs(t));
  });
  if (bad != 0.0) return bad;
  int e;
  (void)__builtin_frexp(top, &e);
  // Sums of terms next to the largest number are taken 2^60 smaller.
  const double unit = e > 1000 ? 0x1p-60 : 1.0, first = __builtin_ldexp(1.0, (e > 1000 ? e - 60 : e) + 6);
#pragma unroll
  for (int q = 0; q < 4; ++q) c[q] = 0.0;
  bool more = true;
#pragma nounroll
  for (double sigma = first; more; sigma = sigma * 0x1p-46) {
    double slice = 0.0;
    more = false;
    each([&](double t) {
      double rest = t * unit;
#pragma nounroll
      for (double s = first; s > sigma; s = s * 0x1p-46) rest = rest - ((s + rest) - s);
      const double part = (sigma + rest) - sigma;
      slice = slice + part;
      more = more || rest != part;
    });
    two_sum(c[0], slice, c[0], slice);
    two_sum(c[1], slice, c[1], slice);
    two_sum(c[2], slice, c[2], slice);
    c[3] = c[3] + slice;
  }
  const double r = rounded_chain(c) * (1.0 / unit);
  return __builtin_isfinite(r) ? r : r - r;
}

// Whether s + e, within `bound` of the exact sum of terms whose magnitudes add
// to mag, fixes its correctly rounded value r: the sum lies between
// r + (rr - bound) and r + (rr + bound) with r + rr = s + e, so r is the
// rounded value when both ends round to r.
__host__ __device__ __forceinline__ bool certified_sum(double s, double e, double mag, double& r) {
#pragma clang fp contract(off)
  double rr;
  two_sum(s, e, r, rr);
  const double eps = 2.220446049250313080847e-16;
  const double bound = 512.0 * eps * eps * mag;
  if (mag == 0.0) {
    r = 0.0;
    return true;
  }
  return r != 0.0 && r + (rr + bound) == r && r + (rr - bound) == r;
}

// a / b with the refined reciprocal y of b: the quotient's residual is exact,
// so one correction rounds it (Markstein 1990).  Callers keep a, b and the
// quotient away from the ends of the exponent range.  The host divides.
__host__ __device__ __forceinline__ double quot(double a, double b, double y) {
#if defined(__HIP_DEVICE_COMPILE__)
  const double q = a * y;
  return __builtin_fma(__builtin_fma(-b, q, a), y, q);
#else
  (void)y;
  return a / b;
#endif
}

template <int W>
__host__ __device__ __forceinline__ bool all_finite(const double* s) {
  bool finite = true;
#pragma unroll
  for (int k = 0; k < W; ++k) finite = finite && __builtin_isfinite(s[k]);
  return finite;
}

template <int W>
struct CentredRow;
template <>
struct CentredRow<8> {
  static constexpr double w[8] = {-191.0, 1879.0, -9531.0, 68323.0, 68323.0, -9531.0, 1879.0, -191.0};
  static constexpr double d = 120960.0;
};
template <>
struct CentredRow<6> {
  static constexpr double w[6] = {11.0, -93.0, 802.0, 802.0, -93.0, 11.0};
  static constexpr double d = 1440.0;
};
template <>
struct CentredRow<4> {
  static constexpr double w[4] = {-1.0, 13.0, 13.0, -1.0};
  static constexpr double d = 24.0;
};
template <>
struct CentredRow<2> {
  static constexpr double w[2] = {1.0, 1.0};
  static constexpr double d = 2.0;
};

// Centred cell average sum_k w_k s_k / d with the numerator correctly rounded
// (mhd_staggering.hpp:59-70): the value of the reference's exact rational
// collocation.  The numerator is a compensated dot product (Ogita, Rump and
// Oishi's Dot2: at most 64 eps^2/4 sum|w s| from the exact sum, bounded by
// certified_sum's 512 eps^2); ties and heavy cancellation take cr_sum_each.
template <int W>
__host__ __device__ __forceinline__ double colloc_centred(const double* s) {
#pragma clang fp contract(off)
  using R = CentredRow<W>;
  double sum = R::w[0] * s[0], e = __builtin_fma(R::w[0], s[0], -sum), mag = __builtin_fabs(sum);
#pragma unroll
  for (int k = 1; k < W; ++k) {
    const double p = R::w[k] * s[k], lo = __builtin_fma(R::w[k], s[k], -p);
    double t;
    two_sum(sum, p, sum, t);
    e = e + (t + lo);
    mag = mag + __builtin_fabs(p);
  }
  if (!__builtin_isfinite(mag) && !all_finite<W>(s)) {
    double acc = 0.0;
#pragma unroll
    for (int k = 0; k < W; ++k) acc = acc + R::w[k] * s[k];
    return acc / R::d;
  }
  double r;
  if (!certified_sum(sum, e, mag, r))
    r = cr_sum_each([&](auto f) {
      const double zero = opaque_zero();
#pragma unroll
      for (int k = 0; k < W; ++k) {
        const double x = s[k] + zero, p = R::w[k] * x;
        f(p);
        f(__builtin_fma(R::w[k], x, -p));
      }
    });
  // A numerator near the bottom of the exponent range leaves no exact residual.
  return __builtin_fabs(r) < 0x1p-900 ? r / R::d : quot(r, R::d, 1.0 / R::d);
}

// The centred rule as a plain fused multiply-add sum (the FP32 forms).
template <int W>
__host__ __device__ __forceinline__ double colloc_centred_fma(const double* s) {
  using R = CentredRow<W>;
  if (W == 2) return 0.5 * (s[0] + s[1]);
  double acc = 0.0;
#pragma unroll
  for (int k = 0; k < W; ++k) acc = fma(R::w[k], s[k], acc);
  return acc * (1.0 / R::d);
}

// One-sided closure of the outer ghost layers (mhd_staggering.hpp:111-173): the
// 4-point Gauss integral over cell `rel` of the barycentric interpolant through
// W consecutive faces, as a correctly rounded sum of the rounded
// product-quotient terms ((w_q b_k) s_k / (x_q - k)) / den_q, den_q the
// correctly rounded sum of b_k / (x_q - k).  den depends on (rel, q) alone and
// is tabulated.  The 4 W terms are summed in double-double and certified; they
// are formed again, by division, for cr_sum_each where that fails, so none is
// stored.  (Formed
// once, stored and expanded in registers with den summed on the device, the
// two ghost strips took 28 us at any grid size, a quarter of a small step.)
template <int W>
__host__ __device__ __forceinline__ double one_sided_den(int rel, int q) {
  static constexpr double den8[8][4] = {
      {0x1.14f137d46e474p+4, 0x1.f8c80074d005bp+2, 0x1.e3d859725c52ap+3, 0x1.6ed7d2561d6f0p+6},
      {-0x1.c0b0434cf8e66p+6, -0x1.3c6f3601b40bdp+5, -0x1.ca7f4af371dd1p+5, -0x1.20535ab48e7fep+8},
      {0x1.41765e1bef6dap+8, 0x1.8104008bc977fp+6, 0x1.c9a41cf316120p+6, 0x1.f2c2483909587p+8},
      {-0x1.02309860b4de3p+9, -0x1.0df8dc157721cp+7, -0x1.0df8dc157721cp+7, -0x1.02309860b4de3p+9},
      {0x1.f2c248390954fp+8, 0x1.c9a41cf316120p+6, 0x1.8104008bc977fp+6, 0x1.41765e1bef6b8p+8},
      {-0x1.20535ab48e7dcp+8, -0x1.ca7f4af371dd1p+5, -0x1.3c6f3601b40bdp+5, -0x1.c0b0434cf8e50p+6},
      {0x1.6ed7d2561d6cfp+6, 0x1.e3d859725c52ep+3, 0x1.f8c80074d005ap+2, 0x1.14f137d46e463p+4},
      {-0x1.824ee835b8992p+3, -0x1.61cd59d5b2438p+0, -0x1.5b7ffefc1a937p-2, -0x1.3659f02596131p-3}};
  static constexpr double den6[6][4] = {
      {0x1.0f05b79641acep+4, 0x1.c687647dc0f8ap+2, 0x1.84ad714acf13ap+3, 0x1.0cbe64ec6cd53p+6},
      {-0x1.38625562bca1bp+6, -0x1.8efd9d3fa7e1bp+4, -0x1.f7e3664b456ffp+4, -0x1.1b3dd70cc1219p+7},
      {0x1.28a9afe25a02dp+7, 0x1.3a39774832ef3p+5, 0x1.3a39774832ef3p+5, 0x1.28a9afe25a02dp+7},
      {-0x1.1b3dd70cc1219p+7, -0x1.f7e3664b456ffp+4, -0x1.8efd9d3fa7e1bp+4, -0x1.38625562bca2ap+6},
      {0x1.0cbe64ec6cd3bp+6, 0x1.84ad714acf13dp+3, 0x1.c687647dc0f89p+2, 0x1.0f05b79641abep+4},
      {-0x1.8aa796fef0833p+3, -0x1.86dbe50cf3676p+0, -0x1.a7472137ee67cp-2, -0x1.96243e36dcae5p-3}};
  static constexpr double den4[4][4] = {
      {0x1.069ea7d427ea4p+4, 0x1.858123c63e0bcp+2, 0x1.18376dbf83e1fp+3, 0x1.4faeffb4b3380p+5},
      {-0x1.67d435f5506d8p+5, -0x1.86f6eebf146a6p+3, -0x1.86f6eebf146a6p+3, -0x1.67d435f5506ecp+5},
      {0x1.4faeffb4b338ap+5, 0x1.18376dbf83e21p+3, 0x1.858123c63e0bcp+2, 0x1.069ea7d427eadp+4},
      {-0x1.97149b513699cp+3, -0x1.c30812c3758b4p+0, -0x1.18327f9fd4d54p-1, -0x1.28e67e0075ea1p-2}};
  static constexpr double den2[2][4] = {
      {0x1.ef456e91b52c8p+3, 0x1.217522dc95a71p+2, 0x1.217522dc95a71p+2, 0x1.ef456e91b52cep+3},
      {-0x1.aef610ccf8cefp+3, -0x1.23a0b30a91550p+1, -0x1.c999f1fda6dfap-1, -0x1.1cfe9e4de8eeep-1}};
  if constexpr (W == 8) return den8[rel][q];
  if constexpr (W == 6) return den6[rel][q];
  if constexpr (W == 4) return den4[rel][q];
  return den2[rel][q];
}

template <int W, bool DIVIDE, class F>
__host__ __device__ __forceinline__ void one_sided_terms(const double* s, int rel, F f) {
#pragma clang fp contract(off)
  constexpr double xq[4] = {0.0694318442029737124, 0.3300094782075718676, 0.6699905217924281324,
                            0.9305681557970262876};
  constexpr double wq[2] = {0.1739274225687269287, 0.3260725774312730713};
#pragma nounroll
  for (int q = 0; q < 4; ++q) {
    const double x = double(rel) + (q < 2 ? (q == 0 ? xq[0] : xq[1]) : (q == 2 ? xq[2] : xq[3]));
    const double wn = (q == 0 || q == 3) ? wq[0] : wq[1];
    const double den = one_sided_den<W>(rel, q), iden = frcp(den);
    double c = 1.0;  // (-1)^k C(W-1, k), exact small integers
#pragma unroll
    for (int k = 0; k < W; ++k) {
      const double xk = x - double(k);
      const double a = (wn * ((k % 2 == 0) ? c : -c)) * s[k];
      f(DIVIDE ? (a / xk) / den : quot(quot(a, xk, frcp(xk)), den, iden));
      c = c * double(W - 1 - k) / double(k + 1);
    }
  }
}

template <int W>
__host__ __device__ __forceinline__ double one_sided(const double* s, int rel) {
#pragma clang fp contract(off)
  bool zero = true;
#pragma unroll
  for (int k = 0; k < W; ++k) zero = zero && s[k] == 0.0;
  if (zero) return 0.0;
  double sum = 0.0, e = 0.0, mag = 0.0;
  one_sided_terms<W, false>(s, rel, [&](double t) {
    double lo;
    two_sum(sum, t, sum, lo);
    e = e + lo;
    mag = mag + __builtin_fabs(t);
  });
  if (!__builtin_isfinite(mag) && !all_finite<W>(s)) {
    // The quotients' residuals are no numbers here: the terms are divided.
    double acc = 0.0;
    one_sided_terms<W, true>(s, rel, [&](double t) { acc = acc + t; });
    return acc;
  }
  // Quotients near the bottom of the exponent range have no exact residual:
  // they are divided.
  double r;
  if (!certified_sum(sum, e, mag, r) || mag < 0x1p-900)
    r = cr_sum_each([&](auto f) { one_sided_terms<W, true>(s, rel, f); });
  return r;
}

// First face of the W-face window of padded cell `cell` (faces and cells
// lo .. hi of the line): centred, moved inside the line at its ends.
template <int W>
__host__ __device__ __forceinline__ int colloc_start(int cell, int lo, int hi) {
  int start = cell - (W / 2 - 1);
  start = start < lo ? lo : start;
  return start + W - 1 > hi ? hi - W + 1 : start;
}

// The centred rule in the form's arithmetic.
template <int W, bool EXACT>
__host__ __device__ __forceinline__ double colloc_centred_as(const double* s) {
  return EXACT ? colloc_centred<W>(s) : colloc_centred_fma<W>(s);
}

// Cell average from the window's faces s, the cell `rel` faces after its first
// face: the centred rule, or the one-sided closure where the window was moved.
template <int W, bool EXACT>
__host__ __device__ __forceinline__ double colloc_window(const double* s, int rel) {
  return rel == W / 2 - 1 ? colloc_centred_as<W, EXACT>(s) : one_sided<W>(s, rel);
}

// Learned form: a face normal to `dir` (x faces dir 0, y faces dir 1) is
// flagged when either of its two cells is.
__host__ __device__ __forceinline__ bool face_flagged(const GridD& g, int dir, const uint8_t* cell_flags, int i, int j) {
  return (cell_flags[idx(g, i, j)] | cell_flags[idx(g, i - (dir == 0), j - (dir == 1))]) != 0;
}

// Whether an unflagged face's interface states are read back: a flagged face
// at most 3 faces away along the face line (the transverse Gauss recovery's
// stencil) reads them.  Faces of the line outside the padded grid are not
// faces of any launch: they read face (0, 0)'s flags, which are masked off.
// Every flag is read and the results are OR'ed without short-circuit, so the
// 14 loads go out together (written as `read_back || face_flagged(...)`
// behind the range test, they were seven round trips one after another).
__host__ __device__ __forceinline__ bool face_states_read_back(const GridD& g, int dir, const uint8_t* cell_flags,
                                                               int i, int j) {
  unsigned any = 0;
#pragma unroll
  for (int d = -3; d <= 3; ++d) {
    int ii = i + (dir == 1 ? d : 0), jj = j + (dir == 0 ? d : 0);
    const bool inside = !(ii < -g.ng || jj < -g.ng || ii >= g.nx + g.ng || jj >= g.ny + g.ng);
    if (!inside) ii = 0, jj = 0;
    const unsigned f = cell_flags[idx(g, ii, jj)] | cell_flags[idx(g, ii - (dir == 0), jj - (dir == 1))];
    any |= inside ? f : 0u;
  }
  return any != 0;
}

// High-order cell average (8/6/4/2 taps, one-sided closures in the outer
// ghosts), mhd_staggering.hpp:175-236.
template <int W>
__host__ __device__ __forceinline__ double face_to_cell_w(const GridD& g, const double* f, int axis, int cell, int fixed) {
  const int n = axis == 0 ? g.nx : g.ny;
  const int start = colloc_start<W>(cell, -g.ng, n + g.ng - 1);
  double s[W];
#pragma unroll
  for (int k = 0; k < W; ++k) s[k] = axis_face(g, f, axis, start + k, fixed);
  return colloc_window<W, true>(s, cell - start);
}

__host__ __device__ inline double face_to_cell(const GridD& g, const double* f, int axis, int cell, int fixed) {
  const int width = colloc_width((axis == 0 ? g.nx : g.ny) + 2 * g.ng, g.ng);
  if (width == 8) return face_to_cell_w<8>(g, f, axis, cell, fixed);
  if (width == 6) return face_to_cell_w<6>(g, f, axis, cell, fixed);
  if (width == 4) return face_to_cell_w<4>(g, f, axis, cell, fixed);
  if (width == 2) return face_to_cell_w<2>(g, f, axis, cell, fixed);
  return axis_face(g, f, axis, cell, fixed);
}

// The same value under the name of the ghost cells' rule (every padded cell
// takes one); for host code that asks for it by that name.
__host__ __device__ inline double face_to_cell_ghost(const GridD& g, const double* f, int axis, int cell, int fixed) {
  return face_to_cell(g, f, axis, cell, fixed);
}

// First-order (two bounding faces) cell average used by the low-order retry.
__host__ __device__ __forceinline__ double face_to_cell_lo(const GridD& g, const double* f, int axis, int cell, int fixed) {
  const int n = axis == 0 ? g.nx : g.ny;
  const double a = axis_face(g, f, axis, cell, fixed);
  if (cell >= n + g.ng - 1) return a;
  const double b = axis_face(g, f, axis, cell + 1, fixed);
  const double s[2] = {a, b};
  return colloc_centred<2>(s);
}

// ---------------------------------------------------------------------------
// Reconstruction.

template <class T>
__host__ __device__ __forceinline__ St<T> load_cell(const GridD& g, const StateView& u, const double* bxc,
                                           const double* byc, int i, int j) {
  const std::size_t k = idx(g, i, j);
  return St<T>{T(u.c[0][k]), T(u.c[1][k]), T(u.c[2][k]), T(u.c[3][k]),
               T(u.c[4][k]), T(bxc[k]),    T(byc[k]),    T(u.c[7][k])};
}

template <class T>
__host__ __device__ __forceinline__ St<T> load_cell_lo(const GridD& g, const StateView& u, int i, int j) {
  const std::size_t k = idx(g, i, j);
  return St<T>{T(u.c[0][k]), T(u.c[1][k]), T(u.c[2][k]), T(u.c[3][k]), T(u.c[4][k]),
               T(face_to_cell_lo(g, u.c[5], 0, i, j)), T(face_to_cell_lo(g, u.c[6], 1, j, i)), T(u.c[7][k])};
}

// Reconstructed-state admissibility (mhd_reconstruct.hip:433-446): finite
// components and primitive velocities, rho > 0, reference pressure > 0.
template <class T>
__host__ __device__ __forceinline__ bool admissible_state(const St<T>& s, T gamma) {
  if (!(fin(s.rho) && s.rho > T(0))) return false;
  if (!(fin(s.mx) && fin(s.my) && fin(s.mz) && fin(s.en) && fin(s.bx) && fin(s.by) && fin(s.bz))) return false;
  if (!(finite_ratio(s.mx, s.rho) && finite_ratio(s.my, s.rho) && finite_ratio(s.mz, s.rho))) return false;
  return pressure_positive(s, gamma);
}

// The reference's decision with its pressure, in p where the state is
// admissible.
template <class T>
__host__ __device__ __forceinline__ bool admissible_state_p(const St<T>& s, T gamma, T& p) {
  if (!(fin(s.rho) && s.rho > T(0))) return false;
  if (!(fin(s.mx) && fin(s.my) && fin(s.mz) && fin(s.en) && fin(s.bx) && fin(s.by) && fin(s.bz))) return false;
  if (!(finite_ratio(s.mx, s.rho) && finite_ratio(s.my, s.rho) && finite_ratio(s.mz, s.rho))) return false;
  const T v = ref_pressure(s, gamma);
  if (!(fin(v) && v > T(0))) return false;
  p = v;
  return true;
}

// Replace the normal field of a face state keeping its pressure: the energy
// gains v^2/2 - bn^2/2 as one correctly rounded sum of the rounded products
// (mhd_reconstruct.hip:141-153).
// The FP32 form takes the plain FP32 sum.
template <class T>
__host__ __device__ __forceinline__ void set_normal_b(St<T>& s, int dir, T v) {
#pragma clang fp contract(off)
  T& bn = dir == 0 ? s.bx : s.by;
  if constexpr (sizeof(T) == 4) {
    s.en = (s.en + v * (T(0.5) * v)) - bn * (T(0.5) * bn);
  } else {
    const double t[3] = {double(s.en), double(v * (T(0.5) * v)), double(bn * (-T(0.5) * bn))};
    s.en = T(cr_sum<3>(t));
  }
  bn = v;
}

template <class T>
__host__ __device__ __forceinline__ T limited_slope(T back, T fwd, int drop) {
  if (drop < 0) return fwd;
  if (drop > 0) return back;
  return minmod2(back, fwd);
}

__host__ __device__ __forceinline__ int slope_drop(int c, int n, int lo, int hi) {
  if (lo != 0 && lo != 4 && c <= 0) return -1;
  if (hi != 0 && hi != 4 && c >= n - 1) return +1;
  return 0;
}

// Second-order MUSCL-minmod in primitive variables (also the MP fallback),
// mhd_reconstruct.hip:96-120, 375-414, in the reference's arithmetic.
// Both states of a face from the primitive cells around it.
template <class T>
__host__ __device__ __forceinline__ void muscl_pair(const Prim<T>* w, int drop_m, int drop_p, T gamma, St<T>& ul,
                                                    St<T>& ur) {
#pragma clang fp contract(off)
  auto face = [&](const Prim<T>& wm, const Prim<T>& wc, const Prim<T>& wp, T sign, int drop) {
    const T h = T(0.5) * sign;
    Prim<T> f;
    f.rho = wc.rho + h * limited_slope(wc.rho - wm.rho, wp.rho - wc.rho, drop);
    f.vx = wc.vx + h * limited_slope(wc.vx - wm.vx, wp.vx - wc.vx, drop);
    f.vy = wc.vy + h * limited_slope(wc.vy - wm.vy, wp.vy - wc.vy, drop);
    f.vz = wc.vz + h * limited_slope(wc.vz - wm.vz, wp.vz - wc.vz, drop);
    f.p = wc.p + h * limited_slope(wc.p - wm.p, wp.p - wc.p, drop);
    f.bx = wc.bx + h * limited_slope(wc.bx - wm.bx, wp.bx - wc.bx, drop);
    f.by = wc.by + h * limited_slope(wc.by - wm.by, wp.by - wc.by, drop);
    f.bz = wc.bz + h * limited_slope(wc.bz - wm.bz, wp.bz - wc.bz, drop);
    return f;
  };
  ul = to_cons(face(w[0], w[1], w[2], T(1), drop_m), gamma);
  ur = to_cons(face(w[1], w[2], w[3], T(-1), drop_p), gamma);
}

template <class T>
__host__ __device__ __noinline__ void muscl_face(const GridD& g, int dir, int i, int j, T gamma, int side_lo,
                                                 int side_hi, const StateView& u, const double* bxc, const double* byc,
                                                 St<T>& ul, St<T>& ur) {
#pragma clang fp contract(off)
  const int di = dir == 0 ? 1 : 0, dj = dir == 0 ? 0 : 1;
  Prim<T> w[4];
  for (int s = 0; s < 4; ++s) w[s] = to_prim(load_cell<T>(g, u, bxc, byc, i + (s - 2) * di, j + (s - 2) * dj), gamma);
  const int n_dir = dir == 0 ? g.nx : g.ny;
  const int drop_m = slope_drop((dir == 0 ? i : j) - 1, n_dir, side_lo, side_hi);
  const int drop_p = slope_drop(dir == 0 ? i : j, n_dir, side_lo, side_hi);
  muscl_pair(w, drop_m, drop_p, gamma, ul, ur);
}

template <class T, int ORDER>
__host__ __device__ __forceinline__ void mp_char_face(const GridD& g, int dir, int i, int j, T gamma, const StateView& u,
                                             const double* bxc, const double* byc, St<T>& ul, St<T>& ur,
                                             T* clip_rel = nullptr) {
  constexpr int H = ORDER == 5 ? 2 : 3;
  constexpr int UW = 2 * H + 2;
  constexpr int W = 2 * H + 1;
  const int di = dir == 0 ? 1 : 0, dj = dir == 0 ? 0 : 1;
  auto cell = [&](int q) {
    return rot(load_cell<T>(g, u, bxc, byc, i + (q - 1 - H) * di, j + (q - 1 - H) * dj), dir);
  };
  St<T> ref;
  {
    const St<T> cl = cell(H), cr = cell(H + 1);
#pragma unroll
    for (int c = 0; c < 8; ++c) set_comp(ref, c, T(0.5) * comp(cl, c) + T(0.5) * comp(cr, c));
  }
  CharBasis<T> B;
  basis_build(ref, gamma, B);
  // Characteristic variables of the union stencil, w[q] = L (U_q - ref) over
  // the 7-vector (rho, mn, mt1, mt2, E, bt1, bt2), cell by cell.
  T wch[UW][7];
#pragma unroll
  for (int q = 0; q < UW; ++q) {
    const St<T> cq = cell(q);
    const T d[7] = {cq.rho - ref.rho, cq.mx - ref.mx, cq.my - ref.my, cq.mz - ref.mz,
                    cq.en - ref.en,   cq.by - ref.by, cq.bz - ref.bz};
    basis_to_char(B, d, wch[q]);
  }
  T wl[7], wr[7];
  T shift = T(0);
  T* const sp = clip_rel ? &shift : nullptr;
#pragma unroll
  for (int k = 0; k < 7; ++k) {
    // Left state: cells 0..W-1 (centre H), right state: reversed cells 1..W.
    T sl[W], sr[W];
#pragma unroll
    for (int s = 0; s < W; ++s) {
      sl[s] = wch[s][k];
      sr[s] = wch[W - s][k];
    }
    const T fl = ORDER == 5 ? mp5_face(sl) : mp7_face(sl);
    const T fr = ORDER == 5 ? mp5_face(sr) : mp7_face(sr);
    constexpr int o = ORDER == 5 ? 0 : 1;
    wl[k] = mp_limit(fl, sl[o], sl[o + 1], sl[o + 2], sl[o + 3], sl[o + 4], sp);
    wr[k] = mp_limit(fr, sr[o], sr[o + 1], sr[o + 2], sr[o + 3], sr[o + 4], sp);
  }
  if (clip_rel) {
    T scale = T(0);
#pragma unroll
    for (int c = 0; c < 8; ++c) scale = fmax(scale, qabs(comp(ref, c)));
    *clip_rel = shift / (scale + Lim<T>::tiny);
  }
  T aL[7], aR[7];
  basis_from_char(B, wl, aL);
  basis_from_char(B, wr, aR);
  St<T> sL{ref.rho + aL[0], ref.mx + aL[1], ref.my + aL[2], ref.mz + aL[3], ref.en + aL[4], ref.bx + T(0), ref.by + aL[5], ref.bz + aL[6]};
  St<T> sR{ref.rho + aR[0], ref.mx + aR[1], ref.my + aR[2], ref.mz + aR[3], ref.en + aR[4], ref.bx + T(0), ref.by + aR[5], ref.bz + aR[6]};
  ul = rot(sL, dir);
  ur = rot(sR, dir);
}

// Path bits of a reconstructed face (the troubled-cell labels): an MP limiter
// changed a face value by more than `tol` of the state's scale, the MUSCL
// fallback or the piecewise-constant fallback (or NaN sentinel) was taken,
// the HLLD and HLL fluxes differ by more than `tol` of the flux scale.
constexpr unsigned kPathMpClip = 1u, kPathMuscl = 2u, kPathConstant = 4u, kPathHllGap = 8u;
struct LabelProbe {
  unsigned bits;
  double tol;
};

// Interface states of one face normal to `dir` at the scheme's order with the
// reference's fallback chain (mhd_reconstruct.hip:465-670): characteristic MP
// -> MUSCL when an MP state is inadmissible; after the normal field is set,
// piecewise-constant cell states, then a NaN sentinel.  `probe` (optional)
// receives the path bits above.
template <class T, int ORDER>
__host__ __device__ __forceinline__ void reconstruct_face(const GridD& g, int dir, int i, int j, T gamma, int side_lo,
                                                          int side_hi, const StateView& u, const double* bxc,
                                                          const double* byc, St<T>& ul, St<T>& ur,
                                                          LabelProbe* probe = nullptr) {
  const int di = dir == 0 ? 1 : 0, dj = dir == 0 ? 0 : 1;
  if (ORDER <= 1) {
    ul = load_cell_lo<T>(g, u, i - di, j - dj);
    ur = load_cell_lo<T>(g, u, i, j);
  } else if (ORDER == 2) {
    muscl_face<T>(g, dir, i, j, gamma, side_lo, side_hi, u, bxc, byc, ul, ur);
  } else {
    T clip = T(0);
    mp_char_face<T, ORDER>(g, dir, i, j, gamma, u, bxc, byc, ul, ur, probe ? &clip : nullptr);
    if (probe && double(clip) > probe->tol) probe->bits |= kPathMpClip;
    if (!admissible_state(ul, gamma) || !admissible_state(ur, gamma)) {
      if (probe) probe->bits |= kPathMuscl;
      muscl_face<T>(g, dir, i, j, gamma, side_lo, side_hi, u, bxc, byc, ul, ur);
    }
  }
  const T bn = T((dir == 0 ? u.c[5] : u.c[6])[idx(g, i, j)]);
  set_normal_b(ul, dir, bn);
  set_normal_b(ur, dir, bn);
  if (!admissible_state(ul, gamma) || !admissible_state(ur, gamma)) {
    if (probe) probe->bits |= kPathConstant;
    if (ORDER <= 1) {
      ul = load_cell_lo<T>(g, u, i - di, j - dj);
      ur = load_cell_lo<T>(g, u, i, j);
    } else {
      ul = load_cell<T>(g, u, bxc, byc, i - di, j - dj);
      ur = load_cell<T>(g, u, bxc, byc, i, j);
    }
    set_normal_b(ul, dir, bn);
    set_normal_b(ur, dir, bn);
  }
  if (!admissible_state(ul, gamma) || !admissible_state(ur, gamma)) {
    const T nan = Lim<T>::nan();
    ul = St<T>{nan, nan, nan, nan, nan, nan, nan, nan};
    ur = ul;
  }
}

// Cell E_z = vy Bx - vx By in the reference's operation order
// (mhd_ct.hip:414-420): velocities by division, two rounded products added
// once.  On the device the quotients come from fdiv (within an ulp of the
// division).  The corner's one-dimensional shortcuts test cell E_z values for
// exact equality: MP5/MP7 cells form theirs as the quadrature's points do
// (average_ez), so that equal states give equal values.
template <class T>
__host__ __device__ __forceinline__ T physical_ez(T rho, T mx, T my, T bx, T by) {
#pragma clang fp contract(off)
  const T vx = fdiv(mx, rho);
  const T vy = fdiv(my, rho);
  return vy * bx + vx * (-by);
}

// ---------------------------------------------------------------------------
// Transverse quadrature (include/quasar/numerics/finite_volume_quadrature.hpp:
// 12-68): a point value (or a Gauss average) from N samples with the exact
// constant-sample shortcut, which returns the centre sample when all N agree.
// The step's kernels form these values from weighted neighbour differences
// (qmhd_face.hpp); this form is what host code holds them against.
template <class T, int N>
__host__ __device__ __forceinline__ T point_from_averages(const T* s, const double* w) {
  T x[N];
#pragma unroll
  for (int t = 0; t < N; ++t) x[t] = s[t];
  bool constant = true;
#pragma unroll
  for (int t = 0; t < N; ++t) constant &= x[t] == x[N / 2];
  if (constant) return x[N / 2];
  T v = T(0);
#pragma unroll
  for (int t = 0; t < N; ++t) v += T(w[t]) * x[t];
  return v;
}

// E_z of a recovered point state when the state is admissible (finite, rho > 0,
// p > 0); false sends the cell to its cell-centre value (mhd_ct.hip:457-632).
template <class T>
__host__ __device__ __forceinline__ bool point_ez(const St<T>& st, T gamma, T& ez) {
  if (!(fin(st.rho) && st.rho > T(0) && fin(st.mx) && fin(st.my) && fin(st.mz) && fin(st.en) && fin(st.bx) &&
        fin(st.by) && fin(st.bz)))
    return false;
  if (!pressure_positive(st, gamma)) return false;
  ez = physical_ez(st.rho, st.mx, st.my, st.bx, st.by);
  return true;
}

// ---------------------------------------------------------------------------
// CT corner EMF at corner (i, j): E_z = ex + ey - e_c, with ex/ey the
// face-average -> edge interpolations of the directional Godunov EMFs
// (-F_x(By), +F_y(Bx)) and e_c the cell-average -> corner tensor interpolation
// of the cell E_z, plus the exact one-dimensional shortcuts
// (mhd_ct.hip:811-878).

// Value at an edge from the averages around it: (-3, 29, -139, 533, 533, ..) /
// 840 and (1, -8, 37, 37, ..) / 60, as the sample before the edge plus half the
// step over it and weighted differences of the other pairs' sums from the inner
// pair's.  Equal samples give that sample exactly with no comparison, and there is
// no division (12 instructions; the quotient of the weighted sum after seven
// comparisons takes 40).  Only the last addition rounds at the size of the value:
// smooth samples are within 1.7 roundings (rms 0.5), with half the inner pair's sum
// in front within 4.5 (1.05), the quotient within 3.4 (0.86).
__host__ __device__ __forceinline__ double edge_interp(int order, const double* e) {
#pragma clang fp contract(off)
  if (order >= 7) {
    const double p = e[3] + e[4], a = e[2] + e[5], b = e[1] + e[6], c = e[0] + e[7];
    const double half = 0.5 * (e[4] - e[3]);
    return e[3] + __builtin_fma(-3.0 / 840.0, c - p, __builtin_fma(29.0 / 840.0, b - p, __builtin_fma(-139.0 / 840.0, a - p, half)));
  }
  if (order >= 5) {
    const double p = e[2] + e[3], a = e[1] + e[4], b = e[0] + e[5];
    const double half = 0.5 * (e[3] - e[2]);
    return e[2] + __builtin_fma(1.0 / 60.0, b - p, __builtin_fma(-8.0 / 60.0, a - p, half));
  }
  return e[0] == e[1] ? e[0] : (e[0] + e[1]) / 2.0;
}

// A corner on a conducting side has no E_z.
__host__ __device__ __forceinline__ bool corner_conducting(const GridD& g, const Flags4& m, int i, int j) {
  return (i == 0 && (m.side[0] == 2 || m.side[0] == 3)) || (i == g.nx && m.side[1] == 2) ||
         (j == 0 && m.side[2] == 2) || (j == g.ny && m.side[3] == 2);
}

template <class T, bool INTERIOR>
__host__ __device__ __forceinline__ double corner_ez_impl(const GridD& g, int order, const Flags4& m, const FluxView<T>& fx,
                                                     const FluxView<T>& fy, const double* cell_ez,
                                                     const int* eqx, const int* eqy, int i, int j) {
  if (corner_conducting(g, m, i, j)) return 0.0;
  const int lo = order >= 7 ? -4 : order >= 5 ? -3 : -1;
  const int nt = order >= 7 ? 8 : order >= 5 ? 6 : 2;
  const int rh = order >= 7 ? 3 : order >= 5 ? 2 : 0;  // transverse recovery half-width
  // Away from the physical boundary every index maps to itself.
  auto mi = [&](int q) { return INTERIOR ? q : face_index(q, g.nx, m.side[0], m.side[1]); };
  auto mj = [&](int q) { return INTERIOR ? q : face_index(q, g.ny, m.side[2], m.side[3]); };
  double e[8];
  for (int t = 0; t < nt; ++t) e[t] = -static_cast<double>(fx.c[6][idx(g, mi(i), mj(j + lo + t))]);
  const double ex = edge_interp(order, e);
  for (int t = 0; t < nt; ++t) e[t] = static_cast<double>(fy.c[5][idx(g, mi(i + lo + t), mj(j))]);
  const double ey = edge_interp(order, e);
  double line[8];
  for (int q = 0; q < nt; ++q) {
    for (int t = 0; t < nt; ++t) e[t] = cell_ez[idx(g, mi(i + lo + t), mj(j + lo + q))];
    line[q] = edge_interp(order, e);
  }
  const double centered = edge_interp(order, line);
  // x-only data: every y-face problem in the stencil has no jump and the cell
  // E_z is constant along y; y-only symmetrically.
  // Face `t` of the interpolation stencil is mapped into the face table first;
  // its point-recovery problem then spans offsets -rh..rh about that mapped
  // face, mapped again (periodic wrap or physical clamp).
  auto no_jump_line = [&](const int* eq, int d) {
    for (int t = 0; t < nt; ++t) {
      const int fi = d == 0 ? mi(i) : mi(i + lo + t);
      const int fj = d == 0 ? mj(j + lo + t) : mj(j);
      for (int off = -rh; off <= rh; ++off) {
        const int ii = d == 0 ? mi(fi) : mi(fi + off);
        const int jj = d == 0 ? mj(fj + off) : mj(fj);
        if (ii < -g.ng || ii >= g.nx + g.ng || jj < -g.ng || jj >= g.ny + g.ng || eq[idx(g, ii, jj)] == 0)
          return false;
      }
    }
    return true;
  };
  auto constant_along = [&](int axis) {
    for (int v = 0; v < nt; ++v) {
      const double ref = axis == 0 ? cell_ez[idx(g, mi(i + lo), mj(j + lo + v))] : cell_ez[idx(g, mi(i + lo + v), mj(j + lo))];
      for (int w = 1; w < nt; ++w) {
        const double c = axis == 0 ? cell_ez[idx(g, mi(i + lo + w), mj(j + lo + v))]
                                   : cell_ez[idx(g, mi(i + lo + v), mj(j + lo + w))];
        if (c != ref) return false;
      }
    }
    return true;
  };
  const bool x_only = no_jump_line(eqy, 1) && constant_along(1);
  const bool y_only = no_jump_line(eqx, 0) && constant_along(0);
  double r;
  if (x_only && !y_only)
    r = ex;
  else if (y_only && !x_only)
    r = ey;
  else
    r = (ex + ey) - centered;
  return r;
}


template <class T>
__host__ __device__ __forceinline__ double corner_ez(const GridD& g, int order, const Flags4& m, const FluxView<T>& fx,
                                                     const FluxView<T>& fy, const double* cell_ez,
                                                     const int* eqx, const int* eqy, int i, int j) {
  const int lo = order >= 7 ? -4 : order >= 5 ? -3 : -1;
  const int nt = order >= 7 ? 8 : order >= 5 ? 6 : 2;
  const int rh = order >= 7 ? 3 : order >= 5 ? 2 : 0;
  // Every face, cell and flag index the corner touches lies in
  // [i+lo-rh, i+lo+nt-1+rh] x [j+lo-rh, j+lo+nt-1+rh].
  const bool interior = i + lo - rh >= 0 && i + lo + nt - 1 + rh < g.nx && j + lo - rh >= 0 &&
                        j + lo + nt - 1 + rh < g.ny && i > 0 && j > 0;
  return interior ? corner_ez_impl<T, true>(g, order, m, fx, fy, cell_ez, eqx, eqy, i, j)
                  : corner_ez_impl<T, false>(g, order, m, fx, fy, cell_ez, eqx, eqy, i, j);
}
}  // namespace qmhd

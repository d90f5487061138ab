// Characteristic MP5/MP7 reconstruction of one face as the reconstruction
// kernels run it.  The reference's face (reconstruct_face, mp_char_face in
// qmhd_stencil.hpp) is bound by instruction issue: 85 IEEE divisions, the
// 1024-epsilon test of L R = I term by term, limiters written with sign
// selects.  Here
//  * the basis comes from the plain closed forms where they are well
//    conditioned, where its usability needs no test (basis_quick); elsewhere
//    from the reference-ordered basis_build;
//  * projections use the pairing of the waves (fast, slow and Alfven pairs
//    share their sums and differences);
//  * the left and right limiters of a wave share their differences, and
//    minmod and median are minima and maxima;
//  * one pressure test with a margin covers both admissibility tests of a
//    state, before and after its normal field is set (setting it keeps the
//    pressure).
// A face that these cannot settle (inadmissible or borderline states, a sum
// that needs the full expansion) is left to reconstruct_face through the
// kernels' fallback list.  Products that fuse are written as fma, contraction
// off: every kernel gives the same bits.
// The closed forms stand where the wave weights are within 2^10 and the units
// (rho, sound speed) near one; 1024^2 FP64, both directions: 160 us there, 217
// where only the weights are not (B = 1e-2 at unit density and pressure), 366 at
// density 100, where the reference's test runs too.
#pragma once

#include "qmhd_face.hpp"

namespace qmhd {

// The basis in the form the projections use.
template <class T>
struct WaveBasis {
  T rho, vn, vt1, vt2, bt1, bt2, half_v2;
  T beta1, beta2;
  // Left rows: fast (q1, t, q4, s), slow, Alfven, entropy.
  T lf1, lf2, lf4, lf5, ls1, ls2, ls4, ls5, la, lb, le;
  // Right columns.
  T rf0, rs0, rf1, rs1, rf2, rs2, rf4, rs4, rf5, rs5, ra, rb;
};

template <class T>
__host__ __device__ __forceinline__ void basis_finish(T rho, T ir, T inv_sq, T sq, T gm1, T a2_ir, T rho_a2, T af, T as,
                                                      T cf, T cs, T a, T sbn, WaveBasis<T>& w) {
#pragma clang fp contract(off)
  // nf = 1 / (2 a^2); Nf/rho folds the momentum's 1/rho and the pressure row's.
  const T nf = T(0.5) * a2_ir, n = nf * ir;
  const T qf = cf * af * sbn, qs = cs * as * sbn, ea = a * sq, ef = ea * af, es = ea * as;
  const T half = T(0.70710678118654752440);
  w.rho = rho;
  w.lf1 = n * af * cf;
  w.lf2 = n * qs;
  w.lf4 = n * af * gm1;
  w.lf5 = n * es;
  w.ls1 = n * as * cs;
  w.ls2 = n * qf;
  w.ls4 = n * as * gm1;
  w.ls5 = n * ef;
  w.la = half * ir;
  w.lb = sbn * half * inv_sq;
  w.le = a2_ir * gm1;
  w.rf0 = rho * af;
  w.rs0 = rho * as;
  w.rf1 = rho * (af * cf);
  w.rs1 = rho * (as * cs);
  w.rf2 = rho * qs;
  w.rs2 = rho * qf;
  const T h = rho_a2 / gm1;
  w.rf4 = af * h;
  w.rs4 = as * h;
  w.rf5 = es;
  w.rs5 = ef;
  w.ra = rho * half;
  w.rb = sbn * half * sq;
}

// The basis about `s` (frame of the face normal) from its closed forms.  True
// when it is certainly the reference's: the pressure positive beyond rounding,
// no wave degenerate, the choice of the transverse direction unambiguous, and
// L R - I certainly inside the reference's bound of 1024 epsilon.  That
// residual is rounding: it grows with the terms that cancel in L R (1 + v^2/a^2
// + b^2/a^2), with (cf^2 + cs^2) / (cf^2 - cs^2), and, the test being absolute,
// with the ratios of the waves' units (1, rho, a).  Over 3e7 random states in
// FP64 and FP32 it stays under 5 epsilon times that product, so the bound of
// 128 on it keeps the residual under 640 epsilon.  alpha_f^2 and alpha_s^2
// under 2^-10 are left to the reference's arithmetic: there they are largely
// its rounding.
// `conditioned`: that bound and the pressure alone hold, so the reference's
// basis is usable whatever its alphas.
template <class T>
__host__ __device__ __forceinline__ bool basis_quick(const St<T>& s, T gamma, WaveBasis<T>& w, bool& conditioned) {
#pragma clang fp contract(off)
  Side<T> o;
  const bool clear = side_of(s, gamma, o);
  const T gm1 = gamma - T(1);
  const T v2 = fm(o.vx, o.vx, fm(o.vy, o.vy, o.vz * o.vz));
  const T a2 = gamma * o.p * o.ir, c2 = o.bn2 * o.ir, t2 = o.bt2 * o.ir;
  const T ca2 = c2 + t2, sum = a2 + ca2;
  T unused, ha, h, inv2;
  const T disc = hi2(fm(sum, sum, T(-4) * (a2 * c2)), Lim<T>::tiny);
  const T root = sqrt_pos(disc, unused);  // cf^2 - cs^2
  const T cf2 = T(0.5) * (sum + root);
  const T icf2 = rcp_near(cf2), iroot = rcp_near(root);
  const T cs2 = a2 * c2 * icf2;
  // (cf^2 - a^2)(cf^2 - c^2) = cf^2 t^2 and (a^2 - cs^2)(c^2 - cs^2) = cs^2 t^2:
  // the smaller weight without cancellation, the other as its complement.
  const bool acoustic = a2 > c2;
  const T num = acoustic ? cf2 : cs2, den = acoustic ? cf2 - c2 : c2 - cs2;
  const T small = num * t2 * iroot * rcp_near(den), large = T(1) - small;
  const T af2 = acoustic ? large : small, as2 = acoustic ? small : large;
  constexpr T geps = T(64) * Lim<T>::eps;
  const T fs2 = hi2(a2, ca2);
  const bool none = t2 <= (T(0.25) * geps * geps) * fs2, some = t2 >= (T(4) * geps * geps) * fs2;
  const T a = sqrt_pos(a2, ha), cf = sqrt_pos(cf2, unused);
  const T ia = T(2) * ha;
  // At most 1 and at least (|v| + |b|) / a, up to its own rounding.
  const T mix = lo2(T(1), ia * (qabs(o.vx) + qabs(o.vy) + qabs(o.vz) + T(2) * cf));
  const T units = hi2(hi2(hi2(s.rho, o.ir), hi2(a, ia)), mix * hi2(s.rho * ia, a * o.ir));
  conditioned = clear && sum * (a2 + v2 + ca2) * units <= T(128) * (root * a2);
  const bool quick = conditioned && (none || some) && small >= T(0x1p-10) && large >= T(0x1p-10);
  const T cs = sqrt_pos(hi2(cs2, Lim<T>::tiny), unused);
  const T af = sqrt_pos(hi2(af2, Lim<T>::tiny), unused);
  const T as = sqrt_pos(hi2(as2, Lim<T>::tiny), unused);
  const T sq = sqrt_pos(s.rho, h);
  (void)sqrt_pos(hi2(o.bt2, Lim<T>::tiny), inv2);
  const T half = T(0.70710678118654752440), ibt = T(2) * inv2;
  w.beta1 = none ? half : s.by * ibt;
  w.beta2 = none ? half : s.bz * ibt;
  w.vn = o.vx;
  w.vt1 = o.vy;
  w.vt2 = o.vz;
  w.bt1 = s.by;
  w.bt2 = s.bz;
  w.half_v2 = T(0.5) * v2;
  basis_finish(s.rho, o.ir, T(2) * h, sq, gm1, ia * ia, gamma * o.p, af, as, cf, cs, a, s.bx >= T(0) ? T(1) : T(-1), w);
  return quick;
}

// The basis in the reference's arithmetic and, unless it is known to be
// usable, its decision; false where it is not usable.
template <class T>
__host__ __device__ __forceinline__ bool basis_exact(const St<T>& s, T gamma, bool conditioned, WaveBasis<T>& w) {
  CharBasis<T> B;
  basis_scalars(s, gamma, B);
  // a from the larger of the two A = a alpha sqrt(rho).
  const bool fast = B.alpha_f >= B.alpha_s;
  const T a = (fast ? B.Af : B.As) / ((fast ? B.alpha_f : B.alpha_s) * B.sqrt_rho);
  w.beta1 = B.beta1;
  w.beta2 = B.beta2;
  w.vn = B.vn;
  w.vt1 = B.vt1;
  w.vt2 = B.vt2;
  w.bt1 = B.bt1;
  w.bt2 = B.bt2;
  w.half_v2 = B.half_v2;
  basis_finish(B.rho, B.inv_rho, T(1) / B.sqrt_rho, B.sqrt_rho, B.gm1, B.inv_a2, B.rho_a2, B.alpha_f, B.alpha_s, B.cf,
               B.cs, a, B.sbn, w);
  return conditioned || basis_usable(B);
}

// Characteristic variables of a conserved difference (rho, mn, mt1, mt2, E,
// bt1, bt2): the fast and slow waves -fast, +fast, -slow, +slow ...
template <class T>
__host__ __device__ __forceinline__ void to_fast_slow(const WaveBasis<T>& B, const T d[7], T w[4]) {
#pragma clang fp contract(off)
  const T q1 = fm(-B.vn, d[0], d[1]), q2 = fm(-B.vt1, d[0], d[2]), q3 = fm(-B.vt2, d[0], d[3]);
  const T q4 = fm(-B.bt2, d[6],
                  fm(-B.bt1, d[5], fm(-B.vt2, d[3], fm(-B.vt1, d[2], fm(-B.vn, d[1], fm(B.half_v2, d[0], d[4]))))));
  const T t = fm(B.beta1, q2, B.beta2 * q3), s = fm(B.beta1, d[5], B.beta2 * d[6]);
  const T af = fm(B.lf4, q4, B.lf5 * s), bf = fm(B.lf1, q1, -(B.lf2 * t));
  const T as = fm(B.ls4, q4, -(B.ls5 * s)), bs = fm(B.ls1, q1, B.ls2 * t);
  w[0] = af - bf;
  w[1] = af + bf;
  w[2] = as - bs;
  w[3] = as + bs;
}

// ... and -Alfven, +Alfven, entropy.
template <class T>
__host__ __device__ __forceinline__ void to_alfven_entropy(const WaveBasis<T>& B, const T d[7], T w[3]) {
#pragma clang fp contract(off)
  const T q2 = fm(-B.vt1, d[0], d[2]), q3 = fm(-B.vt2, d[0], d[3]);
  const T q4 = fm(-B.bt2, d[6],
                  fm(-B.bt1, d[5], fm(-B.vt2, d[3], fm(-B.vt1, d[2], fm(-B.vn, d[1], fm(B.half_v2, d[0], d[4]))))));
  const T aa = B.la * fm(B.beta1, q3, -(B.beta2 * q2)), ba = B.lb * fm(B.beta1, d[6], -(B.beta2 * d[5]));
  w[0] = aa + ba;
  w[1] = aa - ba;
  w[2] = fm(-B.le, q4, d[0]);
}

// Conserved difference of the waves in the order of the two above.
template <class T>
__host__ __device__ __forceinline__ void from_waves(const WaveBasis<T>& B, const T w[7], T out[7]) {
#pragma clang fp contract(off)
  const T pf = w[0] + w[1], mf = w[1] - w[0], ps = w[2] + w[3], ms = w[3] - w[2], pa = w[4] + w[5], ma = w[4] - w[5];
  const T r = fm(B.rf0, pf, fm(B.rs0, ps, w[6]));
  const T m1 = fm(B.rf1, mf, B.rs1 * ms), tt = fm(B.rs2, ms, -(B.rf2 * mf)), tq = B.ra * pa;
  const T m2 = fm(B.beta1, tt, -(B.beta2 * tq)), m3 = fm(B.beta2, tt, B.beta1 * tq);
  const T bb = fm(B.rf5, pf, -(B.rs5 * ps)), bq = B.rb * ma;
  const T b1 = fm(B.beta1, bb, -(B.beta2 * bq)), b2 = fm(B.beta2, bb, B.beta1 * bq);
  out[0] = r;
  out[1] = fm(B.vn, r, m1);
  out[2] = fm(B.vt1, r, m2);
  out[3] = fm(B.vt2, r, m3);
  const T e = fm(B.rf4, pf, B.rs4 * ps);
  out[4] = fm(B.half_v2, r, fm(B.vn, m1, fm(B.vt1, m2, fm(B.vt2, m3, fm(B.bt1, b1, fm(B.bt2, b2, e))))));
  out[5] = b1;
  out[6] = b2;
}

// The argument of least magnitude where all have one sign, else zero.
template <class T>
__host__ __device__ __forceinline__ T minmod_mm(T a, T b) {
  return hi2(lo2(a, b), T(0)) + lo2(hi2(a, b), T(0));
}
// minmod(4a - b, 4b - a, a, b).
template <class T>
__host__ __device__ __forceinline__ T minmod_m4(T a, T b) {
#pragma clang fp contract(off)
  const T p = fm(T(4), a, -b), q = fm(T(4), b, -a);
  const T lo = lo2(lo2(p, q), lo2(a, b)), hi = hi2(hi2(p, q), hi2(a, b));
  return hi2(lo, T(0)) + lo2(hi, T(0));
}

// Whether the unlimited value vl of a cell v0 with differences em = v0 - vm1
// and ep = vp1 - v0 stands: it lies between v0 and v_mp, or within 1e-10 of
// the stencil's variation of doing so.  (A product at or below zero is the
// first rule; the bound of the second is never negative.)
template <class T>
__host__ __device__ __forceinline__ bool mp_keeps(T vl, T v0, T em, T ep) {
#pragma clang fp contract(off)
  const T vmp = v0 + minmod_mm(ep, T(4) * em);
  const T a = vl - v0, b = vl - vmp;
  const T v = hi2(hi2(qabs(em), qabs(ep)), hi2(qabs(a), qabs(b)));
  return a * b <= T(1e-10) * (v * v);
}

// Both face values of one wave: v[0 .. 2H+1] its union stencil, the left value
// from cell H, the right one from cell H + 1 (mp_limit's operations; the
// second differences, the median bound and the pair's extrema are shared).  The
// unlimited value, a sum over its stencil, is not finite where a cell's is not;
// it stands then, since the median's minima and maxima would drop a NaN.
template <class T, int ORDER>
__host__ __device__ __forceinline__ void mp_pair(const T* v, T& left, T& right) {
#pragma clang fp contract(off)
  constexpr int H = ORDER == 5 ? 2 : 3;
  T vl, vr;
  if constexpr (ORDER == 5) {
    constexpr T c[5] = {T(2.0 / 60), T(-13.0 / 60), T(47.0 / 60), T(27.0 / 60), T(-3.0 / 60)};
    vl = fm(c[4], v[4], fm(c[3], v[3], fm(c[2], v[2], fm(c[1], v[1], c[0] * v[0]))));
    vr = fm(c[4], v[1], fm(c[3], v[2], fm(c[2], v[3], fm(c[1], v[4], c[0] * v[5]))));
  } else {
    constexpr T c[7] = {T(-3.0 / 420),  T(25.0 / 420),  T(-101.0 / 420), T(319.0 / 420),
                        T(214.0 / 420), T(-38.0 / 420), T(4.0 / 420)};
    vl = fm(c[6], v[6],
            fm(c[5], v[5], fm(c[4], v[4], fm(c[3], v[3], fm(c[2], v[2], fm(c[1], v[1], c[0] * v[0]))))));
    vr = fm(c[6], v[1],
            fm(c[5], v[2], fm(c[4], v[3], fm(c[3], v[4], fm(c[2], v[5], fm(c[1], v[6], c[0] * v[7]))))));
  }
  const T* m = v + (H - 2);  // m[0..5]: the six cells the limiters read
  const T e0 = m[1] - m[0], e1 = m[2] - m[1], e2 = m[3] - m[2], e3 = m[4] - m[3], e4 = m[5] - m[4];
  const bool kl = mp_keeps(vl, m[2], e1, e2), kr = mp_keeps(vr, m[3], -e3, -e2);
  left = vl;
  right = vr;
  if (kl && kr) return;
  const T d1 = e1 - e0, d2 = e2 - e1, d3 = e3 - e2, d4 = e4 - e3;
  const T md = fm(T(-0.5), minmod_m4(d2, d3), T(0.5) * (m[2] + m[3]));
  const T alo = lo2(lo2(m[2], m[3]), md), ahi = hi2(hi2(m[2], m[3]), md);
  {
    const T ul = fm(T(4), e1, m[2]), lc = fm(T(4.0 / 3.0), minmod_m4(d2, d1), fm(T(0.5), e1, m[2]));
    const T lo = hi2(alo, lo2(lo2(m[2], ul), lc)), hi = lo2(ahi, hi2(hi2(m[2], ul), lc));
    const T med = hi2(lo2(lo, hi), lo2(hi2(lo, hi), vl));
    left = kl || !fin(vl) ? vl : med;
  }
  {
    const T ul = fm(T(-4), e3, m[3]), lc = fm(T(4.0 / 3.0), minmod_m4(d3, d4), fm(T(-0.5), e3, m[3]));
    const T lo = hi2(alo, lo2(lo2(m[3], ul), lc)), hi = lo2(ahi, hi2(hi2(m[3], ul), lc));
    const T med = hi2(lo2(lo, hi), lo2(hi2(lo, hi), vr));
    right = kr || !fin(vr) ? vr : med;
  }
}

// a + b + c rounded once, true when that is certain.  Terms of neighbouring
// exponents: the two rounding errors nearly always add without a third, and then
// t + e rounds the exact sum (on the frequent ties too).  Where b and c are far
// below a (a normal field that is nearly zero) a third error is the rule; it
// moves the result only from within its own size of a midpoint.  (Left to the
// fallback list, such faces took a rotor's reconstruction at 2048^2 from 0.7 to
// 5.8 ms per launch.)
__host__ __device__ __forceinline__ bool sum_of_three(double a, double b, double c, double& sum) {
#pragma clang fp contract(off)
  double t, e1, e2, e, rest, off;
  two_sum(a, b, t, e1);
  two_sum(t, c, t, e2);
  two_sum(e1, e2, e, rest);
  two_sum(t, e, sum, off);
  const double most = fm(2.0, qabs(rest), fm(0x1p-40, qabs(off), qabs(off)));
  return rest == 0.0 || (sum + most == sum && sum - most == sum);
}

// set_normal_b of an admissible face state (frame of the normal); false when
// the state is not admissible beyond rounding before and after, or (FP64) the
// energy's three-term sum is not certain.
template <class T>
__host__ __device__ __forceinline__ bool settle_state(St<T>& s, T v) {
#pragma clang fp contract(off)
  const T ir = rcp_near(s.rho);
  const T ke2 = fm(s.mx, s.mx, fm(s.my, s.my, s.mz * s.mz)) * ir;
  const T b2 = fm(s.bx, s.bx, fm(s.by, s.by, s.bz * s.bz));
  const T q = fm(T(-0.5), b2, fm(T(-0.5), ke2, s.en));
  const T mag = qabs(s.en) + fm(T(0.5), ke2, fm(v, v, b2));
  bool ok = s.rho > T(0) && q > T(64) * Lim<T>::eps * mag;
  const T add = v * (T(0.5) * v), sub = s.bx * (T(0.5) * s.bx);
  if constexpr (sizeof(T) == 4) {
    s.en = (s.en + add) - sub;
  } else {
    const bool sure = sum_of_three(s.en, add, -sub, s.en);
    ok = ok && sure;
  }
  s.bx = v;
  return ok;
}

// set_normal_b to the bit (frame of the normal); false when the state is not
// certainly admissible after it, or (FP64) the energy's three-term sum is not
// certain.
template <class T>
__host__ __device__ __forceinline__ bool settle_exact(St<T>& s, T v, T gamma) {
#pragma clang fp contract(off)
  bool ok = true;
  const T add = v * (T(0.5) * v), sub = s.bx * (T(0.5) * s.bx);
  if constexpr (sizeof(T) == 4) {
    s.en = (s.en + add) - sub;
  } else {
    ok = sum_of_three(s.en, add, -sub, s.en);
  }
  s.bx = v;
  Side<T> o;
  return ok & side_of(s, gamma, o);
}

// Interface states of a face in the frame of its normal; cell(c, q) is
// component c (rho, mn, mt1, mt2, E, bn, bt1, bt2) of cell q of its union
// stencil, bn its own normal field.  False leaves the face to
// reconstruct_face.
template <class T, int ORDER, class Cell>
__host__ __device__ __forceinline__ bool mp_face(Cell cell, T bn, T gamma, St<T>& ul, St<T>& ur) {
#pragma clang fp contract(off)
  constexpr int H = ORDER == 5 ? 2 : 3;
  constexpr int UW = 2 * H + 2;
  St<T> ref;
#pragma unroll
  for (int c = 0; c < 8; ++c) set_comp(ref, c, fm(T(0.5), cell(c, H), T(0.5) * cell(c, H + 1)));
  WaveBasis<T> B;
  bool conditioned, usable = true;
  // The hint keeps the exact basis out of the closed forms' way: 2048^2 FP64, both
  // directions, 671 us without it, 637 with it (656 with the energy sum as it is).
  if (__builtin_expect(!basis_quick(ref, gamma, B, conditioned), 0)) usable = basis_exact(ref, gamma, conditioned, B);
  auto difference = [&](int q, T d[7]) {
    d[0] = cell(0, q) - ref.rho;
    d[1] = cell(1, q) - ref.mx;
    d[2] = cell(2, q) - ref.my;
    d[3] = cell(3, q) - ref.mz;
    d[4] = cell(4, q) - ref.en;
    d[5] = cell(6, q) - ref.by;
    d[6] = cell(7, q) - ref.bz;
  };
  T wl[7], wr[7];
  auto limit = [&](const auto& w, int first, int count) {
#pragma unroll
    for (int n = 0; n < count; ++n) {
      T v[UW];
#pragma unroll
      for (int q = 0; q < UW; ++q) v[q] = w[q][n];
      mp_pair<T, ORDER>(v, wl[first + n], wr[first + n]);
    }
  };
  T a[7], b[7];
  // (Far from unit scales whole waves of faces have no usable basis: 1024^2
  // FP64 at density 1e4, both directions, 419 us with their waves, 352 without.)
  if (any_lane(usable)) {
    // Four waves, then three: the stencil's waves of one group are live at a
    // time (all seven beside the basis are 278 registers in FP64, past two waves
    // per SIMD).
    {
      T w[UW][4];
#pragma unroll
      for (int q = 0; q < UW; ++q) {
        T d[7];
        difference(q, d);
        to_fast_slow(B, d, w[q]);
      }
      limit(w, 0, 4);
    }
    schedule_fence();
    {
      T w[UW][3];
#pragma unroll
      for (int q = 0; q < UW; ++q) {
        T d[7];
        difference(q, d);
        to_alfven_entropy(B, d, w[q]);
      }
      limit(w, 4, 3);
    }
    from_waves(B, wl, a);
    from_waves(B, wr, b);
  }
  if (!usable) {
    // Component-wise limiting of the differences themselves.
#pragma unroll
    for (int n = 0; n < 7; ++n) {
      const int c = n < 5 ? n : n + 1;
      T v[UW];
#pragma unroll
      for (int q = 0; q < UW; ++q) v[q] = cell(c, q) - comp(ref, c);
      mp_pair<T, ORDER>(v, a[n], b[n]);
    }
  }
  ul = St<T>{ref.rho + a[0], ref.mx + a[1], ref.my + a[2], ref.mz + a[3], ref.en + a[4], ref.bx, ref.by + a[5], ref.bz + a[6]};
  ur = St<T>{ref.rho + b[0], ref.mx + b[1], ref.my + b[2], ref.mz + b[3], ref.en + b[4], ref.bx, ref.by + b[5], ref.bz + b[6]};
  const bool okl = settle_state(ul, bn), okr = settle_state(ur, bn);
  return okl && okr;
}

// Cell planes in the frame of the face normal.
struct NormalPlanes {
  const double* c[8];
};
__host__ __device__ __forceinline__ NormalPlanes normal_planes(int dir, const StateView& u, const double* bxc,
                                                               const double* byc) {
  const bool x = dir == 0;
  return NormalPlanes{{u.c[0], x ? u.c[1] : u.c[2], x ? u.c[2] : u.c[1], u.c[3], u.c[4], x ? bxc : byc, x ? byc : bxc,
                       u.c[7]}};
}

}  // namespace qmhd

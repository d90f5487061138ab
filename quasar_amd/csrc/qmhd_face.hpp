// Face solver of the MP5/MP7 flux kernels: point states at the transverse
// Gauss nodes, their admissibility, the face signal speed, the HLLD flux and
// its Gauss average, one node at a time in a rolled loop.
//
// What bounds a face is its FP64 instruction count (two waves per SIMD keep
// the VALU about 70 % busy), so the loop is written for few instructions:
//  * a point value is its face average plus weighted neighbour differences
//    (the recovery rows sum to one), so equal samples give that sample exactly
//    with no comparison, and the differences are formed once per block, not
//    per node;
//  * the Gauss average is a running mean, so equal fluxes give that flux
//    exactly with no comparison;
//  * a state's 1/rho, velocity and pressure are formed once and serve its
//    admissibility, its signal speed and the Riemann fan;
//  * a state whose pressure is clear of rounding needs no finiteness test: a
//    non-finite component fails that comparison;
//  * one solver in the code, not one per node: the four unrolled solves were
//    10.7k instructions, more than the instruction cache of a CU pair holds.
// Every product that may fuse is written as fma and contraction is off, so
// each kernel that includes this gives the same bits: the plain flux, the
// learned form's listed faces and the queue's forms.
#pragma once

#include "qmhd_stencil.hpp"

namespace qmhd {

__host__ __device__ __forceinline__ double fm(double a, double b, double c) { return __builtin_fma(a, b, c); }
__host__ __device__ __forceinline__ float fm(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

__host__ __device__ __forceinline__ double lo2(double a, double b) { return __builtin_fmin(a, b); }
__host__ __device__ __forceinline__ double hi2(double a, double b) { return __builtin_fmax(a, b); }
__host__ __device__ __forceinline__ float lo2(float a, float b) { return __builtin_fminf(a, b); }
__host__ __device__ __forceinline__ float hi2(float a, float b) { return __builtin_fmaxf(a, b); }

// sqrt(x) and 1 / (2 sqrt(x)) of a positive normal x (Goldschmidt from the
// hardware's reciprocal square root).  One Goldschmidt step leaves the inverse
// 19 epsilon off in FP64, so where it is asked for it takes one more against
// the rounded root: within 2 epsilon, as a quotient of the rounded root is (the
// wave basis and the Alfven speeds divide by roots).  2048^2 FP64, both
// directions: flux 997 -> 1012 us for it, reconstruction 643 -> 651.
__host__ __device__ __forceinline__ double sqrt_pos(double x, double& half_inv) {
#if defined(__HIP_DEVICE_COMPILE__)
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  const double r = __builtin_fma(-g, h, 0.5);
  g = __builtin_fma(g, r, g);
  h = __builtin_fma(h, r, h);
  g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
  half_inv = __builtin_fma(h + h, __builtin_fma(-g, h, 0.5), h);
  return g;
#else
  const double g = __builtin_sqrt(x);
  half_inv = 0.5 / g;
  return g;
#endif
}
__host__ __device__ __forceinline__ float sqrt_pos(float x, float& half_inv) {
#if defined(__HIP_DEVICE_COMPILE__)
  const float y = __builtin_amdgcn_rsqf(x);
  const float h = 0.5f * y;
  float g = x * y;
  g = __builtin_fmaf(__builtin_fmaf(-g, g, x), h, g);
  half_inv = __builtin_fmaf(h + h, __builtin_fmaf(-g, h, 0.5f), h);
  return g;
#else
  const float g = __builtin_sqrtf(x);
  half_inv = 0.5f / g;
  return g;
#endif
}

// 1/x as frcp; in FP32 one Newton step on v_rcp_f32 (the face solver's
// divisors are densities and wave-speed differences, far from FP32's ends).
__host__ __device__ __forceinline__ double rcp_near(double x) { return frcp(x); }
__host__ __device__ __forceinline__ float rcp_near(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
  const float r = __builtin_amdgcn_rcpf(x);
  return __builtin_fmaf(__builtin_fmaf(-x, r, 1.0f), r, r);
#else
  return 1.0f / x;
#endif
}

// Nothing moves across it in the device schedule: bounds what is live at once.
__host__ __device__ __forceinline__ void schedule_fence() {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_sched_barrier(0);
#endif
}

// What the solver needs of one state, in the frame of the face normal.
template <class T>
struct Side {
  T ir, vx, vy, vz, p, bt2, bn2, cf;
};

// Fills `o` and returns whether the state is certainly admissible (rho > 0,
// internal energy positive beyond rounding; a NaN or infinity anywhere fails).
template <class T>
__host__ __device__ __forceinline__ bool side_of(const St<T>& s, T gamma, Side<T>& o) {
#pragma clang fp contract(off)
  o.ir = rcp_near(s.rho);
  o.vx = s.mx * o.ir;
  o.vy = s.my * o.ir;
  o.vz = s.mz * o.ir;
  const T ke2 = fm(s.mx, o.vx, fm(s.my, o.vy, s.mz * o.vz));
  o.bt2 = fm(s.by, s.by, s.bz * s.bz);
  o.bn2 = s.bx * s.bx;
  const T b2 = o.bn2 + o.bt2;
  const T q = fm(T(-0.5), b2, fm(T(-0.5), ke2, s.en));
  o.p = (gamma - T(1)) * q;
  return s.rho > T(0) && q > T(32) * Lim<T>::eps * fm(T(0.5), ke2 + b2, qabs(s.en));
}

// Fast magnetosonic speed along the normal.  The discriminant's floor (its
// square root is below any sum's rounding) keeps sqrt_pos off zero.
template <class T>
__host__ __device__ __forceinline__ T fast_of(const Side<T>& s, T bn2, T gamma) {
#pragma clang fp contract(off)
  const T a2 = gamma * hi2(s.p, T(0)) * s.ir, c2 = bn2 * s.ir;
  const T sum = fm(s.bt2, s.ir, a2 + c2);
  T h;
  const T disc = hi2(fm(sum, sum, T(-4) * (a2 * c2)), Lim<T>::tiny);
  return sqrt_pos(T(0.5) * (sum + sqrt_pos(disc, h)), h);
}

// Signal speed of a face from its two sides (order <= 1 takes the larger
// |v| + c); infinite when a side is not admissible.
template <class T>
__host__ __device__ __forceinline__ T rate_of(const Side<T>& l, T cl, const Side<T>& r, T cr, int order) {
#pragma clang fp contract(off)
  const T ul = qabs(l.vx), ur = qabs(r.vx);
  const T v = order <= 1 ? hi2(ul + cl, ur + cr) : hi2(ul, ur) + hi2(cl, cr);
  return l.p > T(0) && r.p > T(0) && fin(v) ? v : Lim<T>::inf();
}

// HLLD (Miyoshi & Kusano 2005) in the face frame with both sides prepared and
// their fast speeds for the averaged normal field bn, falling back to HLL with
// the same Davis speeds (include/quasar/numerics/hlld_core.hpp:157-290).  The
// fan is computed without early exits: each guard clears `ok`, and a value
// that stopped being finite shows in the flux.
template <class T>
__host__ __device__ __forceinline__ St<T> hlld_sides(const St<T>& L, const St<T>& R, const Side<T>& l, const Side<T>& r,
                                                     T bn) {
#pragma clang fp contract(off)
  const T bn2 = bn * bn;
  // Copies: a select between members of two aggregates would index memory.
  const T vxl = l.vx, vyl = l.vy, vzl = l.vz, vxr = r.vx, vyr = r.vy, vzr = r.vz;
  const T rhol = L.rho, mxl = L.mx, myl = L.my, mzl = L.mz, byl = L.by, bzl = L.bz;
  const T rhor = R.rho, mxr = R.mx, myr = R.my, mzr = R.mz, byr = R.by, bzr = R.bz;
  const T enL = fm(T(0.5), bn2 - l.bn2, L.en), enR = fm(T(0.5), bn2 - r.bn2, R.en);
  const T ptL = fm(T(0.5), bn2 + l.bt2, l.p), ptR = fm(T(0.5), bn2 + r.bt2, r.p);
  const T cf = hi2(l.cf, r.cf);
  const T sl = lo2(l.vx, r.vx) - cf, sr = hi2(l.vx, r.vx) + cf;
  const bool equal = L.rho == R.rho && L.mx == R.mx && L.my == R.my && L.mz == R.mz && L.en == R.en && L.bx == R.bx &&
                     L.by == R.by && L.bz == R.bz;
  // Equal states, like a supersonic face, take the physical flux of one side.
  const bool upwind = equal || sl >= T(0) || sr <= T(0);
  bool left = equal || sl >= T(0), inner = false, negligible = false, ok = true;
  T s = T(0), sa = T(0);
  // Star state of the chosen side minus that side's state, and double star
  // minus star.
  T d0 = T(0), d1 = T(0), d2 = T(0), d3 = T(0), d4 = T(0), d6 = T(0), d7 = T(0);
  if (!upwind) {
    const T tol = T(64) * Lim<T>::eps;
    const T smvL = sl - l.vx, smvR = sr - r.vx;
    const T aL = smvL * L.rho, aR = smvR * R.rho;
    const T dM = aR - aL;
    ok = ok && qabs(dM) > tol * (qabs(aR) + qabs(aL));
    const T iM = rcp_near(dM);
    const T sm = (fm(aR, r.vx, -(aL * l.vx)) + (ptL - ptR)) * iM;
    const T pts = fm(aL * aR, r.vx - l.vx, fm(aR, ptL, -(aL * ptR))) * iM;
    const T dL = sl - sm, dR = sr - sm;
    const T wave = tol * (qabs(sl) + qabs(sr) + qabs(sm));
    ok = ok && qabs(dL) > wave && qabs(dR) > wave;
    const T idL = rcp_near(dL), idR = rcp_near(dR);
    const T rhoL = aL * idL, rhoR = aR * idR;
    ok = ok && rhoL > T(0) && rhoR > T(0);
    T vyL, vzL, byL, bzL, vbL, eL, vyR, vzR, byR, bzR, vbR, eR;
    const T smb = sm * bn;
    {
      const T q = aL * dL, den = q - bn2;
      ok = ok && qabs(den) > tol * (qabs(q) + bn2);
      const T id = rcp_near(den), fac = bn * (sm - l.vx) * id, bc = fm(aL, smvL, -bn2) * id;
      vyL = fm(-L.by, fac, l.vy);
      vzL = fm(-L.bz, fac, l.vz);
      byL = L.by * bc;
      bzL = L.bz * bc;
      vbL = fm(vyL, byL, fm(vzL, bzL, smb));
      const T vb = fm(l.vy, L.by, fm(l.vz, L.bz, l.vx * bn));
      eL = fm(smvL, enL, fm(-ptL, l.vx, fm(pts, sm, bn * (vb - vbL)))) * idL;
    }
    {
      const T q = aR * dR, den = q - bn2;
      ok = ok && qabs(den) > tol * (qabs(q) + bn2);
      const T id = rcp_near(den), fac = bn * (sm - r.vx) * id, bc = fm(aR, smvR, -bn2) * id;
      vyR = fm(-R.by, fac, r.vy);
      vzR = fm(-R.bz, fac, r.vz);
      byR = R.by * bc;
      bzR = R.bz * bc;
      vbR = fm(vyR, byR, fm(vzR, bzR, smb));
      const T vb = fm(r.vy, R.by, fm(r.vz, R.bz, r.vx * bn));
      eR = fm(smvR, enR, fm(-ptR, r.vx, fm(pts, sm, bn * (vb - vbR)))) * idR;
    }
    T hL, hR;
    const T sqL = sqrt_pos(rhoL, hL), sqR = sqrt_pos(rhoR, hR);
    const T abn2 = T(2) * qabs(bn);
    const T saL = fm(-abn2, hL, sm), saR = fm(abn2, hR, sm);
    negligible = bn2 <= tol * (qabs(pts) + qabs(ptL) + qabs(ptR) + Lim<T>::tiny);
    if (negligible) {
      left = T(0) <= sm;
    } else if (T(0) <= saL || !(T(0) <= saR)) {
      left = T(0) <= saL;  // outer regions: F + S (U* - U)
    } else {
      inner = true;
      left = T(0) <= sm;
    }
    const T rhos = left ? rhoL : rhoR, es = left ? eL : eR;
    const T vys = left ? vyL : vyR, vzs = left ? vzL : vzR, bys = left ? byL : byR, bzs = left ? bzL : bzR;
    s = left ? sl : sr;
    const T u1 = rhos * sm, u2 = rhos * vys, u3 = rhos * vzs;
    d0 = s * (rhos - (left ? rhol : rhor));
    d1 = s * (u1 - (left ? mxl : mxr));
    d2 = s * (u2 - (left ? myl : myr));
    d3 = s * (u3 - (left ? mzl : mzr));
    d4 = s * (es - (left ? enL : enR));
    d6 = s * (bys - (left ? byl : byr));
    d7 = s * (bzs - (left ? bzl : bzr));
    if (inner) {
      const T isum = rcp_near(sqL + sqR);
      const T sg = bn >= T(0) ? T(1) : T(-1);
      const T qq = sqL * sqR * sg;
      const T vyd = fm(sqL, vyL, fm(sqR, vyR, (byR - byL) * sg)) * isum;
      const T vzd = fm(sqL, vzL, fm(sqR, vzR, (bzR - bzL) * sg)) * isum;
      const T byd = fm(sqL, byR, fm(sqR, byL, qq * (vyR - vyL))) * isum;
      const T bzd = fm(sqL, bzR, fm(sqR, bzL, qq * (vzR - vzL))) * isum;
      const T vbd = fm(vyd, byd, fm(vzd, bzd, smb));
      sa = left ? saL : saR;
      const T sq = left ? -(sqL * sg) : sqR * sg;
      d2 = fm(sa, rhos * vyd - u2, d2);
      d3 = fm(sa, rhos * vzd - u3, d3);
      d4 = fm(sa, sq * ((left ? vbL : vbR) - vbd), d4);
      d6 = fm(sa, byd - bys, d6);
      d7 = fm(sa, bzd - bzs, d7);
    }
  }
  // Physical flux of the chosen side (normal field bn) plus the fan's terms.
  const T ux = left ? vxl : vxr, uy = left ? vyl : vyr, uz = left ? vzl : vzr;
  const T mx = left ? mxl : mxr, by = left ? byl : byr, bz = left ? bzl : bzr;
  const T pt = left ? ptL : ptR, en = left ? enL : enR;
  St<T> f;
  f.rho = mx + d0;
  f.mx = fm(mx, ux, (pt - bn2) + d1);
  f.my = fm(mx, uy, fm(-bn, by, d2));
  f.mz = fm(mx, uz, fm(-bn, bz, d3));
  f.en = fm(ux, (en + pt) - bn2, fm(-bn, fm(uy, by, uz * bz), d4));
  f.bx = T(0);
  f.by = fm(by, ux, fm(-bn, uy, d6));
  f.bz = fm(bz, ux, fm(-bn, uz, d7));
  ok = ok && fin(f.rho) && fin(f.en);
  if (!negligible) ok = ok && fin(f.mx) && fin(f.my) && fin(f.mz) && fin(f.by) && fin(f.bz);
  if (!ok) {
    St<T> a = L, b = R;
    a.en = enL;
    b.en = enR;
    a.bx = b.bx = bn;
    // The speeds' minima and maxima drop a NaN.  The reference's choices keep
    // the right state's, and its speeds then lead to the left state's flux.
    const T right = r.vx + r.cf;
    if (right != right)
      f = phys_flux_of(a, l.ir, l.p);
    else if (!upwind)
      f = hll_combine(a, b, phys_flux_of(a, l.ir, l.p), phys_flux_of(b, r.ir, r.p), sl, sr);
  }
  return f;
}

// HLL with Davis speeds of two states with one normal field, both sides
// prepared, cf the larger of their fast speeds: F_L + w (F_R - F_L) + d (R - L),
// so equal states give their own flux exactly.
template <class T>
__host__ __device__ __forceinline__ St<T> hll_sides(const St<T>& L, const St<T>& R, const Side<T>& l, const Side<T>& r,
                                                    T cf) {
#pragma clang fp contract(off)
  const T sl = lo2(l.vx, r.vx) - cf, sr = hi2(l.vx, r.vx) + cf, width = sr - sl;
  const bool fan = sl < T(0) && sr > T(0) && fin(width);
  const T inv = rcp_near(fan ? width : T(1));
  const T w = fan ? -sl * inv : !(sl >= T(0)) && sr <= T(0) ? T(1) : T(0), d = fan ? sl * sr * inv : T(0);
  auto mix = [&](T a, T b, T x, T y) { return fm(d, y - x, fm(w, b - a, a)); };
  const T bn = L.bx, ptl = fm(T(0.5), l.bt2, l.p), ptr = fm(T(0.5), r.bt2, r.p), hb = T(0.5) * l.bn2;
  St<T> f;
  f.rho = mix(L.mx, R.mx, L.rho, R.rho);
  f.mx = mix(fm(L.mx, l.vx, ptl - hb), fm(R.mx, r.vx, ptr - hb), L.mx, R.mx);
  f.my = mix(fm(L.mx, l.vy, -(bn * L.by)), fm(R.mx, r.vy, -(bn * R.by)), L.my, R.my);
  f.mz = mix(fm(L.mx, l.vz, -(bn * L.bz)), fm(R.mx, r.vz, -(bn * R.bz)), L.mz, R.mz);
  f.en = mix(fm(l.vx, (L.en - hb) + ptl, -(bn * fm(l.vy, L.by, l.vz * L.bz))),
             fm(r.vx, (R.en - hb) + ptr, -(bn * fm(r.vy, R.by, r.vz * R.bz))), L.en, R.en);
  f.bx = T(0);
  f.by = mix(fm(L.by, l.vx, -(bn * l.vy)), fm(R.by, r.vx, -(bn * r.vy)), L.by, R.by);
  f.bz = mix(fm(L.bz, l.vx, -(bn * l.vz)), fm(R.bz, r.vx, -(bn * r.vz)), L.bz, R.bz);
  return f;
}

// The unlimited fifth-order face values of one component from the six cells
// about the face (the MP5 interpolant's weights on its neighbour differences).
template <class T>
__host__ __device__ __forceinline__ void linear_pair(const T v[6], T& left, T& right) {
#pragma clang fp contract(off)
  const T d0 = v[1] - v[0], d1 = v[2] - v[1], d2 = v[3] - v[2], d3 = v[4] - v[3], d4 = v[5] - v[4];
  constexpr T a = T(-2.0 / 60), b = T(11.0 / 60), c = T(24.0 / 60), e = T(-3.0 / 60);
  left = fm(a, d0, fm(b, d1, fm(c, d2, fm(e, d3, v[2]))));
  right = fm(-a, d4, fm(-b, d3, fm(-c, d2, fm(-e, d1, v[3]))));
}

// Flux of one pair of states (in the caller's frame), with the face's signal
// speed folded into smax when RATE.
template <bool LF, class T>
__host__ __device__ __forceinline__ St<T> solve_face(const St<T>& L, const St<T>& R, Side<T>& l, Side<T>& r, int dir,
                                                     int order, T gamma, bool rate, T& smax) {
#pragma clang fp contract(off)
  const T bn = T(0.5) * (L.bx + R.bx), bn2 = bn * bn;
  l.cf = fast_of(l, bn2, gamma);
  r.cf = fast_of(r, bn2, gamma);
  if (rate) {
    // The rate takes each side's own normal field (equal on the solver's
    // faces, where the constrained-transport value is set on both sides).
    T cl = l.cf, cr = r.cf;
    if (L.bx != R.bx) {
      cl = fast_of(l, l.bn2, gamma);
      cr = fast_of(r, r.bn2, gamma);
    }
    smax = hi2(smax, rate_of(l, cl, r, cr, order));
  }
  if constexpr (LF)
    return rot(lf_flux(L, R, l.ir, r.ir, gamma), dir);
  else
    return rot(hlld_sides(L, R, l, r, bn), dir);
}

// E_z = vy Bx - vx By of a recovered point, its components taken in order (rho,
// mx, my, mz, E, Bx, By, Bz) so that four scalars live beside them.
template <class T>
struct PointEz {
  T ir, vx, vy, q, mag, ez;
  bool dense;
  __host__ __device__ __forceinline__ void take(int c, T v) {
#pragma clang fp contract(off)
    switch (c) {
      case 0: ir = rcp_near(v); dense = v > T(0); break;
      case 1: vx = v * ir; mag = v * vx; break;
      case 2: vy = v * ir; mag = fm(v, vy, mag); break;
      case 3: mag = fm(v, v * ir, mag); break;
      case 4: q = fm(T(-0.5), mag, v); mag = fm(T(0.5), mag, qabs(v)); break;
      case 5: ez = vy * v; vy = v * v; break;
      case 6: ez = fm(-vx, v, ez); vy = fm(v, v, vy); break;
      default: vy = fm(v, v, vy); q = fm(T(-0.5), vy, q); mag = fm(T(0.5), vy, mag);
    }
  }
  // Certainly admissible: rho > 0 and the internal energy positive beyond
  // rounding (a NaN or infinity anywhere fails).
  __host__ __device__ __forceinline__ bool sure() const { return dense & (q > T(32) * Lim<T>::eps * mag); }
  // Neither certainly admissible nor certainly not: the internal energy is
  // within rounding of zero.
  __host__ __device__ __forceinline__ bool unsure() const { return dense & (qabs(q) <= T(32) * Lim<T>::eps * mag); }
};

// E_z of a cell average as PointEz forms a point's, so that equal states give
// equal values whichever a cell takes.
template <class T>
__host__ __device__ __forceinline__ T average_ez(T rho, T mx, T my, T bx, T by) {
#pragma clang fp contract(off)
  const T ir = rcp_near(rho), vx = mx * ir, vy = my * ir;
  return fm(-vx, by, vy * bx);
}

// Neighbour-difference rows of the point recovery: point q is
// s[H] + sum_m step[q][m] (s[m+1] - s[m]), and the running-mean weights of the
// Gauss average.
template <class T, int ORDER>
struct NodeRows;
template <>
struct NodeRows<double, 7> {
  static constexpr int NQ = 4, NM = 6;
  static __host__ __device__ __forceinline__ double step(const QuadRows& t, int q, int m) { return t.mp7_step[q][m]; }
  static __host__ __device__ __forceinline__ double mean(const QuadRows& t, int q) { return t.mp7_mean[q]; }
};
template <>
struct NodeRows<double, 5> {
  static constexpr int NQ = 3, NM = 4;
  static __host__ __device__ __forceinline__ double step(const QuadRows& t, int q, int m) { return t.mp5_step[q][m]; }
  static __host__ __device__ __forceinline__ double mean(const QuadRows& t, int q) { return t.mp5_mean[q]; }
};
template <>
struct NodeRows<float, 7> {
  static constexpr int NQ = 4, NM = 6;
  static __host__ __device__ __forceinline__ float step(const QuadRows& t, int q, int m) { return t.mp7_step_f[q][m]; }
  static __host__ __device__ __forceinline__ float mean(const QuadRows& t, int q) { return t.mp7_mean_f[q]; }
};
template <>
struct NodeRows<float, 5> {
  static constexpr int NQ = 3, NM = 4;
  static __host__ __device__ __forceinline__ float step(const QuadRows& t, int q, int m) { return t.mp5_step_f[q][m]; }
  static __host__ __device__ __forceinline__ float mean(const QuadRows& t, int q) { return t.mp5_mean_f[q]; }
};

// side_of of a state u (s: u in the frame of the normal) where it may be within
// rounding of zero pressure: the reference decides, and its pressure serves the
// rate, which asks for its sign again (side_of's, rounded otherwise, is at or
// below zero for some 8 % of the admissible states within 4 ulp of zero: an
// infinite rate, which stops a run).
template <class T>
__host__ __device__ __forceinline__ bool decided_side(const St<T>& u, const St<T>& s, T gamma, Side<T>& o) {
  bool good = side_of(s, gamma, o);
  if (!good) good = admissible_state_p(u, gamma, o.p);
  return good;
}

// Signal speed of a face's averages (infinite when one is not admissible).
template <class T>
__host__ __device__ __forceinline__ T base_rate(const Side<T>& l, bool good_l, const Side<T>& r, bool good_r, int order,
                                                T gamma) {
  const T v = rate_of(l, fast_of(l, l.bn2, gamma), r, fast_of(r, r.bn2, gamma), order);
  return good_l && good_r ? v : Lim<T>::inf();
}

// Flux (and signal speed, when `rate`) of a face at its averages: the orders
// without transverse quadrature.
template <class T, bool LF>
__host__ __device__ __forceinline__ St<T> average_flux(const St<T>& bL, const St<T>& bR, int dir, int order, T gamma,
                                                       bool rate, T& smax) {
  const St<T> a = rot(bL, dir), b = rot(bR, dir);
  Side<T> l, r;
  const bool good_l = decided_side(bL, a, gamma, l), good_r = decided_side(bR, b, gamma, r);
  smax = rate ? base_rate(l, good_l, r, good_r, order, gamma) : T(0);
  T unused = T(0);
  return solve_face<LF>(a, b, l, r, dir, order, gamma, false, unused);
}

// Flux (and signal speed, when `rate`) of an MP5/MP7 face.  bL, bR: its face
// averages; diff[c * cs + m * ms]: the neighbour differences of plane c (L 0..7,
// R 8..15) along the face line.  An inadmissible point sends the face to the
// flux of its averages: one more pass of the same loop, taken by waves that
// hold such a face.
template <class T, int ORDER, bool LF>
__host__ __device__ __forceinline__ St<T> node_flux(const QuadRows& rows, const T* diff, int cs, int ms, const St<T>& bL,
                                           const St<T>& bR, int dir, T gamma, bool rate, T& smax) {
#pragma clang fp contract(off)
  using R = NodeRows<T, ORDER>;
  smax = T(0);
  if (rate) {
    const St<T> a = rot(bL, dir), b = rot(bR, dir);
    Side<T> l, r;
    const bool good_l = decided_side(bL, a, gamma, l), good_r = decided_side(bR, b, gamma, r);
    smax = base_rate(l, good_l, r, good_r, ORDER, gamma);
  }
  St<T> acc;
  bool ok = true;
#pragma nounroll
  for (int q = 0; q <= R::NQ; ++q) {
    if (q == R::NQ && !any_lane(!ok)) break;
    St<T> a = bL, b = bR;
    if (q < R::NQ) {
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        T va = comp(bL, c), vb = comp(bR, c);
#pragma unroll
        for (int m = 0; m < R::NM; ++m) {
          va = fm(R::step(rows, q, m), diff[c * cs + m * ms], va);
          vb = fm(R::step(rows, q, m), diff[(8 + c) * cs + m * ms], vb);
        }
        set_comp(a, c, va);
        set_comp(b, c, vb);
      }
    }
    const St<T> ra = rot(a, dir), rb = rot(b, dir);
    Side<T> l, r;
    const bool cl = side_of(ra, gamma, l), cr = side_of(rb, gamma, r);
    if (q < R::NQ && !(cl && cr)) {
#pragma nounroll
      for (int side = 0; side < 2; ++side) {
        const bool sure = side == 0 ? cl : cr;
        St<T> x = a;
        if (side == 1) x = b;
        T p = side == 0 ? l.p : r.p;
        ok = ok && (sure || admissible_state_p(x, gamma, p));
        if (side == 0)
          l.p = p;
        else
          r.p = p;
      }
    }
    T speed = T(0);
    const St<T> f = solve_face<LF>(ra, rb, l, r, dir, ORDER, gamma, rate, speed);
    // The rate takes every point before the first inadmissible one.
    if (rate && ok && q < R::NQ) smax = hi2(smax, speed);
    const bool take = q < R::NQ || !ok;
    const T w = q == 0 || q == R::NQ ? T(1) : R::mean(rows, q);
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      if (c == 5 + dir) {
        set_comp(acc, c, T(0));  // no flux of the normal field
        continue;
      }
      const T v = comp(f, c);
      if (q == 0)
        set_comp(acc, c, v);
      else if (take)
        set_comp(acc, c, q == R::NQ ? v : fm(w, v - comp(acc, c), comp(acc, c)));
    }
  }
  return acc;
}

}  // namespace qmhd

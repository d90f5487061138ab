// Device numerics for the 2D constrained-transport ideal-MHD step on gfx950:
// equation of state, Suresh-Huynh MP limiter, 7-wave characteristic system,
// Miyoshi-Kusano HLLD with its HLL/LF fallbacks, and the transverse Gauss rows.
//
// Every branch and guard of the reference algorithm is kept (they decide which
// formula a face uses); the arithmetic inside a branch is plain IEEE with fused
// multiply-add where the reference evaluates short dot products through exact
// expansions.  Results therefore agree with the reference to a few ulp per
// operation rather than bit for bit.  Templated on the arithmetic type T so the
// FP32 form shares the code; FP64 instantiations are the parity path.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace qmhd {

template <class T>
struct St {
  T rho, mx, my, mz, en, bx, by, bz;
};

template <class T>
__host__ __device__ __forceinline__ T comp(const St<T>& s, int c) {
  switch (c) {
    case 0: return s.rho;
    case 1: return s.mx;
    case 2: return s.my;
    case 3: return s.mz;
    case 4: return s.en;
    case 5: return s.bx;
    case 6: return s.by;
    default: return s.bz;
  }
}

template <class T>
__host__ __device__ __forceinline__ void set_comp(St<T>& s, int c, T v) {
  switch (c) {
    case 0: s.rho = v; break;
    case 1: s.mx = v; break;
    case 2: s.my = v; break;
    case 3: s.mz = v; break;
    case 4: s.en = v; break;
    case 5: s.bx = v; break;
    case 6: s.by = v; break;
    default: s.bz = v; break;
  }
}

template <class T>
struct Lim;
template <>
struct Lim<double> {
  static constexpr double eps = 2.220446049250313080847e-16;
  static constexpr double tiny = 2.2250738585072014e-308;
  static constexpr double half_max_pow2 = 0x1p1023;  // largest power of two
  static __host__ __device__ __forceinline__ double inf() { return __builtin_huge_val(); }
  static __host__ __device__ __forceinline__ double nan() { return __builtin_nan(""); }
};
template <>
struct Lim<float> {
  static constexpr float eps = 1.1920928955078125e-7f;
  static constexpr float tiny = 1.17549435e-38f;
  static constexpr float half_max_pow2 = 0x1p127f;
  static __host__ __device__ __forceinline__ float inf() { return __builtin_huge_valf(); }
  static __host__ __device__ __forceinline__ float nan() { return __builtin_nanf(""); }
};

template <class T>
__host__ __device__ __forceinline__ bool fin(T x) {
  return __builtin_isfinite(x);
}

// |x| and sqrt(x) in the argument's own precision.
__host__ __device__ __forceinline__ double qabs(double x) { return __builtin_fabs(x); }
__host__ __device__ __forceinline__ float qabs(float x) { return __builtin_fabsf(x); }
__host__ __device__ __forceinline__ double qsqrt(double x) { return __builtin_sqrt(x); }
__host__ __device__ __forceinline__ float qsqrt(float x) { return __builtin_sqrtf(x); }

// Reciprocal, quotient and square root for the face solvers (signal speeds,
// Riemann fans), where a last-bit difference moves no decision the reference
// makes exactly.  The wave basis that rounds as the reference's does keeps
// qsqrt and IEEE division; the closed-form basis, taken where a bound shows
// that the reference's test must pass, divides through sqrt_pos and rcp_near
// (qmhd_face.hpp).  On the device, FP64 starts from the hardware's approximate v_rcp_f64 /
// v_rsq_f64 (about 2^-23 relative error) and refines it with Newton steps.
// On an MI355X, over 2^18 inputs spanning 2^-60..2^60, every refined
// reciprocal and square root was within 0.5 ulp of the exact value, as IEEE
// results are; the compiler's IEEE division and square root add range scaling
// and special-value fixups (about ten and fifteen instructions, against five
// and eleven here).  frcp and fdiv expect a finite, nonzero, normal divisor
// and give a non-finite result otherwise (every caller tests its inputs or
// its result for finiteness); fdiv rounds twice, so it can differ from a/b in
// the last bit.  fsqrt keeps sqrt's results for 0 and +inf.  The host uses the
// IEEE operations, and so do these forms in FP32; the FP32 face solver takes
// rcp_near and sqrt_pos.
__host__ __device__ __forceinline__ double frcp(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  double r = __builtin_amdgcn_rcp(x);
  r = __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
  return __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
#else
  return 1.0 / x;
#endif
}
__host__ __device__ __forceinline__ float frcp(float x) { return 1.0f / x; }
__host__ __device__ __forceinline__ double fdiv(double a, double b) {
#if defined(__HIP_DEVICE_COMPILE__)
  return a * frcp(b);
#else
  return a / b;
#endif
}
__host__ __device__ __forceinline__ float fdiv(float a, float b) { return a / b; }
__host__ __device__ __forceinline__ double fsqrt(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  // Goldschmidt: g -> sqrt(x), h -> 1/(2 sqrt(x)).
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  const double r = __builtin_fma(-g, h, 0.5);
  g = __builtin_fma(g, r, g);
  h = __builtin_fma(h, r, h);
  g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
  return (x == 0.0 || x == __builtin_inf()) ? x : g;
#else
  return __builtin_sqrt(x);
#endif
}
__host__ __device__ __forceinline__ float fsqrt(float x) { return __builtin_sqrtf(x); }

// x/y swap into the +x-normal frame (self-inverse).
template <class T>
__host__ __device__ __forceinline__ St<T> rot(const St<T>& s, int dir) {
  if (dir == 0) return s;
  St<T> r = s;
  r.mx = s.my;
  r.my = s.mx;
  r.bx = s.by;
  r.by = s.bx;
  return r;
}

// ---------------------------------------------------------------------------
// Equation of state.
template <class T>
__host__ __device__ __forceinline__ T half_sq(T x, T y, T z) {
  return T(0.5) * (x * x + y * y + z * z);
}

template <class T>
__host__ __device__ __forceinline__ T pressure(const St<T>& u, T gm1) {
  const T kin = half_sq(u.mx, u.my, u.mz) / u.rho;
  const T mag = half_sq(u.bx, u.by, u.bz);
  return gm1 * ((u.en - kin) - mag);
}

// Pressure with the state's 1/rho supplied (the kinetic energy as a product
// with it, not a quotient): the face kernels evaluate one reciprocal per state
// and share it between the admissibility test, the signal speed and the
// Riemann solve.
template <class T>
__host__ __device__ __forceinline__ T pressure_ir(const St<T>& u, T inv_rho, T gm1) {
  const T kin = half_sq(u.mx, u.my, u.mz) * inv_rho;
  const T mag = half_sq(u.bx, u.by, u.bz);
  return gm1 * ((u.en - kin) - mag);
}

// Fast magnetosonic speed along +x for primitive density/pressure, with
// 1/rho supplied.
template <class T>
__host__ __device__ __forceinline__ T fast_speed_x_ir(T inv_rho, T p, T bx, T by, T bz, T gamma) {
  const T a2 = (p > T(0)) ? gamma * p * inv_rho : T(0);
  const T b2 = (bx * bx + by * by + bz * bz) * inv_rho;
  const T c2 = bx * bx * inv_rho;
  const T sum = a2 + b2;
  T disc = sum * sum - T(4) * a2 * c2;
  disc = disc < T(0) ? T(0) : disc;
  return fsqrt(T(0.5) * (sum + fsqrt(disc)));
}

// Fast magnetosonic speed along +x for primitive density/pressure.
template <class T>
__host__ __device__ __forceinline__ T fast_speed_x(T rho, T p, T bx, T by, T bz, T gamma) {
  const T inv_rho = T(1) / rho;
  const T a2 = (p > T(0)) ? gamma * p * inv_rho : T(0);
  const T b2 = (bx * bx + by * by + bz * bz) * inv_rho;
  const T c2 = bx * bx * inv_rho;
  const T sum = a2 + b2;
  T disc = sum * sum - T(4) * a2 * c2;
  disc = disc < T(0) ? T(0) : disc;
  return qsqrt(T(0.5) * (sum + qsqrt(disc)));
}

// ---------------------------------------------------------------------------
// MP limiter (Suresh & Huynh 1997).
template <class T>
__host__ __device__ __forceinline__ T minmod2(T a, T b) {
  if (a == T(0) || b == T(0) || ((a < T(0)) != (b < T(0)))) return T(0);
  return (qabs(a) < qabs(b)) ? a : b;
}

template <class T>
__host__ __device__ __forceinline__ T sgn0(T a) {
  return (a > T(0)) ? T(1) : ((a < T(0)) ? T(-1) : T(0));
}

template <class T>
__host__ __device__ __forceinline__ T minmod4(T a, T b, T c, T d) {
  const T sa = sgn0(a), sb = sgn0(b), sc = sgn0(c), sd = sgn0(d);
  if (!(sa == sb && sb == sc && sc == sd) || sa == T(0)) return T(0);
  return sa * fmin(fmin(qabs(a), qabs(b)),
                   fmin(qabs(c), qabs(d)));
}

// `shift_max` (optional) receives the largest |limited - unlimited| seen
// (the label of the troubled-cell indicator).
template <class T>
__host__ __device__ __forceinline__ T mp_limit(T vl, T vm2, T vm1, T v0, T vp1, T vp2, T* shift_max = nullptr) {
  const T d_minus = v0 - vm1;
  const T d_plus = vp1 - v0;
  const T vmp = v0 + minmod2(d_plus, T(4) * d_minus);
  const T cfc = vl - v0;
  const T cfm = vl - vmp;
  const bool between = (cfc <= T(0) && cfm >= T(0)) || (cfc >= T(0) && cfm <= T(0));
  const T variation = fmax(fmax(qabs(d_minus), qabs(d_plus)),
                           fmax(qabs(cfc), qabs(cfm)));
  // (|cfc|/v)(|cfm|/v) <= 1e-10, evaluated as |cfc||cfm| <= 1e-10 v^2.
  const bool within = variation > T(0) &&
                      qabs(cfc) * qabs(cfm) <= T(1e-10) * (variation * variation);
  if (between || within) return vl;
  const T dm = (vm2 - vm1) - (vm1 - v0);
  const T d0 = (vm1 - v0) - (v0 - vp1);
  const T dp = (v0 - vp1) - (vp1 - vp2);
  const T djph = minmod4(T(4) * d0 - dp, T(4) * dp - d0, d0, dp);
  const T djmh = minmod4(T(4) * d0 - dm, T(4) * dm - d0, d0, dm);
  const T v_ul = v0 + T(4) * d_minus;
  const T v_md = T(0.5) * (v0 + vp1) - T(0.5) * djph;
  const T v_lc = v0 + T(0.5) * d_minus + (T(4) / T(3)) * djmh;
  const T vmin = fmax(fmin(fmin(v0, vp1), v_md), fmin(fmin(v0, v_ul), v_lc));
  const T vmax = fmin(fmax(fmax(v0, vp1), v_md), fmax(fmax(v0, v_ul), v_lc));
  const T shift = minmod2(vmin - vl, vmax - vl);
  if (shift_max) *shift_max = fmax(*shift_max, qabs(shift));
  return vl + shift;
}

// Finite-volume left-biased face values: MP5 (2,-13,47,27,-3)/60 and
// MP7 (-3,25,-101,319,214,-38,4)/420 applied to cell averages.
template <class T>
__host__ __device__ __forceinline__ T mp5_face(const T* v) {
  const T s = T(2) * v[0] - T(13) * v[1] + T(47) * v[2] + T(27) * v[3] - T(3) * v[4];
  return s * (T(1) / T(60));
}
template <class T>
__host__ __device__ __forceinline__ T mp7_face(const T* v) {
  const T s = -T(3) * v[0] + T(25) * v[1] - T(101) * v[2] + T(319) * v[3] + T(214) * v[4] -
              T(38) * v[5] + T(4) * v[6];
  return s * (T(1) / T(420));
}

// ---------------------------------------------------------------------------
// Seven-wave eigensystem about a reference state, +x normal, in the
// conserved 7-vector (rho, mn, mt1, mt2, E, bt1, bt2) (Stone et al. 2008, App. A).
//
// Whether the characteristic basis is usable is decided by an absolute
// 1024-epsilon test on L R - I (include/quasar/numerics/mhd_eigensystem.hpp:
// 398-431).  Near degenerate states (zero transverse field with a ~ c_ax) the
// residual sits close to that threshold, so the decision depends on how each
// operation rounds.  The whole build therefore follows the reference's
// operation order term by term (its dense M Rp and Lp Minv products reduced to
// their structurally non-zero terms, in the same summation order) with
// multiply-add contraction off, so the decision and the vectors are those of
// the reference arithmetic.

template <class T>
__host__ __device__ __forceinline__ T scaled_norm3(T x, T y, T z) {
#pragma clang fp contract(off)
  const T scale = fmax(qabs(x), fmax(qabs(y), qabs(z)));
  if (scale == T(0)) return T(0);
  const T xs = x / scale, ys = y / scale, zs = z / scale;
  return scale * qsqrt(xs * xs + ys * ys + zs * zs);
}

template <class T>
__host__ __device__ __forceinline__ T half_squared_norm3(T x, T y, T z) {
#pragma clang fp contract(off)
  const T scale = fmax(qabs(x), fmax(qabs(y), qabs(z)));
  if (scale == T(0)) return T(0);
  const T xs = x / scale, ys = y / scale, zs = z / scale;
  const T ns = xs * xs + ys * ys + zs * zs;
  return (T(0.5) * scale) * (scale * ns);
}

template <class T>
__host__ __device__ __forceinline__ T kinetic_from_momentum(T mx, T my, T mz, T rho) {
#pragma clang fp contract(off)
  const T scale = fmax(qabs(mx), fmax(qabs(my), qabs(mz)));
  if (scale == T(0)) return T(0);
  const T xs = mx / scale, ys = my / scale, zs = mz / scale;
  const T q = scale / qsqrt(rho);
  const T ns = xs * xs + ys * ys + zs * zs;
  return (T(0.5) * q) * (q * ns);
}

// Primitive state and the reference's conversions (mhd_state.hpp:183-255):
// velocities by division, kinetic and magnetic energies through the scaled
// norms, no multiply-add contraction.  Reconstructed face states built from
// these compare (L == R) exactly as the reference's do.
template <class T>
struct Prim {
  T rho, vx, vy, vz, p, bx, by, bz;
};

template <class T>
__host__ __device__ __forceinline__ T kinetic_from_velocity(T rho, T vx, T vy, T vz) {
#pragma clang fp contract(off)
  const T scale = fmax(qabs(vx), fmax(qabs(vy), qabs(vz)));
  if (scale == T(0)) return T(0);
  const T xs = vx / scale, ys = vy / scale, zs = vz / scale;
  const T q = qsqrt(rho) * scale;
  const T ns = xs * xs + ys * ys + zs * zs;
  return (T(0.5) * q) * (q * ns);
}

template <class T>
__host__ __device__ __forceinline__ T ref_pressure(const St<T>& u, T gamma) {
#pragma clang fp contract(off)
  return (gamma - T(1)) * ((u.en - kinetic_from_momentum(u.mx, u.my, u.mz, u.rho)) - half_squared_norm3(u.bx, u.by, u.bz));
}

template <class T>
__host__ __device__ __forceinline__ Prim<T> to_prim(const St<T>& u, T gamma) {
#pragma clang fp contract(off)
  return Prim<T>{u.rho, u.mx / u.rho, u.my / u.rho, u.mz / u.rho, ref_pressure(u, gamma), u.bx, u.by, u.bz};
}

template <class T>
__host__ __device__ __forceinline__ St<T> to_cons(const Prim<T>& w, T gamma) {
#pragma clang fp contract(off)
  St<T> u;
  u.rho = w.rho;
  u.mx = w.rho * w.vx;
  u.my = w.rho * w.vy;
  u.mz = w.rho * w.vz;
  u.bx = w.bx;
  u.by = w.by;
  u.bz = w.bz;
  const T kinetic = kinetic_from_velocity(w.rho, w.vx, w.vy, w.vz);
  const T magnetic = half_squared_norm3(w.bx, w.by, w.bz);
  u.en = w.p / (gamma - T(1)) + kinetic + magnetic;
  return u;
}

// Sign of the reference pressure (p > 0 and finite), decided with a fast
// evaluation and a rounding margin: when the fast value is farther from zero
// than 32 epsilon of the magnitudes it cancels, the reference form has the
// same sign; otherwise the reference form decides.
// fin(m / rho) for finite m and finite rho > 0, without the division in the
// common case: |m| < rho * 2^emax (the product is exact or overflows to
// infinity, and then the quotient is at most max/2) bounds |m / rho| below
// 2^emax; otherwise the quotient itself is tested.
template <class T>
__host__ __device__ __forceinline__ bool finite_ratio(T m, T rho) {
  if (qabs(m) < rho * Lim<T>::half_max_pow2) return true;
  return fin(m / rho);
}

template <class T>
__host__ __device__ __forceinline__ bool pressure_positive(const St<T>& u, T gamma) {
  const T kin = fdiv(T(0.5) * (u.mx * u.mx + u.my * u.my + u.mz * u.mz), u.rho);
  const T mag = T(0.5) * (u.bx * u.bx + u.by * u.by + u.bz * u.bz);
  const T gm1 = gamma - T(1);
  const T pf = gm1 * ((u.en - kin) - mag);
  const T margin = T(32) * Lim<T>::eps * gm1 * (qabs(u.en) + kin + mag);
  if (fin(pf) && fin(margin) && pf > margin) return true;
  if (fin(pf) && fin(margin) && pf < -margin) return false;
  const T p = ref_pressure(u, gamma);
  return fin(p) && p > T(0);
}

template <class T>
struct Eig {
  T L[7][7];
  T R[7][7];  // R[var][wave]
};

// The characteristic basis about a reference state in factored form: the
// scalars from which the primitive eigenvector rows Rp[k], Lp[k]
// (var = rho, vn, vt1, vt2, p, bt1, bt2) and the maps M = dU/dW, M^-1
// (mhd_eigensystem.hpp:333-379) are formed on demand.  The conserved
// R = M Rp and L = Lp M^-1 are only materialised for the biorthogonality test,
// which decides `identity`.
template <class T>
struct CharBasis {
  T rho, sqrt_rho, vn, vt1, vt2, bt1, bt2, gm1, half_v2, inv_rho;
  T alpha_f, alpha_s, beta1, beta2, sbn, rs2, cf, cs, qf, qs, Af, As, Nf, inv_a2, rho_a2;
  bool identity;
};

// Primitive right and left rows of wave k (unset entries zero).
template <class T>
__host__ __device__ __forceinline__ void basis_right(const CharBasis<T>& B, int k, T* r) {
#pragma clang fp contract(off)
  const T rho = B.rho, sqrt_rho = B.sqrt_rho, alpha_f = B.alpha_f, alpha_s = B.alpha_s;
  const T beta1 = B.beta1, beta2 = B.beta2, sbn = B.sbn, rs2 = B.rs2, cf = B.cf, cs = B.cs;
  const T qf = B.qf, qs = B.qs, Af = B.Af, As = B.As, rho_a2 = B.rho_a2;
#pragma unroll
  for (int v = 0; v < 7; ++v) r[v] = T(0);
  if (k == 0) {
    r[0] = rho * alpha_f; r[1] = -alpha_f * cf; r[2] = qs * beta1; r[3] = qs * beta2;
    r[4] = alpha_f * rho_a2; r[5] = As * beta1; r[6] = As * beta2;
  } else if (k == 6) {
    r[0] = rho * alpha_f; r[1] = alpha_f * cf; r[2] = -qs * beta1; r[3] = -qs * beta2;
    r[4] = alpha_f * rho_a2; r[5] = As * beta1; r[6] = As * beta2;
  } else if (k == 1) {
    r[2] = -beta2 * rs2; r[3] = beta1 * rs2;
    r[5] = -sbn * beta2 * rs2 * sqrt_rho; r[6] = sbn * beta1 * rs2 * sqrt_rho;
  } else if (k == 5) {
    r[2] = -beta2 * rs2; r[3] = beta1 * rs2;
    r[5] = sbn * beta2 * rs2 * sqrt_rho; r[6] = -sbn * beta1 * rs2 * sqrt_rho;
  } else if (k == 2) {
    r[0] = rho * alpha_s; r[1] = -alpha_s * cs; r[2] = -qf * beta1; r[3] = -qf * beta2;
    r[4] = alpha_s * rho_a2; r[5] = -Af * beta1; r[6] = -Af * beta2;
  } else if (k == 4) {
    r[0] = rho * alpha_s; r[1] = alpha_s * cs; r[2] = qf * beta1; r[3] = qf * beta2;
    r[4] = alpha_s * rho_a2; r[5] = -Af * beta1; r[6] = -Af * beta2;
  } else {
    r[0] = T(1);
  }
}
template <class T>
__host__ __device__ __forceinline__ void basis_left(const CharBasis<T>& B, int k, T* l) {
#pragma clang fp contract(off)
  const T rho = B.rho, sqrt_rho = B.sqrt_rho, alpha_f = B.alpha_f, alpha_s = B.alpha_s;
  const T beta1 = B.beta1, beta2 = B.beta2, sbn = B.sbn, rs2 = B.rs2, cf = B.cf, cs = B.cs;
  const T qf = B.qf, qs = B.qs, Af = B.Af, As = B.As, Nf = B.Nf, inv_a2 = B.inv_a2;
#pragma unroll
  for (int v = 0; v < 7; ++v) l[v] = T(0);
  if (k == 0) {
    l[1] = -Nf * alpha_f * cf; l[2] = Nf * qs * beta1; l[3] = Nf * qs * beta2;
    l[4] = Nf * alpha_f / rho; l[5] = Nf * As * beta1 / rho; l[6] = Nf * As * beta2 / rho;
  } else if (k == 6) {
    l[1] = Nf * alpha_f * cf; l[2] = -Nf * qs * beta1; l[3] = -Nf * qs * beta2;
    l[4] = Nf * alpha_f / rho; l[5] = Nf * As * beta1 / rho; l[6] = Nf * As * beta2 / rho;
  } else if (k == 1) {
    l[2] = -beta2 * rs2; l[3] = beta1 * rs2;
    l[5] = -sbn * beta2 * rs2 / sqrt_rho; l[6] = sbn * beta1 * rs2 / sqrt_rho;
  } else if (k == 5) {
    l[2] = -beta2 * rs2; l[3] = beta1 * rs2;
    l[5] = sbn * beta2 * rs2 / sqrt_rho; l[6] = -sbn * beta1 * rs2 / sqrt_rho;
  } else if (k == 2) {
    l[1] = -Nf * alpha_s * cs; l[2] = -Nf * qf * beta1; l[3] = -Nf * qf * beta2;
    l[4] = Nf * alpha_s / rho; l[5] = -Nf * Af * beta1 / rho; l[6] = -Nf * Af * beta2 / rho;
  } else if (k == 4) {
    l[1] = Nf * alpha_s * cs; l[2] = Nf * qf * beta1; l[3] = Nf * qf * beta2;
    l[4] = Nf * alpha_s / rho; l[5] = -Nf * Af * beta1 / rho; l[6] = -Nf * Af * beta2 / rho;
  } else {
    l[0] = T(1); l[4] = -inv_a2;
  }
}
template <class T>
__host__ __device__ __forceinline__ void basis_rows(const CharBasis<T>& B, int k, T* r, T* l) {
  basis_right(B, k, r);
  basis_left(B, k, l);
}

// Conserved right column R[.][k] = M Rp[k] and left row L[k][.] = Lp[k] M^-1,
// the non-zero entries of M and M^-1 in the reference's summation order.
template <class T>
__host__ __device__ __forceinline__ void basis_rcol(const CharBasis<T>& B, const T* r, T* out) {
#pragma clang fp contract(off)
  const T m41 = B.rho * B.vn, m42 = B.rho * B.vt1, m43 = B.rho * B.vt2, m44 = T(1) / B.gm1;
  out[0] = r[0];
  out[1] = B.vn * r[0] + B.rho * r[1];
  out[2] = B.vt1 * r[0] + B.rho * r[2];
  out[3] = B.vt2 * r[0] + B.rho * r[3];
  out[4] = (((((B.half_v2 * r[0] + m41 * r[1]) + m42 * r[2]) + m43 * r[3]) + m44 * r[4]) + B.bt1 * r[5]) + B.bt2 * r[6];
  out[5] = r[5];
  out[6] = r[6];
}
template <class T>
__host__ __device__ __forceinline__ void basis_lrow(const CharBasis<T>& B, const T* l, T* out) {
#pragma clang fp contract(off)
  const T gm1 = B.gm1, inv_rho = B.inv_rho;
  const T i10 = -B.vn * inv_rho, i20 = -B.vt1 * inv_rho, i30 = -B.vt2 * inv_rho;
  const T i40 = gm1 * B.half_v2, i41 = -gm1 * B.vn, i42 = -gm1 * B.vt1, i43 = -gm1 * B.vt2;
  const T i45 = -gm1 * B.bt1, i46 = -gm1 * B.bt2;
  out[0] = (((l[0] + l[1] * i10) + l[2] * i20) + l[3] * i30) + l[4] * i40;
  out[1] = l[1] * inv_rho + l[4] * i41;
  out[2] = l[2] * inv_rho + l[4] * i42;
  out[3] = l[3] * inv_rho + l[4] * i43;
  out[4] = l[4] * gm1;
  out[5] = l[4] * i45 + l[5];
  out[6] = l[4] * i46 + l[6];
}

// Seven-wave eigensystem about a reference state, +x normal, in the
// conserved 7-vector (rho, mn, mt1, mt2, E, bt1, bt2) (Stone et al. 2008, App. A).
//
// Whether the characteristic basis is usable is decided by an absolute
// 1024-epsilon test on L R - I (include/quasar/numerics/mhd_eigensystem.hpp:
// 398-431).  Near degenerate states (zero transverse field with a ~ c_ax) the
// residual sits close to that threshold, so the decision depends on how each
// operation rounds: the scalars, the rows, M, M^-1 and the test follow the
// reference's operation order term by term (its dense M Rp and Lp M^-1
// products reduced to their structurally non-zero terms, in the same summation
// order) with multiply-add contraction off, so the decision is that of the
// reference arithmetic.
template <class T>
__host__ __device__ __forceinline__ void basis_scalars(const St<T>& s, T gamma, CharBasis<T>& B) {
#pragma clang fp contract(off)
  // Primitive reference state (mhd_state.hpp:183-189, 228-239).
  const T rho = s.rho;
  const T vn = s.mx / rho, vt1 = s.my / rho, vt2 = s.mz / rho;
  T p = (gamma - T(1)) *
        ((s.en - kinetic_from_momentum(s.mx, s.my, s.mz, rho)) - half_squared_norm3(s.bx, s.by, s.bz));
  p = p > T(0) ? p : T(0);
  const T sqrt_rho = qsqrt(rho);
  const T bn = s.bx + T(0), bt1 = s.by + T(0), bt2 = s.bz + T(0);
  // Magnetosonic speeds through the normalised quadratic (mhd_state.hpp:141-180).
  T cf, cs, a, ca;
  {
    a = (p > T(0) && gamma > T(0)) ? qsqrt(gamma) * (qsqrt(p) / sqrt_rho) : T(0);
    const T ax = bn / sqrt_rho, ay = bt1 / sqrt_rho, az = bt2 / sqrt_rho;
    ca = scaled_norm3(ax, ay, az);
    const T cax = qabs(ax);
    const T scale = fmax(a, ca);
    if (!(scale > T(0))) {
      cf = T(0);
      cs = T(0);
    } else {
      const T an = a / scale, bnn = ca / scale, can = cax / scale;
      const T a2n = an * an, b2n = bnn * bnn, can2 = can * can;
      const T sum = a2n + b2n;
      T disc = sum * sum - T(4) * a2n * can2;
      if (disc < T(0)) disc = T(0);
      const T fast2n = T(0.5) * (sum + qsqrt(disc));
      const T slow2n = fast2n > T(0) ? (a2n * can2) / fast2n : T(0);
      cf = scale * qsqrt(fast2n);
      cs = scale * qsqrt(slow2n);
    }
  }
  constexpr T geps = T(64) * Lim<T>::eps;
  const T rs2 = T(1) / qsqrt(T(2));
  T alpha_f, alpha_s;
  {
    const T speed_scale = cf > T(0) ? cf : T(1);
    const T cfn = cf / speed_scale, csn = cs / speed_scale, an = a / speed_scale;
    const T denom = cfn * cfn - csn * csn;
    if (denom <= geps * (cfn * cfn + csn * csn)) {
      alpha_f = rs2;
      alpha_s = rs2;
    } else {
      T af2 = (an * an - csn * csn) / denom;
      T as2 = (cfn * cfn - an * an) / denom;
      if (af2 < T(0)) af2 = T(0);
      if (as2 < T(0)) as2 = T(0);
      alpha_f = qsqrt(af2);
      alpha_s = qsqrt(as2);
    }
  }
  T beta1, beta2;
  {
    const T bt = scaled_norm3(bt1, bt2, T(0));
    const T bt_speed = bt / sqrt_rho;
    const T field_scale = a > ca ? a : ca;
    if (bt == T(0) || bt_speed <= geps * (field_scale + Lim<T>::tiny)) {
      beta1 = rs2;
      beta2 = rs2;
    } else {
      beta1 = bt1 / bt;
      beta2 = bt2 / bt;
    }
  }
  const T sbn = bn >= T(0) ? T(1) : T(-1);
  const T qf = cf * alpha_f * sbn, qs = cs * alpha_s * sbn;
  const T Af = a * alpha_f * sqrt_rho, As = a * alpha_s * sqrt_rho;
  const T inv_a2 = a > T(0) ? (T(1) / a) / a : T(0);
  const T Nf = T(0.5) * inv_a2;
  const T rho_a2 = gamma * p;

  B.rho = rho;
  B.sqrt_rho = sqrt_rho;
  B.vn = vn;
  B.vt1 = vt1;
  B.vt2 = vt2;
  B.bt1 = bt1;
  B.bt2 = bt2;
  B.gm1 = gamma - T(1);
  B.half_v2 = half_squared_norm3(vn, vt1, vt2);
  B.inv_rho = T(1) / rho;
  B.alpha_f = alpha_f;
  B.alpha_s = alpha_s;
  B.beta1 = beta1;
  B.beta2 = beta2;
  B.sbn = sbn;
  B.rs2 = rs2;
  B.cf = cf;
  B.cs = cs;
  B.qf = qf;
  B.qs = qs;
  B.Af = Af;
  B.As = As;
  B.Nf = Nf;
  B.inv_a2 = inv_a2;
  B.rho_a2 = rho_a2;
}

// Whether any lane of the wave has `b` (the host runs one lane).
__host__ __device__ __forceinline__ bool any_lane(bool b) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __any(b);
#else
  return b;
#endif
}

// The waves of a pair (fast 6 / 0, Alfven 5 / 1, slow 4 / 2; the entropy wave 3
// with itself): their primitive rows differ in the sign of entries 1 to 3 (of
// entries 5 and 6 for the Alfven pair), and so do the products that their
// conserved columns and rows are sums of.
__host__ __device__ __forceinline__ int pair_wave(int pair, int side) { return pair == 3 ? 3 : side == 0 ? 6 - pair : pair; }

// Conserved columns of a pair (basis_rcol of both waves to the bit).
template <class T>
__host__ __device__ __forceinline__ void basis_rcol_pair(const CharBasis<T>& B, int pair, T out[2][7]) {
#pragma clang fp contract(off)
  const T m41 = B.rho * B.vn, m42 = B.rho * B.vt1, m43 = B.rho * B.vt2, m44 = T(1) / B.gm1;
  T r[7];
  basis_right(B, pair_wave(pair, 0), r);
  const T p1 = B.rho * r[1], p2 = B.rho * r[2], p3 = B.rho * r[3], q1 = m41 * r[1], q2 = m42 * r[2], q3 = m43 * r[3];
  const T a1 = B.vn * r[0], a2 = B.vt1 * r[0], a3 = B.vt2 * r[0], a4 = B.half_v2 * r[0], e = m44 * r[4];
  const T f = B.bt1 * r[5], g = B.bt2 * r[6];
#pragma unroll
  for (int side = 0; side < 2; ++side) {
    const T mid = side == 1 && (pair == 0 || pair == 2) ? T(-1) : T(1), end = side == 1 && pair == 1 ? T(-1) : T(1);
    out[side][0] = r[0];
    out[side][1] = a1 + mid * p1;
    out[side][2] = a2 + mid * p2;
    out[side][3] = a3 + mid * p3;
    out[side][4] = (((((a4 + mid * q1) + mid * q2) + mid * q3) + e) + end * f) + end * g;
    out[side][5] = end * r[5];
    out[side][6] = end * r[6];
  }
}
// Left rows of a pair (basis_lrow of both waves to the bit).
template <class T>
__host__ __device__ __forceinline__ void basis_lrow_pair(const CharBasis<T>& B, int pair, T out[2][7]) {
#pragma clang fp contract(off)
  const T gm1 = B.gm1, inv_rho = B.inv_rho;
  const T i10 = -B.vn * inv_rho, i20 = -B.vt1 * inv_rho, i30 = -B.vt2 * inv_rho;
  T l[7];
  basis_left(B, pair_wave(pair, 0), l);
  const T x1 = l[1] * i10, x2 = l[2] * i20, x3 = l[3] * i30, x4 = l[4] * (gm1 * B.half_v2);
  const T y1 = l[1] * inv_rho, y2 = l[2] * inv_rho, y3 = l[3] * inv_rho;
  const T z1 = l[4] * (-gm1 * B.vn), z2 = l[4] * (-gm1 * B.vt1), z3 = l[4] * (-gm1 * B.vt2);
  const T z5 = l[4] * (-gm1 * B.bt1), z6 = l[4] * (-gm1 * B.bt2), e = l[4] * gm1;
#pragma unroll
  for (int side = 0; side < 2; ++side) {
    const T mid = side == 1 && (pair == 0 || pair == 2) ? T(-1) : T(1), end = side == 1 && pair == 1 ? T(-1) : T(1);
    out[side][0] = (((l[0] + mid * x1) + mid * x2) + mid * x3) + x4;
    out[side][1] = mid * y1 + z1;
    out[side][2] = mid * y2 + z2;
    out[side][3] = mid * y3 + z3;
    out[side][4] = e;
    out[side][5] = z5 + end * l[5];
    out[side][6] = z6 + end * l[6];
  }
}

// Whether L R = I within the reference's bound; a loss of biorthogonality sends
// the face to component-wise limiting (identity basis).  In FP32 a row of L at a
// time beside the 7 columns of R.  In FP64 those are 98 registers, and set the
// occupancy of every kernel that includes this: pairs of rows against pairs of
// columns, in rolled loops, the two of a pair from shared products.  1024^2 FP64
// at density 100 and unit pressure, where every face takes this test, both
// directions: 442 us with a column at a time formed again for every row, 366
// now (396 for the reference's face per thread, which held all columns).
template <class T>
__host__ __device__ __forceinline__ bool basis_usable(const CharBasis<T>& B) {
#pragma clang fp contract(off)
  bool usable = true;
  auto test = [&](bool same, const T* row, const T* col) {
    T dot = row[0] * col[0];
#pragma unroll
    for (int k = 1; k < 7; ++k) dot = dot + row[k] * col[k];
    const T expect = same ? T(1) : T(0);
    usable = usable && fin(dot) && !(qabs(dot - expect) > T(1024) * Lim<T>::eps);
  };
  if constexpr (sizeof(T) == 4) {
    T cols[7][7];
#pragma unroll
    for (int j = 0; j < 7; ++j) {
      T r[7];
      basis_right(B, j, r);
      basis_rcol(B, r, cols[j]);
    }
#pragma nounroll
    for (int i = 0; i < 7; ++i) {
      T l[7], row[7];
      basis_left(B, i, l);
      basis_lrow(B, l, row);
#pragma unroll
      for (int j = 0; j < 7; ++j) test(i == j, row, cols[j]);
    }
  } else {
#pragma nounroll
    for (int a = 0; a < 4 && any_lane(usable); ++a) {
      T rows[2][7];
      basis_lrow_pair(B, a, rows);
#pragma nounroll
      for (int b = 0; b < 4; ++b) {
        T cols[2][7];
        basis_rcol_pair(B, b, cols);
#pragma unroll
        for (int s = 0; s < 4; ++s) test(pair_wave(a, s >> 1) == pair_wave(b, s & 1), rows[s >> 1], cols[s & 1]);
      }
    }
  }
  return usable;
}

template <class T>
__host__ __device__ __forceinline__ void basis_build(const St<T>& s, T gamma, CharBasis<T>& B) {
  basis_scalars(s, gamma, B);
  B.identity = !basis_usable(B);
}

// The conserved L and R (identity when the basis is not usable).
template <class T>
__host__ __device__ __forceinline__ void eig_build(const St<T>& s, T gamma, Eig<T>& e) {
  CharBasis<T> B;
  basis_build(s, gamma, B);
#pragma unroll
  for (int k = 0; k < 7; ++k) {
    T r[7], l[7], col[7], row[7];
    basis_rows(B, k, r, l);
    basis_rcol(B, r, col);
    basis_lrow(B, l, row);
#pragma unroll
    for (int v = 0; v < 7; ++v) {
      e.R[v][k] = B.identity ? T(v == k ? 1 : 0) : col[v];
      e.L[k][v] = B.identity ? T(v == k ? 1 : 0) : row[v];
    }
  }
}

// Characteristic variables w = L d of a conserved 7-vector difference, as
// Lp (M^-1 d).
template <class T>
__host__ __device__ __forceinline__ void basis_to_char(const CharBasis<T>& B, const T* d, T* w) {
  if (B.identity) {
#pragma unroll
    for (int v = 0; v < 7; ++v) w[v] = d[v];
    return;
  }
  const T gm1 = B.gm1, inv_rho = B.inv_rho;
  T dp[7];
  dp[0] = d[0];
  dp[1] = (d[1] - B.vn * d[0]) * inv_rho;
  dp[2] = (d[2] - B.vt1 * d[0]) * inv_rho;
  dp[3] = (d[3] - B.vt2 * d[0]) * inv_rho;
  dp[4] = gm1 * (((d[4] + B.half_v2 * d[0]) - (B.vn * d[1] + B.vt1 * d[2] + B.vt2 * d[3])) -
                 (B.bt1 * d[5] + B.bt2 * d[6]));
  dp[5] = d[5];
  dp[6] = d[6];
#pragma unroll
  for (int k = 0; k < 7; ++k) {
    T r[7], l[7];
    basis_rows(B, k, r, l);
    T acc = T(0);
#pragma unroll
    for (int v = 0; v < 7; ++v) acc += l[v] * dp[v];
    w[k] = acc;
  }
}

// Conserved 7-vector R w, as M (Rp^T w).
template <class T>
__host__ __device__ __forceinline__ void basis_from_char(const CharBasis<T>& B, const T* w, T* out) {
  if (B.identity) {
#pragma unroll
    for (int v = 0; v < 7; ++v) out[v] = w[v];
    return;
  }
  T ap[7] = {T(0), T(0), T(0), T(0), T(0), T(0), T(0)};
#pragma unroll
  for (int k = 0; k < 7; ++k) {
    T r[7], l[7];
    basis_rows(B, k, r, l);
#pragma unroll
    for (int v = 0; v < 7; ++v) ap[v] += r[v] * w[k];
  }
  out[0] = ap[0];
  out[1] = B.vn * ap[0] + B.rho * ap[1];
  out[2] = B.vt1 * ap[0] + B.rho * ap[2];
  out[3] = B.vt2 * ap[0] + B.rho * ap[3];
  out[4] = B.half_v2 * ap[0] + B.rho * (B.vn * ap[1] + B.vt1 * ap[2] + B.vt2 * ap[3]) + ap[4] / B.gm1 +
           B.bt1 * ap[5] + B.bt2 * ap[6];
  out[5] = ap[5];
  out[6] = ap[6];
}

// ---------------------------------------------------------------------------
// Fluxes along +x.  phys_flux_of takes 1/rho and the pressure of `u` when the
// caller already holds them (the same values phys_flux computes).
template <class T>
__host__ __device__ __forceinline__ St<T> phys_flux_of(const St<T>& u, T inv, T p) {
  const T vx = u.mx * inv, vy = u.my * inv, vz = u.mz * inv;
  const T hbn2 = T(0.5) * u.bx * u.bx;
  const T hbt2 = T(0.5) * (u.by * u.by + u.bz * u.bz);
  St<T> f;
  f.rho = u.mx;
  f.mx = u.mx * vx + p + hbt2 - hbn2;
  f.my = u.mx * vy - u.bx * u.by;
  f.mz = u.mx * vz - u.bx * u.bz;
  const T enth = ((u.en - hbn2) + p) + hbt2;
  f.en = vx * enth - u.bx * (vy * u.by + vz * u.bz);
  f.bx = T(0);
  f.by = u.by * vx - u.bx * vy;
  f.bz = u.bz * vx - u.bx * vz;
  return f;
}

template <class T>
__host__ __device__ __forceinline__ St<T> phys_flux(const St<T>& u, T gm1) {
  return phys_flux_of(u, T(1) / u.rho, pressure(u, gm1));
}

// HLL flux from the two physical fluxes.
template <class T>
__host__ __device__ __forceinline__ St<T> hll_combine(const St<T>& L, const St<T>& R, const St<T>& fl,
                                                      const St<T>& fr, T sl, T sr) {
  if (sl >= T(0)) return fl;
  if (sr <= T(0)) return fr;
  const T scale = fmax(qabs(sl), qabs(sr));
  if (!(scale > T(0)) || !fin(scale)) return fl;
  const T denom = sr - sl;
  if (!(denom > T(0)) || !fin(denom)) return fl;
  const T inv = frcp(denom);
  const T wl = sr * inv, wr = -sl * inv, diss = sl * sr * inv;
  St<T> f;
  f.rho = wl * fl.rho + wr * fr.rho + diss * (R.rho - L.rho);
  f.mx = wl * fl.mx + wr * fr.mx + diss * (R.mx - L.mx);
  f.my = wl * fl.my + wr * fr.my + diss * (R.my - L.my);
  f.mz = wl * fl.mz + wr * fr.mz + diss * (R.mz - L.mz);
  f.en = wl * fl.en + wr * fr.en + diss * (R.en - L.en);
  f.bx = T(0);
  f.by = wl * fl.by + wr * fr.by + diss * (R.by - L.by);
  f.bz = wl * fl.bz + wr * fr.bz + diss * (R.bz - L.bz);
  return f;
}

template <class T>
__host__ __device__ __forceinline__ St<T> hll_flux(const St<T>& L, const St<T>& R, T sl, T sr, T gm1) {
  return hll_combine(L, R, phys_flux(L, gm1), phys_flux(R, gm1), sl, sr);
}

// The Riemann solvers below take each state's 1/rho from the caller (the face
// kernels hold it already); the two-argument forms compute it.
template <class T>
__host__ __device__ __forceinline__ St<T> lf_flux(const St<T>& L, const St<T>& R, T irL, T irR, T gamma) {
  const T gm1 = gamma - T(1);
  const T pL = pressure_ir(L, irL, gm1), pR = pressure_ir(R, irR, gm1);
  const T cfL = fast_speed_x_ir(irL, pL, L.bx, L.by, L.bz, gamma);
  const T cfR = fast_speed_x_ir(irR, pR, R.bx, R.by, R.bz, gamma);
  const T aL = qabs(L.mx * irL) + cfL;
  const T aR = qabs(R.mx * irR) + cfR;
  const T a = aL > aR ? aL : aR;
  return hll_combine(L, R, phys_flux_of(L, irL, pL), phys_flux_of(R, irR, pR), -a, a);
}

template <class T>
__host__ __device__ __forceinline__ St<T> lf_flux(const St<T>& L, const St<T>& R, T gamma) {
  return lf_flux(L, R, frcp(L.rho), frcp(R.rho), gamma);
}

// HLL with the Davis speeds of the HLLD solver below, after the same normal
// field averaging (the flux hlld_flux falls back to on degenerate fans,
// include/quasar/numerics/hlld_core.hpp:157-192, 241-290).  The cheap path
// of the learned form and the HLLD-vs-HLL label use it.
template <class T>
__host__ __device__ __forceinline__ St<T> hll_davis_flux(const St<T>& Lin, const St<T>& Rin, T irL, T irR,
                                                         T gamma) {
  const T gm1 = gamma - T(1);
  const T bn = T(0.5) * (Lin.bx + Rin.bx);
  St<T> L = Lin, R = Rin;
  const T hbn2 = T(0.5) * bn * bn;
  L.en = (L.en - T(0.5) * L.bx * L.bx) + hbn2;
  R.en = (R.en - T(0.5) * R.bx * R.bx) + hbn2;
  L.bx = bn;
  R.bx = bn;
  const T vxL = L.mx * irL, vxR = R.mx * irR;
  const T pL = pressure_ir(L, irL, gm1), pR = pressure_ir(R, irR, gm1);
  const T cfL = fast_speed_x_ir(irL, pL, L.bx, L.by, L.bz, gamma);
  const T cfR = fast_speed_x_ir(irR, pR, R.bx, R.by, R.bz, gamma);
  const T cfmax = cfL > cfR ? cfL : cfR;
  const T sl = (vxL < vxR ? vxL : vxR) - cfmax;
  const T sr = (vxL > vxR ? vxL : vxR) + cfmax;
  return hll_combine(L, R, phys_flux_of(L, irL, pL), phys_flux_of(R, irR, pR), sl, sr);
}

template <class T>
__host__ __device__ __forceinline__ St<T> hll_davis_flux(const St<T>& Lin, const St<T>& Rin, T gamma) {
  return hll_davis_flux(Lin, Rin, frcp(Lin.rho), frcp(Rin.rho), gamma);
}

template <class T>
__host__ __device__ __forceinline__ bool resolved(T value, T scale) {
  return fin(value) && qabs(value) > T(64) * Lim<T>::eps * (scale + Lim<T>::tiny);
}

// HLLD (Miyoshi & Kusano 2005) in the reference's operation order
// (include/quasar/numerics/hlld_core.hpp:213).  Every exit to the HLL flux goes
// through one call site and every physical flux through one evaluation, so the
// four solves a face makes stay small enough for the instruction cache; each
// outcome is computed by the same operations as a solver written with early
// returns.
template <class T>
__host__ __device__ __forceinline__ St<T> hlld_flux(const St<T>& Lin, const St<T>& Rin, T irL, T irR, T gamma) {
  const T gm1 = gamma - T(1);
  const bool equal = Lin.rho == Rin.rho && Lin.mx == Rin.mx && Lin.my == Rin.my && Lin.mz == Rin.mz &&
                     Lin.en == Rin.en && Lin.bx == Rin.bx && Lin.by == Rin.by && Lin.bz == Rin.bz;
  if (equal) return phys_flux_of(Lin, irL, pressure_ir(Lin, irL, gm1));
  const T bn = T(0.5) * (Lin.bx + Rin.bx);
  St<T> L = Lin, R = Rin;
  const T hbn2 = T(0.5) * bn * bn;
  L.en = (L.en - T(0.5) * L.bx * L.bx) + hbn2;
  R.en = (R.en - T(0.5) * R.bx * R.bx) + hbn2;
  L.bx = bn;
  R.bx = bn;
  const T bn2 = T(2) * hbn2;
  const T vxL = L.mx * irL, vyL = L.my * irL, vzL = L.mz * irL;
  const T vxR = R.mx * irR, vyR = R.my * irR, vzR = R.mz * irR;
  const T pL = pressure_ir(L, irL, gm1), pR = pressure_ir(R, irR, gm1);
  const T ptL = pL + half_sq(L.bx, L.by, L.bz);
  const T ptR = pR + half_sq(R.bx, R.by, R.bz);
  const T cfL = fast_speed_x_ir(irL, pL, L.bx, L.by, L.bz, gamma);
  const T cfR = fast_speed_x_ir(irR, pR, R.bx, R.by, R.bz, gamma);
  const T cfmax = cfL > cfR ? cfL : cfR;
  const T sl = (vxL < vxR ? vxL : vxR) - cfmax;
  const T sr = (vxL > vxR ? vxL : vxR) + cfmax;

  // The fan: true with `f` set, false for the HLL flux.  Supersonic faces take
  // the upwind physical flux (f = F(U), region coefficients zero).
  St<T> f;
  auto fan = [&]() -> bool {
    const bool supersonic = sl >= T(0) || sr <= T(0);
    bool left = sl >= T(0);
    // Set on every path that reads them (not supersonic; uss and sa only in
    // the inner regions), so they start unset rather than as zero moves.
    T s, sa;
    St<T> us, uss;
    bool inner = false, negligible = false;
    if (!supersonic) {
      if (!fin(bn2) || !fin(ptL) || !fin(ptR)) return false;
      const T aR = (sr - vxR) * R.rho;
      const T aL = (sl - vxL) * L.rho;
      const T denomM = aR - aL;
      if (!resolved(denomM, qabs(aR) + qabs(aL))) return false;
      const T inv_dM = frcp(denomM);
      const T sm = (aR * vxR - aL * vxL - ptR + ptL) * inv_dM;
      if (!fin(sm)) return false;
      const T pts = (aR * ptL - aL * ptR + aL * aR * (vxR - vxL)) * inv_dM;
      if (!fin(pts)) return false;
      const T dLs = sl - sm, dRs = sr - sm;
      const T wave_scale = qabs(sl) + qabs(sr) + qabs(sm);
      if (!resolved(dLs, wave_scale) || !resolved(dRs, wave_scale)) return false;
      const T idLs = frcp(dLs), idRs = frcp(dRs);
      const T rhoLs = aL * idLs;
      const T rhoRs = aR * idRs;
      if (!(rhoLs > T(0)) || !(rhoRs > T(0))) return false;

      // Single-star states.
      T vyLs, vzLs, byLs, bzLs, eLs, vyRs, vzRs, byRs, bzRs, eRs;
      {
        const T smv = sl - vxL;
        const T q = L.rho * smv * dLs;
        const T den = q - bn2;
        if (!resolved(den, qabs(q) + bn2)) return false;
        const T id = frcp(den);
        const T fac = bn * (sm - vxL) * id;
        vyLs = vyL - L.by * fac;
        vzLs = vzL - L.bz * fac;
        const T bc = (L.rho * smv * smv - bn2) * id;
        byLs = L.by * bc;
        bzLs = L.bz * bc;
        const T vdb = vxL * L.bx + vyL * L.by + vzL * L.bz;
        const T vdbs = sm * bn + vyLs * byLs + vzLs * bzLs;
        eLs = (smv * L.en - ptL * vxL + pts * sm + bn * (vdb - vdbs)) * idLs;
      }
      {
        const T smv = sr - vxR;
        const T q = R.rho * smv * dRs;
        const T den = q - bn2;
        if (!resolved(den, qabs(q) + bn2)) return false;
        const T id = frcp(den);
        const T fac = bn * (sm - vxR) * id;
        vyRs = vyR - R.by * fac;
        vzRs = vzR - R.bz * fac;
        const T bc = (R.rho * smv * smv - bn2) * id;
        byRs = R.by * bc;
        bzRs = R.bz * bc;
        const T vdb = vxR * R.bx + vyR * R.by + vzR * R.bz;
        const T vdbs = sm * bn + vyRs * byRs + vzRs * bzRs;
        eRs = (smv * R.en - ptR * vxR + pts * sm + bn * (vdb - vdbs)) * idRs;
      }
      const T sqL = fsqrt(rhoLs), sqR = fsqrt(rhoRs);
      const T abn = qabs(bn);
      const T saL = sm - fdiv(abn, sqL);
      const T saR = sm + fdiv(abn, sqR);
      negligible = bn2 <= T(64) * Lim<T>::eps * (qabs(pts) + qabs(ptL) + qabs(ptR) + Lim<T>::tiny);
      if (negligible)
        left = sl <= T(0) && T(0) <= sm;
      else if (T(0) <= saL || !(T(0) <= saR))
        left = T(0) <= saL;  // outer regions: F*_{L,R} = F_{L,R} + S_{L,R} (U* - U)
      else {
        inner = true;
        left = T(0) <= sm;
      }
      const St<T> usL{rhoLs, rhoLs * sm, rhoLs * vyLs, rhoLs * vzLs, eLs, bn, byLs, bzLs};
      const St<T> usR{rhoRs, rhoRs * sm, rhoRs * vyRs, rhoRs * vzRs, eRs, bn, byRs, bzRs};
      us = left ? usL : usR;
      s = left ? sl : sr;
      if (inner) {
        const T inv_sum = frcp(sqL + sqR);
        const T sg = bn >= T(0) ? T(1) : T(-1);
        const T vyss = (sqL * vyLs + sqR * vyRs + (byRs - byLs) * sg) * inv_sum;
        const T vzss = (sqL * vzLs + sqR * vzRs + (bzRs - bzLs) * sg) * inv_sum;
        const T byss = (sqL * byRs + sqR * byLs + sqL * sqR * (vyRs - vyLs) * sg) * inv_sum;
        const T bzss = (sqL * bzRs + sqR * bzLs + sqL * sqR * (vzRs - vzLs) * sg) * inv_sum;
        const T vdbss = sm * bn + vyss * byss + vzss * bzss;
        sa = left ? saL : saR;
        const T sq = left ? sqL : sqR;
        const T vys = left ? vyLs : vyRs, vzs = left ? vzLs : vzRs;
        const T bys = left ? byLs : byRs, bzs = left ? bzLs : bzRs;
        const T vdbs = sm * bn + vys * bys + vzs * bzs;
        const T side = left ? T(-1) : T(1);
        uss = St<T>{us.rho, us.rho * sm, us.rho * vyss, us.rho * vzss,
                    us.en + side * sq * sg * (vdbs - vdbss), bn, byss, bzss};
      }
    }
    const St<T>& U = left ? L : R;
    const St<T> fU = phys_flux_of(U, left ? irL : irR, left ? pL : pR);
    if (supersonic) {
      f = fU;
      return true;
    }
    if (inner) {
#pragma unroll
      for (int c = 0; c < 8; ++c)
        set_comp(f, c, comp(fU, c) + sa * (comp(uss, c) - comp(us, c)) + s * (comp(us, c) - comp(U, c)));
    } else {
#pragma unroll
      for (int c = 0; c < 8; ++c) set_comp(f, c, comp(fU, c) + s * (comp(us, c) - comp(U, c)));
    }
    f.bx = T(0);
    if (negligible) return fin(f.rho) && fin(f.en);
    return fin(f.rho) && fin(f.mx) && fin(f.my) && fin(f.mz) && fin(f.en) && fin(f.by) && fin(f.bz);
  };
  if (fan()) return f;
  return hll_combine(L, R, phys_flux_of(L, irL, pL), phys_flux_of(R, irR, pR), sl, sr);
}

template <class T>
__host__ __device__ __forceinline__ St<T> hlld_flux(const St<T>& Lin, const St<T>& Rin, T gamma) {
  return hlld_flux(Lin, Rin, frcp(Lin.rho), frcp(Rin.rho), gamma);
}

// ---------------------------------------------------------------------------
// Transverse Gauss-Legendre rows (3 points for MP5, 4 for MP7) and the
// recovery weights from 5/7 neighbouring face averages.
struct QuadRows {
  double mp5_point[3][5];
  double mp5_gauss[3];
  double mp7_point[4][7];
  double mp7_gauss[4];
  // The point rows as weights of the neighbour differences s[m+1] - s[m]
  // about the centre sample, and the running-mean weights of the Gauss
  // average, w_q / (w_0 + .. + w_q); in FP64 and rounded to FP32.
  double mp5_step[3][4], mp5_mean[3], mp7_step[4][6], mp7_mean[4];
  float mp5_step_f[3][4], mp5_mean_f[3], mp7_step_f[4][6], mp7_mean_f[4];
};

}  // namespace qmhd

// Host build of the face functions of the step kernels (quasar_amd/csrc/
// qmhd_recon.hpp, qmhd_face.hpp): basis decisions, whole reconstructed faces,
// face fluxes and rates, state by state on the CPU.
#include "../../quasar_amd/csrc/qmhd_recon.hpp"

using namespace qmhd;

// The reference's test of L R = I, every row and column formed by itself.
template <class T>
static bool usable_plainly(const CharBasis<T>& B) {
#pragma clang fp contract(off)
  for (int i = 0; i < 7; ++i)
    for (int j = 0; j < 7; ++j) {
      T r[7], l[7], col[7], row[7];
      basis_rows(B, i, r, l);
      basis_lrow(B, l, row);
      basis_rows(B, j, r, l);
      basis_rcol(B, r, col);
      T dot = row[0] * col[0];
      for (int k = 1; k < 7; ++k) dot = dot + row[k] * col[k];
      if (!fin(dot) || qabs(dot - T(i == j ? 1 : 0)) > T(1024) * Lim<T>::eps) return false;
    }
  return true;
}

// Per state of s8 (n rows of rho, mx, my, mz, E, bx, by, bz): bit 0 the closed
// forms stand, bit 1 the basis counts as usable without its test, bit 2 the
// reference-ordered test finds it usable, bit 3 that test without shared
// products does.
template <class T>
static void decisions(long n, const double* s8, double gamma, int32_t* out) {
  for (long t = 0; t < n; ++t) {
    St<T> s;
    for (int c = 0; c < 8; ++c) set_comp(s, c, T(s8[8 * t + c]));
    WaveBasis<T> w;
    bool conditioned;
    const bool quick = basis_quick(s, T(gamma), w, conditioned);
    CharBasis<T> B;
    basis_scalars(s, T(gamma), B);
    out[t] = (quick ? 1 : 0) | (conditioned ? 2 : 0) | (basis_usable(B) ? 4 : 0) | (usable_plainly(B) ? 8 : 0);
  }
}

// Fluxes and signal speeds of n faces: s holds 16 planes (L, R) by the 2 H + 1
// face averages along the face line (one average for orders without nodes).
template <class T, int ORDER, bool LF>
static void fluxes(long n, const double* s, int dir, T gamma, double* flux, double* rate) {
  constexpr int H = ORDER == 7 ? 3 : ORDER == 5 ? 2 : 0, W = 2 * H + 1;
  QuadRows rows;
  build_quad_rows(rows);
  for (long t = 0; t < n; ++t) {
    const double* v = s + static_cast<std::size_t>(t) * 16 * W;
    T diff[16][W] = {};
    St<T> l, r;
    for (int c = 0; c < 16; ++c) {
      for (int m = 0; m + 1 < W; ++m) diff[c][m] = T(v[c * W + m + 1]) - T(v[c * W + m]);
      set_comp(c < 8 ? l : r, c % 8, T(v[c * W + H]));
    }
    T speed;
    St<T> f;
    if constexpr (H > 0)
      f = node_flux<T, ORDER, LF>(rows, &diff[0][0], W, 1, l, r, dir, gamma, true, speed);
    else
      f = average_flux<T, LF>(l, r, dir, ORDER, gamma, true, speed);
    for (int c = 0; c < 8; ++c) flux[8 * t + c] = comp(f, c);
    rate[t] = speed;
  }
}

template <class T>
static void fluxes_of(int order, int lf, long n, const double* s, int dir, double gamma, double* flux, double* rate) {
  if (order == 1)
    lf ? fluxes<T, 1, true>(n, s, dir, T(gamma), flux, rate) : fluxes<T, 1, false>(n, s, dir, T(gamma), flux, rate);
  else if (order == 2)
    fluxes<T, 2, false>(n, s, dir, T(gamma), flux, rate);
  else if (order == 5)
    fluxes<T, 5, false>(n, s, dir, T(gamma), flux, rate);
  else
    fluxes<T, 7, false>(n, s, dir, T(gamma), flux, rate);
}

template <class T, int ORDER>
static void mp_faces(long n, const double* cells, const double* bn, double gamma, double* out16, int32_t* settled) {
  for (long t = 0; t < n; ++t) {
    St<T> l, r;
    const double* v = cells + static_cast<std::size_t>(t) * 8 * (ORDER + 1);
    auto cell = [&](int c, int q) { return T(v[c * (ORDER + 1) + q]); };
    settled[t] = mp_face<T, ORDER>(cell, T(bn[t]), T(gamma), l, r);
    for (int c = 0; c < 8; ++c) {
      out16[16 * t + c] = comp(l, c);
      out16[16 * t + 8 + c] = comp(r, c);
    }
  }
}

// The rows and points of the cell E_z kernel: x values at a node, then y values,
// each a centre and weighted neighbour differences, E_z by running means.
template <class T, int ORDER>
static void cell_ezs(long n, const double* s, double* ez, int32_t* ok) {
  using R = NodeRows<T, ORDER>;
  constexpr int W = R::NM + 1, H = W / 2;
  QuadRows rows;
  build_quad_rows(rows);
  for (long t = 0; t < n; ++t) {
    const double* v = s + static_cast<std::size_t>(t) * 8 * W * W;
    T whole = T(0);
    ok[t] = 1;
    for (int qx = 0; qx < R::NQ; ++qx) {
      T mean = T(0);
      for (int qy = 0; qy < R::NQ; ++qy) {
        PointEz<T> pt;
        for (int c = 0; c < 8; ++c) {
          T column[W];
          for (int y = 0; y < W; ++y) {
            const double* row = v + (c * W + y) * W;
            column[y] = T(row[H]);
            for (int m = 0; m + 1 < W; ++m) column[y] = fm(R::step(rows, qx, m), T(row[m + 1]) - T(row[m]), column[y]);
          }
          T p = column[H];
          for (int m = 0; m + 1 < W; ++m) p = fm(R::step(rows, qy, m), column[m + 1] - column[m], p);
          pt.take(c, p);
        }
        if (!pt.sure()) ok[t] = 0;
        mean = qy == 0 ? pt.ez : fm(R::mean(rows, qy), pt.ez - mean, mean);
      }
      whole = qx == 0 ? mean : fm(R::mean(rows, qx), mean - whole, whole);
    }
    ez[t] = whole;
  }
}

extern "C" {

void fk_fluxes(int fp32, int order, int lf, long n, const double* s, int dir, double gamma, double* flux, double* rate) {
  if (fp32)
    fluxes_of<float>(order, lf, n, s, dir, gamma, flux, rate);
  else
    fluxes_of<double>(order, lf, n, s, dir, gamma, flux, rate);
}

void fk_basis_decisions(int fp32, long n, const double* s8, double gamma, int32_t* out) {
  if (fp32)
    decisions<float>(n, s8, gamma, out);
  else
    decisions<double>(n, s8, gamma, out);
}

// One face per row of `cells` (8 components x order + 1 cells, in the frame of
// the normal); out16 the left and right states, settled whether they stand.
void fk_mp_faces(int order, long n, const double* cells, const double* bn, double gamma, double* out16,
                 int32_t* settled) {
  order == 5 ? mp_faces<double, 5>(n, cells, bn, gamma, out16, settled)
             : mp_faces<double, 7>(n, cells, bn, gamma, out16, settled);
}
void fk_mp_faces_fp32(int order, long n, const double* cells, const double* bn, double gamma, double* out16,
                      int32_t* settled) {
  order == 5 ? mp_faces<float, 5>(n, cells, bn, gamma, out16, settled)
             : mp_faces<float, 7>(n, cells, bn, gamma, out16, settled);
}

// Cell E_z of n cells by the kernel's quadrature: 8 planes by W x W averages
// each (rows, then columns); ok where every point is certainly admissible.
void fk_cell_ez(int order, long n, const double* s, double* ez, int32_t* ok) {
  order == 5 ? cell_ezs<double, 5>(n, s, ez, ok) : cell_ezs<double, 7>(n, s, ez, ok);
}

// The energy's sum when a state takes its face's normal field: the reconstruction's
// (with whether it is certain) and the correctly rounded one.
void fk_sum_of_three(long n, const double* abc, double* sum, int32_t* sure, double* exact) {
  for (long t = 0; t < n; ++t) {
    sure[t] = sum_of_three(abc[3 * t], abc[3 * t + 1], abc[3 * t + 2], sum[t]);
    exact[t] = cr_sum<3>(abc + 3 * t);
  }
}

// Edge values of n rows of order + 1 averages.
void fk_edge_interp(int order, long n, const double* e, double* out) {
  for (long t = 0; t < n; ++t) out[t] = edge_interp(order, e + t * (order + 1));
}

}  // extern "C"

// Host build of the face functions of the MP5/MP7 path (quasar_amd/csrc/
// qmhd_recon.hpp): its basis decisions and whole faces, state by state on the
// CPU.
#include "../../quasar_amd/csrc/qmhd_recon.hpp"

using namespace qmhd;

// Per state of s8 (n rows of rho, mx, my, mz, E, bx, by, bz): bit 0 the closed
// forms stand, bit 1 the basis counts as usable without its test, bit 2 the
// reference-ordered test finds it usable.
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
    out[t] = (quick ? 1 : 0) | (conditioned ? 2 : 0) | (basis_usable(B) ? 4 : 0);
  }
}

extern "C" {

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
  for (long t = 0; t < n; ++t) {
    St<double> l, r;
    const double* v = cells + static_cast<std::size_t>(t) * 8 * (order + 1);
    auto cell = [&](int c, int q) { return v[c * (order + 1) + q]; };
    settled[t] = order == 5 ? mp_face<double, 5>(cell, bn[t], gamma, l, r) : mp_face<double, 7>(cell, bn[t], gamma, l, r);
    for (int c = 0; c < 8; ++c) {
      out16[16 * t + c] = comp(l, c);
      out16[16 * t + 8 + c] = comp(r, c);
    }
  }
}

}  // extern "C"

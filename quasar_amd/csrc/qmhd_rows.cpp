// Host construction of the quadrature tables used by the stencil code:
// transverse point-value rows and Gauss weights of the MP5/MP7 face quadrature
// (include/quasar/numerics/finite_volume_quadrature.hpp:12-68).
#include "qmhd_kernels.hpp"

namespace qmhd {

// step[m]: weight of s[m+1] - s[m] in the row's value less the centre sample:
// the weights beyond the difference on the right of the centre, minus those
// before it on the left.
template <int N>
static void difference_row(const double* w, double* step, float* step_f) {
  constexpr int H = N / 2;
  for (int m = 0; m < N - 1; ++m) {
    long double sum = 0.0L;
    if (m >= H)
      for (int t = m + 1; t < N; ++t) sum += w[t];
    else
      for (int t = 0; t <= m; ++t) sum -= w[t];
    step[m] = static_cast<double>(sum);
    step_f[m] = static_cast<float>(sum);
  }
}

static void mean_row(const double* w, int n, double* mean, float* mean_f) {
  long double sum = 0.0L;
  for (int q = 0; q < n; ++q) {
    sum += w[q];
    mean[q] = static_cast<double>(w[q] / sum);
    mean_f[q] = static_cast<float>(w[q] / sum);
  }
}

void build_quad_rows(QuadRows& r) {
  const double p5[3][5] = {{-0.0392523473402346598, 0.312987195324173573, 0.910833333333333384,
                            -0.216320528657506839, 0.0317523473402346601},
                           {0.00468749999999999983, -0.0604166666666666671, 1.11145833333333344,
                            -0.0604166666666666671, 0.00468749999999999983},
                           {0.0317523473402346601, -0.216320528657506839, 0.910833333333333384,
                            0.312987195324173573, -0.0392523473402346598}};
  const double p7[4][7] = {{0.00860109764472105458, -0.0796691475531970394, 0.415576982717296983,
                            0.849155569794037945, -0.245805403605616202, 0.0591434746546156687,
                            -0.0070025736518584264},
                           {0.00327670662777140203, -0.0266359260617751309, 0.0928282644451935562,
                            1.08046056237311472, -0.183384586025290314, 0.0375843394851378479,
                            -0.00412936084415200903},
                           {-0.00412936084415200903, 0.0375843394851378479, -0.183384586025290314,
                            1.08046056237311472, 0.0928282644451935562, -0.0266359260617751309,
                            0.00327670662777140203},
                           {-0.0070025736518584264, 0.0591434746546156687, -0.245805403605616202,
                            0.849155569794037945, 0.415576982717296983, -0.0796691475531970394,
                            0.00860109764472105458}};
  for (int q = 0; q < 3; ++q)
    for (int t = 0; t < 5; ++t) r.mp5_point[q][t] = p5[q][t];
  for (int q = 0; q < 4; ++q)
    for (int t = 0; t < 7; ++t) r.mp7_point[q][t] = p7[q][t];
  r.mp5_gauss[0] = 5.0 / 18.0;
  r.mp5_gauss[1] = 4.0 / 9.0;
  r.mp5_gauss[2] = 5.0 / 18.0;
  r.mp7_gauss[0] = 0.173927422568726925;
  r.mp7_gauss[1] = 0.326072577431273103;
  r.mp7_gauss[2] = 0.326072577431273103;
  r.mp7_gauss[3] = 0.173927422568726925;
  for (int q = 0; q < 3; ++q) difference_row<5>(r.mp5_point[q], r.mp5_step[q], r.mp5_step_f[q]);
  for (int q = 0; q < 4; ++q) difference_row<7>(r.mp7_point[q], r.mp7_step[q], r.mp7_step_f[q]);
  mean_row(r.mp5_gauss, 3, r.mp5_mean, r.mp5_mean_f);
  mean_row(r.mp7_gauss, 4, r.mp7_mean, r.mp7_mean_f);
}

}  // namespace qmhd

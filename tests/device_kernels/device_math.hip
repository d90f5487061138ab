// The device forms of the face solver's root and reciprocal
// (quasar_amd/csrc/qmhd_face.hpp), value by value, for the tests.
#include "../../quasar_amd/csrc/qmhd_face.hpp"

using namespace qmhd;

template <class T>
__global__ void roots(long n, const T* __restrict__ x, T* __restrict__ root, T* __restrict__ half_inv,
                      T* __restrict__ inv) {
  const long k = blockIdx.x * 256L + threadIdx.x;
  if (k >= n) return;
  T h;
  root[k] = sqrt_pos(x[k], h);
  half_inv[k] = h;
  inv[k] = rcp_near(x[k]);
}

// root, half_inv, inv (n values each, device memory) of x; 0 when launched.
extern "C" int dm_roots(int fp32, long n, const void* x, void* root, void* half_inv, void* inv) {
  const dim3 grid(static_cast<unsigned>((n + 255) / 256));
  if (fp32)
    hipLaunchKernelGGL(roots<float>, grid, dim3(256), 0, nullptr, n, static_cast<const float*>(x),
                       static_cast<float*>(root), static_cast<float*>(half_inv), static_cast<float*>(inv));
  else
    hipLaunchKernelGGL(roots<double>, grid, dim3(256), 0, nullptr, n, static_cast<const double*>(x),
                       static_cast<double*>(root), static_cast<double*>(half_inv), static_cast<double*>(inv));
  return hipDeviceSynchronize() == hipSuccess ? 0 : 1;
}

// Device data views and host launchers for the MHD step kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "qmhd_numerics.hpp"

namespace qmhd {

struct GridD {
  int nx, ny, ng, pitch;
  double dx, dy, ox, oy, lx, ly;
};

struct Flags4 {
  int side[4];
};

struct StateView {
  const double* c[8];
};
struct StateOut {
  double* c[8];
};
template <class T>
struct IfaceView {
  T* c[16];
};
template <class T>
struct FluxView {
  T* c[8];
};

// Device-resident per-step status, reduced with order-independent atomics on
// the bit patterns of non-negative doubles.  The first 128 bytes (one cache
// line of the L2) are what the checks and reductions of a launch update; the
// face-list counters, which a launch's first block clears with plain stores,
// have the next line to themselves.
struct alignas(128) StepStatus {
  unsigned long long theta[4];     // per-stage admissible fraction (min); [3] = stage 2, second collocation
  unsigned long long live_theta0;  // live state, high-order collocation (min)
  unsigned long long live_theta1;  // live state, two-face collocation (min)
  unsigned long long divb_residual;  // max unexplained |div B| (relative check)
  unsigned long long divb_scale;     // max directional scale
  unsigned long long max_rate;       // CFL additive rate (max)
  double dt;                         // device-side dt of the auto-dt loop
  double time;                       // accumulated simulated time
  unsigned long long owned;          // batched steps: the live state is one the solver made (see prep_kernel)
  // Faces listed for the general path (x, y), and again (x, y); see FaceOut.
  alignas(128) unsigned long long lists[4];
};

struct IcSpecD {
  int kind;
  double gamma, magnetic_scale, interface_x;
  double left[8], right[8];
  double rho, pressure, b0, total_b0, amplitude;
  long long wavenumber;
  double magnetic_velocity_scale;
  double b_uniform[3];
  double center[2];
  double r_in, r0, r1, rho_in, rho_out, p_in, p_out, p_core, p_ambient, rho_ambient, u0;
  double ot_rho, ot_p, noise_amplitude;
  unsigned long long noise_seed;
  double blob_half;
};

// launch_prep's solver_owned: the solver made the live state (1), a caller
// seeded it (0), or status.owned says which: a captured step is replayed on
// states of both kinds.
constexpr int kOwnedByStatus = -1;

// Why a batched run stopped (acc[6] of launch_batch_commit; acc[7] the value
// that failed).
enum BatchStop { kStopNone, kStopDivergence, kStopInadmissible, kStopRate };

hipError_t upload_quad_rows(const QuadRows& rows);
void build_quad_rows(QuadRows& rows);

// Launchers (all asynchronous on `stream`).
void launch_prep(const GridD& g, const StateView& u, double* bxc, double* byc, const StateView& base,
                 const double* base_bxc, const double* base_byc, int theta_slot, int theta_co, int theta_both,
                 int live_checks, int solver_owned, StepStatus* status, hipStream_t stream, bool exact = true);
void launch_collocate(const GridD& g, int axis, int co, const double* face, double* cell, hipStream_t stream);
// The face-level launchers are instantiated for T = double (the FP64 form)
// and T = float (the FP32 form: interface states, fluxes and their arithmetic
// in FP32; state, collocation, cell/corner E_z, rates and the update in FP64).
// A counted face list; the count is zero before the launch that fills it.
struct FaceList {
  unsigned long long* count;
  unsigned long long* faces;
};
// One face direction's planes: interface states, L == R flags, fluxes and rates
// (null: no signal speeds wanted), the faces left to the general path and, in
// the learned form, the listed faces left to it.
template <class T>
struct FaceOut {
  IfaceView<T> states;
  int* eq;
  FluxView<T> flux;
  double* rate;
  FaceList list, redo;
};
// Both directions (first 0, count 2) or one (count 1) in one launch each of the
// faces and of the fallback.
template <class T>
void launch_reconstruct(const GridD& g, int order, double gamma, const Flags4& flags, const StateView& u,
                        const double* bxc, const double* byc, const FaceOut<T>* out, int first, int count,
                        hipStream_t stream);
// Zeroes `n` counters (at most 64).
void launch_counter_reset(unsigned long long* counters, int n, hipStream_t stream);
// Learned form (orders 5 and 7), both directions: cheap faces where the
// indicator left both cells unflagged, the plain path over the lists of the
// others; adds the listed counts to *plain_total when given.  The flux launch
// takes the listed faces (the cheap reconstruction stores every other face's
// flux and rate itself).
template <class T>
void launch_flux_learned(const GridD& g, int order, const Flags4& flags, double gamma, const FaceOut<T>* face,
                         const uint8_t* cell_flags, hipStream_t stream, int list_blocks);
template <class T>
void launch_reconstruct_learned(const GridD& g, int order, double gamma, const Flags4& flags, const StateView& u,
                                const double* bxc, const double* byc, const uint8_t* cell_flags,
                                const FaceOut<T>* out, unsigned long long* plain_total, hipStream_t stream,
                                int list_blocks, int cheap_tile);
// `block` shapes the orders without transverse quadrature (MP5/MP7 take their
// LDS tile).
template <class T>
void launch_flux(const GridD& g, int order, int hll_only, const Flags4& flags, double gamma, const FaceOut<T>* face,
                 int first, int count, hipStream_t stream, dim3 block = dim3(64, 4));
void launch_cfl_reduce(const GridD& g, const double* rate_x, const double* rate_y, unsigned long long* max_rate,
                       hipStream_t stream);
// MP5/MP7 cell E_z: `tile` selects the LDS tile, 0: 16x16, 1: 32x8, 2: 8x32
// cells per block.  MP5/MP7 corners: `tiled` selects the 16x16 LDS-tile kernel,
// otherwise one thread per corner in `block`-shaped blocks.  Learned
// reconstruction: `cheap_tile` selects the cheap faces' tile, 0: 64x4, 1: 32x8,
// 2: 128x2, 3: 16x16, 4: 8x32 cells per block.
template <class T>
void launch_cell_emf(const GridD& g, int order, const Flags4& flags, double gamma, const StateView& u,
                     const double* bxc, const double* byc, double* cell_ez, hipStream_t stream,
                     const uint8_t* cell_flags = nullptr, int tile = 0);
template <class T>
void launch_corner(const GridD& g, int order, const Flags4& flags, const FluxView<T>& fx, const FluxView<T>& fy,
                   const double* cell_ez, const int* eqx, const int* eqy, double* ez, hipStream_t stream,
                   dim3 block = dim3(64, 4), bool tiled = true);
template <class T>
void launch_update(const GridD& g, double a, double b, double cw, const double* dt_dev, const StateView& un,
                   const StateView& us, const FluxView<T>& fx, const FluxView<T>& fy, const double* ez,
                   const StateOut& out, hipStream_t stream, dim3 block = dim3(64, 4));
void launch_rk_combine(const GridD& g, double a, double b, double c, const StateView& un, const StateView& us,
                       const StateView& dudt, const StateOut& out, hipStream_t stream);
void launch_ghosts(const GridD& g, const Flags4& fluid, const Flags4& field, const StateOut& u, hipStream_t stream);
void launch_dt(const unsigned long long* max_rate_bits, double effective_cfl, double dx, double dy, double* dt_out,
               double* t_accum, hipStream_t stream);
void launch_seed(const GridD& g, const IcSpecD& s, const StateOut& out, double* raw_mag, int* status,
                 hipStream_t stream);
void launch_divb_linf(const GridD& g, const StateView& u, unsigned long long* out, hipStream_t stream);
void launch_theta(const GridD& g, const StateView& base, const StateView& cand, int co, unsigned long long* out,
                  hipStream_t stream);
void launch_cell_sums(const GridD& g, const StateView& u, double* partials, int blocks, hipStream_t stream);
void launch_eq_flags(const GridD& g, int dir, const IfaceView<double>& in, int* eq, hipStream_t stream);
void launch_flux_difference(const GridD& g, int dir, const FluxView<double>& f, const StateOut& d,
                            hipStream_t stream);
void launch_curl(const GridD& g, const double* ez, double* dbx, double* dby, hipStream_t stream);
void launch_status_reset(StepStatus* s, hipStream_t stream);
// Device-side step commit of the batched launcher: acc[0] accepted steps,
// acc[1] rejected steps, acc[2] fatal (live state invalid), acc[3] simulated
// time, acc[4] the decision of the last step (1 accepted), acc[5] held (a step
// was rejected; later attempts commit nothing until the host clears it).
// Unless the step was accepted, the restore launch copies the live state over
// the candidate, so the next step (which reads the candidate register) starts
// again from the same state.
void launch_batch_commit(StepStatus* status, double* acc, hipStream_t stream);
void launch_batch_restore(const GridD& g, const double* acc, const StateView& live, const StateOut& cand,
                          hipStream_t stream);

// Learned form: troubled-cell indicator network (parameters: FP32 vector of
// mlp::kParams; packed: BF16 MFMA operands from launch_mlp_pack), training
// kernels, features and labels.
void launch_mlp_pack(const float* params, uint16_t* packed, hipStream_t stream);
void launch_mlp_forward(const uint16_t* packed, const float* params, const float* x, long long n, float* logits,
                        hipStream_t stream);
long long mlp_grad_waves(long long n, int chunks);
// grad receives mlp::kParams gradient entries and the loss; partial holds
// mlp_grad_waves(n, chunks) rounded up to 4 rows of mlp::kParams + 1 floats.
void launch_mlp_grad(const uint16_t* packed, const float* params, const float* x, const float* target,
                     const float* weight, const long long* order, long long n, int chunks, float* partial,
                     float* grad, hipStream_t stream);
void launch_mlp_adam(float* params, const float* grad, float* m, float* v, long long step, float lr, float beta1,
                     float beta2, float eps, hipStream_t stream);
void launch_features(const GridD& g, double gamma, const StateView& u, const double* bxc, const double* byc,
                     float* out, hipStream_t stream);
void launch_indicator(const GridD& g, double gamma, const StateView& u, const double* bxc, const double* byc,
                      const uint16_t* packed, const float* params, float threshold, uint8_t* flags,
                      hipStream_t stream);
void launch_labels(const GridD& g, int order, const Flags4& flags, double gamma, const StateView& u,
                   const double* bxc, const double* byc, double label_tol, uint8_t* fx, uint8_t* fy, uint8_t* cell,
                   hipStream_t stream);

}  // namespace qmhd

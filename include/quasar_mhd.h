/* quasar_mhd.h — C ABI of the MI355X (gfx950) implementation of quasar's 2D
 * constrained-transport ideal-MHD step.
 *
 * Two layers, both plain C: pointers, sizes and status codes, no exceptions
 * and no framework types cross it.
 *
 *  1. Launch level: one entry point per operation of the reference launch ABI
 *     (include/quasar/physics/mhd/kernels.hpp, the launch_mhd_* family).
 *     Buffers are caller-owned device arrays of `qmhd_grid_storage(g)` doubles
 *     in the reference's padded Grid2D layout, index (i+ng) + (nx+2ng)*(j+ng);
 *     a state is 8 planes in the order rho, mx, my, mz, energy, bx_face,
 *     by_face, bz_cell; interface states are 16 planes (L then R).  Work
 *     memory is caller-owned too: `scratch` must hold
 *     qmhd_scratch_doubles(g) doubles.  `stream` is a hipStream_t (NULL = the
 *     default stream); calls are stream ordered, and those that return a host
 *     scalar synchronize that stream.
 *
 *  2. Solver level: an opaque handle with the seed / cfl_limit / step /
 *     readback surface of quasar::mhd::MhdSolver2D
 *     (include/quasar/physics/mhd/mhd_solver.hpp:85-173) that the pybind
 *     module _core.mhd exposes (bindings/python/bind_mhd.cpp:571-646).
 *
 * Status codes: QMHD_OK, QMHD_EINVAL (the reference throws
 * std::invalid_argument), QMHD_ERUNTIME (std::runtime_error), QMHD_EHIP (a HIP
 * runtime error; the reference throws backend::DeviceError).
 * qmhd_last_error() returns the message of the calling thread's last failure.
 */
#ifndef QUASAR_MHD_H
#define QUASAR_MHD_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

enum { QMHD_OK = 0, QMHD_EINVAL = 1, QMHD_ERUNTIME = 2, QMHD_EHIP = 3 };

/* Side boundary modes (kernels.hpp:43-51): 0 periodic, 1 outflow, 2 wall,
 * 3 axis, 4 internal.  Side order x_lo, x_hi, y_lo, y_hi. */

/* Mirrors quasar::Grid2D (include/quasar/core/grid.hpp:84-200). */
typedef struct {
  int32_t nx, ny, ng, reserved;
  double lx, ly, origin_x, origin_y, cell_dx, cell_dy;
} qmhd_grid;

/* Mirrors quasar::mhd::MhdInitialConditionSpec
 * (include/quasar/physics/mhd/initial_conditions.hpp:62-124), kind 0 brio_wu,
 * 1 alfven_wave, 2 orszag_tang, 3 blast, 4 rotor, 5 confined_blob (square of
 * half-width blob_half about `center`).  Extensions: ot_rho/ot_p
 * (Orszag-Tang background density/pressure; 0 keeps gamma^2/gamma) and a
 * seeded Philox-4x32-10 white-noise perturbation of amplitude
 * noise_amplitude on rho (relative), vx and vy. */
typedef struct {
  int32_t kind, reserved;
  double gamma, magnetic_scale, interface_x;
  double left[8], right[8];
  double rho, pressure, b0, total_b0, amplitude;
  int64_t wavenumber;
  double magnetic_velocity_scale;
  double b_uniform[3];
  double center[2];
  double r_in, r0, r1, rho_in, rho_out, p_in, p_out, p_core, p_ambient, rho_ambient, u0;
  double ot_rho, ot_p;
  double noise_amplitude;
  uint64_t noise_seed;
  double blob_half;
} qmhd_ic_spec;

const char* qmhd_last_error(void);
const char* qmhd_version(void);
size_t qmhd_grid_storage(const qmhd_grid* g);
size_t qmhd_scratch_doubles(const qmhd_grid* g);

/* ---- launch level ---------------------------------------------------- */

/* launch_mhd_collocate_face_to_cell (kernels.hpp:735-738): face -> cell
 * average of bx_face (axis 0) or by_face (axis 1); collocation 0 = the
 * high-order rule of the grid's halo, 1 = the two-face average. */
int qmhd_collocate_face_to_cell(const qmhd_grid* g, int axis, int collocation, const double* face,
                                double* cell, void* stream);

/* launch_mhd_reconstruct (kernels.hpp:162-166): L/R interface states normal to
 * `dir` for order 1 (piecewise constant), 2 (MUSCL), 5 (MP5), 7 (MP7).
 * Writes out16 on dir 0 faces i in [0,nx], j in [-ng, ny+ng) (dir 1
 * transposed).  The reference's `rate_only` flag (passed by
 * MhdSolver2D::cfl_limit, mhd_solver.cpp:1255-1260) selects an admissibility
 * predicate that forwards to the ordinary one (mhd_solver.cpp:1267-1271), so
 * this one entry point serves both values of it. */
int qmhd_reconstruct(const qmhd_grid* g, int dir, int order, const int32_t* flags4, double gamma,
                     const double* const* u8, double* const* out16, double* scratch, void* stream);

/* launch_mhd_hlld_flux (kernels.hpp:186-194): transverse-Gauss HLLD face flux
 * (Lax-Friedrichs when hll_only) on faces [0,nx] x [0,ny]. */
int qmhd_hlld_flux(const qmhd_grid* g, int dir, int order, int hll_only, const int32_t* flags4, double gamma,
                   const double* const* in16, double* const* flux8, double* scratch, void* stream);

/* launch_mhd_flux_difference (kernels.hpp:203-205): dudt += -(F(i+1)-F(i))/d. */
int qmhd_flux_difference(const qmhd_grid* g, int dir, const double* const* flux8, double* const* dudt8,
                         void* stream);

/* The derived tables of EmfField2D (mhd_field.hpp:107-144) that the corner
 * E_z reads: the cell-average E_z (cell_ez_average), the directional face
 * fluxes the face EMFs come from (x faces: the By flux, face EMF -F_By;
 * y faces: the Bx flux, face EMF +F_Bx; the reference's xface_ez/yface_ez
 * hold the signed EMF) and the per-face no-jump flags (xface_no_jump /
 * yface_no_jump: 1 where the face's L and R states are equal in every
 * component).  Each is one caller-owned plane of qmhd_grid_storage(g)
 * elements. */
typedef struct {
  double* cell_ez;
  double* xface_flux_by;
  double* yface_flux_bx;
  int32_t* xface_no_jump;
  int32_t* yface_no_jump;
} qmhd_emf_tables;

/* launch_mhd_ct_emf_prepare (kernels.hpp:274-281), called by
 * MhdSolver2D::consume_residual_face_records (mhd_solver.cpp:796-798): the
 * tables above from u and the interface states of both directions.  The face
 * fluxes are the transverse-Gauss HLLD fluxes of qmhd_hlld_flux (the
 * Lax-Friedrichs flux when hll_only, which the solver passes for order 1). */
int qmhd_ct_emf_prepare(const qmhd_grid* g, int order, int hll_only, const int32_t* flags4, double gamma,
                        const double* const* u8, const double* const* ifx16, const double* const* ify16,
                        const qmhd_emf_tables* emf, double* scratch, void* stream);

/* launch_mhd_ct_emf_finish (kernels.hpp:282-285), called by
 * MhdSolver2D::finish_ct_emf (mhd_solver.cpp:801-807): corner E_z on corners
 * [0,nx] x [0,ny] from the prepared tables. */
int qmhd_ct_emf_finish(const qmhd_grid* g, int order, const int32_t* flags4, const qmhd_emf_tables* emf,
                       double* ez_edge, void* stream);

/* launch_mhd_ct_emf (kernels.hpp:286-291): prepare and finish back to back.
 * flux_x8 / flux_y8 are optional: the face fluxes of the same interface
 * states when the caller already has them (the solver's own step reuses its
 * update fluxes), NULL to derive them from ifx16 / ify16 as the reference's
 * launcher does (Lax-Friedrichs for order 1). */
int qmhd_ct_emf(const qmhd_grid* g, int order, const int32_t* flags4, double gamma, const double* const* u8,
                const double* const* ifx16, const double* const* ify16, const double* const* flux_x8,
                const double* const* flux_y8, double* ez_edge, double* scratch, void* stream);

/* launch_mhd_emf_curl_rate (kernels.hpp:307-309): face-B rates from E_z. */
int qmhd_emf_curl_rate(const qmhd_grid* g, const double* ez_edge, double* dbx_face, double* dby_face,
                       void* stream);

/* launch_mhd_rk_stage (kernels.hpp:336-338): out = a un + b us + c dudt on
 * cells and physical faces; (1,0,0) is an exact copy. */
int qmhd_rk_stage(const qmhd_grid* g, double a, double b, double c, const double* const* un8,
                  const double* const* us8, const double* const* dudt8, double* const* out8, void* stream);

/* launch_mhd_fill_ghosts_fluid / _field (kernels.hpp:509-533). */
int qmhd_fill_ghosts(const qmhd_grid* g, const int32_t* fluid_flags4, const int32_t* field_flags4,
                     double* const* u8, void* stream);

/* launch_mhd_cfl_max_rate (kernels.hpp:361-366): maximum additive face rate. */
int qmhd_cfl_max_rate(const qmhd_grid* g, int order, const int32_t* flags4, double gamma,
                      const double* const* ifx16, const double* const* ify16, double* host_rate,
                      double* scratch, void* stream);

/* launch_mhd_admissible_fraction (kernels.hpp:397-414). */
int qmhd_admissible_fraction(const qmhd_grid* g, const double* const* base8, const double* const* cand8,
                             int collocation, double* host_theta, double* scratch, void* stream);

/* launch_mhd_ct_divb_linf / _relative_linf (kernels.hpp:483-495). */
int qmhd_divb_linf(const qmhd_grid* g, const double* const* u8, double* host_linf, double* scratch,
                   void* stream);
int qmhd_divb_relative_linf(const qmhd_grid* g, const double* const* u8, int solver_owned, double* host_ratio,
                            double* scratch, void* stream);

/* launch_mhd_conserved_cell_sums (kernels.hpp:545-558): interior mass and
 * energy totals (compensated device partials, exact host fold). */
int qmhd_conserved_cell_sums(const qmhd_grid* g, const double* const* u8, double* mass, double* energy,
                             double* scratch, void* stream);

/* No counterpart in the reference.  For callers that cannot allocate device
 * memory (code under HIP graph capture, tight serving loops, harnesses that
 * forbid hipMalloc): qmhd_conserved_cell_sums with its per-block partials in a
 * static device workspace of the library instead of caller-owned scratch.
 * The workspace is 64 KiB (1024 blocks x 8 doubles) per GPU, held until the
 * process ends; the reduction strides over the cells, so every grid fits (a
 * request beyond the workspace would be refused with QMHD_EINVAL).  It makes
 * no hipMalloc/hipFree call.  All calls on one GPU share its workspace:
 * calls that overlap on one GPU (other streams or threads) race.  Synchronizes
 * `stream`, like the scratch variant. */
int qmhd_conserved_cell_sums_noalloc(const qmhd_grid* g, const double* const* u8, double* mass, double* energy,
                                     void* stream);

/* launch_mhd_seed_initial_state (kernels.hpp:656-660): analytic IC on every
 * padded cell with the collocated magnetic energy. */
int qmhd_seed_initial_state(const qmhd_grid* g, const qmhd_ic_spec* spec, double* const* out8, double* scratch,
                            void* stream);

/* ---- solver level (MhdSolver2D) ---------------------------------------- */

typedef struct qmhd_solver qmhd_solver;

/* MhdConfig (mhd_solver.hpp:50-83).  Scheme names are the reference's
 * registry strings: reconstruction "muscl_minmod" | "mp5" | "mp7", riemann
 * "hlld", integrator "ssprk3", ct "fd_ct_christlieb", positivity
 * "troubled_cell", boundaries "periodic" | "outflow" | "wall".  grid.ng = 0
 * lets the solver size the halo from the reconstruction. */
typedef struct {
  qmhd_grid grid;
  double gamma, cfl, rho_floor, p_floor;
  char reconstruction[32], riemann[32], integrator[32], ct[32], positivity[32], geometry[32];
  char fluid[4][32];
  char field[4][32];
  /* Extension (no reference counterpart): arithmetic of the face work, "fp64"
   * (default, also "") or "fp32".  In "fp32" the interface states, their
   * reconstruction, the Riemann fluxes and the cell E_z quadrature run in
   * FP32; the state, collocation, positivity recompute, CFL rates and
   * reduction, corner E_z, update and conserved sums stay FP64. */
  char arithmetic[32];
  /* Extension (no reference counterpart): troubled-cell indicator, "" or
   * "none" (the plain method) or "mlp" (the learned form, MP5/MP7 only; the
   * network is set with qmhd_solver_set_indicator before the first step). */
  char indicator[32];
} qmhd_solver_config;

int qmhd_solver_create(const qmhd_solver_config* cfg, qmhd_solver** out);
void qmhd_solver_destroy(qmhd_solver* s);
int qmhd_solver_grid(const qmhd_solver* s, qmhd_grid* out);
/* seed_state / state_component_to_host: component "rho", "mx", "my", "mz",
 * "energy", "bx"/"bx_face", "by"/"by_face", "bz"/"bz_cell"; readback of "bx"
 * and "by" is face->cell collocated, "bx_face"/"by_face" raw. */
int qmhd_solver_seed_state(qmhd_solver* s, const char* component, const double* host, size_t n);
int qmhd_solver_state_to_host(qmhd_solver* s, const char* component, double* host, size_t n);
int qmhd_solver_cfl_limit(qmhd_solver* s, double* dt);
int qmhd_solver_step(qmhd_solver* s, double dt);
int qmhd_solver_step_unchecked(qmhd_solver* s, double dt);
int qmhd_solver_advance(qmhd_solver* s, double t_end, double dt);
int qmhd_solver_divergence_b_max(qmhd_solver* s, double* out);
int qmhd_solver_conserved_cell_totals(qmhd_solver* s, double* mass, double* energy);
int qmhd_solver_last_positivity_substeps(const qmhd_solver* s);
/* Test support, the counterpart of the throwing integrators the reference's
 * tests register (tests/unit/physics/mhd/test_mhd_positivity_preservation.cpp:
 * 56-160): the next step / step_unchecked / advance request fails with
 * QMHD_ERUNTIME on its first attempt issued after `pieces` accepted pieces
 * (0: after a complete three-stage attempt, before it is accepted), rolling
 * the whole request back; pieces < 0 disarms. */
int qmhd_solver_fail_after_pieces(qmhd_solver* s, int pieces);
/* The auto-dt run loop (python/quasar/mhd/cli.py:386-491) with the timestep
 * kept on the device: up to `steps` steps or until t_end (t_end <= 0: no end
 * time), one host synchronization per step.  Returns steps taken and the
 * simulated time. */
int qmhd_solver_run(qmhd_solver* s, int steps, double t_end, int* steps_done, double* sim_time);
/* Device pointer of a live-state plane (0..7), for zero-copy consumers. */
int qmhd_solver_state_plane(qmhd_solver* s, int component, double** device_ptr);

/* Launch timing.  No counterpart in the reference (which has no in-process
 * kernel timing); for benchmark harnesses that need per-kernel durations on
 * the solver's own stream.  While enabled, every launch of the step is
 * bracketed by HIP events; qmhd_solver_kernel_time returns the summed
 * milliseconds and launch count of one kind since enabling.  A ghost fill
 * (its x and y launches) is one interval of kind GHOSTS; REDUCE covers the
 * CFL reduction and the device dt kernel. */
enum {
  QMHD_KERNEL_PREP = 0,
  QMHD_KERNEL_RECONSTRUCT = 1,
  QMHD_KERNEL_FLUX = 2,
  QMHD_KERNEL_CELL_EMF = 3,
  QMHD_KERNEL_CORNER = 4,
  QMHD_KERNEL_UPDATE = 5,
  QMHD_KERNEL_GHOSTS = 6,
  QMHD_KERNEL_REDUCE = 7,
  QMHD_KERNEL_INDICATOR = 8,
  QMHD_KERNEL_KINDS = 9
};
int qmhd_solver_set_profiling(qmhd_solver* s, int enable);
int qmhd_solver_kernel_time(qmhd_solver* s, int kind, double* total_ms, long long* launches);
const char* qmhd_kernel_kind_name(int kind);
/* The solver's HIP stream (hipStream_t), on which all its work is ordered. */
void* qmhd_solver_stream(qmhd_solver* s);
/* Wait for all work issued by the solver (device_synchronize in the
 * reference's compute_residual, src/physics/mhd/mhd_solver.cpp:825). */
int qmhd_solver_synchronize(qmhd_solver* s);

/* ---- learned form (no reference counterpart) -------------------------
 * A per-cell troubled-cell indicator: 100 features (the 5x5 stencil of
 * rho, p, |B|, |v|, each as (Q - Q_centre) / (|Q_centre| + max |Q - Q_centre|))
 * into a 100-32-32-1 ReLU network evaluated with BF16 MFMA and FP32
 * accumulation.  A face whose two cells are unflagged takes the unlimited
 * linear fifth-order face values and the HLL flux; every other face takes the
 * plain MP + HLLD path.  Parameters are one FP32 vector: W1[100][32], b1[32],
 * W2[32][32], b2[32], w3[32], b3. */
#define QMHD_MLP_FEATURES 100
#define QMHD_MLP_HIDDEN 32
#define QMHD_MLP_PARAMS 4321
#define QMHD_MLP_PACKED 5632 /* uint16_t BF16 operands */
/* Label bits of a face (cells: OR of their four faces). */
/* label_tol: relative size above which a limiter change (against the largest
 * component of the face's reference state) or an HLLD-HLL flux gap (against
 * the largest HLLD flux component) counts. */
#define QMHD_LABEL_MP_CLIP 1     /* an MP limiter call changed a face value by more than label_tol */
#define QMHD_LABEL_MUSCL 2       /* MUSCL fallback */
#define QMHD_LABEL_CONSTANT 4    /* piecewise-constant fallback or NaN sentinel */
#define QMHD_LABEL_HLL_GAP 8     /* max|F_HLLD - F_HLL| > label_tol * max|F_HLLD| */

/* BF16 operand layout of the network (run after every parameter change). */
int qmhd_mlp_pack(const float* params, uint16_t* packed, void* stream);
/* Logits of n samples (features: n x 100 FP32, row-major). */
int qmhd_mlp_forward(const uint16_t* packed, const float* params, const float* features, int64_t n, float* logits,
                     void* stream);
/* Floats of the `partial` workspace of qmhd_mlp_gradient. */
size_t qmhd_mlp_partial_floats(int64_t n, int chunks);
/* Gradient of sum_s w_s * BCE(logit_s, y_s) over the samples order[0..n)
 * (identity when order is NULL) into grad_and_loss[0..QMHD_MLP_PARAMS), the
 * loss into grad_and_loss[QMHD_MLP_PARAMS]; deterministic; `chunks` passes of
 * 16 samples per wave. */
int qmhd_mlp_gradient(const uint16_t* packed, const float* params, const float* features, const float* targets,
                      const float* weights, const int64_t* order, int64_t n, int chunks, float* partial,
                      float* grad_and_loss, void* stream);
/* One Adam step (bias-corrected, `step` counts from 1). */
int qmhd_mlp_adam(float* params, const float* grad, float* m, float* v, int64_t step, float lr, float beta1,
                  float beta2, float eps, void* stream);
/* Features of every interior cell of a ghost-filled state (nx*ny x 100 FP32,
 * cell (i,j) at row j*nx+i); scratch as qmhd_scratch_doubles. */
int qmhd_cell_features(const qmhd_grid* g, double gamma, const double* const* u8, float* features, double* scratch,
                       void* stream);
/* Label bits of every interior cell (nx*ny bytes) from the plain FP64 MP5/MP7
 * method on a ghost-filled state. */
int qmhd_cell_labels(const qmhd_grid* g, int order, const int32_t* flags4, double gamma, const double* const* u8,
                     double label_tol, uint8_t* cell_bits, double* scratch, void* stream);
/* The solver's indicator on a ghost-filled state: flags (1 = plain path) of
 * every padded cell (storage-size bytes). */
int qmhd_cell_indicator(const qmhd_grid* g, double gamma, const double* const* u8, const uint16_t* packed,
                        const float* params, float threshold_logit, uint8_t* flags, double* scratch, void* stream);
/* Wait for the work queued on `stream` (NULL: the library's null stream). */
int qmhd_stream_synchronize(void* stream);
/* Network of a solver configured with indicator "mlp": cells whose logit is
 * below threshold_logit take the cheap path. */
int qmhd_solver_set_indicator(qmhd_solver* s, const float* host_params, float threshold_logit);
/* Faces sent to the plain path and faces reconstructed since the last call. */
int qmhd_solver_plain_faces(qmhd_solver* s, int64_t* plain, int64_t* total);
/* ---- launch tuning and batched runs (no reference counterpart) --------
 * Tuning vector (QMHD_TUNING_INTS x int32): [0,1] flux block x, y (MUSCL and
 * first order; MP5/MP7 take their LDS tile); [2,3]
 * corner block x, y; [4,5] update block x, y (64..256 threads, multiples of
 * 64); [6] most blocks of a face-list launch of the learned form's plain
 * path; [7] cell E_z tile (0: 16x16, 1: 32x8, 2: 8x32 cells; the learned
 * form takes the full quadrature in whole tiles that hold a flagged cell, so
 * there the tile changes results and the autotuner leaves it at 0); [8] the
 * learned form's cheap-face tile, both directions (0: 64x4, 1: 32x8, 2: 128x2,
 * 3: 16x16, 4: 8x32 cells); [9] MP5/MP7 corner kernel (1: 16x16 LDS tile,
 * 0: one thread per corner in the [2,3] block); [10] accepted as [8], without
 * effect (the y faces of a cell are taken with its x faces); [11] reserved (0).
 * qmhd_solver_autotune times every candidate of each knob that shapes a launch
 * of the run's scheme over `trial_steps` steps (the live state is restored
 * afterwards) and keeps the fastest. */
#define QMHD_TUNING_INTS 12
int qmhd_solver_autotune(qmhd_solver* s, int trial_steps, int32_t* tuning_out);
int qmhd_solver_set_tuning(qmhd_solver* s, const int32_t* tuning);
int qmhd_solver_get_tuning(const qmhd_solver* s, int32_t* tuning);

/* Many independent runs stepped together: the auto-dt step of every run
 * (each on its own stream, with the accept/reject decision and commit on the
 * device) is captured into a HIP graph, and one graph launch advances every
 * run by one step.  qmhd_batch_run launches the graph in segments of up to
 * 16 steps.  A rejected step (an inadmissible stage) leaves that run's state
 * unchanged, is counted, and holds the run for the rest of the segment;
 * after each segment, every held run's steps of that segment are finished
 * through its own positivity controller (the retries of
 * mhd_solver.cpp:965-1143) and the run rejoins the graph, so each run that is
 * not fatal ends the call with the requested number of accepted steps.  A run whose live state is invalid
 * (or whose controller fails) stops and is flagged fatal.  The runs stay owned
 * by the caller and must be stepped only through the batch while it exists
 * (readbacks are fine). */
typedef struct qmhd_batch qmhd_batch;
int qmhd_batch_create(qmhd_solver* const* runs, int count, qmhd_batch** out);
/* Tile work-queue batch: every run's step is recorded once, and each launch
 * of the step becomes one launch over the tiles of all runs (per-run argument
 * records and tile ranges in device memory; a workgroup finds its tile's
 * run among the runs' first tiles), so a graph launch advances every run with
 * as many kernel launches as one run's step makes.  The runs must use the same
 * scheme, form and launch shapes (set one tuning on all of them).
 * queue_blocks: 0 for one workgroup per tile, where each run ends bit for
 * bit where its own loop would; else a persistent grid of that many
 * workgroups, each taking tiles blockIdx.x, blockIdx.x + gridDim.x, ...,
 * where each run ends there to rounding (the compiler fuses some multiplies
 * and adds differently in the persistent kernels; a launch with fewer tiles
 * than queue_blocks runs one workgroup per tile). */
int qmhd_batch_create_queued(qmhd_solver* const* runs, int count, int queue_blocks, qmhd_batch** out);
/* Queue mode: times each candidate queue_blocks (0, 256 .. 8192) over
 * trial_steps steps, puts every run back in its state and keeps the fastest. */
int qmhd_batch_autotune(qmhd_batch* b, int trial_steps, int* queue_blocks);
void qmhd_batch_destroy(qmhd_batch* b);
int qmhd_batch_run(qmhd_batch* b, int steps);
/* Runs found fatal by the calls so far, and why (and after how many accepted
 * steps) run `run` stopped: "" for a run that has not (text owned by the
 * batch, valid until it is destroyed). */
int qmhd_batch_fatal_runs(const qmhd_batch* b);
const char* qmhd_batch_run_failure(const qmhd_batch* b, int run);
int qmhd_batch_run_status(qmhd_batch* b, int run, int64_t* accepted, int64_t* rejected, int* fatal,
                          double* sim_time);

/* Features / label bits of the live state (device outputs, as above). */
int qmhd_solver_cell_features(qmhd_solver* s, float* features);
int qmhd_solver_cell_labels(qmhd_solver* s, double label_tol, uint8_t* cell_bits);

#ifdef __cplusplus
}
#endif

#endif /* QUASAR_MHD_H */

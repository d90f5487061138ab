// HIP kernels (gfx950) for one SSP-RK3 stage of the 2D constrained-transport
// ideal-MHD step: staggered-field collocation with the admissibility and
// div(B) preflights, characteristic MP5/MP7 (MUSCL, piecewise-constant)
// reconstruction, transverse-Gauss HLLD face fluxes with the CFL face rate,
// the cell-average E_z tensor quadrature (LDS tile), the upwind CT corner EMF,
// the fused flux-difference + EMF-curl + Shu-Osher update, ghost fills and the
// analytic initial conditions.
//
// Storage: every plane is a padded row-major array, index (i+ng) + pitch*(j+ng),
// pitch = nx + 2 ng, identical to the reference's Grid2D so seeds and
// readbacks are byte compatible.  State planes are FP64; interface states and
// fluxes are of the kernel's arithmetic type T.

#include "qmhd_face.hpp"
#include "qmhd_kernels.hpp"
#include "qmhd_queue.hpp"
#include "qmhd_recon.hpp"
#include "qmhd_stencil.hpp"

#include <algorithm>
#include <cstdint>
#include <stdexcept>
#include <type_traits>

namespace qmhd {

__constant__ QuadRows c_rows;

// ---------------------------------------------------------------------------
// Small helpers.

// Non-negative doubles order like their bit patterns: min/max through
// 64-bit integer atomics is exact and order independent.
__device__ __forceinline__ void atomic_min_nonneg(unsigned long long* slot, double v) {
  atomicMin(slot, static_cast<unsigned long long>(__double_as_longlong(v)));
}
__device__ __forceinline__ void atomic_max_nonneg(unsigned long long* slot, double v) {
  atomicMax(slot, static_cast<unsigned long long>(__double_as_longlong(v)));
}

// Wave-level reductions (64 lanes) before one atomic per wave.
__device__ __forceinline__ double wave_min(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmin(v, __shfl_xor(v, off, 64));
  return v;
}
__device__ __forceinline__ double wave_max(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off, 64));
  return v;
}
__device__ __forceinline__ bool lane_leader() { return (threadIdx.x + blockDim.x * threadIdx.y) % 64 == 0; }

// Reduction over a 256-thread block (4 waves): wave shuffles, then the four
// wave results through LDS.  Every thread of the block must call it; the
// result is returned to all of them.  Blocks that reduce cover many cells
// (kRowsPerThread rows per thread), so one atomic per block keeps the status
// slots free of contention.
constexpr int kRowsPerThread = 8;
template <bool MAX>
__device__ __forceinline__ double block_reduce(double v, double* lds4) {
  v = MAX ? wave_max(v) : wave_min(v);
  const int tid = threadIdx.x + blockDim.x * threadIdx.y;
  if (tid % 64 == 0) lds4[tid / 64] = v;
  __syncthreads();
  double r = lds4[0];
#pragma unroll
  for (int w = 1; w < 4; ++w) r = MAX ? fmax(r, lds4[w]) : fmin(r, lds4[w]);
  __syncthreads();
  return r;
}
__device__ __forceinline__ bool block_leader() { return threadIdx.x == 0 && threadIdx.y == 0; }

// Internal energy q = E - K - M of a convex combination (the admissible set
// rho > 0, q > 0 is convex).
// Internal energy q = E - K - M of a convex combination (the admissible set
// rho > 0, q > 0 is convex), in the reference's arithmetic
// (mhd_reduce.hip:99-123): its sign decides the positivity controller.
__device__ __forceinline__ double convex_q(const St<double>& a, const St<double>& b, double th) {
#pragma clang fp contract(off)
  const double om = 1.0 - th;
  const double rho = om * a.rho + th * b.rho;
  if (!(rho > 0.0) || !fin(rho)) return -Lim<double>::inf();
  const double mx = om * a.mx + th * b.mx, my = om * a.my + th * b.my, mz = om * a.mz + th * b.mz;
  const double e = om * a.en + th * b.en;
  const double bx = om * a.bx + th * b.bx, by = om * a.by + th * b.by, bz = om * a.bz + th * b.bz;
  const double q = (e - kinetic_from_momentum(mx, my, mz, rho)) - half_squared_norm3(bx, by, bz);
  return fin(q) ? q : -Lim<double>::inf();
}

// Largest theta in [0,1] keeping rho > 0 and q > 0 on the segment a -> b.
__device__ double admissible_theta(const St<double>& a, const St<double>& b) {
  const double qa = convex_q(a, b, 0.0);
  if (!(a.rho > 0.0) || !(qa > 0.0) || !fin(a.rho) || !fin(qa)) return 0.0;
  if (!fin(b.rho) || !fin(b.mx) || !fin(b.my) || !fin(b.mz) || !fin(b.en) || !fin(b.bx) || !fin(b.by) || !fin(b.bz))
    return 0.0;
  double hi = 1.0;
  if (b.rho <= 0.0) {
    const double d = a.rho - b.rho;
    hi = d > 0.0 ? a.rho / d : 0.0;
    hi = hi < 0.0 ? 0.0 : (hi > 1.0 ? 1.0 : hi);
  }
  if (convex_q(a, b, hi) > 0.0) return hi;
  double lo = 0.0;
  for (int it = 0; it < 56; ++it) {
    const double mid = 0.5 * (lo + hi);
    if (convex_q(a, b, mid) > 0.0)
      lo = mid;
    else
      hi = mid;
  }
  return lo;
}

__device__ __forceinline__ St<double> cell_state(const GridD& g, const StateView& u, std::size_t k, double bx, double by) {
  return St<double>{u.c[0][k], u.c[1][k], u.c[2][k], u.c[3][k], u.c[4][k], bx, by, u.c[7][k]};
}

// ulp of a binary64 value as used by the solenoidality roundoff budget.
__device__ __forceinline__ double ulp_of(double v) {
  if (!fin(v)) return Lim<double>::inf();
  const double m = __builtin_fabs(v);
  if (m < Lim<double>::tiny) return 4.9406564584124654e-324;
  int e = 0;
  (void)frexp(m, &e);
  return ldexp(0.5, e - 52);
}

// Whether a cell state is finite with rho > 0 and internal energy q > 0 beyond
// any rounding of q: then convex_q's q, which rounds in another order, is
// positive too.  (False only says that convex_q has to decide.)
__device__ __forceinline__ bool clearly_admissible(const St<double>& s, double bx, double by) {
  const double kin = 0.5 * (s.mx * s.mx + s.my * s.my + s.mz * s.mz) * frcp(s.rho);
  const double mag = 0.5 * (bx * bx + by * by + s.bz * s.bz);
  const double q = (s.en - kin) - mag;
  return s.rho > 0.0 && q > 32.0 * Lim<double>::eps * (__builtin_fabs(s.en) + kin + mag) + 1e-290;
}

__device__ __forceinline__ double ok_or_zero(double v) { return fin(v) ? v : 0.0; }

// Collocated Bx/By of `u` on every padded cell (W faces; EXACT: correctly
// rounded, the FP64 form; otherwise a fused multiply-add sum), and on the
// interior cells the admissible fraction of a stage candidate against its base
// (status.theta[slot]; with theta_both the other collocation into theta[3])
// and the live-state preflights (admissibility under both collocations, the
// relative div B residual).  One pass: 8 planes read, 2 written.  At 2048^2 a
// stage's collocation, ghost strips and checks as three kernels, the checks
// reading the candidate and its base (16 planes) and bisecting with divisions
// in every cell, took 262 us; now 106 us.  A division-free sign test decides
// all but the cells at the edge of the admissible set; those read the base.
// The one-sided closures of the outer ghost cells, a serial chain of some 600
// instructions each, have blocks of their own, a thread per closure: taken by
// the wave that holds the cell, nearly every wave of a small grid ran one per
// axis behind its centred sums (64^2 FP64 16 -> 6.3 us per launch, learned rotor
// 768^2 21 -> 17, a queue of 24 runs 24 -> 18).

// Blocks of the closures' part of a prep launch.
template <int W>
__host__ __device__ __forceinline__ int prep_strip_blocks(const GridD& g) {
  return ((W - 1) * (g.nx + g.ny + 4 * g.ng) + 255) / 256;
}

template <bool EXACT, int W>
__device__ __forceinline__ void prep_kernel_tile(
    const Blk& qb, const GridD& g, const StateView& u, double* __restrict__ bxc, double* __restrict__ byc,
    const StateView& base, const double* __restrict__ base_bxc, const double* __restrict__ base_byc, int theta_slot,
    int theta_co, int theta_both, int live_checks, int solver_owned, StepStatus* __restrict__ status) {
#include "tiles/prep_kernel.inc"
}

template <bool EXACT, int W>
__global__ __launch_bounds__(256) void prep_kernel(GridD g, StateView u, double* __restrict__ bxc,
                                                   double* __restrict__ byc, StateView base,
                                                   const double* __restrict__ base_bxc,
                                                   const double* __restrict__ base_byc, int theta_slot,
                                                   int theta_co, int theta_both, int live_checks,
                                                   int solver_owned, StepStatus* __restrict__ status) {
  [[maybe_unused]] const Blk qb = Blk::xcd_tiled();
#include "tiles/prep_kernel.inc"
}

// Queue form of prep_kernel (one launch over the tiles of many runs).
template <bool EXACT, int W>
struct prep_kernel_q {
  static constexpr int kWindow = W;
  struct Args {
    GridD g;
    StateView u;
    double* bxc;
    double* byc;
    StateView base;
    const double* base_bxc;
    const double* base_byc;
    int theta_slot;
    int theta_co;
    int theta_both;
    int live_checks;
    int solver_owned;
    StepStatus* status;
  };
  static __device__ __forceinline__ void run(const Blk& qb, const Args& a) {
    prep_kernel_tile<EXACT, W>(qb, queue_arg(a.g), queue_arg(a.u), queue_arg(a.bxc), queue_arg(a.byc), queue_arg(a.base),
                     queue_arg(a.base_bxc), queue_arg(a.base_byc), queue_arg(a.theta_slot), queue_arg(a.theta_co),
                     queue_arg(a.theta_both), queue_arg(a.live_checks), queue_arg(a.solver_owned), queue_arg(a.status));
  }
  static void launch(dim3 grid, dim3 block, hipStream_t s, const Args& a) {
    hipLaunchKernelGGL((prep_kernel<EXACT, W>), grid, block, 0, s, a.g, a.u, a.bxc, a.byc, a.base, a.base_bxc, a.base_byc,
                       a.theta_slot, a.theta_co, a.theta_both, a.live_checks, a.solver_owned, a.status);
  }
  static const void* tag() {
    static const char t = 0;
    return &t;
  }
};

// prep_kernel over the tile queue, one workgroup per tile: the same text, the
// arguments read from the tile's run record.
template <bool EXACT, int W>
__global__ __launch_bounds__(256) void prep_kernel_queue(
    const typename prep_kernel_q<EXACT, W>::Args* __restrict__ qargs, const QueueRun* __restrict__ qruns, int qnruns) {
  const QueueTile qtile = queue_tile(qruns, qnruns);
  [[maybe_unused]] const Blk qb = qtile.blk;
  const typename prep_kernel_q<EXACT, W>::Args& qa = qargs[qtile.run];
  GridD g = qa.g;
  StateView u = queue_arg(qa.u);
  double* __restrict__ bxc = queue_arg(qa.bxc);
  double* __restrict__ byc = queue_arg(qa.byc);
  StateView base = queue_arg(qa.base);
  const double* __restrict__ base_bxc = queue_arg(qa.base_bxc);
  const double* __restrict__ base_byc = queue_arg(qa.base_byc);
  int theta_slot = qa.theta_slot;
  int theta_co = qa.theta_co;
  int theta_both = qa.theta_both;
  int live_checks = qa.live_checks;
  int solver_owned = qa.solver_owned;
  StepStatus* __restrict__ status = queue_arg(qa.status);
#include "tiles/prep_kernel.inc"
}
template <bool EXACT, int W>
struct QueueTiles<prep_kernel_q<EXACT, W>> {
  static constexpr auto kernel = &prep_kernel_queue<EXACT, W>;
};

// Stand-alone collocation (readback of bx/by and the launch-level ABI).
__global__ __launch_bounds__(256) void collocate_kernel(GridD g, int axis, int co, const double* __restrict__ face,
                                                        double* __restrict__ cell) {
  const int i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x) - g.ng;
  const int j = static_cast<int>(blockIdx.y * blockDim.y + threadIdx.y) - g.ng;
  if (i >= g.nx + g.ng || j >= g.ny + g.ng) return;
  double v;
  if (axis == 0)
    v = co == 1 ? face_to_cell_lo(g, face, 0, i, j) : face_to_cell(g, face, 0, i, j);
  else
    v = co == 1 ? face_to_cell_lo(g, face, 1, j, i) : face_to_cell(g, face, 1, j, i);
  cell[idx(g, i, j)] = v;
}

// Writes a face's L (0..7) and R (8..15) interface planes, from states in the
// frame of its normal, and its "L == R" flag used by the CT 1-D shortcut.
template <class T>
__device__ __forceinline__ void write_faces(const IfaceView<T>& out, int dir, int* eq_flag, std::size_t k,
                                            const St<T>& ul, const St<T>& ur) {
  // Plane of component c: x and y components exchanged for y faces.
  const int plane[8] = {0, dir == 0 ? 1 : 2, dir == 0 ? 2 : 1, 3, 4, dir == 0 ? 5 : 6, dir == 0 ? 6 : 5, 7};
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    out.c[plane[c]][k] = comp(ul, c);
    out.c[8 + plane[c]][k] = comp(ur, c);
  }
  bool eq = true;
#pragma unroll
  for (int c = 0; c < 8; ++c) eq = eq && (comp(ul, c) == comp(ur, c));
  eq_flag[k] = eq ? 1 : 0;
}

// Appends face k of every lane with `need` to a list (one atomic per wave;
// every lane of the wave calls it).
__device__ __forceinline__ void list_faces(bool need, std::size_t k, unsigned long long* __restrict__ count,
                                           unsigned long long* __restrict__ list) {
  const unsigned long long mask = __ballot(need);
  if (mask == 0ull) return;
  const int lane = static_cast<int>(__lane_id());
  const int leader = __ffsll(static_cast<long long>(mask)) - 1;
  unsigned long long base = 0;
  if (lane == leader) base = atomicAdd(count, static_cast<unsigned long long>(__popcll(mask)));
  base = __shfl(base, leader, 64);
  if (need) list[base + __popcll(mask & ((1ull << lane) - 1ull))] = k;
}

// Face (i, j) of a reconstruction launch over dir 0 faces i in [0,nx],
// j in [-ng, ny+ng) (dir 1 transposed); false outside.
__device__ __forceinline__ bool recon_face_of(const GridD& g, int dir, int li, int lj, int& i, int& j) {
  i = dir == 1 ? li - g.ng : li;
  j = dir == 0 ? lj - g.ng : lj;
  if (dir == 0) return li <= g.nx && lj < g.ny + 2 * g.ng;
  return li < g.nx + 2 * g.ng && lj <= g.ny;
}

// Waves per SIMD of the MP reconstruction: in FP64 two (256 registers; it would
// take 264, mostly in the rarely taken exact basis: 563 against 327 us per x
// launch at 2048^2), in FP32 four (49 us per 1024^2 launch; 54 with no bound).
// The listed faces' kernel is left unbounded: it holds the whole stencil in
// registers and its time is one face's latency (learned rotor 768^2 16 us; 29
// with the bound).
template <class T>
constexpr int kReconWaves = sizeof(T) == 4 ? 4 : 2;
// Faces per block of the MP5/MP7 reconstruction (x faces, y faces) and the
// cells the larger of the two stages.
constexpr int kReconTiles[2][2] = {{64, 4}, {32, 8}};
template <int ORDER>
constexpr int recon_tile_cells() {
  constexpr int more = ORDER == 2 ? 3 : ORDER == 5 ? 5 : 7;
  constexpr int x = (kReconTiles[0][0] + more) * kReconTiles[0][1], y = kReconTiles[1][0] * (kReconTiles[1][1] + more);
  return x > y ? x : y;
}

// One thread per face normal to `dir`.  For MP5/MP7 this kernel takes the
// characteristic MP path of qmhd_recon.hpp; a face that does not settle there is
// appended to `fb_list` and redone, fallback chain included, by the fallback
// kernel.  2048^2, x / y faces: 700 us each with the reference's face per thread
// and its cells read from global memory (5.2k VALU instructions in the code, its
// L R = I loop seven times), 327 us now in FP64 (2.0k besides the exact basis;
// 494 / 523 with the cells read from global memory); FP32 at 1024^2 132 -> 49 us.
template <class T, int ORDER>
__device__ __forceinline__ void reconstruct_kernel_tile(
    const Blk& qb, const GridD& g, int dir, T gamma, int side_lo, int side_hi, const StateView& u,
    const double* __restrict__ bxc, const double* __restrict__ byc, const IfaceView<T>& out, int* __restrict__ eq_flag,
    unsigned long long* __restrict__ fb_count, unsigned long long* __restrict__ fb_list) {
#include "tiles/reconstruct_kernel.inc"
}

// Queue form of reconstruct_kernel (one launch over the tiles of many runs).
template <class T, int ORDER>
struct reconstruct_kernel_q {
  struct Args {
    GridD g;
    int dir;
    T gamma;
    int side_lo;
    int side_hi;
    StateView u;
    const double* bxc;
    const double* byc;
    IfaceView<T> out;
    int* eq_flag;
    unsigned long long* fb_count;
    unsigned long long* fb_list;
  };
  static __device__ __forceinline__ void run(const Blk& qb, const Args& a) {
    reconstruct_kernel_tile<T, ORDER>(qb, queue_arg(a.g), queue_arg(a.dir), queue_arg(a.gamma), queue_arg(a.side_lo),
                                      queue_arg(a.side_hi), queue_arg(a.u), queue_arg(a.bxc), queue_arg(a.byc),
                                      queue_arg(a.out), queue_arg(a.eq_flag), queue_arg(a.fb_count),
                                      queue_arg(a.fb_list));
  }
  static const void* tag() {
    static const char t = 0;
    return &t;
  }
};

// reconstruct_kernel over the tile queue, one workgroup per tile: the same text, the
// arguments read from the tile's run record.
template <class T, int ORDER>
__global__ __launch_bounds__(256, kReconWaves<T>) void reconstruct_kernel_queue(
    const typename reconstruct_kernel_q<T, ORDER>::Args* __restrict__ qargs, const QueueRun* __restrict__ qruns,
    int qnruns,
    Pair<typename reconstruct_kernel_q<T, ORDER>::Args>) {
  const auto qtile = tile_of(qargs, qruns, qnruns);
  [[maybe_unused]] const Blk qb = qtile.blk;
  const auto& qa = qtile.args;
  GridD g = qa.g;
  int dir = qa.dir;
  T gamma = qa.gamma;
  int side_lo = qa.side_lo;
  int side_hi = qa.side_hi;
  StateView u = queue_arg(qa.u);
  const double* __restrict__ bxc = queue_arg(qa.bxc);
  const double* __restrict__ byc = queue_arg(qa.byc);
  IfaceView<T> out = queue_arg(qa.out);
  int* __restrict__ eq_flag = queue_arg(qa.eq_flag);
  unsigned long long* __restrict__ fb_count = queue_arg(qa.fb_count);
  unsigned long long* __restrict__ fb_list = queue_arg(qa.fb_list);
#include "tiles/reconstruct_kernel.inc"
}
template <class T, int ORDER>
struct Paired<reconstruct_kernel_q<T, ORDER>> {
  static constexpr bool value = true;
  static constexpr unsigned xcd = 1u;
};
template <class T, int ORDER>
struct QueueTiles<reconstruct_kernel_q<T, ORDER>> {
  static constexpr auto kernel = &reconstruct_kernel_queue<T, ORDER>;
};

// Learned form: the characteristic MP states of the faces on the cheap
// reconstruction's list (a bounded grid strides over the list); a face whose MP states (or their normal-field update) are not
// admissible goes on the second list, for the full fallback chain.
template <class T, int ORDER>
__device__ __forceinline__ void reconstruct_list_kernel_tile(
    const Blk& qb, const GridD& g, int dir, T gamma, const StateView& u, const double* __restrict__ bxc,
    const double* __restrict__ byc, const IfaceView<T>& out, int* __restrict__ eq_flag,
    const unsigned long long* __restrict__ list_count, const unsigned long long* __restrict__ list,
    unsigned long long* __restrict__ fb_count, unsigned long long* __restrict__ fb_list,
    unsigned long long* __restrict__ plain_total) {
#include "tiles/reconstruct_list_kernel.inc"
}

// Queue form of reconstruct_list_kernel (one launch over the tiles of many runs).
template <class T, int ORDER>
struct reconstruct_list_kernel_q {
  struct Args {
    GridD g;
    int dir;
    T gamma;
    StateView u;
    const double* bxc;
    const double* byc;
    IfaceView<T> out;
    int* eq_flag;
    const unsigned long long* list_count;
    const unsigned long long* list;
    unsigned long long* fb_count;
    unsigned long long* fb_list;
    unsigned long long* plain_total;
  };
  static __device__ __forceinline__ void run(const Blk& qb, const Args& a) {
    reconstruct_list_kernel_tile<T, ORDER>(qb, queue_arg(a.g), queue_arg(a.dir), queue_arg(a.gamma), queue_arg(a.u),
                                           queue_arg(a.bxc), queue_arg(a.byc), queue_arg(a.out), queue_arg(a.eq_flag),
                                           queue_arg(a.list_count), queue_arg(a.list), queue_arg(a.fb_count),
                                           queue_arg(a.fb_list), queue_arg(a.plain_total));
  }
  static const void* tag() {
    static const char t = 0;
    return &t;
  }
};

// reconstruct_list_kernel over the tile queue, one workgroup per tile: the same text, the
// arguments read from the tile's run record.
template <class T, int ORDER>
__global__ __launch_bounds__(256) void reconstruct_list_kernel_queue(
    const typename reconstruct_list_kernel_q<T, ORDER>::Args* __restrict__ qargs, const QueueRun* __restrict__ qruns,
    int qnruns,
    Pair<typename reconstruct_list_kernel_q<T, ORDER>::Args>) {
  const auto qtile = tile_of(qargs, qruns, qnruns);
  [[maybe_unused]] const Blk qb = qtile.blk;
  const auto& qa = qtile.args;
  GridD g = qa.g;
  int dir = qa.dir;
  T gamma = qa.gamma;
  StateView u = queue_arg(qa.u);
  const double* __restrict__ bxc = queue_arg(qa.bxc);
  const double* __restrict__ byc = queue_arg(qa.byc);
  IfaceView<T> out = queue_arg(qa.out);
  int* __restrict__ eq_flag = queue_arg(qa.eq_flag);
  const unsigned long long* __restrict__ list_count = queue_arg(qa.list_count);
  const unsigned long long* __restrict__ list = queue_arg(qa.list);
  unsigned long long* __restrict__ fb_count = queue_arg(qa.fb_count);
  unsigned long long* __restrict__ fb_list = queue_arg(qa.fb_list);
  unsigned long long* __restrict__ plain_total = queue_arg(qa.plain_total);
#include "tiles/reconstruct_list_kernel.inc"
}
template <class T, int ORDER>
struct Paired<reconstruct_list_kernel_q<T, ORDER>> {
  static constexpr bool value = true;
  static constexpr unsigned xcd = 0u;
};
template <class T, int ORDER>
struct QueueTiles<reconstruct_list_kernel_q<T, ORDER>> {
  static constexpr auto kernel = &reconstruct_list_kernel_queue<T, ORDER>;
};

// The full fallback chain for the faces the MP kernel listed; a small
// grid-stride launch.
template <class T, int ORDER>
__device__ __forceinline__ void reconstruct_fallback_kernel_tile(
    const Blk& qb, const GridD& g, int dir, T gamma, int side_lo, int side_hi, const StateView& u,
    const double* __restrict__ bxc, const double* __restrict__ byc, const IfaceView<T>& out, int* __restrict__ eq_flag,
    const unsigned long long* __restrict__ fb_count, const unsigned long long* __restrict__ fb_list) {
#include "tiles/reconstruct_fallback_kernel.inc"
}

// Queue form of reconstruct_fallback_kernel (one launch over the tiles of many runs).
template <class T, int ORDER>
struct reconstruct_fallback_kernel_q {
  struct Args {
    GridD g;
    int dir;
    T gamma;
    int side_lo;
    int side_hi;
    StateView u;
    const double* bxc;
    const double* byc;
    IfaceView<T> out;
    int* eq_flag;
    const unsigned long long* fb_count;
    const unsigned long long* fb_list;
  };
  static __device__ __forceinline__ void run(const Blk& qb, const Args& a) {
    reconstruct_fallback_kernel_tile<T, ORDER>(qb, queue_arg(a.g), queue_arg(a.dir), queue_arg(a.gamma),
                                               queue_arg(a.side_lo), queue_arg(a.side_hi), queue_arg(a.u),
                                               queue_arg(a.bxc), queue_arg(a.byc), queue_arg(a.out),
                                               queue_arg(a.eq_flag), queue_arg(a.fb_count), queue_arg(a.fb_list));
  }
  static const void* tag() {
    static const char t = 0;
    return &t;
  }
};

// reconstruct_fallback_kernel over the tile queue, one workgroup per tile: the same text, the
// arguments read from the tile's run record.
template <class T, int ORDER>
__global__ __launch_bounds__(256) void reconstruct_fallback_kernel_queue(
    const typename reconstruct_fallback_kernel_q<T, ORDER>::Args* __restrict__ qargs,
    const QueueRun* __restrict__ qruns, int qnruns,
    Pair<typename reconstruct_fallback_kernel_q<T, ORDER>::Args>) {
  const auto qtile = tile_of(qargs, qruns, qnruns);
  [[maybe_unused]] const Blk qb = qtile.blk;
  const auto& qa = qtile.args;
  GridD g = qa.g;
  int dir = qa.dir;
  T gamma = qa.gamma;
  int side_lo = qa.side_lo;
  int side_hi = qa.side_hi;
  StateView u = queue_arg(qa.u);
  const double* __restrict__ bxc = queue_arg(qa.bxc);
  const double* __restrict__ byc = queue_arg(qa.byc);
  IfaceView<T> out = queue_arg(qa.out);
  int* __restrict__ eq_flag = queue_arg(qa.eq_flag);
  const unsigned long long* __restrict__ fb_count = queue_arg(qa.fb_count);
  const unsigned long long* __restrict__ fb_list = queue_arg(qa.fb_list);
#include "tiles/reconstruct_fallback_kernel.inc"
}
template <class T, int ORDER>
struct Paired<reconstruct_fallback_kernel_q<T, ORDER>> {
  static constexpr bool value = true;
  static constexpr unsigned xcd = 0u;
};
template <class T, int ORDER>
struct QueueTiles<reconstruct_fallback_kernel_q<T, ORDER>> {
  static constexpr auto kernel = &reconstruct_fallback_kernel_queue<T, ORDER>;
};
// Zeroes face-list counters (the solver's own are zeroed by its prep launches).
__global__ void counter_reset_kernel(unsigned long long* __restrict__ c, int n) {
  if (static_cast<int>(threadIdx.x) < n) c[threadIdx.x] = 0ull;
}

// Learned form, one thread per face: a face whose two cells the indicator
// left unflagged takes the linear fifth-order upwind-biased face values (the
// unlimited MP5 interpolant, include/quasar/numerics/mp_limiter.hpp:182-191)
// of the conserved cell averages, component by component, and the face normal
// field.  Flagged faces, and cheap states that are not admissible, are listed
// for the plain path (characteristic MP with its fallback chain).  A block takes
// a tile of cells and the low x and low y face of each from one staged set of
// cells (32 x 8: 37 x 13).  Bound by memory: 64 B of state and 80 B of outputs
// per cell in FP32, about 470 us per 4096^2 launch at a copy's rate.  Where no
// flag is near the block none is read per face, and each state's 1/rho,
// velocity and pressure serve its admissibility, its speed and its flux.
// 4096^2, both directions: 1060 us with a launch per direction at 1.2k VALU
// instructions a face (16 flag reads with range tests, index quotients by a
// run-time width, tests, speeds and fluxes formed apart); 944 with the
// instructions cut, 854 with the blocks of one XCD adjacent, 741 in one
// launch.
template <class T>
__device__ __forceinline__ void cheap_face_flux(const St<T>& L, const St<T>& R, const Side<T>& l, const Side<T>& r,
                                                int dir, T gamma, bool rate, St<T>& f, T& smax);
template <class T>
__device__ __forceinline__ void store_face(const GridD& g, int dir, const FluxView<T>& flux, double* __restrict__ rate,
                                           std::size_t ko, const St<T>& f, T smax);

// One direction's outputs of the cheap faces.
template <class T>
struct CheapFace {
  IfaceView<T> out;
  int* eq;
  unsigned long long* count;
  unsigned long long* list;
  FluxView<T> flux;
  double* rate;
  int periodic;
};
template <class T>
__device__ __forceinline__ CheapFace<T> queue_arg(const CheapFace<T>& f) {
  return CheapFace<T>{queue_arg(f.out), queue_arg(f.eq), queue_arg(f.count), queue_arg(f.list), queue_arg(f.flux),
                      queue_arg(f.rate), f.periodic};
}

// Cheap-reconstruction tiles (cells per block, TX x TY = 256 threads): the
// autotuner picks one of kCheapTiles.  The tile stages TX + 5 by TY + 5 cells:
// the squarer ones stage fewest (4096^2, reconstruction of a stage: 32 x 8 773 us,
// 16 x 16 817, 64 x 4 834, 128 x 2 878, 8 x 32 947).
constexpr int kCheapTileCount = 5;
constexpr int kCheapTiles[kCheapTileCount][2] = {{64, 4}, {32, 8}, {128, 2}, {16, 16}, {8, 32}};

template <class T, int TX, int TY>
__device__ __forceinline__ void cheap_reconstruct_kernel_tile(
    const Blk& qb, const GridD& g, T gamma, const StateView& u, const double* __restrict__ bxc,
    const double* __restrict__ byc, const uint8_t* __restrict__ cell_flags, const CheapFace<T>& cheap_x,
    const CheapFace<T>& cheap_y) {
#include "tiles/cheap_reconstruct_kernel.inc"
}

template <class T, int TX, int TY>
__global__ __launch_bounds__(256) void cheap_reconstruct_kernel(GridD g, T gamma, StateView u,
                                                                const double* __restrict__ bxc,
                                                                const double* __restrict__ byc,
                                                                const uint8_t* __restrict__ cell_flags,
                                                                CheapFace<T> cheap_x, CheapFace<T> cheap_y) {
  [[maybe_unused]] const Blk qb = Blk::xcd_tiled();
#include "tiles/cheap_reconstruct_kernel.inc"
}

// Queue form of cheap_reconstruct_kernel (one launch over the tiles of many runs).
template <class T, int TX, int TY>
struct cheap_reconstruct_kernel_q {
  struct Args {
    GridD g;
    T gamma;
    StateView u;
    const double* bxc;
    const double* byc;
    const uint8_t* cell_flags;
    CheapFace<T> cheap_x;
    CheapFace<T> cheap_y;
  };
  static __device__ __forceinline__ void run(const Blk& qb, const Args& a) {
    cheap_reconstruct_kernel_tile<T, TX, TY>(qb, queue_arg(a.g), queue_arg(a.gamma), queue_arg(a.u), queue_arg(a.bxc),
                                             queue_arg(a.byc), queue_arg(a.cell_flags), queue_arg(a.cheap_x),
                                             queue_arg(a.cheap_y));
  }
  static void launch(dim3 grid, dim3 block, hipStream_t s, const Args& a) {
    hipLaunchKernelGGL((cheap_reconstruct_kernel<T, TX, TY>), grid, block, 0, s, a.g, a.gamma, a.u, a.bxc, a.byc,
                       a.cell_flags, a.cheap_x, a.cheap_y);
  }
  static const void* tag() {
    static const char t = 0;
    return &t;
  }
};

// cheap_reconstruct_kernel over the tile queue, one workgroup per tile: the same text, the
// arguments read from the tile's run record.
template <class T, int TX, int TY>
__global__ __launch_bounds__(256) void cheap_reconstruct_kernel_queue(
    const typename cheap_reconstruct_kernel_q<T, TX, TY>::Args* __restrict__ qargs, const QueueRun* __restrict__ qruns,
    int qnruns) {
  const QueueTile qtile = queue_tile(qruns, qnruns);
  [[maybe_unused]] const Blk qb = qtile.blk;
  const typename cheap_reconstruct_kernel_q<T, TX, TY>::Args& qa = qargs[qtile.run];
  GridD g = qa.g;
  T gamma = qa.gamma;
  StateView u = queue_arg(qa.u);
  const double* __restrict__ bxc = queue_arg(qa.bxc);
  const double* __restrict__ byc = queue_arg(qa.byc);
  const uint8_t* __restrict__ cell_flags = queue_arg(qa.cell_flags);
  const CheapFace<T> cheap_x = queue_arg(qa.cheap_x), cheap_y = queue_arg(qa.cheap_y);
#include "tiles/cheap_reconstruct_kernel.inc"
}
template <class T, int TX, int TY>
struct QueueTiles<cheap_reconstruct_kernel_q<T, TX, TY>> {
  static constexpr auto kernel = &cheap_reconstruct_kernel_queue<T, TX, TY>;
};


// ---------------------------------------------------------------------------
// Face flux with transverse Gauss quadrature and the CFL face rate.

// The learned form's flux of a face whose two cells the indicator left
// unflagged: one HLL flux (Davis speeds) at its face-average states (in the
// frame of the normal, both with the face's own normal field), the rate from
// those states.  The plain list's flux and the cheap-face kernel share it, so
// both give the same bits.
template <class T>
__device__ __forceinline__ void cheap_face_flux(const St<T>& L, const St<T>& R, const Side<T>& l, const Side<T>& r,
                                                int dir, T gamma, bool rate, St<T>& f, T& smax) {
  const T cl = fast_of(l, l.bn2, gamma), cr = fast_of(r, r.bn2, gamma);
  smax = rate ? rate_of(l, cl, r, cr, 5) : T(0);
  f = rot(hll_sides(L, R, l, r, hi2(cl, cr)), dir);
}

// Face flux and, with a rate plane, the face rate (0.5 * signal speed /
// spacing) of face ko.
template <class T>
__device__ __forceinline__ void store_face(const GridD& g, int dir, const FluxView<T>& flux, double* __restrict__ rate,
                                           std::size_t ko, const St<T>& f, T smax) {
#pragma unroll
  for (int c = 0; c < 8; ++c) flux.c[c][ko] = comp(f, c);
  if (!rate) return;
  const double sp = static_cast<double>(smax);
  const double spacing = dir == 0 ? g.dx : g.dy;
  rate[ko] = (fin(sp) && sp >= 0.0) ? (sp * 0.5) / spacing : Lim<double>::inf();
}

// Flux and, with a rate plane, the signal speed max(|v_n|) + max(c_f) over the
// face average and every Gauss point, scaled by 0.5/spacing, of the faces
// [0,nx] x [0,ny], one thread each.  (The learned form's unflagged faces take
// cheap_face_flux instead.)  MP5/MP7: qmhd_face.hpp's node loop over the
// block's neighbour differences in LDS.  The tiles keep the differences under
// 43 KB in FP64 and give every half-wave 32 consecutive LDS words: 16 x 16 for
// x faces (lines along y), 32 x 8 for y faces.  2048^2 FP64,
// x / y faces: 955 / 861 us with one unrolled solve per node and the samples
// read from global memory (238 VGPRs, 5.7k VALU instructions a face), 553 / 535
// us now with the rate and 540 / 519 us without (219 / 243 VGPRs, about 3.3k),
// both at two waves per SIMD; forced to three it spills 22 VGPRs and takes 819
// / 795 us.  In the hardware's tile order the x faces take 565 us.
constexpr int kFluxTiles[2][2] = {{16, 16}, {32, 8}};
constexpr int kFluxListBlock = 64;
// Waves per SIMD of the face flux: both directions in one kernel take 147
// registers in FP32 (119 / 127 apart), past four waves.
template <class T>
constexpr int kFluxWaves = sizeof(T) == 4 ? 4 : 2;
template <int ORDER>
constexpr int flux_tile_values() {
  constexpr int more = ORDER == 5 ? 3 : 5;
  constexpr int x = kFluxTiles[0][0] * (kFluxTiles[0][1] + more), y = (kFluxTiles[1][0] + more) * kFluxTiles[1][1];
  return 16 * (x > y ? x : y);
}

template <class T, int ORDER, bool LF>
__device__ __forceinline__ void flux_kernel_tile(
    const Blk& qb, const GridD& g, int dir, int periodic_dir, T gamma, const IfaceView<T>& in, const FluxView<T>& flux,
    double* __restrict__ rate) {
#include "tiles/flux_kernel.inc"
}

// Queue form of flux_kernel (one launch over the tiles of many runs).
template <class T, int ORDER, bool LF>
struct flux_kernel_q {
  struct Args {
    GridD g;
    int dir;
    int periodic_dir;
    T gamma;
    IfaceView<T> in;
    FluxView<T> flux;
    double* rate;
  };
  static __device__ __forceinline__ void run(const Blk& qb, const Args& a) {
    flux_kernel_tile<T, ORDER, LF>(qb, queue_arg(a.g), queue_arg(a.dir), queue_arg(a.periodic_dir), queue_arg(a.gamma),
                                        queue_arg(a.in), queue_arg(a.flux), queue_arg(a.rate));
  }
  static const void* tag() {
    static const char t = 0;
    return &t;
  }
};

// flux_kernel over the tile queue, one workgroup per tile: the same text, the
// arguments read from the tile's run record.
template <class T, int ORDER, bool LF>
__global__ __launch_bounds__(256, kFluxWaves<T>) void flux_kernel_queue(
    const typename flux_kernel_q<T, ORDER, LF>::Args* __restrict__ qargs, const QueueRun* __restrict__ qruns,
    int qnruns,
    Pair<typename flux_kernel_q<T, ORDER, LF>::Args>) {
  const auto qtile = tile_of(qargs, qruns, qnruns);
  [[maybe_unused]] const Blk qb = qtile.blk;
  const auto& qa = qtile.args;
  GridD g = qa.g;
  const int dir = qa.dir;
  int periodic_dir = qa.periodic_dir;
  T gamma = qa.gamma;
  IfaceView<T> in = queue_arg(qa.in);
  FluxView<T> flux = queue_arg(qa.flux);
  double* __restrict__ rate = queue_arg(qa.rate);
#include "tiles/flux_kernel.inc"
}
template <class T, int ORDER, bool LF>
struct Paired<flux_kernel_q<T, ORDER, LF>> {
  static constexpr bool value = true;
  static constexpr unsigned xcd = 1u;
};
template <class T, int ORDER, bool LF>
struct QueueTiles<flux_kernel_q<T, ORDER, LF>> {
  static constexpr auto kernel = &flux_kernel_queue<T, ORDER, LF>;
};

// Learned form: the flux of the faces on the plain reconstruction's list,
// after that list's states are written.  The list holds every flagged face of
// the launch (plain flux) and the unflagged faces whose cheap states were
// inadmissible (the cheap flux of their plain states); the cheap
// reconstruction stored every other face's flux.  Ghost-row entries are
// skipped; a periodic high face takes its low partner's flux.  A bounded grid
// strides over the list; one wave per block, its lanes' neighbour differences
// in LDS (24 KB in FP32).
template <class T, int ORDER>
__device__ __forceinline__ void flux_plain_list_kernel_tile(const Blk& qb, const GridD& g, int dir, int periodic_dir, T gamma,
                                                              const IfaceView<T>& in, const FluxView<T>& flux,
                                                              double* __restrict__ rate,
                                                              const uint8_t* __restrict__ cell_flags,
                                                              const unsigned long long* __restrict__ fb_count,
                                                              const unsigned long long* __restrict__ fb_list) {
#include "tiles/flux_plain_list_kernel.inc"
}

// Queue form of flux_plain_list_kernel (one launch over the tiles of many runs).
template <class T, int ORDER>
struct flux_plain_list_kernel_q {
  struct Args {
    GridD g;
    int dir;
    int periodic_dir;
    T gamma;
    IfaceView<T> in;
    FluxView<T> flux;
    double* rate;
    const uint8_t* cell_flags;
    const unsigned long long* fb_count;
    const unsigned long long* fb_list;
  };
  static __device__ __forceinline__ void run(const Blk& qb, const Args& a) {
    flux_plain_list_kernel_tile<T, ORDER>(qb, queue_arg(a.g), queue_arg(a.dir), queue_arg(a.periodic_dir), queue_arg(a.gamma),
                                               queue_arg(a.in), queue_arg(a.flux), queue_arg(a.rate),
                                               queue_arg(a.cell_flags), queue_arg(a.fb_count), queue_arg(a.fb_list));
  }
  static const void* tag() {
    static const char t = 0;
    return &t;
  }
};

// flux_plain_list_kernel over the tile queue, one workgroup per tile: the same text, the
// arguments read from the tile's run record.
template <class T, int ORDER>
__global__ __launch_bounds__(kFluxListBlock) void flux_plain_list_kernel_queue(
    const typename flux_plain_list_kernel_q<T, ORDER>::Args* __restrict__ qargs,
    const QueueRun* __restrict__ qruns, int qnruns,
    Pair<typename flux_plain_list_kernel_q<T, ORDER>::Args>) {
  const auto qtile = tile_of(qargs, qruns, qnruns);
  [[maybe_unused]] const Blk qb = qtile.blk;
  const auto& qa = qtile.args;
  GridD g = qa.g;
  const int dir = qa.dir;
  int periodic_dir = qa.periodic_dir;
  T gamma = qa.gamma;
  IfaceView<T> in = queue_arg(qa.in);
  FluxView<T> flux = queue_arg(qa.flux);
  double* __restrict__ rate = queue_arg(qa.rate);
  const uint8_t* __restrict__ cell_flags = queue_arg(qa.cell_flags);
  const unsigned long long* __restrict__ fb_count = queue_arg(qa.fb_count);
  const unsigned long long* __restrict__ fb_list = queue_arg(qa.fb_list);
#include "tiles/flux_plain_list_kernel.inc"
}
template <class T, int ORDER>
struct Paired<flux_plain_list_kernel_q<T, ORDER>> {
  static constexpr bool value = true;
  static constexpr unsigned xcd = 0u;
};
template <class T, int ORDER>
struct QueueTiles<flux_plain_list_kernel_q<T, ORDER>> {
  static constexpr auto kernel = &flux_plain_list_kernel_queue<T, ORDER>;
};

// Additive cell CFL rate from the incident face rates, reduced to the maximum.
__device__ __forceinline__ void cfl_reduce_kernel_tile(const Blk& qb, const GridD& g, const double* __restrict__ rate_x,
                                                         const double* __restrict__ rate_y,
                                                         unsigned long long* __restrict__ max_rate) {
#include "tiles/cfl_reduce_kernel.inc"
}

__global__ __launch_bounds__(256) void cfl_reduce_kernel(GridD g, const double* __restrict__ rate_x,
                                                         const double* __restrict__ rate_y,
                                                         unsigned long long* __restrict__ max_rate) {
  [[maybe_unused]] const Blk qb = Blk::native();
#include "tiles/cfl_reduce_kernel.inc"
}

// Queue form of cfl_reduce_kernel (one launch over the tiles of many runs).
struct cfl_reduce_kernel_q {
  struct Args {
    GridD g;
    const double* rate_x;
    const double* rate_y;
    unsigned long long* max_rate;
  };
  static __device__ __forceinline__ void run(const Blk& qb, const Args& a) {
    cfl_reduce_kernel_tile(qb, queue_arg(a.g), queue_arg(a.rate_x), queue_arg(a.rate_y), queue_arg(a.max_rate));
  }
  static void launch(dim3 grid, dim3 block, hipStream_t s, const Args& a) {
    hipLaunchKernelGGL((cfl_reduce_kernel), grid, block, 0, s, a.g, a.rate_x, a.rate_y, a.max_rate);
  }
  static const void* tag() {
    static const char t = 0;
    return &t;
  }
};

// cfl_reduce_kernel over the tile queue, one workgroup per tile: the same text, the
// arguments read from the tile's run record.
__global__ __launch_bounds__(256) void cfl_reduce_kernel_queue(const cfl_reduce_kernel_q::Args* __restrict__ qargs,
    const QueueRun* __restrict__ qruns, int qnruns) {
  const QueueTile qtile = queue_tile(qruns, qnruns);
  [[maybe_unused]] const Blk qb = qtile.blk;
  const cfl_reduce_kernel_q::Args& qa = qargs[qtile.run];
  GridD g = qa.g;
  const double* __restrict__ rate_x = queue_arg(qa.rate_x);
  const double* __restrict__ rate_y = queue_arg(qa.rate_y);
  unsigned long long* __restrict__ max_rate = queue_arg(qa.max_rate);
#include "tiles/cfl_reduce_kernel.inc"
}
template <>
struct QueueTiles<cfl_reduce_kernel_q> {
  static constexpr auto kernel = &cfl_reduce_kernel_queue;
};

// ---------------------------------------------------------------------------
// Cell-average E_z = vy Bx - vx By by tensor Gauss recovery (MP5: 3x3 points
// from a 5x5 stencil, MP7: 4x4 from 7x7).
//
// Bound by instruction issue (about 2000 VALU instructions per 64 cells in
// FP64) with the LDS reads of the x pass behind it.  A wave owns 16 columns by
// the NQ x nodes and marches up its rows: a row's 22 x 8 values go through a
// wave-private LDS line (loaded one row ahead, no block barrier), its x point
// values enter a window of 2H + 1 rows in registers, and the y values, E_z and
// pressure test of the row below come from the window.  Point values are
// weighted neighbour differences about the centre, so equal samples give that
// sample with no comparison; a point is admissible when its internal energy is
// positive beyond rounding, and rows with one that is within rounding of zero
// are decided again, in the oracle's operations, after the march.  2048^2 FP64
// 702 -> 391 us, 1024^2 FP32 119 -> 69 us, 64^2 FP64 28 -> 12 us, learned rotor
// 768^2 35 -> 24 us, a queue of 24 learned runs 55 -> 30 us, against both passes
// through LDS by 16 x 16 cells.

// Cell E_z tiles: a block covers kEmfTiles[.][0] (at least 16) columns and
// march times kEmfTiles[.][1] rows; the autotuner picks one.  With LEARNED a
// BX x BY tile none of whose cells the indicator flagged takes the cell-average
// E_z (second order) in every cell.
constexpr int kEmfTiles[3][2] = {{16, 16}, {32, 8}, {8, 32}};

// A wave that marches m rows spends m + 2H rows of x passes, a quarter of its
// work per row: waves march four times as far (16 rows) when that leaves at
// least this many blocks (two waves per SIMD), twice or once as far below
// (64^2: 10 row steps one after the other, 12 us, in place of 22).
constexpr unsigned kEmfBlocks = 512;

// Orders this wave's LDS writes before its reads of other lanes' values (the
// LDS serves a wave's accesses in order; this keeps the compiler to it).
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

template <class T, int ORDER, bool LEARNED, int BX, int BY>
__device__ __forceinline__ void cell_emf_kernel_tile(
    const Blk& qb, const GridD& g, int phys_x_high, int phys_y_high, T gamma, const StateView& u,
    const double* __restrict__ bxc, const double* __restrict__ byc, double* __restrict__ cell_ez,
    const uint8_t* __restrict__ cell_flags, int march) {
#include "tiles/cell_emf_kernel.inc"
}

template <class T, int ORDER, bool LEARNED, int BX, int BY>
__global__ __launch_bounds__(256) void cell_emf_kernel(GridD g, int phys_x_high, int phys_y_high, T gamma,
                                                       StateView u, const double* __restrict__ bxc,
                                                       const double* __restrict__ byc, double* __restrict__ cell_ez,
                                                       const uint8_t* __restrict__ cell_flags, int march) {
  [[maybe_unused]] const Blk qb = Blk::xcd_tiled();
#include "tiles/cell_emf_kernel.inc"
}

// Queue form of cell_emf_kernel (one launch over the tiles of many runs).
template <class T, int ORDER, bool LEARNED, int BX, int BY>
struct cell_emf_kernel_q {
  struct Args {
    GridD g;
    int phys_x_high;
    int phys_y_high;
    T gamma;
    StateView u;
    const double* bxc;
    const double* byc;
    double* cell_ez;
    const uint8_t* cell_flags;
    int march;
  };
  static __device__ __forceinline__ void run(const Blk& qb, const Args& a) {
    cell_emf_kernel_tile<T, ORDER, LEARNED, BX, BY>(qb, queue_arg(a.g), queue_arg(a.phys_x_high),
                                                    queue_arg(a.phys_y_high), queue_arg(a.gamma), queue_arg(a.u),
                                                    queue_arg(a.bxc), queue_arg(a.byc), queue_arg(a.cell_ez),
                                                    queue_arg(a.cell_flags), queue_arg(a.march));
  }
  static void launch(dim3 grid, dim3 block, hipStream_t s, const Args& a) {
    hipLaunchKernelGGL((cell_emf_kernel<T, ORDER, LEARNED, BX, BY>), grid, block, 0, s, a.g, a.phys_x_high,
                       a.phys_y_high, a.gamma, a.u, a.bxc, a.byc, a.cell_ez, a.cell_flags, a.march);
  }
  static const void* tag() {
    static const char t = 0;
    return &t;
  }
};

// cell_emf_kernel over the tile queue, one workgroup per tile: the same text, the
// arguments read from the tile's run record.
template <class T, int ORDER, bool LEARNED, int BX, int BY>
__global__ __launch_bounds__(256) void cell_emf_kernel_queue(
    const typename cell_emf_kernel_q<T, ORDER, LEARNED, BX, BY>::Args* __restrict__ qargs,
    const QueueRun* __restrict__ qruns, int qnruns) {
  const QueueTile qtile = queue_tile(qruns, qnruns);
  [[maybe_unused]] const Blk qb = qtile.blk;
  const typename cell_emf_kernel_q<T, ORDER, LEARNED, BX, BY>::Args& qa = qargs[qtile.run];
  GridD g = qa.g;
  int phys_x_high = qa.phys_x_high;
  int phys_y_high = qa.phys_y_high;
  T gamma = qa.gamma;
  StateView u = queue_arg(qa.u);
  const double* __restrict__ bxc = queue_arg(qa.bxc);
  const double* __restrict__ byc = queue_arg(qa.byc);
  double* __restrict__ cell_ez = queue_arg(qa.cell_ez);
  const uint8_t* __restrict__ cell_flags = queue_arg(qa.cell_flags);
  int march = qa.march;
#include "tiles/cell_emf_kernel.inc"
}
template <class T, int ORDER, bool LEARNED, int BX, int BY>
struct QueueTiles<cell_emf_kernel_q<T, ORDER, LEARNED, BX, BY>> {
  static constexpr auto kernel = &cell_emf_kernel_queue<T, ORDER, LEARNED, BX, BY>;
};

// Low-order (direct) cell E_z with the two-face collocation.
__device__ __forceinline__ void cell_emf_lo_kernel_tile(
    const Blk& qb, const GridD& g, int phys_x_high, int phys_y_high, int co, const StateView& u,
    const double* __restrict__ bxc, const double* __restrict__ byc, double* __restrict__ cell_ez) {
#include "tiles/cell_emf_lo_kernel.inc"
}

__global__ __launch_bounds__(256) void cell_emf_lo_kernel(
    GridD g, int phys_x_high, int phys_y_high, int co, StateView u, const double* __restrict__ bxc,
    const double* __restrict__ byc, double* __restrict__ cell_ez) {
  [[maybe_unused]] const Blk qb = Blk::native();
#include "tiles/cell_emf_lo_kernel.inc"
}

// Queue form of cell_emf_lo_kernel (one launch over the tiles of many runs).
struct cell_emf_lo_kernel_q {
  struct Args {
    GridD g;
    int phys_x_high;
    int phys_y_high;
    int co;
    StateView u;
    const double* bxc;
    const double* byc;
    double* cell_ez;
  };
  static __device__ __forceinline__ void run(const Blk& qb, const Args& a) {
    cell_emf_lo_kernel_tile(qb, queue_arg(a.g), queue_arg(a.phys_x_high), queue_arg(a.phys_y_high), queue_arg(a.co),
                            queue_arg(a.u), queue_arg(a.bxc), queue_arg(a.byc), queue_arg(a.cell_ez));
  }
  static void launch(dim3 grid, dim3 block, hipStream_t s, const Args& a) {
    hipLaunchKernelGGL((cell_emf_lo_kernel), grid, block, 0, s, a.g, a.phys_x_high, a.phys_y_high, a.co, a.u, a.bxc,
                       a.byc, a.cell_ez);
  }
  static const void* tag() {
    static const char t = 0;
    return &t;
  }
};

// cell_emf_lo_kernel over the tile queue, one workgroup per tile: the same text, the
// arguments read from the tile's run record.
__global__ __launch_bounds__(256) void cell_emf_lo_kernel_queue(const cell_emf_lo_kernel_q::Args* __restrict__ qargs,
    const QueueRun* __restrict__ qruns, int qnruns) {
  const QueueTile qtile = queue_tile(qruns, qnruns);
  [[maybe_unused]] const Blk qb = qtile.blk;
  const cell_emf_lo_kernel_q::Args& qa = qargs[qtile.run];
  GridD g = qa.g;
  int phys_x_high = qa.phys_x_high;
  int phys_y_high = qa.phys_y_high;
  int co = qa.co;
  StateView u = queue_arg(qa.u);
  const double* __restrict__ bxc = queue_arg(qa.bxc);
  const double* __restrict__ byc = queue_arg(qa.byc);
  double* __restrict__ cell_ez = queue_arg(qa.cell_ez);
#include "tiles/cell_emf_lo_kernel.inc"
}
template <>
struct QueueTiles<cell_emf_lo_kernel_q> {
  static constexpr auto kernel = &cell_emf_lo_kernel_queue;
};

// ---------------------------------------------------------------------------
// CT corner EMF: E_z = ex + ey - e_c, with ex/ey the face-average -> edge
// interpolations of the directional Godunov EMFs (-F_x(By), +F_y(Bx)) and e_c
// the cell-average -> corner tensor interpolation of the cell E_z, plus the
// exact one-dimensional shortcuts.

template <class T>
__device__ __forceinline__ void corner_kernel_tile(
    const Blk& qb, const GridD& g, int order, const Flags4& m, const FluxView<T>& fx, const FluxView<T>& fy,
    const double* __restrict__ cell_ez, const int* __restrict__ eqx, const int* __restrict__ eqy,
    double* __restrict__ ez) {
#include "tiles/corner_kernel.inc"
}

template <class T>
__global__ __launch_bounds__(256) void corner_kernel(GridD g, int order, Flags4 m, FluxView<T> fx, FluxView<T> fy,
                                                     const double* __restrict__ cell_ez, const int* __restrict__ eqx,
                                                     const int* __restrict__ eqy, double* __restrict__ ez) {
  [[maybe_unused]] const Blk qb = Blk::native();
#include "tiles/corner_kernel.inc"
}

// Queue form of corner_kernel (one launch over the tiles of many runs).
template <class T>
struct corner_kernel_q {
  struct Args {
    GridD g;
    int order;
    Flags4 m;
    FluxView<T> fx;
    FluxView<T> fy;
    const double* cell_ez;
    const int* eqx;
    const int* eqy;
    double* ez;
  };
  static __device__ __forceinline__ void run(const Blk& qb, const Args& a) {
    corner_kernel_tile<T>(qb, queue_arg(a.g), queue_arg(a.order), queue_arg(a.m), queue_arg(a.fx), queue_arg(a.fy),
                          queue_arg(a.cell_ez), queue_arg(a.eqx), queue_arg(a.eqy), queue_arg(a.ez));
  }
  static void launch(dim3 grid, dim3 block, hipStream_t s, const Args& a) {
    hipLaunchKernelGGL((corner_kernel<T>), grid, block, 0, s, a.g, a.order, a.m, a.fx, a.fy, a.cell_ez, a.eqx, a.eqy,
                       a.ez);
  }
  static const void* tag() {
    static const char t = 0;
    return &t;
  }
};

// corner_kernel over the tile queue, one workgroup per tile: the same text, the
// arguments read from the tile's run record.
template <class T>
__global__ __launch_bounds__(256) void corner_kernel_queue(const typename corner_kernel_q<T>::Args* __restrict__ qargs,
    const QueueRun* __restrict__ qruns, int qnruns) {
  const QueueTile qtile = queue_tile(qruns, qnruns);
  [[maybe_unused]] const Blk qb = qtile.blk;
  const typename corner_kernel_q<T>::Args& qa = qargs[qtile.run];
  GridD g = qa.g;
  int order = qa.order;
  Flags4 m = qa.m;
  FluxView<T> fx = queue_arg(qa.fx);
  FluxView<T> fy = queue_arg(qa.fy);
  const double* __restrict__ cell_ez = queue_arg(qa.cell_ez);
  const int* __restrict__ eqx = queue_arg(qa.eqx);
  const int* __restrict__ eqy = queue_arg(qa.eqy);
  double* __restrict__ ez = queue_arg(qa.ez);
#include "tiles/corner_kernel.inc"
}
template <class T>
struct QueueTiles<corner_kernel_q<T>> {
  static constexpr auto kernel = &corner_kernel_queue<T>;
};

// MP5/MP7 corners, 16x16 per block: the cell E_z and the directional EMF samples
// the block reads are staged in LDS, every index mapped as corner_ez maps it,
// and the cell -> corner interpolation is formed separably (the x-direction one
// of every tile row once, then the y-direction one per corner: corner_ez's
// operations on the same values).  Bound by its reads and writes (40 B per
// corner in FP64, 33 us per 2048^2 launch at a copy's rate).  Blocks at the
// boundary took corner_ez per corner before, eight serial gathers of eight and
// the shortcut scans: a floor of 25 us under any launch.  2048^2 FP64 100 -> 47
// us, 4096^2 FP32 285 -> 174, 1024^2 FP32 42 -> 15, 64^2 FP64 29 -> 5, a queue of
// 24 runs 42 -> 13.
template <class T, int ORDER>
__device__ __forceinline__ void corner_tiled_kernel_tile(
    const Blk& qb, const GridD& g, const Flags4& m, const FluxView<T>& fx, const FluxView<T>& fy,
    const double* __restrict__ cell_ez, const int* __restrict__ eqx, const int* __restrict__ eqy,
    double* __restrict__ ez) {
#include "tiles/corner_tiled_kernel.inc"
}

template <class T, int ORDER>
__global__ __launch_bounds__(256) void corner_tiled_kernel(GridD g, Flags4 m, FluxView<T> fx, FluxView<T> fy,
                                                           const double* __restrict__ cell_ez,
                                                           const int* __restrict__ eqx, const int* __restrict__ eqy,
                                                           double* __restrict__ ez) {
  [[maybe_unused]] const Blk qb = Blk::xcd_tiled();
#include "tiles/corner_tiled_kernel.inc"
}

// Queue form of corner_tiled_kernel (one launch over the tiles of many runs).
template <class T, int ORDER>
struct corner_tiled_kernel_q {
  struct Args {
    GridD g;
    Flags4 m;
    FluxView<T> fx;
    FluxView<T> fy;
    const double* cell_ez;
    const int* eqx;
    const int* eqy;
    double* ez;
  };
  static __device__ __forceinline__ void run(const Blk& qb, const Args& a) {
    corner_tiled_kernel_tile<T, ORDER>(qb, queue_arg(a.g), queue_arg(a.m), queue_arg(a.fx), queue_arg(a.fy),
                                       queue_arg(a.cell_ez), queue_arg(a.eqx), queue_arg(a.eqy), queue_arg(a.ez));
  }
  static void launch(dim3 grid, dim3 block, hipStream_t s, const Args& a) {
    hipLaunchKernelGGL((corner_tiled_kernel<T, ORDER>), grid, block, 0, s, a.g, a.m, a.fx, a.fy, a.cell_ez, a.eqx,
                       a.eqy, a.ez);
  }
  static const void* tag() {
    static const char t = 0;
    return &t;
  }
};

// corner_tiled_kernel over the tile queue, one workgroup per tile: the same text, the
// arguments read from the tile's run record.
template <class T, int ORDER>
__global__ __launch_bounds__(256) void corner_tiled_kernel_queue(
    const typename corner_tiled_kernel_q<T, ORDER>::Args* __restrict__ qargs, const QueueRun* __restrict__ qruns,
    int qnruns) {
  const QueueTile qtile = queue_tile(qruns, qnruns);
  [[maybe_unused]] const Blk qb = qtile.blk;
  const typename corner_tiled_kernel_q<T, ORDER>::Args& qa = qargs[qtile.run];
  GridD g = qa.g;
  Flags4 m = qa.m;
  FluxView<T> fx = queue_arg(qa.fx);
  FluxView<T> fy = queue_arg(qa.fy);
  const double* __restrict__ cell_ez = queue_arg(qa.cell_ez);
  const int* __restrict__ eqx = queue_arg(qa.eqx);
  const int* __restrict__ eqy = queue_arg(qa.eqy);
  double* __restrict__ ez = queue_arg(qa.ez);
#include "tiles/corner_tiled_kernel.inc"
}
template <class T, int ORDER>
struct QueueTiles<corner_tiled_kernel_q<T, ORDER>> {
  static constexpr auto kernel = &corner_tiled_kernel_queue<T, ORDER>;
};

// ---------------------------------------------------------------------------
// Fused residual + Shu-Osher stage: out = a Un + b Us + c L(U) with
// L = -div F for the cell components and the EMF curl for the faces.  A zero
// weight never reads its operand (rejected stages may hold NaN).

__device__ __forceinline__ double rk_combine(double a, double un, double b, double us, double c, double d) {
  const bool ua = a != 0.0, ub = b != 0.0, uc = c != 0.0;
  if (ua) {
    if (ub) return uc ? fma(c, d, fma(b, us, a * un)) : fma(b, us, a * un);
    return uc ? fma(c, d, a * un) : a * un;
  }
  if (ub) return uc ? fma(c, d, b * us) : b * us;
  return uc ? c * d : 0.0;
}

template <class T>
__device__ __forceinline__ void update_kernel_tile(
    const Blk& qb, const GridD& g, double a, double b, double cw, const double* __restrict__ dt_dev,
    const StateView& un, const StateView& us, const FluxView<T>& fx, const FluxView<T>& fy,
    const double* __restrict__ ez, const StateOut& out) {
#include "tiles/update_kernel.inc"
}

template <class T>
__global__ __launch_bounds__(256) void update_kernel(GridD g, double a, double b, double cw,
                                                     const double* __restrict__ dt_dev, StateView un, StateView us,
                                                     FluxView<T> fx, FluxView<T> fy, const double* __restrict__ ez,
                                                     StateOut out) {
  [[maybe_unused]] const Blk qb = Blk::xcd_tiled();
#include "tiles/update_kernel.inc"
}

// Queue form of update_kernel (one launch over the tiles of many runs).
template <class T>
struct update_kernel_q {
  struct Args {
    GridD g;
    double a;
    double b;
    double cw;
    const double* dt_dev;
    StateView un;
    StateView us;
    FluxView<T> fx;
    FluxView<T> fy;
    const double* ez;
    StateOut out;
  };
  static __device__ __forceinline__ void run(const Blk& qb, const Args& a) {
    update_kernel_tile<T>(qb, queue_arg(a.g), queue_arg(a.a), queue_arg(a.b), queue_arg(a.cw), queue_arg(a.dt_dev),
                          queue_arg(a.un), queue_arg(a.us), queue_arg(a.fx), queue_arg(a.fy), queue_arg(a.ez),
                          queue_arg(a.out));
  }
  static void launch(dim3 grid, dim3 block, hipStream_t s, const Args& a) {
    hipLaunchKernelGGL((update_kernel<T>), grid, block, 0, s, a.g, a.a, a.b, a.cw, a.dt_dev, a.un, a.us, a.fx, a.fy,
                       a.ez, a.out);
  }
  static const void* tag() {
    static const char t = 0;
    return &t;
  }
};

// update_kernel over the tile queue, one workgroup per tile: the same text, the
// arguments read from the tile's run record.
template <class T>
__global__ __launch_bounds__(256) void update_kernel_queue(const typename update_kernel_q<T>::Args* __restrict__ qargs,
    const QueueRun* __restrict__ qruns, int qnruns) {
  const QueueTile qtile = queue_tile(qruns, qnruns);
  [[maybe_unused]] const Blk qb = qtile.blk;
  const typename update_kernel_q<T>::Args& qa = qargs[qtile.run];
  GridD g = qa.g;
  double a = qa.a;
  double b = qa.b;
  double cw = qa.cw;
  const double* __restrict__ dt_dev = queue_arg(qa.dt_dev);
  StateView un = queue_arg(qa.un);
  StateView us = queue_arg(qa.us);
  FluxView<T> fx = queue_arg(qa.fx);
  FluxView<T> fy = queue_arg(qa.fy);
  const double* __restrict__ ez = queue_arg(qa.ez);
  StateOut out = queue_arg(qa.out);
#include "tiles/update_kernel.inc"
}
template <class T>
struct QueueTiles<update_kernel_q<T>> {
  static constexpr auto kernel = &update_kernel_queue<T>;
};

// ---------------------------------------------------------------------------
// Ghost fills: periodic / outflow / wall / axis maps per side, full padded
// transverse range so corner blocks are closed by the later y pass.

__device__ __forceinline__ void ghost_map(int n, int layer, bool lo, int mode, int& gi, int& si) {
  gi = lo ? -layer : n - 1 + layer;
  if (mode == 0)
    si = lo ? n - layer : layer - 1;
  else if (mode == 1)
    si = lo ? 0 : n - 1;
  else
    si = lo ? layer - 1 : n - layer;
}

__device__ __forceinline__ void ghost_kernel_tile(const Blk& qb, const GridD& g, int axis, const Flags4& fluid,
                                                  const Flags4& field, const StateOut& u) {
#include "tiles/ghost_kernel.inc"
}

__global__ __launch_bounds__(256) void ghost_kernel(GridD g, int axis, Flags4 fluid, Flags4 field, StateOut u) {
  [[maybe_unused]] const Blk qb = Blk::native();
#include "tiles/ghost_kernel.inc"
}

// Queue form of ghost_kernel (one launch over the tiles of many runs).
struct ghost_kernel_q {
  struct Args {
    GridD g;
    int axis;
    Flags4 fluid;
    Flags4 field;
    StateOut u;
  };
  static __device__ __forceinline__ void run(const Blk& qb, const Args& a) {
    ghost_kernel_tile(qb, queue_arg(a.g), queue_arg(a.axis), queue_arg(a.fluid), queue_arg(a.field), queue_arg(a.u));
  }
  static void launch(dim3 grid, dim3 block, hipStream_t s, const Args& a) {
    hipLaunchKernelGGL((ghost_kernel), grid, block, 0, s, a.g, a.axis, a.fluid, a.field, a.u);
  }
  static const void* tag() {
    static const char t = 0;
    return &t;
  }
};

// ghost_kernel over the tile queue, one workgroup per tile: the same text, the
// arguments read from the tile's run record.
__global__ __launch_bounds__(256) void ghost_kernel_queue(const ghost_kernel_q::Args* __restrict__ qargs,
    const QueueRun* __restrict__ qruns, int qnruns) {
  const QueueTile qtile = queue_tile(qruns, qnruns);
  [[maybe_unused]] const Blk qb = qtile.blk;
  const ghost_kernel_q::Args& qa = qargs[qtile.run];
  GridD g = qa.g;
  int axis = qa.axis;
  Flags4 fluid = qa.fluid;
  Flags4 field = qa.field;
  StateOut u = queue_arg(qa.u);
#include "tiles/ghost_kernel.inc"
}
template <>
struct QueueTiles<ghost_kernel_q> {
  static constexpr auto kernel = &ghost_kernel_queue;
};

// ---------------------------------------------------------------------------
// dt from the reduced rate (device side, for the auto-dt stepping loop).
__device__ __forceinline__ void dt_kernel_tile(
    const Blk& qb, const unsigned long long* __restrict__ max_rate_bits, double effective_cfl, double dx, double dy,
    double* __restrict__ dt_out, double* __restrict__ t_accum) {
#include "tiles/dt_kernel.inc"
}

__global__ void dt_kernel(const unsigned long long* __restrict__ max_rate_bits, double effective_cfl, double dx,
                          double dy, double* __restrict__ dt_out, double* __restrict__ t_accum) {
  [[maybe_unused]] const Blk qb = Blk::native();
#include "tiles/dt_kernel.inc"
}

// Queue form of dt_kernel (one launch over the tiles of many runs).
struct dt_kernel_q {
  struct Args {
    const unsigned long long* max_rate_bits;
    double effective_cfl;
    double dx;
    double dy;
    double* dt_out;
    double* t_accum;
  };
  static __device__ __forceinline__ void run(const Blk& qb, const Args& a) {
    dt_kernel_tile(qb, queue_arg(a.max_rate_bits), queue_arg(a.effective_cfl), queue_arg(a.dx), queue_arg(a.dy),
                   queue_arg(a.dt_out), queue_arg(a.t_accum));
  }
  static void launch(dim3 grid, dim3 block, hipStream_t s, const Args& a) {
    hipLaunchKernelGGL((dt_kernel), grid, block, 0, s, a.max_rate_bits, a.effective_cfl, a.dx, a.dy, a.dt_out, a.t_accum);
  }
  static const void* tag() {
    static const char t = 0;
    return &t;
  }
};

// dt_kernel over the tile queue, one workgroup per tile: the same text, the
// arguments read from the tile's run record.
__global__ void dt_kernel_queue(const dt_kernel_q::Args* __restrict__ qargs,
    const QueueRun* __restrict__ qruns, int qnruns) {
  const QueueTile qtile = queue_tile(qruns, qnruns);
  [[maybe_unused]] const Blk qb = qtile.blk;
  const dt_kernel_q::Args& qa = qargs[qtile.run];
  const unsigned long long* __restrict__ max_rate_bits = queue_arg(qa.max_rate_bits);
  double effective_cfl = qa.effective_cfl;
  double dx = qa.dx;
  double dy = qa.dy;
  double* __restrict__ dt_out = queue_arg(qa.dt_out);
  double* __restrict__ t_accum = queue_arg(qa.t_accum);
#include "tiles/dt_kernel.inc"
}
template <>
struct QueueTiles<dt_kernel_q> {
  static constexpr auto kernel = &dt_kernel_queue;
};

// ---------------------------------------------------------------------------
// Analytic initial conditions (two passes: primitives -> conserved with the raw
// magnetic energy, then energy re-formed with the collocated field).

__device__ __forceinline__ std::uint64_t mulhilo32(std::uint32_t a, std::uint32_t b, std::uint32_t& hi) {
  const std::uint64_t p = static_cast<std::uint64_t>(a) * b;
  hi = static_cast<std::uint32_t>(p >> 32);
  return p;
}

// Philox-4x32-10 (Salmon, Moraes, Dror, Shaw 2011): uniform on [-1, 1) from the
// 53 high bits of the first two output words.
__device__ double philox_pm1(std::uint64_t seed, std::uint32_t comp_id, std::uint64_t cell) {
  std::uint32_t c0 = static_cast<std::uint32_t>(cell), c1 = static_cast<std::uint32_t>(cell >> 32), c2 = comp_id, c3 = 0;
  std::uint32_t k0 = static_cast<std::uint32_t>(seed), k1 = static_cast<std::uint32_t>(seed >> 32);
  for (int r = 0; r < 10; ++r) {
    if (r > 0) {
      k0 += 0x9E3779B9u;
      k1 += 0xBB67AE85u;
    }
    std::uint32_t hi0, hi1;
    const std::uint32_t lo0 = static_cast<std::uint32_t>(mulhilo32(0xD2511F53u, c0, hi0));
    const std::uint32_t lo1 = static_cast<std::uint32_t>(mulhilo32(0xCD9E8D57u, c2, hi1));
    const std::uint32_t n0 = hi1 ^ c1 ^ k0, n2 = hi0 ^ c3 ^ k1;
    c0 = n0;
    c1 = lo1;
    c2 = n2;
    c3 = lo0;
  }
  const std::uint64_t bits = (static_cast<std::uint64_t>(c1) << 32) | c0;
  return 2.0 * (static_cast<double>(bits >> 11) * 0x1.0p-53) - 1.0;
}

__global__ __launch_bounds__(256) void seed_kernel(GridD g, IcSpecD s, StateOut out, double* __restrict__ raw_mag,
                                                   int* __restrict__ status) {
  const int i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x) - g.ng;
  const int j = static_cast<int>(blockIdx.y * blockDim.y + threadIdx.y) - g.ng;
  if (i >= g.nx + g.ng || j >= g.ny + g.ng) return;
  const double pi = 3.141592653589793238462643383279502884;
  const double xc = fma(static_cast<double>(i) + 0.5, g.dx, g.ox);
  const double yc = fma(static_cast<double>(j) + 0.5, g.dy, g.oy);
  double rho = 1, p = 1, vx = 0, vy = 0, vz = 0, bx = 0, by = 0, bz = 0, eoff = 0;
  switch (s.kind) {
    case 0: {
      const double* side = xc < s.interface_x ? s.left : s.right;
      rho = side[0]; p = side[1]; vx = side[2]; vy = side[3]; vz = side[4]; bx = side[5]; by = side[6]; bz = side[7];
      break;
    }
    case 1: {
      const double n = static_cast<double>(s.wavenumber);
      const double kw = 2.0 * pi * n / g.lx;
      const double phase = kw * (xc - g.ox);
      const double q = n / static_cast<double>(g.nx);
      const double fv = q == 0.0 ? 1.0 : sin(pi * q) / (pi * q);
      const double isr = copysign(s.magnetic_velocity_scale, s.total_b0) / sqrt(s.rho);
      rho = s.rho; p = s.pressure;
      vy = -s.amplitude * isr * fv * sin(phase);
      vz = -s.amplitude * isr * fv * cos(phase);
      bx = s.b0; by = s.amplitude * fv * sin(phase); bz = s.amplitude * fv * cos(phase);
      const double sa = s.amplitude * s.magnetic_velocity_scale;
      eoff = sa * sa * (1.0 - fv * fv);
      break;
    }
    case 2: {
      const double xi = (xc - g.ox) / g.lx, eta = (yc - g.oy) / g.ly;
      const double two_pi = 2.0 * pi;
      const double b0 = s.b_uniform[0];
      rho = s.ot_rho != 0.0 ? s.ot_rho : s.gamma * s.gamma;
      p = s.ot_p != 0.0 ? s.ot_p : s.gamma;
      vx = -sin(two_pi * eta);
      vy = sin(two_pi * xi);
      bx = -b0 * sin(two_pi * eta);
      by = b0 * sin(2.0 * two_pi * xi);
      break;
    }
    case 3: {
      const double r = hypot(xc - s.center[0], yc - s.center[1]);
      rho = s.rho_ambient; p = r < s.r_in ? s.p_core : s.p_ambient;
      bx = s.b_uniform[0]; by = s.b_uniform[1]; bz = s.b_uniform[2];
      break;
    }
    case 4: {
      const double rx = xc - s.center[0], ry = yc - s.center[1];
      const double r = hypot(rx, ry);
      double f = (s.r1 - r) / (s.r1 - s.r0);
      f = fmin(fmax(f, 0.0), 1.0);
      const bool inside = r <= s.r0;
      if (inside) f = 1.0;
      if (r >= s.r1) f = 0.0;
      double speed = 0.0;
      if (inside)
        speed = s.u0 / s.r0;
      else if (r < s.r1)
        speed = f * s.u0 / r;
      rho = s.rho_out + f * (s.rho_in - s.rho_out);
      p = s.p_ambient;
      vx = -speed * ry;
      vy = speed * rx;
      bx = s.b_uniform[0]; by = s.b_uniform[1]; bz = s.b_uniform[2];
      break;
    }
    case 5: {  // confined_blob (mhd_initial_conditions.hip:190-207): in-plane field zero
      const bool inside = fabs(xc - s.center[0]) <= s.blob_half && fabs(yc - s.center[1]) <= s.blob_half;
      rho = inside ? s.rho_in : s.rho_out;
      p = inside ? s.p_in : s.p_out;
      bz = s.b_uniform[2];
      break;
    }
    default:
      atomicOr(status, 1);
      return;
  }
  if (s.noise_amplitude != 0.0) {
    int wi = i % g.nx;
    if (wi < 0) wi += g.nx;
    int wj = j % g.ny;
    if (wj < 0) wj += g.ny;
    const std::uint64_t cell = static_cast<std::uint64_t>(wj) * static_cast<std::uint64_t>(g.nx) + static_cast<std::uint64_t>(wi);
    rho = rho * (1.0 + s.noise_amplitude * philox_pm1(s.noise_seed, 0, cell));
    vx = vx + s.noise_amplitude * philox_pm1(s.noise_seed, 1, cell);
    vy = vy + s.noise_amplitude * philox_pm1(s.noise_seed, 2, cell);
  }
  if (!(fin(rho) && rho > 0.0)) {
    atomicOr(status, 2);
    return;
  }
  if (!(fin(p) && p > 0.0)) {
    atomicOr(status, 4);
    return;
  }
  // Scaled forms of rho|v|^2/2 and |B|^2/2 as the reference seeds them.
  auto kin_v = [](double r, double x, double y, double z) {
    const double sc = fmax(fabs(x), fmax(fabs(y), fabs(z)));
    if (sc == 0.0) return 0.0;
    const double xs = x / sc, ys = y / sc, zs = z / sc;
    const double q = sqrt(r) * sc;
    return (0.5 * q) * (q * (xs * xs + ys * ys + zs * zs));
  };
  auto hsq = [](double x, double y, double z) {
    const double sc = fmax(fabs(x), fmax(fabs(y), fabs(z)));
    if (sc == 0.0) return 0.0;
    const double xs = x / sc, ys = y / sc, zs = z / sc;
    return (0.5 * sc) * (sc * (xs * xs + ys * ys + zs * zs));
  };
  const double kin = kin_v(rho, vx, vy, vz);
  const double mag = hsq(bx, by, bz);
  const std::size_t k = idx(g, i, j);
  out.c[0][k] = rho;
  out.c[1][k] = rho * vx;
  out.c[2][k] = rho * vy;
  out.c[3][k] = rho * vz;
  out.c[4][k] = p / (s.gamma - 1.0) + kin + mag + eoff;
  out.c[5][k] = s.magnetic_scale * bx;
  out.c[6][k] = s.magnetic_scale * by;
  out.c[7][k] = s.magnetic_scale * bz;
  raw_mag[k] = mag;
}

__global__ __launch_bounds__(256) void recollocate_kernel(
    GridD g, double gamma, StateOut out, const double* __restrict__ raw_mag, int* __restrict__ status) {
  const int i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x) - g.ng;
  const int j = static_cast<int>(blockIdx.y * blockDim.y + threadIdx.y) - g.ng;
  if (i >= g.nx + g.ng || j >= g.ny + g.ng) return;
  const std::size_t k = idx(g, i, j);
  const double bxc = face_to_cell(g, out.c[5], 0, i, j);
  const double byc = face_to_cell(g, out.c[6], 1, j, i);
  const double bz = out.c[7][k];
  const double sc = fmax(fabs(bxc), fmax(fabs(byc), fabs(bz)));
  double mag = 0.0;
  if (sc != 0.0) {
    const double xs = bxc / sc, ys = byc / sc, zs = bz / sc;
    mag = (0.5 * sc) * (sc * (xs * xs + ys * ys + zs * zs));
  }
  const double e = (out.c[4][k] - raw_mag[k]) + mag;
  out.c[4][k] = e;
  const St<double> st{out.c[0][k], out.c[1][k], out.c[2][k], out.c[3][k], e, bxc, byc, bz};
  if (!(pressure(st, gamma - 1.0) > 0.0)) atomicOr(status, 4);
}

// ---------------------------------------------------------------------------
// Launch-level helpers mirroring the reference ABI.

__global__ __launch_bounds__(256) void rk_combine_kernel(GridD g, double a, double b, double c, StateView un,
                                                         StateView us, StateView dudt, StateOut out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y * blockDim.y + threadIdx.y;
  if (i > g.nx || j > g.ny) return;
  const bool copy = a == 1.0 && b == 0.0 && c == 0.0;
  const std::size_t k = idx(g, i, j);
  for (int cc = 0; cc < 8; ++cc) {
    const bool active = cc == 5 ? j < g.ny : cc == 6 ? i < g.nx : (i < g.nx && j < g.ny);
    if (!active) continue;
    out.c[cc][k] = copy ? un.c[cc][k]
                        : rk_combine(a, un.c[cc][k], b, b != 0.0 ? us.c[cc][k] : 0.0, c,
                                     c != 0.0 ? dudt.c[cc][k] : 0.0);
  }
}

__global__ __launch_bounds__(256) void divb_linf_kernel(GridD g, StateView u, unsigned long long* out) {
  __shared__ double lds[4];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double local = 0.0;
  for (int r = 0; r < kRowsPerThread; ++r) {
    const int j = (blockIdx.y * kRowsPerThread + r) * blockDim.y + threadIdx.y;
    if (i < g.nx && j < g.ny) {
      const double d = (u.c[5][idx(g, i + 1, j)] - u.c[5][idx(g, i, j)]) / g.dx +
                       (u.c[6][idx(g, i, j + 1)] - u.c[6][idx(g, i, j)]) / g.dy;
      local = fmax(local, fin(d) ? __builtin_fabs(d) : Lim<double>::inf());
    }
  }
  local = block_reduce<true>(local, lds);
  if (block_leader()) atomic_max_nonneg(out, local);
}

__global__ __launch_bounds__(256) void theta_kernel(GridD g, StateView base, StateView cand, int co,
                                                    unsigned long long* out) {
  __shared__ double lds[4];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double th = 1.0;
  for (int r = 0; r < kRowsPerThread; ++r) {
    const int j = (blockIdx.y * kRowsPerThread + r) * blockDim.y + threadIdx.y;
    if (i < g.nx && j < g.ny) {
      const std::size_t k = idx(g, i, j);
      const double bxa = co == 1 ? face_to_cell_lo(g, base.c[5], 0, i, j) : face_to_cell(g, base.c[5], 0, i, j);
      const double bya = co == 1 ? face_to_cell_lo(g, base.c[6], 1, j, i) : face_to_cell(g, base.c[6], 1, j, i);
      const double bxb = co == 1 ? face_to_cell_lo(g, cand.c[5], 0, i, j) : face_to_cell(g, cand.c[5], 0, i, j);
      const double byb = co == 1 ? face_to_cell_lo(g, cand.c[6], 1, j, i) : face_to_cell(g, cand.c[6], 1, j, i);
      th = fmin(th, ok_or_zero(admissible_theta(cell_state(g, base, k, bxa, bya), cell_state(g, cand, k, bxb, byb))));
    }
  }
  th = block_reduce<false>(th, lds);
  if (block_leader()) atomic_min_nonneg(out, th);
}

// Per-block compensated (two-sum) partial sums of mass and energy; the host
// folds the 2x2 partials per block exactly.
__global__ __launch_bounds__(256) void cell_sums_kernel(GridD g, StateView u, double* __restrict__ partials) {
  __shared__ double s_val[4][256];
  const int tid = threadIdx.x;
  double sm = 0.0, cm = 0.0, se = 0.0, ce = 0.0;
  const long long cells = static_cast<long long>(g.nx) * g.ny;
  for (long long c = blockIdx.x * 256LL + tid; c < cells; c += static_cast<long long>(gridDim.x) * 256) {
    const int i = static_cast<int>(c % g.nx), j = static_cast<int>(c / g.nx);
    const std::size_t k = idx(g, i, j);
    {
      const double x = u.c[0][k];
      const double t = sm + x;
      const double bp = t - sm;
      cm += (sm - (t - bp)) + (x - bp);
      sm = t;
    }
    {
      const double x = u.c[4][k];
      const double t = se + x;
      const double bp = t - se;
      ce += (se - (t - bp)) + (x - bp);
      se = t;
    }
  }
  s_val[0][tid] = sm;
  s_val[1][tid] = cm;
  s_val[2][tid] = se;
  s_val[3][tid] = ce;
  __syncthreads();
  if (tid < 4) {
    // Exact-enough per-block fold of 256 (sum, correction) pairs with two-sum.
    double s = 0.0, comp_acc = 0.0;
    for (int t = 0; t < 256; ++t) {
      const double x = s_val[tid][t];
      const double r = s + x;
      const double bp = r - s;
      comp_acc += (s - (r - bp)) + (x - bp);
      s = r;
    }
    partials[(blockIdx.x * 4 + tid) * 2 + 0] = s;
    partials[(blockIdx.x * 4 + tid) * 2 + 1] = comp_acc;
  }
}

__global__ __launch_bounds__(256) void eq_flag_kernel(GridD g, int dir, IfaceView<double> in, int* __restrict__ eq) {
  const int li = blockIdx.x * blockDim.x + threadIdx.x;
  const int lj = blockIdx.y * blockDim.y + threadIdx.y;
  const int i = dir == 1 ? li - g.ng : li;
  const int j = dir == 0 ? lj - g.ng : lj;
  if (dir == 0) {
    if (li > g.nx || lj >= g.ny + 2 * g.ng) return;
  } else {
    if (li >= g.nx + 2 * g.ng || lj > g.ny) return;
  }
  const std::size_t k = idx(g, i, j);
  bool e = true;
  for (int c = 0; c < 8; ++c) e = e && (in.c[c][k] == in.c[8 + c][k]);
  eq[k] = e ? 1 : 0;
}

__global__ __launch_bounds__(256) void flux_diff_kernel(GridD g, int dir, FluxView<double> f, StateOut d) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y * blockDim.y + threadIdx.y;
  if (i >= g.nx || j >= g.ny) return;
  const std::size_t k = idx(g, i, j);
  const std::size_t kp = dir == 0 ? idx(g, i + 1, j) : idx(g, i, j + 1);
  const double sp = dir == 0 ? g.dx : g.dy;
  for (int c = 0; c < 8; ++c) d.c[c][k] += -((f.c[c][kp] - f.c[c][k]) / sp);
}

__global__ __launch_bounds__(256) void curl_kernel(GridD g, const double* __restrict__ ez, double* __restrict__ dbx,
                                                   double* __restrict__ dby) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y * blockDim.y + threadIdx.y;
  if (i > g.nx || j > g.ny) return;
  const std::size_t k = idx(g, i, j);
  if (j < g.ny) dbx[k] = (ez[k] - ez[idx(g, i, j + 1)]) / g.dy;
  if (i < g.nx) dby[k] = (ez[idx(g, i + 1, j)] - ez[k]) / g.dx;
}

// Reset of the step status block by a kernel (no memset node in a captured graph).
__device__ __forceinline__ void status_reset_kernel_tile(const Blk& qb, StepStatus* s) {
#include "tiles/status_reset_kernel.inc"
}

__global__ void status_reset_kernel(StepStatus* s) {
  [[maybe_unused]] const Blk qb = Blk::native();
#include "tiles/status_reset_kernel.inc"
}

// Queue form of status_reset_kernel (one launch over the tiles of many runs).
struct status_reset_kernel_q {
  struct Args {
    StepStatus* s;
  };
  static __device__ __forceinline__ void run(const Blk& qb, const Args& a) {
    status_reset_kernel_tile(qb, queue_arg(a.s));
  }
  static void launch(dim3 grid, dim3 block, hipStream_t s, const Args& a) {
    hipLaunchKernelGGL((status_reset_kernel), grid, block, 0, s, a.s);
  }
  static const void* tag() {
    static const char t = 0;
    return &t;
  }
};

// status_reset_kernel over the tile queue, one workgroup per tile: the same text, the
// arguments read from the tile's run record.
__global__ void status_reset_kernel_queue(const status_reset_kernel_q::Args* __restrict__ qargs,
    const QueueRun* __restrict__ qruns, int qnruns) {
  const QueueTile qtile = queue_tile(qruns, qnruns);
  [[maybe_unused]] const Blk qb = qtile.blk;
  const status_reset_kernel_q::Args& qa = qargs[qtile.run];
  StepStatus* s = queue_arg(qa.s);
#include "tiles/status_reset_kernel.inc"
}
template <>
struct QueueTiles<status_reset_kernel_q> {
  static constexpr auto kernel = &status_reset_kernel_queue;
};

// Batched launcher: accept or reject the attempt on the device with the
// host run loop's rule (python/quasar/mhd/cli.py:386-491 with
// src/physics/mhd/mhd_solver.cpp:965-1143): the live state must be
// admissible and discretely solenoidal and the CFL rate finite (otherwise the
// run is stopped), and every stage of the attempt admissible (otherwise the
// step is rejected and the run is held: its later attempts in the same batch
// call commit nothing, and the host's positivity controller finishes its
// steps after the graph launches).
__device__ __forceinline__ void batch_commit_kernel_tile(const Blk& qb, StepStatus* __restrict__ st,
                                                         double* __restrict__ acc) {
#include "tiles/batch_commit_kernel.inc"
}

__global__ void batch_commit_kernel(StepStatus* __restrict__ st, double* __restrict__ acc) {
  [[maybe_unused]] const Blk qb = Blk::native();
#include "tiles/batch_commit_kernel.inc"
}

// Queue form of batch_commit_kernel (one launch over the tiles of many runs).
struct batch_commit_kernel_q {
  struct Args {
    StepStatus* st;
    double* acc;
  };
  static __device__ __forceinline__ void run(const Blk& qb, const Args& a) {
    batch_commit_kernel_tile(qb, queue_arg(a.st), queue_arg(a.acc));
  }
  static void launch(dim3 grid, dim3 block, hipStream_t s, const Args& a) {
    hipLaunchKernelGGL((batch_commit_kernel), grid, block, 0, s, a.st, a.acc);
  }
  static const void* tag() {
    static const char t = 0;
    return &t;
  }
};

// batch_commit_kernel over the tile queue, one workgroup per tile: the same text, the
// arguments read from the tile's run record.
__global__ void batch_commit_kernel_queue(const batch_commit_kernel_q::Args* __restrict__ qargs,
    const QueueRun* __restrict__ qruns, int qnruns) {
  const QueueTile qtile = queue_tile(qruns, qnruns);
  [[maybe_unused]] const Blk qb = qtile.blk;
  const batch_commit_kernel_q::Args& qa = qargs[qtile.run];
  StepStatus* __restrict__ st = queue_arg(qa.st);
  double* __restrict__ acc = queue_arg(qa.acc);
#include "tiles/batch_commit_kernel.inc"
}
template <>
struct QueueTiles<batch_commit_kernel_q> {
  static constexpr auto kernel = &batch_commit_kernel_queue;
};

__device__ __forceinline__ void batch_restore_kernel_tile(const Blk& qb, std::size_t n, const double* __restrict__ acc,
                                                            const StateView& live, const StateOut& cand) {
#include "tiles/batch_restore_kernel.inc"
}

__global__ __launch_bounds__(256) void batch_restore_kernel(std::size_t n, const double* __restrict__ acc,
                                                            StateView live, StateOut cand) {
  [[maybe_unused]] const Blk qb = Blk::native();
#include "tiles/batch_restore_kernel.inc"
}

// Queue form of batch_restore_kernel (one launch over the tiles of many runs).
struct batch_restore_kernel_q {
  struct Args {
    std::size_t n;
    const double* acc;
    StateView live;
    StateOut cand;
  };
  static __device__ __forceinline__ void run(const Blk& qb, const Args& a) {
    batch_restore_kernel_tile(qb, queue_arg(a.n), queue_arg(a.acc), queue_arg(a.live), queue_arg(a.cand));
  }
  static void launch(dim3 grid, dim3 block, hipStream_t s, const Args& a) {
    hipLaunchKernelGGL((batch_restore_kernel), grid, block, 0, s, a.n, a.acc, a.live, a.cand);
  }
  static const void* tag() {
    static const char t = 0;
    return &t;
  }
};

// batch_restore_kernel over the tile queue, one workgroup per tile: the same text, the
// arguments read from the tile's run record.
__global__ __launch_bounds__(256) void batch_restore_kernel_queue(
    const batch_restore_kernel_q::Args* __restrict__ qargs, const QueueRun* __restrict__ qruns, int qnruns) {
  const QueueTile qtile = queue_tile(qruns, qnruns);
  [[maybe_unused]] const Blk qb = qtile.blk;
  const batch_restore_kernel_q::Args& qa = qargs[qtile.run];
  std::size_t n = qa.n;
  const double* __restrict__ acc = queue_arg(qa.acc);
  StateView live = queue_arg(qa.live);
  StateOut cand = queue_arg(qa.cand);
#include "tiles/batch_restore_kernel.inc"
}
template <>
struct QueueTiles<batch_restore_kernel_q> {
  static constexpr auto kernel = &batch_restore_kernel_queue;
};

// ---------------------------------------------------------------------------
// Host launchers.

void launch_batch_commit(StepStatus* status, double* acc, hipStream_t stream) {
  go<batch_commit_kernel_q>(dim3(1), dim3(64), stream, status, acc);
}

void launch_batch_restore(const GridD& g, const double* acc, const StateView& live, const StateOut& cand,
                          hipStream_t stream) {
  const std::size_t n = static_cast<std::size_t>(g.pitch) * (g.ny + 2 * g.ng);
  go<batch_restore_kernel_q>(dim3(256), dim3(256), stream, n, acc, live, cand);
}

void launch_eq_flags(const GridD& g, int dir, const IfaceView<double>& in, int* eq, hipStream_t stream) {
  const dim3 b(64, 4);
  const int lx = dir == 0 ? g.nx + 1 : g.nx + 2 * g.ng;
  const int ly = dir == 0 ? g.ny + 2 * g.ng : g.ny + 1;
  hipLaunchKernelGGL(eq_flag_kernel, dim3((lx + 63) / 64, (ly + 3) / 4), b, 0, stream, g, dir, in, eq);
}

void launch_flux_difference(const GridD& g, int dir, const FluxView<double>& f, const StateOut& d,
                            hipStream_t stream) {
  const dim3 b(64, 4);
  hipLaunchKernelGGL(flux_diff_kernel, dim3((g.nx + 63) / 64, (g.ny + 3) / 4), b, 0, stream, g, dir, f, d);
}

void launch_curl(const GridD& g, const double* ez, double* dbx, double* dby, hipStream_t stream) {
  const dim3 b(64, 4);
  hipLaunchKernelGGL(curl_kernel, dim3((g.nx + 64) / 64, (g.ny + 4) / 4), b, 0, stream, g, ez, dbx, dby);
}

void launch_status_reset(StepStatus* s, hipStream_t stream) {
  go<status_reset_kernel_q>(dim3(1), dim3(64), stream, s);
}

namespace {
inline dim3 blocks2d(int nx, int ny, dim3 b) { return dim3((nx + b.x - 1) / b.x, (ny + b.y - 1) / b.y); }
}  // namespace

void launch_prep(const GridD& g, const StateView& u, double* bxc, double* byc, const StateView& base,
                 const double* base_bxc, const double* base_byc, int theta_slot, int theta_co, int theta_both,
                 int live_checks, int solver_owned, StepStatus* status, hipStream_t stream, bool exact) {
  const dim3 b(64, 4);
  const dim3 cells = blocks2d(g.nx + 2 * g.ng, g.ny + 2 * g.ng, b);
  auto prep = [&](auto q) {
    const int strips = prep_strip_blocks<decltype(q)::kWindow>(g);
    go<decltype(q)>(dim3(strips + cells.x * cells.y), b, stream, g, u, bxc, byc, base, base_bxc, base_byc, theta_slot, theta_co, theta_both,
                    live_checks, solver_owned, status);
  };
  // The padded extents hold the halo's full window (2 ng + 1 cells at least).
  auto by_form = [&](auto exact_q, auto fma_q) { exact ? prep(exact_q) : prep(fma_q); };
  if (g.ng >= 4)
    by_form(prep_kernel_q<true, 8>{}, prep_kernel_q<false, 8>{});
  else if (g.ng == 3)
    by_form(prep_kernel_q<true, 6>{}, prep_kernel_q<false, 6>{});
  else if (g.ng == 2)
    by_form(prep_kernel_q<true, 4>{}, prep_kernel_q<false, 4>{});
  else
    by_form(prep_kernel_q<true, 2>{}, prep_kernel_q<false, 2>{});
}

void launch_collocate(const GridD& g, int axis, int co, const double* face, double* cell, hipStream_t stream) {
  const dim3 b(64, 4);
  hipLaunchKernelGGL(collocate_kernel, blocks2d(g.nx + 2 * g.ng, g.ny + 2 * g.ng, b), b, 0, stream, g, axis, co, face,
                     cell);
}

void launch_counter_reset(unsigned long long* counters, int n, hipStream_t stream) {
  hipLaunchKernelGGL(counter_reset_kernel, dim3(1), dim3(64), 0, stream, counters, n);
}

// Faces of a reconstruction launch along x and y.
static dim3 recon_faces(const GridD& g, int dir) {
  return dir == 0 ? dim3(g.nx + 1, g.ny + 2 * g.ng) : dim3(g.nx + 2 * g.ng, g.ny + 1);
}
// Blocks over a face list: no more than it can fill (a queue batch launches
// every run's).
static dim3 list_blocks_of(const GridD& g, int dir, std::size_t most) {
  const dim3 l = recon_faces(g, dir);
  return dim3(static_cast<unsigned>(std::min<std::size_t>(most, (static_cast<std::size_t>(l.x) * l.y + 255) / 256)));
}
static int periodic_of(const Flags4& flags, int dir) {
  return flags.side[2 * dir] == 0 && flags.side[2 * dir + 1] == 0;
}

template <class T>
void launch_reconstruct(const GridD& g, int order, double gamma, const Flags4& flags, const StateView& u,
                        const double* bxc, const double* byc, const FaceOut<T>* out, int first, int count,
                        hipStream_t stream) {
  const T gamma_t = T(gamma);
  auto launch = [&](auto faces, auto fallback) {
    using F = decltype(faces);
    using B = decltype(fallback);
    dim3 grid[2]{dim3(0, 0), dim3(0, 0)}, fb_grid[2]{dim3(0, 0), dim3(0, 0)};
    typename F::Args a[2];
    typename B::Args b[2];
    for (int k = 0; k < 2; ++k) {
      const int dir = k < count ? first + k : first;
      const FaceOut<T>& o = out[k < count ? k : 0];
      const int slo = flags.side[2 * dir], shi = flags.side[2 * dir + 1];
      a[k] = {g, dir, gamma_t, slo, shi, u, bxc, byc, o.states, o.eq, o.list.count, o.list.faces};
      b[k] = {g, dir, gamma_t, slo, shi, u, bxc, byc, o.states, o.eq, o.list.count, o.list.faces};
      if (k >= count) continue;
      const dim3 l = recon_faces(g, dir);
      grid[k] = blocks2d(l.x, l.y, dim3(kReconTiles[dir][0], kReconTiles[dir][1]));
      fb_grid[k] = list_blocks_of(g, dir, 64);
    }
    go_pair<F>(grid[0], a[0], grid[1], a[1], dim3(256), stream);
    if (order >= 2) go_pair<B>(fb_grid[0], b[0], fb_grid[1], b[1], dim3(256), stream);
  };
  switch (order) {
    case 1: launch(reconstruct_kernel_q<T, 1>{}, reconstruct_fallback_kernel_q<T, 5>{}); break;
    case 2: launch(reconstruct_kernel_q<T, 2>{}, reconstruct_fallback_kernel_q<T, 2>{}); break;
    case 5: launch(reconstruct_kernel_q<T, 5>{}, reconstruct_fallback_kernel_q<T, 5>{}); break;
    default: launch(reconstruct_kernel_q<T, 7>{}, reconstruct_fallback_kernel_q<T, 7>{}); break;
  }
}

template <class T>
void launch_reconstruct_learned(const GridD& g, int order, double gamma, const Flags4& flags, const StateView& u,
                                const double* bxc, const double* byc, const uint8_t* cell_flags,
                                const FaceOut<T>* out, unsigned long long* plain_total, hipStream_t stream,
                                int list_blocks, int cheap_tile) {
  const T gamma_t = T(gamma);
  if (cheap_tile < 0 || cheap_tile >= kCheapTileCount)
    throw std::invalid_argument("reconstruct launch: cheap tile choice is 0..4");
  const dim3 cb(kCheapTiles[cheap_tile][0], kCheapTiles[cheap_tile][1]);
  auto side = [&](int dir) {
    const FaceOut<T>& o = out[dir];
    return CheapFace<T>{o.states, o.eq, o.list.count, o.list.faces, o.flux, o.rate, periodic_of(flags, dir)};
  };
  auto cheap = [&](auto q) {
    go<decltype(q)>(blocks2d(g.nx + 2 * g.ng, g.ny + 2 * g.ng, cb), cb, stream, g, gamma_t, u, bxc, byc, cell_flags,
                    side(0), side(1));
  };
  switch (cheap_tile) {
    case 0: cheap(cheap_reconstruct_kernel_q<T, kCheapTiles[0][0], kCheapTiles[0][1]>{}); break;
    case 1: cheap(cheap_reconstruct_kernel_q<T, kCheapTiles[1][0], kCheapTiles[1][1]>{}); break;
    case 2: cheap(cheap_reconstruct_kernel_q<T, kCheapTiles[2][0], kCheapTiles[2][1]>{}); break;
    case 3: cheap(cheap_reconstruct_kernel_q<T, kCheapTiles[3][0], kCheapTiles[3][1]>{}); break;
    default: cheap(cheap_reconstruct_kernel_q<T, kCheapTiles[4][0], kCheapTiles[4][1]>{}); break;
  }
  // Enough blocks to fill the device at the MP kernel's occupancy (the plain
  // list can hold a large share of the faces), no more than the list can fill:
  // one block per possible slot spent 25 us at 4096^2 on blocks without work.
  auto launch = [&](auto listed, auto fallback) {
    using F = decltype(listed);
    using B = decltype(fallback);
    dim3 grid[2];
    typename F::Args a[2];
    typename B::Args b[2];
    for (int dir = 0; dir < 2; ++dir) {
      const FaceOut<T>& o = out[dir];
      grid[dir] = list_blocks_of(g, dir, list_blocks);
      a[dir] = {g, dir, gamma_t, u, bxc, byc, o.states, o.eq, o.list.count, o.list.faces, o.redo.count, o.redo.faces,
                plain_total};
      b[dir] = {g, dir, gamma_t, flags.side[2 * dir], flags.side[2 * dir + 1], u, bxc, byc, o.states, o.eq,
                o.redo.count, o.redo.faces};
    }
    go_pair<F>(grid[0], a[0], grid[1], a[1], dim3(256), stream);
    go_pair<B>(grid[0], b[0], grid[1], b[1], dim3(256), stream);
  };
  if (order == 5)
    launch(reconstruct_list_kernel_q<T, 5>{}, reconstruct_fallback_kernel_q<T, 5>{});
  else
    launch(reconstruct_list_kernel_q<T, 7>{}, reconstruct_fallback_kernel_q<T, 7>{});
}

template <class T>
void launch_flux(const GridD& g, int order, int hll_only, const Flags4& flags, double gamma, const FaceOut<T>* face,
                 int first, int count, hipStream_t stream, dim3 b) {
  const bool mp = order != 1 && order != 2;
  auto launch = [&](auto q) {
    using F = decltype(q);
    dim3 grid[2]{dim3(0, 0), dim3(0, 0)};
    typename F::Args a[2];
    for (int k = 0; k < 2; ++k) {
      const int dir = k < count ? first + k : first;
      const FaceOut<T>& o = face[k < count ? k : 0];
      a[k] = {g, dir, periodic_of(flags, dir), T(gamma), o.states, o.flux, o.rate};
      if (k < count)
        grid[k] = blocks2d(g.nx + 1, g.ny + 1, mp ? dim3(kFluxTiles[dir][0], kFluxTiles[dir][1]) : b);
    }
    go_pair<F>(grid[0], a[0], grid[1], a[1], mp ? dim3(256) : b, stream);
  };
  switch (order) {
    case 1: hll_only ? launch(flux_kernel_q<T, 1, true>{}) : launch(flux_kernel_q<T, 1, false>{}); break;
    case 2: hll_only ? launch(flux_kernel_q<T, 2, true>{}) : launch(flux_kernel_q<T, 2, false>{}); break;
    case 5: hll_only ? launch(flux_kernel_q<T, 5, true>{}) : launch(flux_kernel_q<T, 5, false>{}); break;
    default: hll_only ? launch(flux_kernel_q<T, 7, true>{}) : launch(flux_kernel_q<T, 7, false>{}); break;
  }
}

template <class T>
void launch_flux_learned(const GridD& g, int order, const Flags4& flags, double gamma, const FaceOut<T>* face,
                         const uint8_t* cell_flags, hipStream_t stream, int list_blocks) {
  if (order != 5 && order != 7) throw std::invalid_argument("flux launch: the learned form runs MP5/MP7");
  auto launch = [&](auto q) {
    using F = decltype(q);
    dim3 grid[2];
    typename F::Args a[2];
    for (int dir = 0; dir < 2; ++dir) {
      const FaceOut<T>& o = face[dir];
      const dim3 l = recon_faces(g, dir);
      const std::size_t most = (static_cast<std::size_t>(l.x) * l.y + kFluxListBlock - 1) / kFluxListBlock;
      grid[dir] = dim3(static_cast<unsigned>(std::min(static_cast<std::size_t>(list_blocks) * 256 / kFluxListBlock, most)));
      a[dir] = {g, dir, periodic_of(flags, dir), T(gamma), o.states, o.flux, o.rate, cell_flags, o.list.count,
                o.list.faces};
    }
    go_pair<F>(grid[0], a[0], grid[1], a[1], dim3(kFluxListBlock), stream);
  };
  if (order == 5)
    launch(flux_plain_list_kernel_q<T, 5>{});
  else
    launch(flux_plain_list_kernel_q<T, 7>{});
}

void launch_cfl_reduce(const GridD& g, const double* rate_x, const double* rate_y, unsigned long long* max_rate,
                       hipStream_t stream) {
  const dim3 b(64, 4);
  go<cfl_reduce_kernel_q>(blocks2d(g.nx, g.ny, dim3(64, 4 * kRowsPerThread)), b, stream, g, rate_x, rate_y, max_rate);
}

template <class T>
void launch_cell_emf(const GridD& g, int order, const Flags4& flags, double gamma, const StateView& u,
                     const double* bxc, const double* byc, double* cell_ez, hipStream_t stream,
                     const uint8_t* cell_flags, int tile) {
  const int pxh = flags.side[1] != 0 && flags.side[1] != 4;
  const int pyh = flags.side[3] != 0 && flags.side[3] != 4;
  if (order == 5 || order == 7) {
    if (tile < 0 || tile > 2) throw std::invalid_argument("cell E_z launch: tile choice is 0..2");
    const int columns = std::max(16, kEmfTiles[tile][0]);
    auto blocks = [&](int m) { return blocks2d(g.nx + 1, g.ny + 1, dim3(columns, m * kEmfTiles[tile][1])); };
    auto many = [&](int m) { return blocks(m).x * blocks(m).y >= kEmfBlocks; };
    const int march = cell_flags ? 1 : many(4) ? 4 : many(2) ? 2 : 1;
    const dim3 b(256), grid = blocks(march);
    auto launch = [&](auto q) {
      go<decltype(q)>(grid, b, stream, g, pxh, pyh, T(gamma), u, bxc, byc, cell_ez, cell_flags, march);
    };
    // ORDER x learned x tile.
    auto by_tile = [&](auto k0, auto k1, auto k2) { tile == 0 ? launch(k0) : tile == 1 ? launch(k1) : launch(k2); };
#define QMHD_EMF_TILES(O, L)                                                                        \
  by_tile(cell_emf_kernel_q<T, O, L, kEmfTiles[0][0], kEmfTiles[0][1]>{},                           \
          cell_emf_kernel_q<T, O, L, kEmfTiles[1][0], kEmfTiles[1][1]>{},                           \
          cell_emf_kernel_q<T, O, L, kEmfTiles[2][0], kEmfTiles[2][1]>{})
    if (cell_flags) {
      if (order == 5)
        QMHD_EMF_TILES(5, true);
      else
        QMHD_EMF_TILES(7, true);
    } else if (order == 5) {
      QMHD_EMF_TILES(5, false);
    } else {
      QMHD_EMF_TILES(7, false);
    }
#undef QMHD_EMF_TILES
  } else {
    const dim3 b(64, 4);
    go<cell_emf_lo_kernel_q>(blocks2d(g.nx + 1, g.ny + 1, b), b, stream, g, pxh, pyh, order <= 1 ? 1 : 0, u, bxc,
                             byc, cell_ez);
  }
}

template <class T>
void launch_corner(const GridD& g, int order, const Flags4& flags, const FluxView<T>& fx, const FluxView<T>& fy,
                   const double* cell_ez, const int* eqx, const int* eqy, double* ez, hipStream_t stream, dim3 b,
                   bool tiled) {
  if ((order == 5 || order == 7) && tiled) {
    const dim3 tb(16, 16);
    if (order == 7)
      go<corner_tiled_kernel_q<T, 7>>(blocks2d(g.nx + 1, g.ny + 1, tb), tb, stream, g, flags, fx, fy, cell_ez, eqx,
                                      eqy, ez);
    else
      go<corner_tiled_kernel_q<T, 5>>(blocks2d(g.nx + 1, g.ny + 1, tb), tb, stream, g, flags, fx, fy, cell_ez, eqx,
                                      eqy, ez);
    return;
  }
  go<corner_kernel_q<T>>(blocks2d(g.nx + 1, g.ny + 1, b), b, stream, g, order, flags, fx, fy, cell_ez, eqx, eqy, ez);
}

template <class T>
void launch_update(const GridD& g, double a, double b_, double cw, const double* dt_dev, const StateView& un,
                   const StateView& us, const FluxView<T>& fx, const FluxView<T>& fy, const double* ez,
                   const StateOut& out, hipStream_t stream, dim3 b) {
  go<update_kernel_q<T>>(blocks2d(g.nx + 1, g.ny + 1, b), b, stream, g, a, b_, cw, dt_dev, un, us, fx, fy, ez, out);
}

void launch_rk_combine(const GridD& g, double a, double b_, double c, const StateView& un, const StateView& us,
                       const StateView& dudt, const StateOut& out, hipStream_t stream) {
  const dim3 b(64, 4);
  hipLaunchKernelGGL(rk_combine_kernel, blocks2d(g.nx + 1, g.ny + 1, b), b, 0, stream, g, a, b_, c, un, us, dudt, out);
}

void launch_ghosts(const GridD& g, const Flags4& fluid, const Flags4& field, const StateOut& u, hipStream_t stream) {
  for (int axis = 0; axis < 2; ++axis) {
    const int lines = axis == 0 ? g.ny + 2 * g.ng : g.nx + 2 * g.ng;
    const int total = 2 * g.ng * lines;
    go<ghost_kernel_q>(dim3((total + 255) / 256), dim3(256), stream, g, axis, fluid, field, u);
  }
}

void launch_dt(const unsigned long long* max_rate_bits, double effective_cfl, double dx, double dy, double* dt_out,
               double* t_accum, hipStream_t stream) {
  go<dt_kernel_q>(dim3(1), dim3(1), stream, max_rate_bits, effective_cfl, dx, dy, dt_out, t_accum);
}

void launch_seed(const GridD& g, const IcSpecD& s, const StateOut& out, double* raw_mag, int* status,
                 hipStream_t stream) {
  const dim3 b(64, 4);
  const dim3 grid = blocks2d(g.nx + 2 * g.ng, g.ny + 2 * g.ng, b);
  hipLaunchKernelGGL(seed_kernel, grid, b, 0, stream, g, s, out, raw_mag, status);
  hipLaunchKernelGGL(recollocate_kernel, grid, b, 0, stream, g, s.gamma, out, raw_mag, status);
}

void launch_divb_linf(const GridD& g, const StateView& u, unsigned long long* out, hipStream_t stream) {
  const dim3 b(64, 4);
  hipLaunchKernelGGL(divb_linf_kernel, blocks2d(g.nx, g.ny, dim3(64, 4 * kRowsPerThread)), b, 0, stream, g, u, out);
}

void launch_theta(const GridD& g, const StateView& base, const StateView& cand, int co, unsigned long long* out,
                  hipStream_t stream) {
  const dim3 b(64, 4);
  hipLaunchKernelGGL(theta_kernel, blocks2d(g.nx, g.ny, dim3(64, 4 * kRowsPerThread)), b, 0, stream, g, base, cand, co,
                     out);
}

void launch_cell_sums(const GridD& g, const StateView& u, double* partials, int blocks, hipStream_t stream) {
  hipLaunchKernelGGL(cell_sums_kernel, dim3(blocks), dim3(256), 0, stream, g, u, partials);
}

// Transverse Gauss rows and the outer-ghost one-sided face->cell rows.  The
// one-sided row integrates the degree-(w-1) interpolant through w equally
// spaced face samples over one cell by 4-point Gauss-Legendre quadrature of
// its barycentric form; evaluated in long double and rounded once.
hipError_t upload_quad_rows(const QuadRows& rows) {
  return hipMemcpyToSymbol(HIP_SYMBOL(c_rows), &rows, sizeof(QuadRows));
}


// FP64 and FP32 forms of the face-level launchers.
#define QMHD_INSTANTIATE(T)                                                                                        \
  template void launch_reconstruct<T>(const GridD&, int, double, const Flags4&, const StateView&, const double*,     \
                                      const double*, const FaceOut<T>*, int, int, hipStream_t);                     \
  template void launch_flux<T>(const GridD&, int, int, const Flags4&, double, const FaceOut<T>*, int, int,          \
                               hipStream_t, dim3);                                                                 \
  template void launch_cell_emf<T>(const GridD&, int, const Flags4&, double, const StateView&, const double*,     \
                                   const double*, double*, hipStream_t, const uint8_t*, int);                     \
  template void launch_corner<T>(const GridD&, int, const Flags4&, const FluxView<T>&, const FluxView<T>&,        \
                                 const double*, const int*, const int*, double*, hipStream_t, dim3, bool);        \
  template void launch_update<T>(const GridD&, double, double, double, const double*, const StateView&,           \
                                 const StateView&, const FluxView<T>&, const FluxView<T>&, const double*,         \
                                 const StateOut&, hipStream_t, dim3);
#define QMHD_INSTANTIATE_LEARNED(T)                                                                                \
  template void launch_flux_learned<T>(const GridD&, int, const Flags4&, double, const FaceOut<T>*,                \
                                       const uint8_t*, hipStream_t, int);                                         \
  template void launch_reconstruct_learned<T>(const GridD&, int, double, const Flags4&, const StateView&,           \
                                              const double*, const double*, const uint8_t*, const FaceOut<T>*,     \
                                              unsigned long long*, hipStream_t, int, int);
QMHD_INSTANTIATE_LEARNED(double)
QMHD_INSTANTIATE_LEARNED(float)
#undef QMHD_INSTANTIATE_LEARNED
QMHD_INSTANTIATE(double)
QMHD_INSTANTIATE(float)
#undef QMHD_INSTANTIATE

}  // namespace qmhd

// Host side of the MI355X MHD step: the MhdSolver2D driver and the C ABI
// (include/quasar_mhd.h).
//
// One SSP-RK3 step is issued as one speculative three-stage attempt with the
// per-stage positivity fractions, the live-state admissibility and the div(B)
// preflight reduced on the device and read back with a single synchronization.
// The reference (src/physics/mhd/mhd_solver.cpp:965-1143) checks each stage on
// the host as it goes; because a rejected candidate never touches the live
// register here, evaluating the later stages speculatively and rejecting the
// attempt at its first failing stage yields the same accepted state and the
// same retry decisions.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <limits>
#include <memory>
#include <sstream>
#include <stdexcept>
#include <string>
#include <vector>

#include "../../include/quasar_mhd.h"
#include "qmhd_host.hpp"
#include "qmhd_kernels.hpp"
#include "qmhd_mlp.hpp"
#include "qmhd_queue.hpp"

namespace qmhd {

thread_local std::string g_error;

namespace {

// Per-kind launch timing with HIP events recorded on the solver's stream
// around each launch (a ghost fill's x and y launches form one interval).
// Intervals are harvested after every stream synchronization the solver
// makes; the pool of event pairs grows to the launches of one step.
class KernelClock {
 public:
  ~KernelClock() {
    for (auto& p : pool_) {
      (void)hipEventDestroy(p.a);
      (void)hipEventDestroy(p.b);
    }
  }
  void enable(bool on) {
    on_ = on;
    used_ = 0;
    for (int k = 0; k < QMHD_KERNEL_KINDS; ++k) {
      ms_[k] = 0.0;
      count_[k] = 0;
    }
  }
  template <class F>
  void timed(int kind, hipStream_t s, F&& launch) {
    if (!on_) {
      launch();
      return;
    }
    if (used_ == pool_.size()) {
      Pair p{};
      QMHD_HIP(hipEventCreate(&p.a));
      QMHD_HIP(hipEventCreate(&p.b));
      pool_.push_back(p);
    }
    Pair& p = pool_[used_++];
    p.kind = kind;
    QMHD_HIP(hipEventRecord(p.a, s));
    launch();
    QMHD_HIP(hipEventRecord(p.b, s));
  }
  // Call only after the stream has been synchronized.
  void harvest() {
    for (std::size_t i = 0; i < used_; ++i) {
      float ms = 0.f;
      QMHD_HIP(hipEventElapsedTime(&ms, pool_[i].a, pool_[i].b));
      ms_[pool_[i].kind] += ms;
      ++count_[pool_[i].kind];
    }
    used_ = 0;
  }
  double total_ms(int k) const { return ms_[k]; }
  long long launches(int k) const { return count_[k]; }
  bool enabled() const { return on_; }

 private:
  struct Pair {
    hipEvent_t a, b;
    int kind;
  };
  bool on_{false};
  std::vector<Pair> pool_;
  std::size_t used_{0};
  double ms_[QMHD_KERNEL_KINDS]{};
  long long count_[QMHD_KERNEL_KINDS]{};
};

bool quad_rows_uploaded = false;

void ensure_quad_rows() {
  if (quad_rows_uploaded) return;
  QuadRows rows;
  build_quad_rows(rows);
  QMHD_HIP(upload_quad_rows(rows));
  quad_rows_uploaded = true;
}


std::size_t storage(const GridD& g) {
  return static_cast<std::size_t>(g.nx + 2 * g.ng) * static_cast<std::size_t>(g.ny + 2 * g.ng);
}

Flags4 flags_of(const int32_t* f) {
  Flags4 out{};
  for (int s = 0; s < 4; ++s) out.side[s] = f ? f[s] : 0;
  return out;
}

StateOut outv(double* const* p) {
  StateOut v;
  for (int c = 0; c < 8; ++c) v.c[c] = p[c];
  return v;
}
IfaceView<double> iface(double* const* p) {
  IfaceView<double> v;
  for (int c = 0; c < 16; ++c) v.c[c] = p[c];
  return v;
}
FluxView<double> fluxv(double* const* p) {
  FluxView<double> v;
  for (int c = 0; c < 8; ++c) v.c[c] = p[c];
  return v;
}
// Views of the solver's face planes in the arithmetic type of the face work
// (FP32 planes occupy the first half of each FP64-sized buffer).
template <class T>
IfaceView<T> iface_as(double* const* p) {
  IfaceView<T> v;
  for (int c = 0; c < 16; ++c) v.c[c] = reinterpret_cast<T*>(p[c]);
  return v;
}
template <class T>
FluxView<T> flux_as(double* const* p) {
  FluxView<T> v;
  for (int c = 0; c < 8; ++c) v.c[c] = reinterpret_cast<T*>(p[c]);
  return v;
}

double bits_to_double(unsigned long long b) {
  double d;
  std::memcpy(&d, &b, sizeof d);
  return d;
}

int order_of(const std::string& name) {
  if (name == "muscl_minmod") return 2;
  if (name == "mp5") return 5;
  if (name == "mp7") return 7;
  throw std::invalid_argument(
      "MhdSolver2D: device evolution supports only reconstruction='muscl_minmod', 'mp5', or 'mp7'");
}

int halo_of(int order) { return order == 7 ? 4 : order == 5 ? 3 : 2; }

int boundary_mode(const std::string& name) {
  if (name == "periodic") return 0;
  if (name == "outflow") return 1;
  if (name == "wall") return 2;
  if (name == "axis") return 3;
  // "internal" (4) marks guards exchanged by the distributed tile runtime,
  // which this single-GPU build does not provide.
  throw std::invalid_argument("MhdSolver2D: unknown boundary '" + name + "'");
}

// Owned device array.
struct DBuf {
  double* p{nullptr};
  std::size_t n{0};
  DBuf() = default;
  explicit DBuf(std::size_t count) : n(count) {
    QMHD_HIP(hipMalloc(&p, count * sizeof(double)));
    QMHD_HIP(hipMemset(p, 0, count * sizeof(double)));
  }
  DBuf(const DBuf&) = delete;
  DBuf& operator=(const DBuf&) = delete;
  DBuf(DBuf&& o) noexcept : p(o.p), n(o.n) {
    o.p = nullptr;
    o.n = 0;
  }
  DBuf& operator=(DBuf&& o) noexcept {
    std::swap(p, o.p);
    std::swap(n, o.n);
    return *this;
  }
  ~DBuf() {
    if (p) (void)hipFree(p);
  }
};

// One state register with its collocated Bx/By.
struct Register {
  DBuf c[8];
  DBuf bxc, byc;
  void allocate(std::size_t n) {
    for (auto& b : c) b = DBuf(n);
    bxc = DBuf(n);
    byc = DBuf(n);
  }
  StateView view() const {
    StateView v;
    for (int k = 0; k < 8; ++k) v.c[k] = c[k].p;
    return v;
  }
  StateOut out() {
    StateOut v;
    for (int k = 0; k < 8; ++k) v.c[k] = c[k].p;
    return v;
  }
};

struct PositivityRetry {
  double theta;
};

int component_index(const std::string& c) {
  if (c == "rho") return 0;
  if (c == "mx") return 1;
  if (c == "my") return 2;
  if (c == "mz") return 3;
  if (c == "energy") return 4;
  if (c == "bx" || c == "bx_face") return 5;
  if (c == "by" || c == "by_face") return 6;
  if (c == "bz" || c == "bz_cell") return 7;
  throw std::invalid_argument("MhdSolver2D: unknown state component '" + c + "'");
}

}  // namespace

GridD to_grid(const qmhd_grid& g) {
  if (g.nx <= 0 || g.ny <= 0) throw std::invalid_argument("Grid2D: nx and ny must be positive");
  if (!(std::isfinite(g.lx) && std::isfinite(g.ly)) || g.lx <= 0 || g.ly <= 0)
    throw std::invalid_argument("Grid2D: lx and ly must be finite and positive");
  if (g.ng < 1) throw std::invalid_argument("Grid2D: nghost must be positive");
  GridD d;
  d.nx = g.nx;
  d.ny = g.ny;
  d.ng = g.ng;
  d.pitch = g.nx + 2 * g.ng;
  d.dx = g.cell_dx > 0 ? g.cell_dx : g.lx / static_cast<double>(g.nx);
  d.dy = g.cell_dy > 0 ? g.cell_dy : g.ly / static_cast<double>(g.ny);
  d.ox = g.origin_x;
  d.oy = g.origin_y;
  d.lx = g.lx;
  d.ly = g.ly;
  return d;
}

StateView view(const double* const* p) {
  StateView v;
  for (int c = 0; c < 8; ++c) v.c[c] = p[c];
  return v;
}

class Solver {
 public:
  explicit Solver(const qmhd_solver_config& cfg) {
    gamma_ = cfg.gamma;
    cfl_ = cfg.cfl;
    if (!(std::isfinite(gamma_) && gamma_ > 1.0))
      throw std::invalid_argument("MhdSolver2D: gamma must be finite and greater than one");
    if (!(std::isfinite(cfg.rho_floor) && cfg.rho_floor > 0))
      throw std::invalid_argument("MhdSolver2D: rho_floor must be finite and positive");
    if (!(std::isfinite(cfg.p_floor) && cfg.p_floor > 0))
      throw std::invalid_argument("MhdSolver2D: p_floor must be finite and positive");
    if (!(std::isfinite(cfl_) && cfl_ > 0 && cfl_ <= 1))
      throw std::invalid_argument("MhdSolver2D: cfl must be finite and in (0,1]");
    const std::string geometry = cfg.geometry[0] ? cfg.geometry : "cartesian";
    if (geometry != "cartesian")
      throw std::invalid_argument("MhdSolver2D: this build implements geometry 'cartesian'");
    order_ = order_of(cfg.reconstruction);
    const std::string arithmetic = cfg.arithmetic[0] ? cfg.arithmetic : "fp64";
    if (arithmetic == "fp32")
      fp32_ = true;
    else if (arithmetic != "fp64")
      throw std::invalid_argument("MhdSolver2D: arithmetic must be 'fp64' or 'fp32'");
    const std::string indicator = cfg.indicator;
    if (indicator == "mlp") {
      if (order_ != 5 && order_ != 7)
        throw std::invalid_argument("MhdSolver2D: the learned indicator needs reconstruction 'mp5' or 'mp7'");
      learned_ = true;
    } else if (!indicator.empty() && indicator != "none") {
      throw std::invalid_argument("MhdSolver2D: indicator must be 'none' or 'mlp'");
    }
    if (std::string(cfg.riemann) != "hlld")
      throw std::invalid_argument("MhdSolver2D: device evolution supports only riemann='hlld'");
    if (std::string(cfg.ct) != "fd_ct_christlieb")
      throw std::invalid_argument("MhdSolver2D: device evolution supports only ct='fd_ct_christlieb'");
    if (std::string(cfg.integrator) != "ssprk3")
      throw std::invalid_argument("MhdSolver2D: unknown integrator '" + std::string(cfg.integrator) + "'");
    if (std::string(cfg.positivity) != "troubled_cell")
      throw std::invalid_argument("MhdSolver2D: unknown positivity limiter '" + std::string(cfg.positivity) + "'");
    for (int s = 0; s < 4; ++s) {
      fluid_.side[s] = boundary_mode(cfg.fluid[s]);
      field_.side[s] = boundary_mode(cfg.field[s]);
      if ((fluid_.side[s] == 0) != (field_.side[s] == 0) || (fluid_.side[s] == 4) != (field_.side[s] == 4))
        throw std::invalid_argument("MhdSolver2D: fluid and field topology must match on every side");
      if (fluid_.side[s] == 3 || field_.side[s] == 3)
        throw std::invalid_argument("MhdSolver2D: the 'axis' boundary is valid only at cylindrical r=0 (x_lo)");
    }
    for (int a = 0; a < 2; ++a)
      if ((fluid_.side[2 * a] == 0) != (fluid_.side[2 * a + 1] == 0))
        throw std::invalid_argument("MhdSolver2D: periodic boundaries must be selected on both sides of an axis");
    qmhd_grid gg = cfg.grid;
    const int required = halo_of(order_);
    if (gg.ng > 0 && gg.ng < required)
      throw std::invalid_argument("MhdSolver2D: grid nghost is smaller than the reconstruction scheme's required halo");
    gg.ng = std::max(gg.ng, required);
    g_ = to_grid(gg);
    grid_pub_ = gg;
    ensure_quad_rows();
    QMHD_HIP(hipStreamCreate(&stream_));
    const std::size_t n = storage(g_);
    for (auto& r : reg_) r.allocate(n);
    // Both directions' interface planes in one allocation (32 more of them took
    // 2 ms of a solver's construction).
    const std::size_t stride = (n + 31) / 32 * 32;
    iface_mem_ = DBuf(32 * stride);
    for (int c = 0; c < 32; ++c) iface_[c / 16][c % 16] = iface_mem_.p + c * stride;
    for (auto& p : fx_) p = DBuf(n);
    for (auto& p : fy_) p = DBuf(n);
    rate_x_ = DBuf(n);
    rate_y_ = DBuf(n);
    eqx_ = DBuf(n);
    eqy_ = DBuf(n);
    cell_ez_ = DBuf(n);
    ez_ = DBuf(n);
    for (int dir = 0; dir < 2; ++dir) {
      fb_list_[dir] = DBuf(n);
      if (learned_) fb2_list_[dir] = DBuf(n);
    }
    if (learned_) {
      mlp_params_ = DBuf((mlp::kParams + 1) / 2);
      mlp_packed_ = DBuf((mlp::kPackTotal + 3) / 4);
      cell_flags_ = DBuf((n + 7) / 8);
      plain_total_ = DBuf(1);
      QMHD_HIP(hipMemset(plain_total_.p, 0, sizeof(double)));
    }
    QMHD_HIP(hipMalloc(&status_, sizeof(StepStatus)));
    QMHD_HIP(hipMemset(status_, 0, sizeof(StepStatus)));
    QMHD_HIP(hipHostMalloc(&host_status_, sizeof(StepStatus), hipHostMallocDefault));
  }

  ~Solver() {
    if (status_) (void)hipFree(status_);
    if (host_status_) (void)hipHostFree(host_status_);
    if (stream_) (void)hipStreamDestroy(stream_);
  }

  const qmhd_grid& grid() const { return grid_pub_; }
  int last_substeps() const { return last_substeps_; }
  // Test support: the next positivity-controlled request (step,
  // step_unchecked, advance) throws std::runtime_error on its first attempt
  // issued after `pieces` accepted pieces; negative disarms.
  void fail_after_pieces(int pieces) { fail_after_pieces_ = pieces; }

  void seed(const std::string& comp, const double* host, std::size_t n) {
    const int c = component_index(comp);
    if (n != storage(g_))
      throw std::invalid_argument("MhdSolver2D::seed_state: host buffer size does not match the component storage size");
    for (std::size_t k = 0; k < n; ++k)
      if (!std::isfinite(host[k]))
        throw std::invalid_argument("MhdSolver2D::seed_state: host buffer must contain only finite values");
    QMHD_HIP(hipMemcpyAsync(reg_[L_].c[c].p, host, n * sizeof(double), hipMemcpyHostToDevice, stream_));
    QMHD_HIP(hipStreamSynchronize(stream_));
    cache_order_ = -1;
    solver_owned_ = false;
  }

  void to_host(const std::string& comp, double* host, std::size_t n) {
    const int c = component_index(comp);
    if (n != storage(g_)) throw std::invalid_argument("MhdSolver2D: host buffer size does not match storage size");
    const double* src = reg_[L_].c[c].p;
    if (comp == "bx" || comp == "by") {
      launch_collocate(g_, comp == "bx" ? 0 : 1, 0, src, cell_ez_.p, stream_);
      QMHD_HIP(hipGetLastError());
      src = cell_ez_.p;
    }
    QMHD_HIP(hipMemcpyAsync(host, src, n * sizeof(double), hipMemcpyDeviceToHost, stream_));
    QMHD_HIP(hipStreamSynchronize(stream_));
  }

  double* plane(int c) { return reg_[L_].c[c].p; }

  // mhd_solver.cpp:1228-1321
  double cfl_limit(int co = 0) {
    const int order = co > 0 ? 1 : order_;
    issue_rate_phase(order);
    read_status();
    check_live(co);
    const double rate = bits_to_double(host_status_->max_rate);
    const double eff = order >= 5 ? std::min(cfl_, 0.2) : cfl_;
    if (!std::isfinite(rate)) throw std::runtime_error("MhdSolver2D: non-finite state encountered in CFL reduction");
    if (!(rate > 0)) {
      const double hmin = std::min(g_.dx, g_.dy), hmax = std::max(g_.dx, g_.dy);
      return eff * (hmin / (1.0 + hmin / hmax));
    }
    const double dt = eff / rate;
    if (!(dt > 0) || !std::isfinite(dt))
      throw std::runtime_error("MhdSolver2D: no finite positive CFL timestep is representable");
    return dt;
  }

  void step(double dt) {
    if (!(dt > 0) || !std::isfinite(dt)) throw std::invalid_argument("MhdSolver2D: dt must be finite and positive");
    if (dt > cfl_limit(0))
      throw std::invalid_argument("MhdSolver2D: dt exceeds the CFL stability limit for this grid and scheme");
    advance_positive(dt, /*checked_live=*/false);
  }

  void step_unchecked(double dt) {
    if (!(dt > 0) || !std::isfinite(dt)) throw std::invalid_argument("MhdSolver2D: dt must be finite and positive");
    advance_positive(dt, /*checked_live=*/false);
  }

  void advance(double t_end, double dt) {
    if (!(t_end >= 0) || !std::isfinite(t_end))
      throw std::invalid_argument("MhdSolver2D::advance: t_end must be finite and non-negative");
    if (!(dt > 0) || !std::isfinite(dt)) throw std::invalid_argument("MhdSolver2D::advance: dt must be finite and positive");
    double t = 0;
    while (t < t_end) {
      const double remaining = t_end - t;
      const double d = std::min(dt, remaining);
      if (!(d > 0)) throw std::runtime_error("MhdSolver2D::advance: timestep made no finite forward progress");
      step(d);
      if (d == remaining) {
        t = t_end;
      } else {
        const double next = t + d;
        if (!(next > t)) throw std::runtime_error("MhdSolver2D::advance: timestep made no finite forward progress");
        t = next;
      }
    }
  }

  double divergence_b_max() {
    launch_ghosts(g_, fluid_, field_, reg_[L_].out(), stream_);
    launch_status_reset(status_, stream_);
    launch_divb_linf(g_, reg_[L_].view(), &status_->max_rate, stream_);
    QMHD_HIP(hipGetLastError());
    read_status();
    return bits_to_double(host_status_->max_rate);
  }

  void totals(double* mass, double* energy);

  // The auto-dt loop with the timestep kept on the device.
  void run(int steps, double t_end, int* done, double* sim_time);

 private:
  // -- phases -------------------------------------------------------------
  void issue_faces(int slot, int order, bool want_rates) {
    const int hll = order <= 1 ? 1 : 0;
    Register& r = reg_[slot];
    if (learned_ && order == order_) {
      if (!indicator_set_)
        throw std::invalid_argument("MhdSolver2D: indicator 'mlp' needs its network (set_indicator) before stepping");
      // Once per step, on the live state: within one step a feature moves by
      // at most the CFL fraction of a cell, well inside the neighbourhood the
      // flags cover (the face rule takes either neighbour's flag).
      if (slot == L_)
        clock_.timed(QMHD_KERNEL_INDICATOR, stream_, [&] {
          launch_indicator(g_, gamma_, r.view(), r.bxc.p, r.byc.p, packed(), params(), threshold_, flags(),
                           stream_);
        });
      faces_issued_ += static_cast<long long>(g_.nx + 1) * (g_.ny + 2 * g_.ng) +
                       static_cast<long long>(g_.nx + 2 * g_.ng) * (g_.ny + 1);
    }
    if (fp32_)
      issue_faces_as<float>(r, order, hll, want_rates);
    else
      issue_faces_as<double>(r, order, hll, want_rates);
  }

  // Reconstruction and fluxes of both directions, each in one launch (the
  // lists' counters were zeroed by the register's prep launch).
  template <class T>
  void issue_faces_as(Register& r, int order, int hll, bool want_rates) {
    const bool learned = learned_ && order == order_;
    FaceOut<T> out[2];
    for (int dir = 0; dir < 2; ++dir) {
      double* ip[16];
      double* fp[8];
      for (int c = 0; c < 16; ++c) ip[c] = iface_[dir][c];
      for (int c = 0; c < 8; ++c) fp[c] = (dir == 0 ? fx_ : fy_)[c].p;
      unsigned long long* lists = status_->lists;
      out[dir] = FaceOut<T>{iface_as<T>(ip), reinterpret_cast<int*>((dir == 0 ? eqx_ : eqy_).p), flux_as<T>(fp),
                            // Only the live state's face rates are reduced to a timestep.
                            want_rates ? (dir == 0 ? rate_x_ : rate_y_).p : nullptr,
                            FaceList{lists + dir, reinterpret_cast<unsigned long long*>(fb_list_[dir].p)},
                            FaceList{lists + 2 + dir, reinterpret_cast<unsigned long long*>(fb2_list_[dir].p)}};
    }
    clock_.timed(QMHD_KERNEL_RECONSTRUCT, stream_, [&] {
      if (learned)
        launch_reconstruct_learned<T>(g_, order, gamma_, field_, r.view(), r.bxc.p, r.byc.p, flags(), out, plain_total(),
                                      stream_, tuning_.list_blocks, tuning_.cheap_tile);
      else
        launch_reconstruct<T>(g_, order, gamma_, field_, r.view(), r.bxc.p, r.byc.p, out, 0, 2, stream_);
    });
    clock_.timed(QMHD_KERNEL_FLUX, stream_, [&] {
      if (learned)
        launch_flux_learned<T>(g_, order, field_, gamma_, out, flags(), stream_, tuning_.list_blocks);
      else
        launch_flux<T>(g_, order, hll, field_, gamma_, out, 0, 2, stream_, tuning_.flux);
    });
  }

  // Cell E_z, corner E_z and the fused update of one stage.
  template <class T>
  void issue_ct_update(Register& in, Register& out, double a, double b, double c_host, const double* dt_dev,
                       const Register& us, int order, double* const* fxp, double* const* fyp) {
    const uint8_t* cf = learned_ && order == order_ ? flags() : nullptr;
    clock_.timed(QMHD_KERNEL_CELL_EMF, stream_, [&] {
      launch_cell_emf<T>(g_, order, field_, gamma_, in.view(), in.bxc.p, in.byc.p, cell_ez_.p, stream_, cf,
                         tuning_.emf_tile);
    });
    clock_.timed(QMHD_KERNEL_CORNER, stream_, [&] {
      launch_corner<T>(g_, order, field_, flux_as<T>(fxp), flux_as<T>(fyp), cell_ez_.p,
                       reinterpret_cast<int*>(eqx_.p), reinterpret_cast<int*>(eqy_.p), ez_.p, stream_,
                       tuning_.corner, tuning_.corner_tiled != 0);
    });
    clock_.timed(QMHD_KERNEL_UPDATE, stream_, [&] {
      launch_update<T>(g_, a, b, c_host, dt_dev, reg_[L_].view(), us.view(), flux_as<T>(fxp), flux_as<T>(fyp),
                       ez_.p, out.out(), stream_, tuning_.update);
    });
  }

  // Ghost fill, collocation + live checks, reconstruction and fluxes of the live
  // register at `order`, additive CFL rate reduction.  Leaves the flux cache
  // valid for `order`.
  void issue_rate_phase(int order) { issue_rate_phase(order, solver_owned_ ? 1 : 0); }
  void issue_rate_phase(int order, int owned) {
    launch_status_reset(status_, stream_);
    issue_live_prep(owned);
    issue_faces(L_, order, true);
    clock_.timed(QMHD_KERNEL_REDUCE, stream_,
                 [&] { launch_cfl_reduce(g_, rate_x_.p, rate_y_.p, &status_->max_rate, stream_); });
    QMHD_HIP(hipGetLastError());
    cache_order_ = order;
  }

  // Three speculative stages from the live register into reg_[C_].  When
  // `fresh`, the status block is reset and the live-state checks and stage-0
  // faces are (re)issued; otherwise a rate phase at the same order preceded.
  void issue_attempt(double dt, const double* dt_dev, int pos_order, bool fresh) {
    const int order = pos_order > 0 ? 1 : order_;
    if (fresh || cache_order_ != order) {
      launch_status_reset(status_, stream_);
      issue_live_prep();
      issue_faces(L_, order, false);
    }
    const double a[3] = {1.0, 3.0 / 4.0, 1.0 / 3.0};
    const double b[3] = {0.0, 1.0 / 4.0, 2.0 / 3.0};
    const double cw[3] = {1.0, 1.0 / 4.0, 2.0 / 3.0};
    const int in_slot[3] = {L_, S1_, S2_};
    const int out_slot[3] = {S1_, S2_, C_};
    double* fxp[8];
    double* fyp[8];
    for (int c = 0; c < 8; ++c) {
      fxp[c] = fx_[c].p;
      fyp[c] = fy_[c].p;
    }
    for (int s = 0; s < 3; ++s) {
      Register& in = reg_[in_slot[s]];
      Register& out = reg_[out_slot[s]];
      if (s > 0) issue_faces(in_slot[s], order, false);
      const double c_host = dt_dev ? cw[s] : (s == 0 ? dt : cw[s] * dt);
      const Register& us = reg_[s == 2 ? S2_ : S1_];
      if (fp32_)
        issue_ct_update<float>(in, out, a[s], b[s], c_host, dt_dev, us, order, fxp, fyp);
      else
        issue_ct_update<double>(in, out, a[s], b[s], c_host, dt_dev, us, order, fxp, fyp);
      clock_.timed(QMHD_KERNEL_GHOSTS, stream_, [&] { launch_ghosts(g_, fluid_, field_, out.out(), stream_); });
      clock_.timed(QMHD_KERNEL_PREP, stream_, [&] {
        launch_prep(g_, out.view(), out.bxc.p, out.byc.p, reg_[L_].view(), reg_[L_].bxc.p, reg_[L_].byc.p, s,
                    pos_order, s == 2 ? 1 : 0, 0, 0, status_, stream_, !fp32_);
      });
    }
    QMHD_HIP(hipGetLastError());
    cache_order_ = -1;
  }

  // Ghost fill and live-state preparation of the live register.
  void issue_live_prep() { issue_live_prep(solver_owned_ ? 1 : 0); }
  void issue_live_prep(int owned) {
    clock_.timed(QMHD_KERNEL_GHOSTS, stream_, [&] { launch_ghosts(g_, fluid_, field_, reg_[L_].out(), stream_); });
    clock_.timed(QMHD_KERNEL_PREP, stream_, [&] {
      launch_prep(g_, reg_[L_].view(), reg_[L_].bxc.p, reg_[L_].byc.p, reg_[L_].view(), reg_[L_].bxc.p,
                  reg_[L_].byc.p, -1, 0, 0, 1, owned, status_, stream_, !fp32_);
    });
  }

  void read_status() {
    QMHD_HIP(hipMemcpyAsync(host_status_, status_, sizeof(StepStatus), hipMemcpyDeviceToHost, stream_));
    QMHD_HIP(hipStreamSynchronize(stream_));
    clock_.harvest();
  }

 public:
  void set_profiling(bool on) {
    QMHD_HIP(hipStreamSynchronize(stream_));
    clock_.enable(on);
  }
  void kernel_time(int kind, double* total_ms, long long* launches) {
    if (kind < 0 || kind >= QMHD_KERNEL_KINDS) throw std::invalid_argument("unknown kernel kind");
    QMHD_HIP(hipStreamSynchronize(stream_));
    clock_.harvest();
    *total_ms = clock_.total_ms(kind);
    *launches = clock_.launches(kind);
  }
  void* stream() const { return stream_; }

  // -- learned form ---------------------------------------------------------
  void set_indicator(const float* host_params, float threshold) {
    if (!learned_) throw std::invalid_argument("MhdSolver2D: set_indicator needs indicator 'mlp' in the config");
    for (int k = 0; k < mlp::kParams; ++k)
      if (!std::isfinite(host_params[k])) throw std::invalid_argument("MhdSolver2D: non-finite indicator parameter");
    if (std::isnan(threshold)) throw std::invalid_argument("MhdSolver2D: indicator threshold is NaN");
    QMHD_HIP(hipMemcpyAsync(params(), host_params, sizeof(float) * mlp::kParams, hipMemcpyHostToDevice, stream_));
    launch_mlp_pack(params(), packed(), stream_);
    QMHD_HIP(hipGetLastError());
    QMHD_HIP(hipStreamSynchronize(stream_));
    threshold_ = threshold;
    indicator_set_ = true;
  }
  void plain_faces(long long* plain, long long* total) {
    if (!learned_) {
      *plain = *total = 0;
      return;
    }
    unsigned long long v = 0;
    QMHD_HIP(hipMemcpyAsync(&v, plain_total_.p, sizeof v, hipMemcpyDeviceToHost, stream_));
    QMHD_HIP(hipMemsetAsync(plain_total_.p, 0, sizeof v, stream_));
    QMHD_HIP(hipStreamSynchronize(stream_));
    *plain = static_cast<long long>(v);
    *total = faces_issued_;
    faces_issued_ = 0;
  }
  void cell_features(float* dev_out) {
    issue_live_prep();
    launch_features(g_, gamma_, reg_[L_].view(), reg_[L_].bxc.p, reg_[L_].byc.p, dev_out, stream_);
    QMHD_HIP(hipGetLastError());
    QMHD_HIP(hipStreamSynchronize(stream_));
  }
  // -- launch tuning ---------------------------------------------------------
  // Block shapes of the flux, corner and update launches and the grid of the
  // persistent list launches (waves per CU of the plain path over its list).
  // Launch shapes (the QMHD_TUNING_INTS vector of include/quasar_mhd.h).
  struct Tuning {
    dim3 flux{64, 4}, corner{64, 4}, update{64, 4};
    int list_blocks{1024};
    int emf_tile{0};      // cell E_z LDS tile: 16x16, 32x8, 8x32
    int cheap_tile{1};    // learned form's cheap-face tile: 64x4, 32x8, 128x2, 16x16, 8x32
    int cheap_tile_y{1};  // kept and validated; both directions run in cheap_tile's tile
    int corner_tiled{1};  // MP5/MP7 corners: LDS tile (1) or one thread per corner in `corner` blocks (0)
  };
  static bool valid_block(int bx, int by) {
    return bx >= 1 && by >= 1 && bx * by <= 256 && (bx * by) % 64 == 0;
  }
  void set_tuning(const int32_t* t) {
    if (!valid_block(t[0], t[1]) || !valid_block(t[2], t[3]) || !valid_block(t[4], t[5]) || t[6] < 1 ||
        t[6] > 65535)
      throw std::invalid_argument("MhdSolver2D: tuning needs blocks of 64..256 threads (multiples of 64) and "
                                  "1..65535 list blocks");
    if (t[7] < 0 || t[7] > 2 || t[8] < 0 || t[8] > 4 || (t[9] != 0 && t[9] != 1) || t[10] < 0 || t[10] > 4)
      throw std::invalid_argument("MhdSolver2D: tuning tile choices are 0..2 (cell E_z), 0..4 (cheap faces) and "
                                  "0/1 (corner tile)");
    tuning_.flux = dim3(t[0], t[1]);
    tuning_.corner = dim3(t[2], t[3]);
    tuning_.update = dim3(t[4], t[5]);
    tuning_.list_blocks = t[6];
    tuning_.emf_tile = t[7];
    tuning_.cheap_tile = t[8];
    tuning_.corner_tiled = t[9];
    tuning_.cheap_tile_y = t[10];
  }
  void get_tuning(int32_t* t) const {
    t[0] = tuning_.flux.x, t[1] = tuning_.flux.y, t[2] = tuning_.corner.x, t[3] = tuning_.corner.y;
    t[4] = tuning_.update.x, t[5] = tuning_.update.y, t[6] = tuning_.list_blocks;
    t[7] = tuning_.emf_tile, t[8] = tuning_.cheap_tile, t[9] = tuning_.corner_tiled, t[10] = tuning_.cheap_tile_y;
    t[11] = 0;
  }

  // Times every candidate of each knob over `trial_steps` steps (after one
  // warm-up step) with the kernel clock, keeps the fastest, and restores the
  // live state: the run continues from where it was.
  void autotune(int trial_steps) {
    if (trial_steps < 1) throw std::invalid_argument("MhdSolver2D::autotune: trial_steps must be positive");
    copy_live_to_backup();
    QMHD_HIP(hipStreamSynchronize(stream_));
    const int prev_owned = solver_owned_;
    const dim3 shapes[] = {dim3(64, 4), dim3(32, 8), dim3(128, 2), dim3(256, 1), dim3(16, 16), dim3(64, 1)};
    auto trial = [&](int kind) {
      int done = 0;
      double t = 0.0;
      run(1, 0.0, &done, &t);
      clock_.enable(true);
      run(trial_steps, 0.0, &done, &t);
      QMHD_HIP(hipStreamSynchronize(stream_));
      clock_.harvest();
      const double ms = clock_.total_ms(kind);
      clock_.enable(false);
      restore_backup();
      solver_owned_ = prev_owned;
      return ms;
    };
    dim3* knobs[3] = {&tuning_.flux, &tuning_.update, &tuning_.corner};
    const int kinds[3] = {QMHD_KERNEL_FLUX, QMHD_KERNEL_UPDATE, QMHD_KERNEL_CORNER};
    // MP5/MP7 corners: the LDS tile, or one thread per corner in the best block.
    if (order_ >= 5) tuning_.corner_tiled = 0;
    // (MP5/MP7 take the fluxes in their own tiles, the flux block shapes the
    // other orders' launches only.)
    for (int k = order_ >= 5 ? 1 : 0; k < 3; ++k) {
      dim3 best = *knobs[k];
      double best_ms = std::numeric_limits<double>::infinity();
      for (const dim3& c : shapes) {
        *knobs[k] = c;
        const double ms = trial(kinds[k]);
        if (ms < best_ms) {
          best_ms = ms;
          best = c;
        }
      }
      *knobs[k] = best;
    }
    // Choice knobs: (value, candidates, timed kind).
    auto choose = [&](int& knob, std::initializer_list<int> candidates, int kind) {
      int best = knob;
      double best_ms = std::numeric_limits<double>::infinity();
      for (int c : candidates) {
        knob = c;
        const double ms = trial(kind);
        if (ms < best_ms) {
          best_ms = ms;
          best = c;
        }
      }
      knob = best;
    };
    if (order_ >= 5) choose(tuning_.corner_tiled, {0, 1}, QMHD_KERNEL_CORNER);
    // The learned cell E_z takes the full quadrature in every block that holds
    // a flagged cell, so its tile decides which unflagged cells get it: the
    // tile is a knob of the plain method only.
    if (order_ >= 5 && !learned_) choose(tuning_.emf_tile, {0, 1, 2}, QMHD_KERNEL_CELL_EMF);
    if (learned_) choose(tuning_.cheap_tile, {0, 1, 2, 3, 4}, QMHD_KERNEL_RECONSTRUCT);
    if (learned_) {
      const int grids[] = {256, 512, 1024, 2048, 4096};
      int best = tuning_.list_blocks;
      double best_ms = std::numeric_limits<double>::infinity();
      for (int c : grids) {
        tuning_.list_blocks = c;
        const double ms = trial(QMHD_KERNEL_RECONSTRUCT);
        if (ms < best_ms) {
          best_ms = ms;
          best = c;
        }
      }
      tuning_.list_blocks = best;
    }
  }

  // -- batched, graph-captured stepping ------------------------------------
  // One auto-dt step with no host synchronization: the accept/reject decision
  // and the commit happen on the device (acc = per-run accumulators), and the
  // live/candidate roles swap on the host as bookkeeping only, so a capture of
  // two consecutive steps replays forever.
  double* batch_acc() {
    if (!batch_acc_.p) {
      batch_acc_ = DBuf(8);
      QMHD_HIP(hipMemset(batch_acc_.p, 0, 8 * sizeof(double)));
    }
    return batch_acc_.p;
  }
  void issue_batch_step() {
    if (learned_ && !indicator_set_)
      throw std::invalid_argument("MhdSolver2D: indicator 'mlp' needs its network (set_indicator) before stepping");
    double* acc = batch_acc();
    const double eff = order_ >= 5 ? std::min(cfl_, 0.2) : cfl_;
    issue_rate_phase(order_, kOwnedByStatus);
    launch_dt(&status_->max_rate, eff, g_.dx, g_.dy, &status_->dt, nullptr, stream_);
    issue_attempt(0.0, &status_->dt, 0, false);
    launch_batch_commit(status_, acc, stream_);
    launch_batch_restore(g_, acc, reg_[L_].view(), reg_[C_].out(), stream_);
    QMHD_HIP(hipGetLastError());
    swap_roles();
  }
  void swap_roles() {
    std::swap(L_, C_);
    cache_order_ = -1;
  }
  // Whether the live state is one the solver made: the host's word for it, and
  // the batched step's (status.owned, which an accepted step sets).
  bool owned() const { return solver_owned_; }
  void set_owned(bool v) { solver_owned_ = v; }
  void set_status_owned(bool v) {
    const unsigned long long word = v ? 1ull : 0ull;
    QMHD_HIP(hipMemcpyAsync(&status_->owned, &word, sizeof word, hipMemcpyHostToDevice, stream_));
    QMHD_HIP(hipStreamSynchronize(stream_));
  }
  void batch_status(long long* accepted, long long* rejected, int* fatal, double* sim_time) {
    double h[8];
    QMHD_HIP(hipMemcpyAsync(h, batch_acc(), sizeof h, hipMemcpyDeviceToHost, stream_));
    QMHD_HIP(hipStreamSynchronize(stream_));
    *accepted = static_cast<long long>(h[0]);
    *rejected = static_cast<long long>(h[1]);
    *fatal = h[2] != 0.0 ? 1 : 0;
    *sim_time = h[3];
  }
  // The batch's device counters (see launch_batch_commit).
  void batch_counters(double h[8]) {
    QMHD_HIP(hipMemcpyAsync(h, batch_acc(), 8 * sizeof(double), hipMemcpyDeviceToHost, stream_));
    QMHD_HIP(hipStreamSynchronize(stream_));
  }
  void batch_set_counter(int k, double v) {
    QMHD_HIP(hipMemcpyAsync(batch_acc() + k, &v, sizeof v, hipMemcpyHostToDevice, stream_));
    QMHD_HIP(hipStreamSynchronize(stream_));
  }
  // Batched-run autotuning: the live state and the batch counters saved, and
  // put back with the saved live register live again.
  void batch_snapshot() {
    if (!snap_) {
      snap_.reset(new Register);
      snap_->allocate(storage(g_));
    }
    const std::size_t bytes = storage(g_) * sizeof(double);
    for (int c = 0; c < 8; ++c)
      QMHD_HIP(hipMemcpyAsync(snap_->c[c].p, reg_[L_].c[c].p, bytes, hipMemcpyDeviceToDevice, stream_));
    QMHD_HIP(hipMemcpyAsync(snap_acc_, batch_acc(), sizeof snap_acc_, hipMemcpyDeviceToHost, stream_));
    QMHD_HIP(hipStreamSynchronize(stream_));
    snap_live_ = L_;
  }
  void batch_rewind() {
    if (!snap_) throw std::logic_error("MhdSolver2D: no batch snapshot to rewind to");
    if (L_ != snap_live_) {
      if (C_ != snap_live_) throw std::logic_error("MhdSolver2D: register is not the live/candidate pair");
      std::swap(L_, C_);
    }
    const std::size_t bytes = storage(g_) * sizeof(double);
    for (int c = 0; c < 8; ++c)
      QMHD_HIP(hipMemcpyAsync(reg_[L_].c[c].p, snap_->c[c].p, bytes, hipMemcpyDeviceToDevice, stream_));
    QMHD_HIP(hipMemcpyAsync(batch_acc(), snap_acc_, sizeof snap_acc_, hipMemcpyHostToDevice, stream_));
    QMHD_HIP(hipStreamSynchronize(stream_));
    cache_order_ = -1;
  }
  hipStream_t hip_stream() const { return stream_; }
  bool profiling() const { return clock_.enabled(); }
  int live_index() const { return L_; }
  int candidate_index() const { return C_; }
  // Make register `want` of the live/candidate pair the live one, copying
  // the live state (and its collocated field planes) across when it is not.
  void set_live_register(int want) {
    if (L_ == want) return;
    if (C_ != want) throw std::logic_error("MhdSolver2D: register is not the live/candidate pair");
    const std::size_t bytes = storage(g_) * sizeof(double);
    Register& src = reg_[L_];
    Register& dst = reg_[C_];
    for (int c = 0; c < 8; ++c)
      QMHD_HIP(hipMemcpyAsync(dst.c[c].p, src.c[c].p, bytes, hipMemcpyDeviceToDevice, stream_));
    QMHD_HIP(hipMemcpyAsync(dst.bxc.p, src.bxc.p, bytes, hipMemcpyDeviceToDevice, stream_));
    QMHD_HIP(hipMemcpyAsync(dst.byc.p, src.byc.p, bytes, hipMemcpyDeviceToDevice, stream_));
    QMHD_HIP(hipStreamSynchronize(stream_));
    std::swap(L_, C_);
    cache_order_ = -1;
  }

  void cell_labels(double tol, uint8_t* dev_out) {
    issue_live_prep();
    uint8_t* fx = reinterpret_cast<uint8_t*>(cell_ez_.p);
    uint8_t* fy = reinterpret_cast<uint8_t*>(ez_.p);
    launch_labels(g_, order_, field_, gamma_, reg_[L_].view(), reg_[L_].bxc.p, reg_[L_].byc.p, tol, fx, fy, dev_out,
                  stream_);
    QMHD_HIP(hipGetLastError());
    QMHD_HIP(hipStreamSynchronize(stream_));
  }

 private:

  double divb_ratio() const {
    const double res = bits_to_double(host_status_->divb_residual);
    const double scl = bits_to_double(host_status_->divb_scale);
    if (!(std::isfinite(res) && std::isfinite(scl))) return std::numeric_limits<double>::infinity();
    if (res == 0.0) return 0.0;
    if (!(scl > 0.0)) return std::numeric_limits<double>::infinity();
    return res / scl;
  }

  // ensure_live_state_solenoidal / ensure_live_state_admissible
  // (mhd_solver.cpp:1178-1222) on the status of the last live prep.
  void check_admissible(int co) const {
    const double th = bits_to_double(co == 1 ? host_status_->live_theta1 : host_status_->live_theta0);
    if (!(th >= 1.0))
      throw std::invalid_argument(
          "MhdSolver2D: live state must have finite components, rho > 0, and gas pressure > 0 in every interior "
          "cell");
  }
  void check_solenoidal() const {
    const double rel = divb_ratio();
    if (!(std::isfinite(rel) && rel <= 1024.0 * std::numeric_limits<double>::epsilon()))
      throw std::invalid_argument("MhdSolver2D: live magnetic field is not discretely divergence-free");
  }
  void check_live(int co) const {
    check_solenoidal();
    check_admissible(co);
  }

  // First failing stage theta (>= 1 when every stage is admissible).
  double attempt_theta(int pos_order, bool low_anchor) const {
    for (int s = 0; s < 3; ++s) {
      double th = bits_to_double(host_status_->theta[s]);
      if (s == 2) {
        const double other = bits_to_double(host_status_->theta[3]);
        if (pos_order == 1 || low_anchor) th = std::min(th, other);
      }
      if (!std::isfinite(th)) th = 0.0;
      if (!(th >= 1.0)) return th;
    }
    return 1.0;
  }

  void accept() {
    std::swap(L_, C_);
    cache_order_ = -1;
    solver_owned_ = true;
  }

  void copy_live_to_backup() {
    if (!backup_) {
      backup_.reset(new Register);
      backup_->allocate(storage(g_));
    }
    for (int c = 0; c < 8; ++c)
      QMHD_HIP(hipMemcpyAsync(backup_->c[c].p, reg_[L_].c[c].p, storage(g_) * sizeof(double),
                              hipMemcpyDeviceToDevice, stream_));
  }
  void restore_backup() {
    for (int c = 0; c < 8; ++c)
      QMHD_HIP(hipMemcpyAsync(reg_[L_].c[c].p, backup_->c[c].p, storage(g_) * sizeof(double),
                              hipMemcpyDeviceToDevice, stream_));
    QMHD_HIP(hipStreamSynchronize(stream_));
    cache_order_ = -1;
  }

  // mhd_solver.cpp:965-1143.  `first` carries an attempt already issued with
  // dt_dev (auto-dt loop); otherwise each attempt is issued here.
  void advance_positive(double dt, bool attempt_issued) {
    const int prev_substeps = last_substeps_;
    const bool prev_owned = solver_owned_;
    bool backed_up = false;
    try {
      double remaining = dt, trial = dt;
      bool low_interval = false;
      int retries = 0, attempts = 0, pos_order = 0;
      bool low_anchor = false;
      bool first = true;
      last_substeps_ = 0;
      while (remaining > 0) {
        if (++attempts > 100000)
          throw std::runtime_error("MhdSolver2D: positivity controller exceeded its substep limit");
        trial = std::min(trial, remaining);
        if (!(first && attempt_issued)) issue_attempt(trial, nullptr, pos_order, false);
        read_status();
        if (fail_after_pieces_ >= 0 && last_substeps_ >= fail_after_pieces_) {
          fail_after_pieces_ = -1;
          throw std::runtime_error("MhdSolver2D: injected integrator failure (test hook)");
        }
        const int co = (pos_order > 0 ? 1 : order_) <= 1 ? 1 : 0;
        if (first) {
          // step_unchecked's preflight, then the advance's low-order anchor.
          check_admissible(0);
          low_anchor = bits_to_double(host_status_->live_theta1) >= 1.0;
          first = false;
        }
        check_live(co);
        const double theta = attempt_theta(pos_order, low_anchor);
        if (!(theta >= 1.0)) {
          const bool high_order_attempt = pos_order == 0;
          pos_order = 0;
          if (++retries > 80) throw std::runtime_error("MhdSolver2D: unable to find a positive conservative substep");
          if (high_order_attempt && bits_to_double(host_status_->live_theta1) >= 1.0) {
            low_anchor = true;
            low_interval = true;
            pos_order = 1;
            trial = std::min(trial, cfl_limit(1));
            if (!(trial > 0) || !std::isfinite(trial) || !(remaining - trial < remaining))
              throw std::runtime_error("MhdSolver2D: low-order CFL substep cannot advance time");
            continue;
          }
          const double factor = std::max(0.05, std::min(0.8, 0.8 * theta));
          trial *= factor;
          pos_order = low_interval ? 1 : 0;
          if (!(trial > 0) || !std::isfinite(trial) || !(remaining - trial < remaining))
            throw std::runtime_error("MhdSolver2D: positive conservative substep cannot advance time");
          continue;
        }
        const bool final_piece = trial == remaining;
        if (!final_piece && !backed_up) {
          copy_live_to_backup();
          backed_up = true;
        }
        accept();
        retries = 0;
        ++last_substeps_;
        pos_order = low_interval ? 1 : 0;
        if (final_piece) break;
        const double next = remaining - trial;
        if (!(next > 0) || !(next < remaining))
          throw std::runtime_error("MhdSolver2D: positivity substep made no finite time progress");
        remaining = next;
        trial = std::min(std::min(2.0 * trial, remaining), cfl_limit(low_interval ? 1 : 0));
      }
    } catch (...) {
      last_substeps_ = prev_substeps;
      if (backed_up) restore_backup();
      solver_owned_ = prev_owned;
      throw;
    }
  }

  GridD g_{};
  qmhd_grid grid_pub_{};
  double gamma_{5.0 / 3.0}, cfl_{0.4};
  int order_{7};
  bool fp32_{false};  // FP32 face arithmetic (reconstruction, fluxes, cell E_z quadrature)
  // Learned form: indicator network, its BF16 operands, per-cell flags and
  // the running count of faces sent to the plain path.
  bool learned_{false}, indicator_set_{false};
  float threshold_{0.f};
  long long faces_issued_{0};
  DBuf mlp_params_, mlp_packed_, cell_flags_, plain_total_;
  Tuning tuning_;
  DBuf batch_acc_;
  float* params() { return reinterpret_cast<float*>(mlp_params_.p); }
  uint16_t* packed() { return reinterpret_cast<uint16_t*>(mlp_packed_.p); }
  uint8_t* flags() { return reinterpret_cast<uint8_t*>(cell_flags_.p); }
  unsigned long long* plain_total() { return reinterpret_cast<unsigned long long*>(plain_total_.p); }
  Flags4 fluid_{}, field_{};
  hipStream_t stream_{nullptr};
  Register reg_[4];
  int L_{0}, S1_{1}, S2_{2}, C_{3};
  std::unique_ptr<Register> backup_;
  std::unique_ptr<Register> snap_;  // batch autotuning snapshot
  double snap_acc_[8]{};
  int snap_live_{0};
  DBuf iface_mem_, fx_[8], fy_[8];
  double* iface_[2][16];
  DBuf rate_x_, rate_y_, eqx_, eqy_, cell_ez_, ez_;
  // Faces whose MP states need the fallback chain (list + count).
  DBuf fb_list_[2], fb2_list_[2];
  StepStatus* status_{nullptr};
  StepStatus* host_status_{nullptr};
  int cache_order_{-1};
  bool solver_owned_{false};
  int last_substeps_{0};
  int fail_after_pieces_{-1};
  KernelClock clock_;
};

// Exact fold of compensated per-block partials (Shewchuk partials with the
// half-even finalisation), in fixed storage: the partials of a sum of doubles
// never overlap, so their count is bounded by the exponent range over the
// 53-bit significand (about 40).
static double exact_fold(const double* v, std::size_t count) {
  constexpr std::size_t kCap = 128;
  double partials[kCap];
  std::size_t np = 0;
  for (std::size_t k = 0; k < count; ++k) {
    double x = v[k];
    if (x == 0.0) continue;
    std::size_t i = 0;
    for (std::size_t p = 0; p < np; ++p) {
      double y = partials[p];
      if (std::fabs(x) < std::fabs(y)) std::swap(x, y);
      const double hi = x + y;
      const double lo = y - (hi - x);
      if (lo != 0.0) partials[i++] = lo;
      x = hi;
    }
    if (i >= kCap) throw std::logic_error("exact_fold: partials exceed their bound");
    partials[i++] = x;
    np = i;
  }
  if (np == 0) return 0.0;
  std::size_t n = np;
  double hi = partials[--n], lo = 0.0;
  while (n > 0) {
    const double x = hi, y = partials[--n];
    hi = x + y;
    lo = y - (hi - x);
    if (lo != 0.0) break;
  }
  if (n > 0 && ((lo < 0 && partials[n - 1] < 0) || (lo > 0 && partials[n - 1] > 0))) {
    const double y = lo * 2, x = hi + y;
    if (y == x - hi) hi = x;
  }
  return hi;
}

int cell_sum_blocks(const GridD& g) {
  const long long cells = static_cast<long long>(g.nx) * g.ny;
  return static_cast<int>(std::min<long long>(kCellSumMaxBlocks, (cells + 255) / 256));
}

void fold_cell_partials(const double* host, int blocks, double* mass, double* energy) {
  // Per block: 2 (sum, correction) pairs of mass, then 2 of energy.
  double m[4 * kCellSumMaxBlocks], e[4 * kCellSumMaxBlocks];
  std::size_t n = 0;
  for (int b = 0; b < blocks; ++b)
    for (int q = 0; q < 2; ++q)
      for (int t = 0; t < 2; ++t) {
        m[n] = host[(b * 4 + q) * 2 + t];
        e[n] = host[(b * 4 + 2 + q) * 2 + t];
        ++n;
      }
  *mass = exact_fold(m, n);
  *energy = exact_fold(e, n);
}

static void cell_sums(const GridD& g, const StateView& u, double* scratch, hipStream_t stream, double* mass,
                      double* energy) {
  const int blocks = cell_sum_blocks(g);
  launch_cell_sums(g, u, scratch, blocks, stream);
  QMHD_HIP(hipGetLastError());
  std::vector<double> host(static_cast<std::size_t>(blocks) * kCellSumDoublesPerBlock);
  QMHD_HIP(hipMemcpyAsync(host.data(), scratch, host.size() * sizeof(double), hipMemcpyDeviceToHost, stream));
  QMHD_HIP(hipStreamSynchronize(stream));
  fold_cell_partials(host.data(), blocks, mass, energy);
}

void Solver::totals(double* mass, double* energy) { cell_sums(g_, reg_[L_].view(), ez_.p, stream_, mass, energy); }

void Solver::run(int steps, double t_end, int* done, double* sim_time) {
  int k = 0;
  double t = 0.0;
  double* dt_dev = &status_->dt;
  const double eff = order_ >= 5 ? std::min(cfl_, 0.2) : cfl_;
  while (k < steps && (t_end <= 0 || t < t_end)) {
    issue_rate_phase(order_);
    clock_.timed(QMHD_KERNEL_REDUCE, stream_,
                 [&] { launch_dt(&status_->max_rate, eff, g_.dx, g_.dy, dt_dev, nullptr, stream_); });
    // dt clipped to the end time on the host-known remaining interval is
    // reproduced on the device: the attempt reads status.dt.
    if (t_end > 0) {
      // Clip on the host only when it can bind: read the rate first.
      read_status();
      check_live(0);
      const double rate = bits_to_double(host_status_->max_rate);
      if (!std::isfinite(rate)) throw std::runtime_error("MhdSolver2D: non-finite state encountered in CFL reduction");
      double dt = host_status_->dt;
      const double remaining = t_end - t;
      const bool clipped = dt >= remaining;
      if (clipped) dt = remaining;
      advance_positive(dt, false);
      t = clipped ? t_end : t + dt;
    } else {
      issue_attempt(0.0, dt_dev, 0, false);
      read_status();
      check_live(0);
      const double rate = bits_to_double(host_status_->max_rate);
      if (!std::isfinite(rate)) throw std::runtime_error("MhdSolver2D: non-finite state encountered in CFL reduction");
      const double dt = host_status_->dt;
      if (attempt_theta(0, bits_to_double(host_status_->live_theta1) >= 1.0) >= 1.0) {
        accept();
        last_substeps_ = 1;
      } else {
        advance_positive(dt, false);
      }
      t += dt;
    }
    ++k;
  }
  *done = k;
  *sim_time = t;
}

}  // namespace qmhd

// ===========================================================================
// C ABI.

using qmhd::guarded;

struct qmhd_solver {
  qmhd::Solver impl;
  explicit qmhd_solver(const qmhd_solver_config& c) : impl(c) {}
};

namespace {

struct Scratch {
  // Layout of the caller-owned launch-level scratch: kPlanes planes + 64 doubles.
  static constexpr std::size_t kPlanes = 12;
  double* plane(std::size_t k) const { return base + k * n; }
  double* tail() const { return base + kPlanes * n; }
  double* base;
  std::size_t n;
};

Scratch scratch_of(const qmhd_grid* g, double* s) {
  const qmhd::GridD d = qmhd::to_grid(*g);
  if (!s) throw std::invalid_argument("scratch workspace must be provided (qmhd_scratch_doubles)");
  return Scratch{s, qmhd::storage(d)};
}

hipStream_t st(void* s) { return static_cast<hipStream_t>(s); }

double fetch_bits_as_double(const unsigned long long* dev, hipStream_t stream) {
  unsigned long long bits = 0;
  qmhd::hip_check(hipMemcpyAsync(&bits, dev, sizeof bits, hipMemcpyDeviceToHost, stream), "hipMemcpyAsync");
  qmhd::hip_check(hipStreamSynchronize(stream), "hipStreamSynchronize");
  return qmhd::bits_to_double(bits);
}

void set_bits(unsigned long long* dev, double v, hipStream_t stream) {
  unsigned long long b;
  std::memcpy(&b, &v, sizeof b);
  qmhd::hip_check(hipMemcpyAsync(dev, &b, sizeof b, hipMemcpyHostToDevice, stream), "hipMemcpyAsync");
}

// One direction's face fluxes (and rates, when given) from its interface states.
void face_flux(const qmhd::GridD& d, int dir, int order, int hll_only, const qmhd::Flags4& f, double gamma,
               const double* const* if16, double* const* flux8, double* rate, hipStream_t stream) {
  const qmhd::FaceOut<double> o{qmhd::iface(const_cast<double* const*>(if16)), nullptr, qmhd::fluxv(flux8), rate, {}, {}};
  qmhd::launch_flux<double>(d, order, hll_only, f, gamma, &o, dir, 1, stream);
}

// The EMF tables of the CT corner (cell E_z, face fluxes, no-jump flags)
// from u and both directions' interface states.  Work planes: scratch 0..7.
void prepare_emf_tables(const qmhd::GridD& d, int order, bool hll_only, const qmhd::Flags4& f, double gamma,
                        const double* const* u8, const double* const* ifx16, const double* const* ify16,
                        const qmhd_emf_tables& t, const Scratch& s, hipStream_t stream) {
  qmhd::launch_collocate(d, 0, 0, u8[5], s.plane(0), stream);
  qmhd::launch_collocate(d, 1, 0, u8[6], s.plane(1), stream);
  qmhd::launch_cell_emf<double>(d, order, f, gamma, qmhd::view(u8), s.plane(0), s.plane(1), t.cell_ez, stream);
  qmhd::launch_eq_flags(d, 0, qmhd::iface(const_cast<double* const*>(ifx16)), t.xface_no_jump, stream);
  qmhd::launch_eq_flags(d, 1, qmhd::iface(const_cast<double* const*>(ify16)), t.yface_no_jump, stream);
  // The face kernel writes all eight flux components: the
  // By (x faces) and Bx (y faces) components go to the tables, the rest to
  // work planes (two components share a plane; only the table is read).
  double* fx[8] = {s.plane(0), s.plane(1), s.plane(2), s.plane(3), s.plane(4), s.plane(5), t.xface_flux_by, s.plane(6)};
  face_flux(d, 0, order, hll_only ? 1 : 0, f, gamma, ifx16, fx, nullptr, stream);
  double* fy[8] = {s.plane(0), s.plane(1), s.plane(2), s.plane(3), s.plane(4), t.yface_flux_bx, s.plane(5), s.plane(6)};
  face_flux(d, 1, order, hll_only ? 1 : 0, f, gamma, ify16, fy, nullptr, stream);
}

// Corner E_z from prepared tables: the corner reads only the By flux of the
// x faces and the Bx flux of the y faces.
void finish_emf(const qmhd::GridD& d, int order, const qmhd::Flags4& f, const qmhd_emf_tables& t, double* ez_edge,
                hipStream_t stream) {
  double* fx[8] = {nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, t.xface_flux_by, nullptr};
  double* fy[8] = {nullptr, nullptr, nullptr, nullptr, nullptr, t.yface_flux_bx, nullptr, nullptr};
  qmhd::launch_corner(d, order, f, qmhd::fluxv(fx), qmhd::fluxv(fy), t.cell_ez, t.xface_no_jump, t.yface_no_jump,
                      ez_edge, stream);
}

}  // namespace

extern "C" {

const char* qmhd_last_error(void) { return qmhd::g_error.c_str(); }
const char* qmhd_version(void) { return "quasar-mhd-mi355x 0.1 (gfx950)"; }

size_t qmhd_grid_storage(const qmhd_grid* g) {
  if (!g || g->nx <= 0 || g->ny <= 0 || g->ng < 0) return 0;
  return static_cast<size_t>(g->nx + 2 * g->ng) * static_cast<size_t>(g->ny + 2 * g->ng);
}
size_t qmhd_scratch_doubles(const qmhd_grid* g) { return Scratch::kPlanes * qmhd_grid_storage(g) + 64; }

int qmhd_collocate_face_to_cell(const qmhd_grid* g, int axis, int collocation, const double* face, double* cell,
                                void* stream) {
  return guarded([&] {
    const qmhd::GridD d = qmhd::to_grid(*g);
    qmhd::ensure_quad_rows();
    qmhd::launch_collocate(d, axis, collocation, face, cell, st(stream));
    qmhd::hip_check(hipGetLastError(), "collocate");
  });
}

int qmhd_reconstruct(const qmhd_grid* g, int dir, int order, const int32_t* flags4, double gamma,
                     const double* const* u8, double* const* out16, double* scratch, void* stream) {
  return guarded([&] {
    const qmhd::GridD d = qmhd::to_grid(*g);
    if (order != 1 && order != 2 && order != 5 && order != 7) throw std::invalid_argument("order must be 1, 2, 5 or 7");
    qmhd::ensure_quad_rows();
    const Scratch s = scratch_of(g, scratch);
    const qmhd::StateView u = qmhd::view(u8);
    qmhd::launch_collocate(d, 0, 0, u8[5], s.plane(0), st(stream));
    qmhd::launch_collocate(d, 1, 0, u8[6], s.plane(1), st(stream));
    const qmhd::FaceList list{reinterpret_cast<unsigned long long*>(s.tail()),
                              reinterpret_cast<unsigned long long*>(s.plane(3))};
    const qmhd::FaceOut<double> o{qmhd::iface(out16), reinterpret_cast<int*>(s.plane(2)), {}, nullptr, list, {}};
    if (order >= 2) qmhd::launch_counter_reset(list.count, 1, st(stream));
    qmhd::launch_reconstruct<double>(d, order, gamma, qmhd::flags_of(flags4), u, s.plane(0), s.plane(1), &o,
                                     dir == 0 ? 0 : 1, 1, st(stream));
    qmhd::hip_check(hipGetLastError(), "reconstruct");
  });
}

int qmhd_hlld_flux(const qmhd_grid* g, int dir, int order, int hll_only, const int32_t* flags4, double gamma,
                   const double* const* in16, double* const* flux8, double* scratch, void* stream) {
  return guarded([&] {
    const qmhd::GridD d = qmhd::to_grid(*g);
    qmhd::ensure_quad_rows();
    (void)scratch_of(g, scratch);  // a missing workspace stays refused
    face_flux(d, dir == 0 ? 0 : 1, order, hll_only, qmhd::flags_of(flags4), gamma, in16, flux8, nullptr, st(stream));
    qmhd::hip_check(hipGetLastError(), "hlld_flux");
  });
}

int qmhd_flux_difference(const qmhd_grid* g, int dir, const double* const* flux8, double* const* dudt8,
                         void* stream) {
  return guarded([&] {
    const qmhd::GridD d = qmhd::to_grid(*g);
    qmhd::launch_flux_difference(d, dir, qmhd::fluxv(const_cast<double* const*>(flux8)), qmhd::outv(dudt8),
                                 st(stream));
    qmhd::hip_check(hipGetLastError(), "flux_difference");
  });
}

int qmhd_ct_emf_prepare(const qmhd_grid* g, int order, int hll_only, const int32_t* flags4, double gamma,
                        const double* const* u8, const double* const* ifx16, const double* const* ify16,
                        const qmhd_emf_tables* emf, double* scratch, void* stream) {
  return guarded([&] {
    const qmhd::GridD d = qmhd::to_grid(*g);
    if (!emf || !emf->cell_ez || !emf->xface_flux_by || !emf->yface_flux_bx || !emf->xface_no_jump ||
        !emf->yface_no_jump)
      throw std::invalid_argument("qmhd_ct_emf_prepare: every EMF table must be provided");
    qmhd::ensure_quad_rows();
    const Scratch s = scratch_of(g, scratch);
    prepare_emf_tables(d, order, hll_only != 0, qmhd::flags_of(flags4), gamma, u8, ifx16, ify16, *emf, s,
                       st(stream));
    qmhd::hip_check(hipGetLastError(), "ct_emf_prepare");
  });
}

int qmhd_ct_emf_finish(const qmhd_grid* g, int order, const int32_t* flags4, const qmhd_emf_tables* emf,
                       double* ez_edge, void* stream) {
  return guarded([&] {
    const qmhd::GridD d = qmhd::to_grid(*g);
    if (!emf || !emf->cell_ez || !emf->xface_flux_by || !emf->yface_flux_bx || !emf->xface_no_jump ||
        !emf->yface_no_jump)
      throw std::invalid_argument("qmhd_ct_emf_finish: every EMF table must be provided");
    finish_emf(d, order, qmhd::flags_of(flags4), *emf, ez_edge, st(stream));
    qmhd::hip_check(hipGetLastError(), "ct_emf_finish");
  });
}

int qmhd_ct_emf(const qmhd_grid* g, int order, const int32_t* flags4, double gamma, const double* const* u8,
                const double* const* ifx16, const double* const* ify16, const double* const* flux_x8,
                const double* const* flux_y8, double* ez_edge, double* scratch, void* stream) {
  return guarded([&] {
    const qmhd::GridD d = qmhd::to_grid(*g);
    qmhd::ensure_quad_rows();
    const Scratch s = scratch_of(g, scratch);
    const qmhd::Flags4 f = qmhd::flags_of(flags4);
    if (!flux_x8 || !flux_y8) {
      // Tables in scratch planes 8..11 (both flag tables share plane 11);
      // the preparation works in planes 0..7.
      int32_t* flags_plane = reinterpret_cast<int32_t*>(s.plane(11));
      const qmhd_emf_tables t{s.plane(8), s.plane(9), s.plane(10), flags_plane, flags_plane + s.n};
      prepare_emf_tables(d, order, order <= 1, f, gamma, u8, ifx16, ify16, t, s, st(stream));
      finish_emf(d, order, f, t, ez_edge, st(stream));
      qmhd::hip_check(hipGetLastError(), "ct_emf");
      return;
    }
    // Fast path: the caller's face fluxes of these interface states.
    qmhd::launch_collocate(d, 0, 0, u8[5], s.plane(0), st(stream));
    qmhd::launch_collocate(d, 1, 0, u8[6], s.plane(1), st(stream));
    int* eqx = reinterpret_cast<int*>(s.plane(3));
    int* eqy = reinterpret_cast<int*>(s.plane(4));
    qmhd::launch_eq_flags(d, 0, qmhd::iface(const_cast<double* const*>(ifx16)), eqx, st(stream));
    qmhd::launch_eq_flags(d, 1, qmhd::iface(const_cast<double* const*>(ify16)), eqy, st(stream));
    qmhd::launch_cell_emf<double>(d, order, f, gamma, qmhd::view(u8), s.plane(0), s.plane(1), s.plane(2), st(stream));
    qmhd::launch_corner(d, order, f, qmhd::fluxv(const_cast<double* const*>(flux_x8)),
                        qmhd::fluxv(const_cast<double* const*>(flux_y8)), s.plane(2), eqx, eqy, ez_edge,
                        st(stream));
    qmhd::hip_check(hipGetLastError(), "ct_emf");
  });
}

int qmhd_emf_curl_rate(const qmhd_grid* g, const double* ez_edge, double* dbx_face, double* dby_face,
                       void* stream) {
  return guarded([&] {
    const qmhd::GridD d = qmhd::to_grid(*g);
    qmhd::launch_curl(d, ez_edge, dbx_face, dby_face, st(stream));
    qmhd::hip_check(hipGetLastError(), "emf_curl_rate");
  });
}

int qmhd_rk_stage(const qmhd_grid* g, double a, double b, double c, const double* const* un8,
                  const double* const* us8, const double* const* dudt8, double* const* out8, void* stream) {
  return guarded([&] {
    const qmhd::GridD d = qmhd::to_grid(*g);
    qmhd::launch_rk_combine(d, a, b, c, qmhd::view(un8), qmhd::view(us8), qmhd::view(dudt8), qmhd::outv(out8),
                            st(stream));
    qmhd::hip_check(hipGetLastError(), "rk_stage");
  });
}

int qmhd_fill_ghosts(const qmhd_grid* g, const int32_t* fluid_flags4, const int32_t* field_flags4,
                     double* const* u8, void* stream) {
  return guarded([&] {
    const qmhd::GridD d = qmhd::to_grid(*g);
    qmhd::launch_ghosts(d, qmhd::flags_of(fluid_flags4), qmhd::flags_of(field_flags4), qmhd::outv(u8), st(stream));
    qmhd::hip_check(hipGetLastError(), "fill_ghosts");
  });
}

int qmhd_cfl_max_rate(const qmhd_grid* g, int order, const int32_t* flags4, double gamma,
                      const double* const* ifx16, const double* const* ify16, double* host_rate, double* scratch,
                      void* stream) {
  return guarded([&] {
    const qmhd::GridD d = qmhd::to_grid(*g);
    qmhd::ensure_quad_rows();
    const Scratch s = scratch_of(g, scratch);
    const qmhd::Flags4 f = qmhd::flags_of(flags4);
    // The face kernels write fluxes too; route them to scratch planes 2..7 and
    // the two rate planes to 0..1 (flux planes 6,7 share scratch tail-free).
    double* fl[8] = {s.plane(2), s.plane(3), s.plane(4), s.plane(5), s.plane(6), s.plane(7), s.plane(6), s.plane(7)};
    face_flux(d, 0, order, order <= 1, f, gamma, ifx16, fl, s.plane(0), st(stream));
    face_flux(d, 1, order, order <= 1, f, gamma, ify16, fl, s.plane(1), st(stream));
    auto* slot = reinterpret_cast<unsigned long long*>(s.tail());
    set_bits(slot, 0.0, st(stream));
    qmhd::launch_cfl_reduce(d, s.plane(0), s.plane(1), slot, st(stream));
    qmhd::hip_check(hipGetLastError(), "cfl_max_rate");
    *host_rate = fetch_bits_as_double(slot, st(stream));
  });
}

int qmhd_admissible_fraction(const qmhd_grid* g, const double* const* base8, const double* const* cand8,
                             int collocation, double* host_theta, double* scratch, void* stream) {
  return guarded([&] {
    const qmhd::GridD d = qmhd::to_grid(*g);
    qmhd::ensure_quad_rows();
    const Scratch s = scratch_of(g, scratch);
    auto* slot = reinterpret_cast<unsigned long long*>(s.tail());
    set_bits(slot, 1.0, st(stream));
    qmhd::launch_theta(d, qmhd::view(base8), qmhd::view(cand8), collocation, slot, st(stream));
    qmhd::hip_check(hipGetLastError(), "admissible_fraction");
    const double th = fetch_bits_as_double(slot, st(stream));
    *host_theta = std::fmax(0.0, std::fmin(1.0, std::isfinite(th) ? th : 0.0));
  });
}

int qmhd_divb_linf(const qmhd_grid* g, const double* const* u8, double* host_linf, double* scratch, void* stream) {
  return guarded([&] {
    const qmhd::GridD d = qmhd::to_grid(*g);
    const Scratch s = scratch_of(g, scratch);
    auto* slot = reinterpret_cast<unsigned long long*>(s.tail());
    set_bits(slot, 0.0, st(stream));
    qmhd::launch_divb_linf(d, qmhd::view(u8), slot, st(stream));
    qmhd::hip_check(hipGetLastError(), "divb_linf");
    *host_linf = fetch_bits_as_double(slot, st(stream));
  });
}

int qmhd_divb_relative_linf(const qmhd_grid* g, const double* const* u8, int solver_owned, double* host_ratio,
                            double* scratch, void* stream) {
  return guarded([&] {
    const qmhd::GridD d = qmhd::to_grid(*g);
    qmhd::ensure_quad_rows();
    const Scratch s = scratch_of(g, scratch);
    auto* status = reinterpret_cast<qmhd::StepStatus*>(s.tail());
    qmhd::launch_status_reset(status, st(stream));
    const qmhd::StateView u = qmhd::view(u8);
    qmhd::launch_prep(d, u, s.plane(0), s.plane(1), u, s.plane(0), s.plane(1), -1, 0, 0, 1, solver_owned, status,
                      st(stream));
    qmhd::hip_check(hipGetLastError(), "divb_relative_linf");
    qmhd::StepStatus host{};
    qmhd::hip_check(hipMemcpyAsync(&host, status, sizeof host, hipMemcpyDeviceToHost, st(stream)), "copy");
    qmhd::hip_check(hipStreamSynchronize(st(stream)), "sync");
    const double res = qmhd::bits_to_double(host.divb_residual), scl = qmhd::bits_to_double(host.divb_scale);
    double r;
    if (!(std::isfinite(res) && std::isfinite(scl)))
      r = std::numeric_limits<double>::infinity();
    else if (res == 0.0)
      r = 0.0;
    else if (!(scl > 0.0))
      r = std::numeric_limits<double>::infinity();
    else
      r = res / scl;
    *host_ratio = r;
  });
}

int qmhd_conserved_cell_sums(const qmhd_grid* g, const double* const* u8, double* mass, double* energy,
                             double* scratch, void* stream) {
  return guarded([&] {
    const qmhd::GridD d = qmhd::to_grid(*g);
    const Scratch s = scratch_of(g, scratch);
    qmhd::cell_sums(d, qmhd::view(u8), s.plane(0), st(stream), mass, energy);
  });
}

int qmhd_seed_initial_state(const qmhd_grid* g, const qmhd_ic_spec* spec, double* const* out8, double* scratch,
                            void* stream) {
  return guarded([&] {
    const qmhd::GridD d = qmhd::to_grid(*g);
    qmhd::ensure_quad_rows();
    const Scratch s = scratch_of(g, scratch);
    if (spec->kind < 0 || spec->kind > 5) throw std::invalid_argument("unknown initial condition kind");
    if (!(spec->gamma > 1.0)) throw std::invalid_argument("gamma must be greater than one");
    qmhd::IcSpecD k{};
    k.kind = spec->kind;
    k.gamma = spec->gamma;
    k.magnetic_scale = spec->magnetic_scale;
    k.interface_x = spec->interface_x;
    for (int q = 0; q < 8; ++q) {
      k.left[q] = spec->left[q];
      k.right[q] = spec->right[q];
    }
    k.rho = spec->rho;
    k.pressure = spec->pressure;
    k.b0 = spec->b0;
    k.total_b0 = spec->total_b0;
    k.amplitude = spec->amplitude;
    k.wavenumber = spec->wavenumber;
    k.magnetic_velocity_scale = spec->magnetic_velocity_scale;
    for (int q = 0; q < 3; ++q) k.b_uniform[q] = spec->b_uniform[q];
    k.center[0] = spec->center[0];
    k.center[1] = spec->center[1];
    k.r_in = spec->r_in;
    k.r0 = spec->r0;
    k.r1 = spec->r1;
    k.rho_in = spec->rho_in;
    k.rho_out = spec->rho_out;
    k.p_in = spec->p_in;
    k.p_out = spec->p_out;
    k.p_core = spec->p_core;
    k.p_ambient = spec->p_ambient;
    k.rho_ambient = spec->rho_ambient;
    k.u0 = spec->u0;
    k.ot_rho = spec->ot_rho;
    k.ot_p = spec->ot_p;
    k.noise_amplitude = spec->noise_amplitude;
    k.noise_seed = spec->noise_seed;
    k.blob_half = spec->blob_half;
    int* status = reinterpret_cast<int*>(s.tail());
    qmhd::hip_check(hipMemsetAsync(status, 0, sizeof(int), st(stream)), "memset");
    qmhd::launch_seed(d, k, qmhd::outv(out8), s.plane(0), status, st(stream));
    qmhd::hip_check(hipGetLastError(), "seed");
    int host = 0;
    qmhd::hip_check(hipMemcpyAsync(&host, status, sizeof host, hipMemcpyDeviceToHost, st(stream)), "copy");
    qmhd::hip_check(hipStreamSynchronize(st(stream)), "sync");
    if (host & 2) throw std::invalid_argument("initial state: density is not positive");
    if (host & 4) throw std::invalid_argument("initial state: pressure is not positive");
    if (host & 1) throw std::invalid_argument("initial state: unknown generator");
  });
}

int qmhd_solver_create(const qmhd_solver_config* cfg, qmhd_solver** out) {
  return guarded([&] {
    if (!cfg || !out) throw std::invalid_argument("null argument");
    *out = new qmhd_solver(*cfg);
  });
}
void qmhd_solver_destroy(qmhd_solver* s) { delete s; }
int qmhd_solver_grid(const qmhd_solver* s, qmhd_grid* out) {
  return guarded([&] { *out = s->impl.grid(); });
}
int qmhd_solver_seed_state(qmhd_solver* s, const char* component, const double* host, size_t n) {
  return guarded([&] { s->impl.seed(component, host, n); });
}
int qmhd_solver_state_to_host(qmhd_solver* s, const char* component, double* host, size_t n) {
  return guarded([&] { s->impl.to_host(component, host, n); });
}
int qmhd_solver_cfl_limit(qmhd_solver* s, double* dt) {
  return guarded([&] { *dt = s->impl.cfl_limit(0); });
}
int qmhd_solver_step(qmhd_solver* s, double dt) {
  return guarded([&] { s->impl.step(dt); });
}
int qmhd_solver_step_unchecked(qmhd_solver* s, double dt) {
  return guarded([&] { s->impl.step_unchecked(dt); });
}
int qmhd_solver_advance(qmhd_solver* s, double t_end, double dt) {
  return guarded([&] { s->impl.advance(t_end, dt); });
}
int qmhd_solver_divergence_b_max(qmhd_solver* s, double* out) {
  return guarded([&] { *out = s->impl.divergence_b_max(); });
}
int qmhd_solver_conserved_cell_totals(qmhd_solver* s, double* mass, double* energy) {
  return guarded([&] { s->impl.totals(mass, energy); });
}
int qmhd_solver_last_positivity_substeps(const qmhd_solver* s) { return s->impl.last_substeps(); }

int qmhd_solver_fail_after_pieces(qmhd_solver* s, int pieces) {
  return guarded([&] { s->impl.fail_after_pieces(pieces); });
}
int qmhd_solver_run(qmhd_solver* s, int steps, double t_end, int* steps_done, double* sim_time) {
  return guarded([&] { s->impl.run(steps, t_end, steps_done, sim_time); });
}
int qmhd_solver_set_profiling(qmhd_solver* s, int enable) {
  return guarded([&] { s->impl.set_profiling(enable != 0); });
}
int qmhd_solver_kernel_time(qmhd_solver* s, int kind, double* total_ms, long long* launches) {
  return guarded([&] {
    if (!total_ms || !launches) throw std::invalid_argument("null argument");
    s->impl.kernel_time(kind, total_ms, launches);
  });
}
const char* qmhd_kernel_kind_name(int kind) {
  static const char* names[QMHD_KERNEL_KINDS] = {"prep",   "reconstruct", "flux",   "cell_emf", "corner",
                                                 "update", "ghosts",      "reduce", "indicator"};
  return kind >= 0 && kind < QMHD_KERNEL_KINDS ? names[kind] : "";
}
void* qmhd_solver_stream(qmhd_solver* s) { return s->impl.stream(); }
int qmhd_solver_synchronize(qmhd_solver* s) {
  return guarded([&] { qmhd::hip_check(hipStreamSynchronize(static_cast<hipStream_t>(s->impl.stream())), "sync"); });
}
int qmhd_solver_state_plane(qmhd_solver* s, int component, double** device_ptr) {
  return guarded([&] {
    if (component < 0 || component > 7) throw std::invalid_argument("component must be 0..7");
    *device_ptr = s->impl.plane(component);
  });
}


// ---- learned form -------------------------------------------------------

int qmhd_mlp_pack(const float* params, uint16_t* packed, void* stream) {
  return guarded([&] {
    qmhd::launch_mlp_pack(params, packed, st(stream));
    qmhd::hip_check(hipGetLastError(), "mlp pack");
  });
}

int qmhd_mlp_forward(const uint16_t* packed, const float* params, const float* features, int64_t n, float* logits,
                     void* stream) {
  return guarded([&] {
    if (n < 0) throw std::invalid_argument("qmhd_mlp_forward: negative sample count");
    if (n == 0) return;
    qmhd::launch_mlp_forward(packed, params, features, n, logits, st(stream));
    qmhd::hip_check(hipGetLastError(), "mlp forward");
  });
}

size_t qmhd_mlp_partial_floats(int64_t n, int chunks) {
  if (n <= 0 || chunks <= 0) return 0;
  const long long waves = qmhd::mlp_grad_waves(n, chunks);
  return static_cast<size_t>((waves + 3) / 4 * 4) * (qmhd::mlp::kParams + 1);
}

int qmhd_mlp_gradient(const uint16_t* packed, const float* params, const float* features, const float* targets,
                      const float* weights, const int64_t* order, int64_t n, int chunks, float* partial,
                      float* grad_and_loss, void* stream) {
  return guarded([&] {
    if (n <= 0 || chunks <= 0) throw std::invalid_argument("qmhd_mlp_gradient: n and chunks must be positive");
    qmhd::launch_mlp_grad(packed, params, features, targets, weights, reinterpret_cast<const long long*>(order), n,
                          chunks, partial, grad_and_loss, st(stream));
    qmhd::hip_check(hipGetLastError(), "mlp gradient");
  });
}

int qmhd_mlp_adam(float* params, const float* grad, float* m, float* v, int64_t step, float lr, float beta1,
                  float beta2, float eps, void* stream) {
  return guarded([&] {
    if (step < 1) throw std::invalid_argument("qmhd_mlp_adam: step counts from 1");
    qmhd::launch_mlp_adam(params, grad, m, v, step, lr, beta1, beta2, eps, st(stream));
    qmhd::hip_check(hipGetLastError(), "mlp adam");
  });
}

int qmhd_cell_features(const qmhd_grid* g, double gamma, const double* const* u8, float* features, double* scratch,
                       void* stream) {
  return guarded([&] {
    const qmhd::GridD d = qmhd::to_grid(*g);
    if (d.ng < qmhd::mlp::kHalo) throw std::invalid_argument("qmhd_cell_features: nghost must be at least 2");
    const Scratch s = scratch_of(g, scratch);
    qmhd::ensure_quad_rows();
    qmhd::launch_collocate(d, 0, 0, u8[5], s.plane(0), st(stream));
    qmhd::launch_collocate(d, 1, 0, u8[6], s.plane(1), st(stream));
    qmhd::launch_features(d, gamma, qmhd::view(u8), s.plane(0), s.plane(1), features, st(stream));
    qmhd::hip_check(hipGetLastError(), "cell features");
  });
}

int qmhd_cell_labels(const qmhd_grid* g, int order, const int32_t* flags4, double gamma, const double* const* u8,
                     double label_tol, uint8_t* cell_bits, double* scratch, void* stream) {
  return guarded([&] {
    const qmhd::GridD d = qmhd::to_grid(*g);
    if (order != 5 && order != 7) throw std::invalid_argument("qmhd_cell_labels: order must be 5 or 7");
    if (d.ng < (order == 7 ? 4 : 3)) throw std::invalid_argument("qmhd_cell_labels: nghost too small for the order");
    const Scratch s = scratch_of(g, scratch);
    qmhd::ensure_quad_rows();
    qmhd::launch_collocate(d, 0, 0, u8[5], s.plane(0), st(stream));
    qmhd::launch_collocate(d, 1, 0, u8[6], s.plane(1), st(stream));
    qmhd::launch_labels(d, order, qmhd::flags_of(flags4), gamma, qmhd::view(u8), s.plane(0), s.plane(1), label_tol,
                        reinterpret_cast<uint8_t*>(s.plane(2)), reinterpret_cast<uint8_t*>(s.plane(3)), cell_bits,
                        st(stream));
    qmhd::hip_check(hipGetLastError(), "cell labels");
  });
}

int qmhd_cell_indicator(const qmhd_grid* g, double gamma, const double* const* u8, const uint16_t* packed,
                        const float* params, float threshold_logit, uint8_t* flags, double* scratch, void* stream) {
  return guarded([&] {
    const qmhd::GridD d = qmhd::to_grid(*g);
    if (d.ng < qmhd::mlp::kHalo) throw std::invalid_argument("qmhd_cell_indicator: nghost must be at least 2");
    const Scratch s = scratch_of(g, scratch);
    qmhd::ensure_quad_rows();
    qmhd::launch_collocate(d, 0, 0, u8[5], s.plane(0), st(stream));
    qmhd::launch_collocate(d, 1, 0, u8[6], s.plane(1), st(stream));
    qmhd::launch_indicator(d, gamma, qmhd::view(u8), s.plane(0), s.plane(1), packed, params, threshold_logit, flags,
                           st(stream));
    qmhd::hip_check(hipGetLastError(), "cell indicator");
  });
}

int qmhd_stream_synchronize(void* stream) {
  return guarded([&] { qmhd::hip_check(hipStreamSynchronize(st(stream)), "hipStreamSynchronize"); });
}

int qmhd_solver_autotune(qmhd_solver* s, int trial_steps, int32_t* tuning_out) {
  return guarded([&] {
    s->impl.autotune(trial_steps);
    if (tuning_out) s->impl.get_tuning(tuning_out);
  });
}

int qmhd_solver_set_tuning(qmhd_solver* s, const int32_t* tuning) {
  return guarded([&] { s->impl.set_tuning(tuning); });
}

int qmhd_solver_get_tuning(const qmhd_solver* s, int32_t* tuning) {
  return guarded([&] { s->impl.get_tuning(tuning); });
}

// ---- batched runs ---------------------------------------------------------

struct qmhd_batch {
  std::vector<qmhd::Solver*> runs;
  hipStream_t master{nullptr};
  hipEvent_t fork{nullptr};
  std::vector<hipEvent_t> joins;
  hipGraph_t graph[2]{nullptr, nullptr};
  hipGraphExec_t exec[2]{nullptr, nullptr};
  std::vector<int> live0;  // each run's live register index at parity 0
  std::vector<int> cand0;  // ... and its candidate register (live at parity 1)
  // Steps asked of every run, and those a run finished through its own
  // positivity controller after a rejected step held it.
  std::vector<long long> requested, host_accepted;
  std::vector<double> host_time;
  // Steps the device had accepted when last looked at, what status.owned of a
  // run holds, and why a run stopped.
  std::vector<double> seen;
  std::vector<char> status_owned;
  std::vector<std::string> failure;
  int fatal_runs{0};
  int parity{0};           // parity of the next step
  int solver_parity{0};    // parity the runs' register roles reflect
  // Tile work-queue mode: the recorded launch slots of each parity (one
  // queue launch each over the tiles of every run), their argument records
  // and run tables in one device allocation, and the workgroups per queue
  // launch (0: one per tile).
  bool queued{false};
  unsigned queue_blocks{0};
  struct Slot {
    qmhd::QueueLaunch launch;
    dim3 block;
    std::size_t args_off, runs_off;
    int nruns;
    unsigned total;
  };
  std::vector<Slot> slots[2];
  unsigned char* queue_mem{nullptr};

  ~qmhd_batch() {
    if (queue_mem) (void)hipFree(queue_mem);
    for (int p = 0; p < 2; ++p) {
      if (exec[p]) (void)hipGraphExecDestroy(exec[p]);
      if (graph[p]) (void)hipGraphDestroy(graph[p]);
    }
    for (hipEvent_t e : joins) (void)hipEventDestroy(e);
    if (fork) (void)hipEventDestroy(fork);
    if (master) (void)hipStreamDestroy(master);
  }

  void align_roles(int want) {
    if (solver_parity == want) return;
    for (qmhd::Solver* r : runs) r->swap_roles();
    solver_parity = want;
  }

  // Brings status.owned of run k in line with the run's own word.
  void tell_owned(std::size_t k) {
    runs[k]->set_status_owned(runs[k]->owned());
    status_owned[k] = runs[k]->owned() ? 1 : 0;
  }

  // Streams mode: the step of every run, each on its own stream, forked from
  // and joined back to the master stream, captured as one graph per register
  // parity.  Queue mode: every run's step recorded, and each launch slot
  // captured as one queue launch over all runs' tiles.
  void build() {
    qmhd::hip_check(hipStreamCreate(&master), "hipStreamCreate");
    qmhd::hip_check(hipEventCreateWithFlags(&fork, hipEventDisableTiming), "hipEventCreate");
    joins.resize(runs.size());
    for (auto& e : joins) qmhd::hip_check(hipEventCreateWithFlags(&e, hipEventDisableTiming), "hipEventCreate");
    for (qmhd::Solver* r : runs) {
      if (r->profiling()) throw std::invalid_argument("qmhd_batch: turn kernel profiling off on every run");
      (void)r->batch_acc();
      qmhd::hip_check(hipStreamSynchronize(r->hip_stream()), "hipStreamSynchronize");
      live0.push_back(r->live_index());
      cand0.push_back(r->candidate_index());
    }
    requested.assign(runs.size(), 0);
    host_accepted.assign(runs.size(), 0);
    host_time.assign(runs.size(), 0.0);
    seen.assign(runs.size(), 0.0);
    failure.assign(runs.size(), std::string());
    status_owned.assign(runs.size(), 0);
    for (std::size_t k = 0; k < runs.size(); ++k) tell_owned(k);
    if (queued) {
      record_queue();
      capture_queue();
      return;
    }
    for (int p = 0; p < 2; ++p) {
      qmhd::hip_check(hipStreamBeginCapture(master, hipStreamCaptureModeRelaxed), "hipStreamBeginCapture");
      try {
        qmhd::hip_check(hipEventRecord(fork, master), "hipEventRecord");
        for (std::size_t k = 0; k < runs.size(); ++k) {
          qmhd::hip_check(hipStreamWaitEvent(runs[k]->hip_stream(), fork, 0), "hipStreamWaitEvent");
          runs[k]->issue_batch_step();
          qmhd::hip_check(hipEventRecord(joins[k], runs[k]->hip_stream()), "hipEventRecord");
          qmhd::hip_check(hipStreamWaitEvent(master, joins[k], 0), "hipStreamWaitEvent");
        }
      } catch (...) {
        hipGraph_t g = nullptr;
        (void)hipStreamEndCapture(master, &g);
        if (g) (void)hipGraphDestroy(g);
        throw;
      }
      qmhd::hip_check(hipStreamEndCapture(master, &graph[p]), "hipStreamEndCapture");
      qmhd::hip_check(hipGraphInstantiate(&exec[p], graph[p], nullptr, nullptr, 0), "hipGraphInstantiate");
    }
    // Each capture swapped every run's roles once: back at parity 0.
    solver_parity = 0;
  }

  // Records both parities' steps of every run and lays out the queue's
  // argument records and run tables.
  void record_queue() {
    std::vector<unsigned char> blob;
    auto align = [&](std::size_t a) { blob.resize((blob.size() + a - 1) / a * a); };
    const int nruns = static_cast<int>(runs.size());
    for (int p = 0; p < 2; ++p) {
      std::vector<std::vector<qmhd::Recorder::Entry>> rec(runs.size());
      for (std::size_t k = 0; k < runs.size(); ++k) {
        qmhd::Recorder r;
        qmhd::g_recorder = &r;
        try {
          runs[k]->issue_batch_step();
        } catch (...) {
          qmhd::g_recorder = nullptr;
          throw;
        }
        qmhd::g_recorder = nullptr;
        rec[k] = std::move(r.entries);
      }
      const std::size_t n = rec[0].size();
      for (std::size_t k = 1; k < runs.size(); ++k)
        if (rec[k].size() != n)
          throw std::invalid_argument("qmhd_batch: queue mode needs runs with the same scheme, form and launch shapes");
      for (std::size_t i = 0; i < n; ++i) {
        const qmhd::Recorder::Entry& e0 = rec[0][i];
        // A joining entry's tiles follow its predecessor's in one launch.
        const std::size_t last = i + 1 < n && rec[0][i + 1].joins ? i + 1 : i;
        for (std::size_t q = i; q <= last; ++q)
          for (std::size_t k = 0; k < runs.size(); ++k) {
            const qmhd::Recorder::Entry& e = rec[k][q];
            if (e.tag != e0.tag || e.joins != (q > i) || e.block.x != e0.block.x || e.block.y != e0.block.y ||
                e.block.z != e0.block.z || e.args.size() != e0.args.size())
              throw std::invalid_argument(
                  "qmhd_batch: queue mode needs runs with the same scheme, form and launch shapes");
          }
        Slot s;
        s.launch = e0.launch;
        s.block = e0.block;
        align(256);
        s.args_off = blob.size();
        for (std::size_t q = i; q <= last; ++q)
          for (std::size_t k = 0; k < runs.size(); ++k)
            blob.insert(blob.end(), rec[k][q].args.begin(), rec[k][q].args.end());
        align(16);
        s.runs_off = blob.size();
        s.nruns = static_cast<int>((last - i + 1) * runs.size());
        unsigned long long total = 0;
        for (std::size_t q = i; q <= last; ++q)
          for (std::size_t k = 0; k < runs.size(); ++k) {
            const dim3 gr = rec[k][q].grid;
            if (gr.z != 1 || gr.x == 0 || gr.y == 0)
              throw std::logic_error("qmhd_batch: queue slot with an empty or 3-D grid");
            const qmhd::QueueRun qr{static_cast<unsigned>(total), gr.x, gr.y, 0u};
            const unsigned char* b = reinterpret_cast<const unsigned char*>(&qr);
            blob.insert(blob.end(), b, b + sizeof qr);
            total += static_cast<unsigned long long>(gr.x) * gr.y;
          }
        if (total > 0xFFFFFFFFull) throw std::invalid_argument("qmhd_batch: too many tiles in one queue launch");
        s.total = static_cast<unsigned>(total);
        slots[p].push_back(s);
        i = last;
      }
      (void)nruns;
    }
    // Each recording swapped every run's roles once: back at parity 0.
    solver_parity = 0;
    qmhd::hip_check(hipMalloc(&queue_mem, blob.size()), "hipMalloc");
    qmhd::hip_check(hipMemcpy(queue_mem, blob.data(), blob.size(), hipMemcpyHostToDevice), "hipMemcpy");
  }

  // One graph per parity: the slots' queue launches in order on the master stream.
  void capture_queue() {
    for (int p = 0; p < 2; ++p) {
      if (exec[p]) qmhd::hip_check(hipGraphExecDestroy(exec[p]), "hipGraphExecDestroy");
      if (graph[p]) qmhd::hip_check(hipGraphDestroy(graph[p]), "hipGraphDestroy");
      exec[p] = nullptr;
      graph[p] = nullptr;
      qmhd::hip_check(hipStreamBeginCapture(master, hipStreamCaptureModeRelaxed), "hipStreamBeginCapture");
      for (const Slot& s : slots[p]) {
        s.launch(queue_mem + s.args_off, reinterpret_cast<const qmhd::QueueRun*>(queue_mem + s.runs_off),
                 s.nruns, s.total, queue_blocks, s.block, master);
      }
      hipGraph_t g = nullptr;
      const hipError_t e = hipStreamEndCapture(master, &g);
      if (e != hipSuccess) {
        if (g) (void)hipGraphDestroy(g);
        qmhd::hip_check(e, "hipStreamEndCapture");
      }
      graph[p] = g;
      qmhd::hip_check(hipGraphInstantiate(&exec[p], graph[p], nullptr, nullptr, 0), "hipGraphInstantiate");
    }
  }

  // Queue mode: times each candidate number of workgroups per queue launch
  // over `trial_steps` steps from the batch's current state, which every run
  // gets back afterwards, and keeps the fastest.
  unsigned autotune_queue(int trial_steps) {
    if (!queued) throw std::invalid_argument("qmhd_batch_autotune: the batch is not in queue mode");
    if (trial_steps < 1) throw std::invalid_argument("qmhd_batch_autotune: trial_steps must be positive");
    align_roles(parity);
    for (qmhd::Solver* r : runs) r->batch_snapshot();
    const int parity0 = parity;
    const auto req0 = requested, acc0 = host_accepted;
    const auto time0 = host_time;
    const unsigned candidates[] = {0u, 256u, 512u, 1024u, 2048u, 4096u, 8192u};
    unsigned best = queue_blocks;
    float best_ms = 0.f;
    bool have = false;
    hipEvent_t a = nullptr, b = nullptr;
    qmhd::hip_check(hipEventCreate(&a), "hipEventCreate");
    qmhd::hip_check(hipEventCreate(&b), "hipEventCreate");
    try {
      for (unsigned c : candidates) {
        queue_blocks = c;
        capture_queue();
        qmhd::hip_check(hipGraphLaunch(exec[parity], master), "hipGraphLaunch");  // warm-up
        parity ^= 1;
        qmhd::hip_check(hipEventRecord(a, master), "hipEventRecord");
        for (int k = 0; k < trial_steps; ++k) {
          qmhd::hip_check(hipGraphLaunch(exec[parity], master), "hipGraphLaunch");
          parity ^= 1;
        }
        qmhd::hip_check(hipEventRecord(b, master), "hipEventRecord");
        qmhd::hip_check(hipEventSynchronize(b), "hipEventSynchronize");
        float ms = 0.f;
        qmhd::hip_check(hipEventElapsedTime(&ms, a, b), "hipEventElapsedTime");
        if (!have || ms < best_ms) {
          best_ms = ms;
          best = c;
          have = true;
        }
        align_roles(parity);
        for (qmhd::Solver* r : runs) r->batch_rewind();
        // The rewound live registers are the ones of the starting parity.
        solver_parity = parity0;
        parity = parity0;
      }
    } catch (...) {
      (void)hipEventDestroy(a);
      (void)hipEventDestroy(b);
      throw;
    }
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    requested = req0;
    host_accepted = acc0;
    host_time = time0;
    for (std::size_t k = 0; k < runs.size(); ++k) tell_owned(k);
    queue_blocks = best;
    capture_queue();
    return best;
  }

  void run(int steps) {
    if (steps < 0) throw std::invalid_argument("qmhd_batch_run: steps must be non-negative");
    align_roles(parity);
    for (std::size_t k = 0; k < runs.size(); ++k) {
      const int expect = parity == 0 ? live0[k] : cand0[k];
      if (runs[k]->live_index() != expect)
        throw std::invalid_argument("qmhd_batch_run: a run was stepped outside the batch");
      if (runs[k]->owned() != (status_owned[k] != 0)) tell_owned(k);
    }
    // Segments of at most kSegment graph launches: a run held by a rejected
    // step waits at most one segment before its own loop finishes that
    // segment's steps and it rejoins the batch.
    constexpr int kSegment = 16;
    for (int done = 0; done < steps;) {
      const int seg = std::min(kSegment, steps - done);
      for (int k = 0; k < seg; ++k) {
        qmhd::hip_check(hipGraphLaunch(exec[parity], master), "hipGraphLaunch");
        parity ^= 1;
      }
      qmhd::hip_check(hipStreamSynchronize(master), "hipStreamSynchronize");
      align_roles(parity);
      for (std::size_t k = 0; k < runs.size(); ++k) {
        requested[k] += seg;
        finish_held(k);
      }
      done += seg;
    }
  }

  // Keeps what stopped run k (told once).
  void stopped(std::size_t k, const double acc[8], const char* controller = nullptr) {
    if (!failure[k].empty()) return;
    ++fatal_runs;
    std::ostringstream why;
    why << "after " << static_cast<long long>(acc[0]) + host_accepted[k] << " accepted steps: ";
    switch (static_cast<int>(acc[6])) {
      case qmhd::kStopDivergence:
        why << "live magnetic field is not discretely divergence-free (relative residual " << acc[7] << ")";
        break;
      case qmhd::kStopInadmissible: why << "live state is not admissible (fraction " << acc[7] << ")"; break;
      case qmhd::kStopRate: why << "non-finite CFL rate (" << acc[7] << ")"; break;
      default: why << (controller ? controller : "stopped before this batch"); break;
    }
    failure[k] = why.str();
  }

  // A run held by a rejected step finishes its requested steps through its
  // own auto-dt loop, whose positivity controller takes the retries
  // (mhd_solver.cpp:965-1143), and rejoins the batch on the register the
  // next graph launch reads.  A run whose controller fails is marked fatal.
  void finish_held(std::size_t k) {
    qmhd::Solver* r = runs[k];
    double acc[8];
    r->batch_counters(acc);
    if (acc[0] > seen[k]) {
      seen[k] = acc[0];
      r->set_owned(true);
      status_owned[k] = 1;
    }
    if (acc[2] != 0.0) stopped(k, acc);
    if (acc[2] != 0.0 || acc[5] == 0.0) return;
    const long long remaining = requested[k] - static_cast<long long>(acc[0]) - host_accepted[k];
    if (remaining > 0) {
      int done = 0;
      double t = 0.0;
      try {
        r->run(static_cast<int>(remaining), 0.0, &done, &t);
      } catch (const std::exception& e) {
        r->batch_set_counter(2, 1.0);
        acc[2] = 1.0;
        acc[6] = qmhd::kStopNone;
        stopped(k, acc, e.what());
        r->set_live_register(parity == 0 ? live0[k] : cand0[k]);
        return;
      }
      host_accepted[k] += done;
      host_time[k] += t;
      if (!status_owned[k]) tell_owned(k);
    }
    r->batch_set_counter(5, 0.0);
    r->set_live_register(parity == 0 ? live0[k] : cand0[k]);
  }
};

namespace {
int batch_create(qmhd_solver* const* runs, int count, bool queued, int queue_blocks, qmhd_batch** out) {
  return guarded([&] {
    if (count < 1 || !runs || !out) throw std::invalid_argument("qmhd_batch_create: need at least one run");
    if (queue_blocks < 0) throw std::invalid_argument("qmhd_batch_create_queued: queue_blocks must be >= 0");
    std::unique_ptr<qmhd_batch> b(new qmhd_batch);
    b->queued = queued;
    b->queue_blocks = static_cast<unsigned>(queue_blocks);
    for (int k = 0; k < count; ++k) {
      if (!runs[k]) throw std::invalid_argument("qmhd_batch_create: null run");
      for (int q = 0; q < k; ++q)
        if (runs[q] == runs[k]) throw std::invalid_argument("qmhd_batch_create: a run appears twice");
      b->runs.push_back(&runs[k]->impl);
    }
    b->build();
    *out = b.release();
  });
}
}  // namespace

int qmhd_batch_create(qmhd_solver* const* runs, int count, qmhd_batch** out) {
  return batch_create(runs, count, false, 0, out);
}

int qmhd_batch_create_queued(qmhd_solver* const* runs, int count, int queue_blocks, qmhd_batch** out) {
  return batch_create(runs, count, true, queue_blocks, out);
}

int qmhd_batch_autotune(qmhd_batch* b, int trial_steps, int* queue_blocks) {
  return guarded([&] {
    const unsigned best = b->autotune_queue(trial_steps);
    if (queue_blocks) *queue_blocks = static_cast<int>(best);
  });
}

void qmhd_batch_destroy(qmhd_batch* b) { delete b; }

int qmhd_batch_run(qmhd_batch* b, int steps) {
  return guarded([&] { b->run(steps); });
}

int qmhd_batch_fatal_runs(const qmhd_batch* b) { return b->fatal_runs; }

const char* qmhd_batch_run_failure(const qmhd_batch* b, int run) {
  if (run < 0 || run >= static_cast<int>(b->runs.size())) return "";
  return b->failure[run].c_str();
}

int qmhd_batch_run_status(qmhd_batch* b, int run, int64_t* accepted, int64_t* rejected, int* fatal,
                          double* sim_time) {
  return guarded([&] {
    if (run < 0 || run >= static_cast<int>(b->runs.size()))
      throw std::invalid_argument("qmhd_batch_run_status: run index out of range");
    long long a = 0, r = 0;
    b->runs[run]->batch_status(&a, &r, fatal, sim_time);
    *accepted = a + b->host_accepted[run];
    *rejected = r;
    *sim_time += b->host_time[run];
  });
}

int qmhd_solver_set_indicator(qmhd_solver* s, const float* host_params, float threshold_logit) {
  return guarded([&] { s->impl.set_indicator(host_params, threshold_logit); });
}

int qmhd_solver_plain_faces(qmhd_solver* s, int64_t* plain, int64_t* total) {
  return guarded([&] {
    long long p = 0, t = 0;
    s->impl.plain_faces(&p, &t);
    *plain = p;
    *total = t;
  });
}

int qmhd_solver_cell_features(qmhd_solver* s, float* features) {
  return guarded([&] { s->impl.cell_features(features); });
}

int qmhd_solver_cell_labels(qmhd_solver* s, double label_tol, uint8_t* cell_bits) {
  return guarded([&] { s->impl.cell_labels(label_tol, cell_bits); });
}

}  // extern "C"

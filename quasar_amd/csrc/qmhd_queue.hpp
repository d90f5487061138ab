// Tile work queue over many runs: one launch per step phase covers the tiles
// of every run of a batch.
//
// Each step kernel's text lives in tiles/<kernel>.inc and reads its block
// coordinates from a Blk named qb.  The kernel includes that text directly,
// with qb taken from the hardware block index, so it compiles as a kernel
// written without the queue (written as a call to an inlined body function
// instead, the MP7 cell E_z kernel compiled to 210 VGPRs instead of 145).  A
// tile function <kernel>_tile includes the same text for the queue, and a
// queue functor <kernel>_q names the tile function, its argument record and
// the single-run launch.  Launchers go through go<Q>(): normally it launches
// the kernel; while a Recorder is active on the calling thread it appends the
// launch (kernel, grid, block, argument record) instead.  The batch records
// every run's step, checks that the runs issue the same kernels with the same
// block shapes, and replays each launch slot as one launch over the
// concatenated tiles of all runs, each workgroup mapping its tile to its run
// by binary search over the runs' first tiles: one workgroup per tile
// (<kernel>_queue), or a persistent grid of `cap` workgroups looping over the
// tiles (queue_kernel<Q>, through the tile function).
#pragma once

#include <hip/hip_runtime.h>

#include "qmhd_kernels.hpp"

#include <cstddef>
#include <cstring>
#include <vector>

namespace qmhd {

// Block index and grid size of one tile as the body sees them.
// The hardware hands the workgroups of a launch to the eight XCDs in turn
// (linear workgroup b, x fastest, to XCD b mod 8), and each XCD has its own
// L2.  native() is the hardware order.  xcd_tiled() gives XCD k the k-th
// contiguous eighth of the tiles in row-major order, in order, so tiles that
// share halo rows and columns are read through the same L2.  It suits a tile
// grid whose every tile has work: on the 2048^2 step it took the update
// kernel from 4.45 to 4.30 ms and the learned cell E_z from 111 to 97 us per
// launch.  It does not suit launches where only the first workgroups have
// work (the compact face lists, where it put every active workgroup on one
// XCD: 2-3x slower).
constexpr unsigned kXcds = 8;

struct Blk {
  unsigned x, y, gx, gy;
  static __device__ __forceinline__ Blk native() { return Blk{blockIdx.x, blockIdx.y, gridDim.x, gridDim.y}; }
  static __device__ __forceinline__ Blk xcd_tiled();
};

// The tile (row-major index) that linear workgroup b of an n-workgroup launch
// takes in the XCD-aware order.
__host__ __device__ inline unsigned xcd_tile(unsigned b, unsigned n) {
  const unsigned per = n / kXcds, extra = n % kXcds, xcd = b % kXcds, slot = b / kXcds;
  return xcd * per + (xcd < extra ? xcd : extra) + slot;
}

__device__ __forceinline__ Blk Blk::xcd_tiled() {
  const unsigned gx = gridDim.x, gy = gridDim.y;
  const unsigned t = xcd_tile(blockIdx.y * gx + blockIdx.x, gx * gy);
  return Blk{t % gx, t / gx, gx, gy};
}

// Run r owns the queue's tiles [first, next run's first); its own grid is gx x gy.
struct QueueRun {
  unsigned first, gx, gy, pad;
};

// Arguments as a tile function receives them from an argument record.  A
// pointer read from memory is generic, so the compiler would address through
// it with flat instructions; taking it through an integer into the global
// address space gives it the global loads and stores a kernel argument gets
// (the views' pointers likewise, copied into registers).  Everything else is
// passed through.
template <class E>
__device__ __forceinline__ E* queue_arg(E* p) {
  return (E*)(__attribute__((address_space(1))) E*)(__UINTPTR_TYPE__)p;
}
template <class V, int N = sizeof(V::c) / sizeof(V::c[0])>
__device__ __forceinline__ V global_view(const V& v) {
  V o;
#pragma unroll
  for (int k = 0; k < N; ++k) o.c[k] = queue_arg(v.c[k]);
  return o;
}
__device__ __forceinline__ StateView queue_arg(const StateView& v) { return global_view(v); }
__device__ __forceinline__ StateOut queue_arg(const StateOut& v) { return global_view(v); }
template <class T>
__device__ __forceinline__ IfaceView<T> queue_arg(const IfaceView<T>& v) { return global_view(v); }
template <class T>
__device__ __forceinline__ FluxView<T> queue_arg(const FluxView<T>& v) { return global_view(v); }
template <class X>
__device__ __forceinline__ const X& queue_arg(const X& x) { return x; }

// Run owning queue tile t: the last run whose first tile is <= t.
__host__ __device__ inline int queue_run_of(const QueueRun* __restrict__ runs, int nruns, unsigned t) {
  int lo = 0, hi = nruns - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (runs[mid].first <= t)
      lo = mid;
    else
      hi = mid - 1;
  }
  return lo;
}

// The tile of a one-workgroup-per-tile queue launch (the grid is every
// run's tiles): its run and its block coordinates in that run's grid.
struct QueueTile {
  int run;
  Blk blk;
};
__device__ __forceinline__ QueueTile queue_tile(const QueueRun* __restrict__ runs, int nruns) {
  const int r = queue_run_of(runs, nruns, blockIdx.x);
  const QueueRun run = runs[r];
  const unsigned local = blockIdx.x - run.first;
  return QueueTile{r, Blk{local % run.gx, local / run.gx, run.gx, run.gy}};
}

// QueueTiles<Q>::kernel: the kernel <name>_queue, which includes the step
// kernel's text itself (a call to the tile function costs registers: the MP7
// cell E_z tile function takes 210 VGPRs where the text takes 145) and takes
// one tile per workgroup.
template <class Q>
struct QueueTiles;

// Persistent form: `cap` workgroups, each taking tiles blockIdx.x,
// blockIdx.x + gridDim.x, ...  The loop around the tile function costs
// registers: the FP64 MP7 flux tile takes 256 VGPRs plus spills here (one wave
// per SIMD) against 249 (two waves) in its one-tile-per-workgroup kernel.
template <class Q>
__global__ __launch_bounds__(256) void queue_kernel(const typename Q::Args* __restrict__ args,
                                                    const QueueRun* __restrict__ runs, int nruns, unsigned total) {
  for (unsigned t = blockIdx.x; t < total; t += gridDim.x) {
    const int r = queue_run_of(runs, nruns, t);
    const QueueRun run = runs[r];
    const unsigned local = t - run.first;
    Q::run(Blk{local % run.gx, local / run.gx, run.gx, run.gy}, args[r]);
    // The next tile may rewrite this block's LDS.
    __syncthreads();
  }
}

using QueueLaunch = void (*)(const void* dev_args, const QueueRun* dev_runs, int nruns, unsigned total, unsigned cap,
                             dim3 block, hipStream_t stream);

// cap = 0, or cap >= total: one workgroup per tile; else the persistent form
// over cap workgroups.
template <class Q>
void queue_launch(const void* dev_args, const QueueRun* dev_runs, int nruns, unsigned total, unsigned cap, dim3 block,
                  hipStream_t stream) {
  if (total == 0) return;
  const auto* args = static_cast<const typename Q::Args*>(dev_args);
  if (cap == 0 || cap >= total)
    hipLaunchKernelGGL(QueueTiles<Q>::kernel, dim3(total), block, 0, stream, args, dev_runs, nruns);
  else
    hipLaunchKernelGGL((queue_kernel<Q>), dim3(cap), block, 0, stream, args, dev_runs, nruns, total);
}

// Launches recorded instead of issued (one run's step at a time).
struct Recorder {
  struct Entry {
    const void* tag;
    dim3 grid, block;
    std::vector<unsigned char> args;
    QueueLaunch launch;
  };
  std::vector<Entry> entries;

  template <class Q>
  void add(dim3 grid, dim3 block, const typename Q::Args& a) {
    Entry e;
    e.tag = Q::tag();
    e.grid = grid;
    e.block = block;
    e.args.resize(sizeof a);
    std::memcpy(e.args.data(), &a, sizeof a);
    e.launch = &queue_launch<Q>;
    entries.push_back(std::move(e));
  }
};

inline thread_local Recorder* g_recorder = nullptr;

// Launch of a step kernel through its queue functor.
template <class Q, class... A>
void go(dim3 grid, dim3 block, hipStream_t stream, A... a) {
  const typename Q::Args args{a...};
  if (g_recorder)
    g_recorder->add<Q>(grid, block, args);
  else
    Q::launch(grid, block, stream, args);
}

}  // namespace qmhd

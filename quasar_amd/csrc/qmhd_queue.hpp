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
// by a ballot over the runs' first tiles: one workgroup per tile
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

// Run r owns the queue's tiles [first, next run's first); its own grid is gx x
// gy.  xcd: a Pair's half takes its tiles in the XCD-aware order.
struct QueueRun {
  unsigned first, gx, gy, xcd;
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
  // The last run whose first tile is not past this one, 64 runs per read (the
  // binary search is five reads one after another for 24 runs, 4 us in front of
  // every launch; a block of less than a wave keeps it).
  int r = -1;
  if (blockDim.x * blockDim.y < 64) {
    r = queue_run_of(runs, nruns, blockIdx.x);
  } else {
    for (int base = 0; base < nruns; base += 64) {
      const int k = base + static_cast<int>(__lane_id());
      r += __popcll(__ballot(k < nruns && runs[k < nruns ? k : 0].first <= blockIdx.x));
    }
  }
  r = __builtin_amdgcn_readfirstlane(r);
  const QueueRun run = runs[r];
  const unsigned local = blockIdx.x - run.first;
  return QueueTile{r, Blk{local % run.gx, local / run.gx, run.gx, run.gy}};
}

// Two launches of one kernel taken as one: the records and tile ranges of both
// (r[1].first is the first tile of the second), passed by value.  A kernel that
// can run so takes a Pair behind its queue arguments and is launched with null
// ones.  Small grids spend most of a step on launches that fill a fraction of
// the device; a pair costs one of them, and its halves run side by side: 64^2
// FP64, x and y faces, reconstruction 9.6 + 9.6 -> 9.4 us, flux 14 + 14 -> 14,
// fallback 2.9 + 2.9 -> 4.1; learned rotor 768^2 lists 16.6 + 16.6 -> 22.6, their
// fluxes 17.6 + 14.2 -> 21.4; large grids within 2 %.
template <class A>
struct Pair {
  A a[2];
  QueueRun r[2];
};
template <class A>
struct TileOf {
  const A& args;
  Blk blk;
};
// Records are read through the constant address space: scalar loads, and no
// private copy of the by-value ones.
template <class A>
__device__ __forceinline__ const A* constant_space(const A* p) {
  return (const A*)(const __attribute__((address_space(4))) A*)(__UINTPTR_TYPE__)p;
}
template <class A>
__device__ __forceinline__ TileOf<A> tile_of(const A* __restrict__ args, const QueueRun* __restrict__ runs, int nruns) {
  if (runs) {
    const QueueTile t = queue_tile(runs, nruns);
    return TileOf<A>{*constant_space(args + t.run), t.blk};
  }
  // The Pair follows two pointers and an int in the kernel's arguments.
  static_assert(alignof(Pair<A>) == 8, "the pair's offset in the kernel arguments");
  const Pair<A>* own = constant_space(
      (const Pair<A>*)((__UINTPTR_TYPE__)__builtin_amdgcn_kernarg_segment_ptr() + 24));
  const int second = blockIdx.x >= own->r[1].first ? 1 : 0;
  const QueueRun run = own->r[second];
  const unsigned b = blockIdx.x - run.first, t = run.xcd ? xcd_tile(b, run.gx * run.gy) : b;
  return TileOf<A>{own->a[second], Blk{t % run.gx, t / run.gx, run.gx, run.gy}};
}

// QueueTiles<Q>::kernel: the kernel <name>_queue, which includes the step
// kernel's text itself (a call to the tile function costs registers: the MP7
// cell E_z tile function takes 210 VGPRs where the text takes 145) and takes
// one tile per workgroup.
template <class Q>
struct QueueTiles;
// Whether that kernel takes a Pair.
template <class Q>
struct Paired {
  static constexpr bool value = false;
};

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
  if (cap == 0 || cap >= total) {
    if constexpr (Paired<Q>::value)
      hipLaunchKernelGGL(QueueTiles<Q>::kernel, dim3(total), block, 0, stream, args, dev_runs, nruns,
                         Pair<typename Q::Args>{});
    else
      hipLaunchKernelGGL(QueueTiles<Q>::kernel, dim3(total), block, 0, stream, args, dev_runs, nruns);
  } else
    hipLaunchKernelGGL((queue_kernel<Q>), dim3(cap), block, 0, stream, args, dev_runs, nruns, total);
}

// Launches recorded instead of issued (one run's step at a time).
struct Recorder {
  struct Entry {
    const void* tag;
    dim3 grid, block;
    std::vector<unsigned char> args;
    QueueLaunch launch;
    bool joins;  // runs beside the entry before it, in one launch
  };
  std::vector<Entry> entries;

  template <class Q>
  void add(dim3 grid, dim3 block, const typename Q::Args& a, bool joins = false) {
    Entry e;
    e.tag = Q::tag();
    e.grid = grid;
    e.block = block;
    e.args.resize(sizeof a);
    std::memcpy(e.args.data(), &a, sizeof a);
    e.launch = &queue_launch<Q>;
    e.joins = joins;
    entries.push_back(std::move(e));
  }
};

inline thread_local Recorder* g_recorder = nullptr;

// One launch over the tiles of both grids (the second may be empty).  Q's tiles
// go out in the XCD-aware order when neighbours share cells; a face list, whose
// first tiles hold all its work, in the hardware's, which deals them over the
// XCDs (in the other order the 1024-block launches of the learned rotor 768^2
// had their faces on one XCD: 59 against 21 us).
template <class Q>
void go_pair(dim3 grid0, const typename Q::Args& a0, dim3 grid1, const typename Q::Args& a1, dim3 block,
             hipStream_t stream) {
  if (g_recorder) {
    g_recorder->add<Q>(grid0, block, a0);
    g_recorder->add<Q>(grid1, block, a1, true);
    return;
  }
  const unsigned n0 = grid0.x * grid0.y, n1 = grid1.x * grid1.y;
  hipLaunchKernelGGL(QueueTiles<Q>::kernel, dim3(n0 + n1), block, 0, stream, nullptr, nullptr, 0,
                     Pair<typename Q::Args>{{a0, a1},
                                            {{0u, grid0.x, grid0.y, Paired<Q>::xcd}, {n0, grid1.x, grid1.y, Paired<Q>::xcd}}});
}

// Launch of a step kernel through its queue functor.
template <class Q, class... A>
void go(dim3 grid, dim3 block, hipStream_t stream, A... a) {
  const typename Q::Args args{a...};
  if (g_recorder)
    g_recorder->add<Q>(grid, block, args);
  else if constexpr (Paired<Q>::value)
    go_pair<Q>(grid, args, dim3(0, 0), args, block, stream);
  else
    Q::launch(grid, block, stream, args);
}

}  // namespace qmhd

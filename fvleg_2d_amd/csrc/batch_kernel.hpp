// Batched form: many independent solves (any grid size, flux, limiter) advanced
// by ONE persistent launch per RK stage.  Each workgroup walks a contiguous
// slice of the (solve, tile) work list of its XCD and dispatches the solve's
// (flux, limiter) variant of the fused stage tile; all variants share one LDS
// buffer sized for the largest.  Solves whose time loop is done are skipped,
// and the host drops them from the work list at its next poll.
#pragma once

#include "aux_kernels.hpp"

namespace cato {

// Each work cursor has a cache line of its own.  With the eight of a stage in one
// line, the atomics of all XCDs queued up on it: some 12,000 of them in a stage of
// 32 solves of side 64 to 256, whose waves waited for 75 % of their time.  That
// batch took 43.7 ms for 64 steps (168 us a stage) and takes 31.9 ms with this
// line, fewer atomics (batch_stage_kernel) and scalar arguments (table); 8 served
// requests of side 128 to 384 took 40.4 ms and take 23.6 ms.  (25.9 and 23.4 ms now,
// with the order of build_work_list and the loads ahead of stage_tile's barrier.)
constexpr int kCursorStride = 32;
constexpr int kCursorInts = kNumXcd * kCursorStride;  // per stage

struct BatchItem {
  int solve;
  int tile;
};

struct BatchSolveRef {
  double *block_min;
  int *block_err;
  LoopState *loop;
  int ntiles;
  int pad;
};

struct BatchStageArgs {
  const StageArgs *args;   // per solve, this stage
  const int *variant;      // per solve: flux * LIM_COUNT + limiter
  const BatchItem *items;  // work list (build_work_list)
  const int *slices;       // its kNumXcd slices: slice x is entries slices[x] to slices[x + 1] (device-resident:
                           // graph replays see updates)
  int *cursor;             // kNumXcd work cursors of this stage, kCursorStride apart: zero at launch, reset by
                           // the finalize kernel
};

template <typename R, int TX, int TY> constexpr size_t batch_smem_bytes() {
  size_t a = sizeof(TileSmem<LIM_MINMOD, R, TX, TY>);
  size_t b = sizeof(TileSmem<LIM_MLP5, R, TX, TY>);
  return a > b ? a : b;
}

// A table the launch only reads, through the constant address space: with a
// workgroup-uniform index its fields come by scalar loads wherever they are used,
// as kernel arguments do.  As plain global memory the stage arguments were fetched
// again by vector loads after every store and barrier of a tile, and the arrays
// they point at by flat accesses.
template <typename T> using ConstPtr = const __attribute__((address_space(4))) T *;
template <typename T> __device__ inline ConstPtr<T> table(const T *p) { return (ConstPtr<T>)p; }

#define CATO_BATCH_CASE(F, L)                                                                                 \
  case (F) * LIM_COUNT + (L):                                                                                 \
    stage_tile<F, L, R, TX, TY, true>(a, tile, dt, *reinterpret_cast<TileSmem<L, R, TX, TY> *>(smem), red); \
    break;
#define CATO_BATCH_FLUX(F)   \
  CATO_BATCH_CASE(F, 0)      \
  CATO_BATCH_CASE(F, 1)      \
  CATO_BATCH_CASE(F, 2)      \
  CATO_BATCH_CASE(F, 3)      \
  CATO_BATCH_CASE(F, 4)

// Waves per SIMD the LDS footprint allows (at most 4): the register budget is
// capped to match, since the forty variants merged in one body would
// otherwise claim far more registers than any single variant needs.  (More waves
// of the precision form, whose LDS would hold eight, spill: 32 solves of side 64 to
// 256 take 46 us a stage with four, 52 us with six or eight.)
template <typename R, int TX, int TY> constexpr int batch_waves_per_simd() {
  constexpr size_t lds = batch_smem_bytes<R, TX, TY>() + sizeof(RedSmem);
  constexpr int fit = (int)((160 * 1024) / lds);
  return fit < 1 ? 1 : (fit > 4 ? 4 : fit);
}

template <typename R, int TX, int TY>
__global__ __launch_bounds__(kThreads, (batch_waves_per_simd<R, TX, TY>())) void batch_stage_kernel(BatchStageArgs b) {
  __shared__ __attribute__((aligned(16))) char smem[batch_smem_bytes<R, TX, TY>()];
  __shared__ RedSmem red;
  __shared__ int s_item;
  // The work list is cut into kNumXcd slices.  Workgroups of XCD x
  // take items of slice x (neighbouring tiles stay in one L2), the first of them
  // by position and the others through the slice's cursor, then help the other
  // slices: items differ in cost by variant, so a static split would leave XCDs
  // idle while others finish.  Thread 0 asks for the next item before the
  // workgroup starts on the one it has and looks at the answer after it, so that
  // the atomic's round trip lies under the tile's work; and it looks at another
  // slice's cursor before it adds to it, so that drained slices cost a load.
  const int x0 = blockIdx.x % kNumXcd, nwg = gridDim.x / kNumXcd;
  auto slice = [&](int x) { return table(b.slices)[x]; };
  auto cursor = [&](int x) { return b.cursor + x * kCursorStride; };
  int x = x0, helped = 0, base = slice(x0), taken = (int)blockIdx.x / kNumXcd;  // of thread 0: item base + taken
  while (true) {
    __syncthreads();  // the previous item (its LDS and s_item) is finished
    if (threadIdx.x == 0) {
      while (base + taken >= slice(x + 1) && ++helped < kNumXcd) {
        x = (x0 + helped) % kNumXcd;
        base = slice(x) + nwg;
        taken = __hip_atomic_load(cursor(x), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (base + taken < slice(x + 1)) taken = atomicAdd(cursor(x), 1);
      }
      s_item = helped < kNumXcd ? base + taken : -1;
    }
    __syncthreads();
    const int w = __builtin_amdgcn_readfirstlane(s_item);
    if (w < 0) break;
    if (threadIdx.x == 0) {
      base = slice(x) + nwg;
      taken = atomicAdd(cursor(x), 1);
    }
    {
      const int solve = table(b.items)[w].solve, tile = table(b.items)[w].tile;
      auto &a = table(b.args)[solve];
      auto loop = table(a.loop);
      if (a.loop && loop->done) continue;
      const double dt = a.loop ? loop->dt : a.dt_value;
      switch (table(b.variant)[solve]) {
        CATO_BATCH_FLUX(0)
        CATO_BATCH_FLUX(1)
        CATO_BATCH_FLUX(2)
        CATO_BATCH_FLUX(3)
        CATO_BATCH_FLUX(4)
        CATO_BATCH_FLUX(5)
        CATO_BATCH_FLUX(6)
        CATO_BATCH_FLUX(7)
        CATO_BATCH_FLUX(8)
        default: break;
      }
    }
  }
}

#undef CATO_BATCH_CASE
#undef CATO_BATCH_FLUX

// Per-solve end-of-step reduction: one workgroup per solve.  Workgroup 0 also
// zeroes the stage work cursors for the next step (all stages have finished).
static __global__ __launch_bounds__(kThreads) void batch_finalize_kernel(const BatchSolveRef *refs, int mode,
                                                                       int *cursors, int ncursors) {
  if (blockIdx.x == 0)
    for (int k = threadIdx.x; k < ncursors; k += kThreads) cursors[k] = 0;
  auto &r = table(refs)[blockIdx.x];
  close_step<kThreads, 4>(r.ntiles, r.block_min, r.block_err, nullptr, r.loop, mode);
}

}  // namespace cato

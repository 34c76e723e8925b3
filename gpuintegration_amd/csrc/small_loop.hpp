// small_loop.hpp -- the iteration loop of short lists in one workgroup
// (small_loop.hip): the launch and the rule for the lists it takes.
#pragma once

#include <hip/hip_runtime.h>

#include "ws_internal.hpp"

namespace pagani {
namespace internal {

// Lists of at most this many regions: two chunks, whether the list has
// parents or not.
constexpr std::size_t kSmallMax = 2 * phases::kChunk;
// Iterations per launch: the first launch of a segment, and later ones
// (replayed from a graph); both fit the trace of a round.
constexpr int kSmallFirst = 24, kSmallNext = 8;

// The workspace's buffers the loop works in (those of the device-resident
// loop), and the launch constants.
struct SmallBufs {
  double *L[2], *H[2];
  std::uint8_t* pdim[2];
  double *est, *err0, *err1, *pest;
  std::uint8_t *dim, *active;
  std::uint64_t *off, *foff;
  phases::Scalars* scal;
  phases::Levels lv;
};

// Largest list the loop takes for a family at dimension d (0: never).
std::size_t small_cap(int family, int d);

// One launch: at most `iterations` iterations of the loop whose state is at
// `loop` (pinned host memory, read at the start and written back at the end).
// split > 0: the list is the run's first, split^ndim equal regions, not
// formed yet.
hipError_t launch_small_loop(hipStream_t s, const pagani_genz& g, DevLoop* loop, int iterations,
                             int split, const SmallBufs& b, const pagani_eval_consts& C);

}  // namespace internal
}  // namespace pagani

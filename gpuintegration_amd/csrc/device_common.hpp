// device_common.hpp -- deterministic reductions, the per-region refinement
// and the move of a kept region, shared by the phase kernels (phases.hip),
// the batch's segment kernel (segments.hip) and the small-list loop
// (small_loop.hip).  Compile with -ffp-contract=off: the
// refinement is plain IEEE double in the reference's operation order.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "phases.hpp"

namespace pagani {
namespace phases {

struct DD {
  double hi, lo;
};

// Compensated addition (two-sum of the leading parts, then the tails).
// Non-finite sums fall back to the plain sum so inf/NaN propagate as in an
// uncompensated reduction.
__device__ __forceinline__ DD dd_add(DD a, DD b)
{
  const double s = a.hi + b.hi;
  if (!__builtin_isfinite(s)) return DD{s, 0.0};
  const double bb = s - a.hi;
  double e = (a.hi - (s - bb)) + (b.hi - bb);
  e += a.lo + b.lo;
  const double hi = s + e;
  return DD{hi, e - (hi - s)};
}

__device__ __forceinline__ DD dd_add(DD a, double b) { return dd_add(a, DD{b, 0.0}); }

__device__ __forceinline__ DD wave_reduce(DD v)
{
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    DD o;
    o.hi = __shfl_xor(v.hi, off, 64);
    o.lo = __shfl_xor(v.lo, off, 64);
    v = dd_add(v, o);
  }
  return v;
}

// Four sums over a wave at once: the steps of wave_reduce, interleaved.
__device__ __forceinline__ void wave_reduce4(DD (&v)[4])
{
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    DD o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      o[i].hi = __shfl_xor(v[i].hi, off, 64);
      o[i].lo = __shfl_xor(v[i].lo, off, 64);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = dd_add(v[i], o[i]);
  }
}

// Four DDs over a 256-thread block: block_reduce's steps, interleaved, with
// one barrier (sh is the caller's, used once).
__device__ __forceinline__ void block_reduce4(DD (&v)[4], DD (&sh)[4][kThreads / 64])
{
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  wave_reduce4(v);
  if (lane == 0)
#pragma unroll
    for (int i = 0; i < 4; ++i) sh[i][wave] = v[i];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[i] = sh[i][0];
#pragma unroll
    for (int w = 1; w < kThreads / 64; ++w) v[i] = dd_add(v[i], sh[i][w]);
  }
}

// Records that the workgroup finishing last reads in the same launch: stored
// and loaded at agent scope, which is where every XCD sees them, and counted
// by a ticket taken when the stores have arrived there.  A release fence
// would also write back everything else in the XCD's L2.
__device__ __forceinline__ void store_agent(double* p, double v)
{
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double load_agent(const double* p)
{
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The calling wave's stores have arrived.
__device__ __forceinline__ void wait_stores() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// The workgroup's place in the order of finishing, one lane of the wave that
// stored its record.
__device__ __forceinline__ std::uint32_t take_ticket(std::uint32_t* ticket)
{
  wait_stores();
  const std::uint32_t t =
      __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  asm volatile("" ::: "memory");
  return t;
}

// Reduce a DD over a 256-thread block; every thread gets the result.
__device__ __forceinline__ DD block_reduce(DD v, DD* sh)
{
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  v = wave_reduce(v);
  if (lane == 0) sh[wave] = v;
  __syncthreads();
  DD r = sh[0];
#pragma unroll
  for (int w = 1; w < kThreads / 64; ++w) r = dd_add(r, sh[w]);
  __syncthreads();
  return r;
}

__device__ __forceinline__ std::uint32_t block_count(std::uint32_t c, std::uint32_t* sh)
{
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off, 64);
  if (lane == 0) sh[wave] = c;
  __syncthreads();
  std::uint32_t r = 0;
#pragma unroll
  for (int w = 0; w < kThreads / 64; ++w) r += sh[w];
  __syncthreads();
  return r;
}

// RefineError (Phases.cuh:219-268) of one region (estimate e, error r)
// with its sibling (es, rs) and their parent's estimate pe, and the relerr
// classification: r_out the refined error, active unless relerr finishes it.
__device__ __forceinline__ void refine_region(double e, double r, double es, double rs, double pe,
                                              double epsrel, int relerr, double& r_out,
                                              bool& active)
{
#pragma clang fp contract(off)
  const double diff = fabs(.25 * ((es + e) - pe));
  const double E = r + rs;
  if (E > 0.0) {
    const double cc = 1 + 2 * diff / E;
    r *= cc;
  }
  r += diff;
  const bool pass = relerr && r < fmax(epsrel * fabs(e), 1e-200);
  r_out = r;
  active = !pass;
}

// Row `row` of a list's bounds along axis j at stride `stride`: lower bound
// and width (from the level when lv.on), and the width's level.
__device__ __forceinline__ void read_row(const double* __restrict__ L,
                                         const double* __restrict__ H, const Levels& lv,
                                         std::size_t o, int j, double& l, double& w, int& lev)
{
  l = L[o];
  if (lv.on) {
    lev = reinterpret_cast<const std::uint16_t*>(H)[o];
    w = __builtin_ldexp(lv.h0[j], -lev);
  } else {
    lev = 0;
    w = H[o];
  }
}

// The kept region t of an n-region list (split form when pdim is given)
// becomes parent i of the next list's m: its own bounds, derived from its
// parent's as the evaluation derives them, at [j*m + i], the axis it is to
// be halved along (dim[t]) and its estimate.
template <int D>
__device__ __forceinline__ void move_region(
    std::size_t n, std::size_t m, std::size_t t, std::size_t i, const double* __restrict__ L,
    const double* __restrict__ H, const std::uint8_t* __restrict__ pdim,
    const double* __restrict__ est, const std::uint8_t* __restrict__ dim, double* __restrict__ L2,
    double* __restrict__ H2, std::uint8_t* __restrict__ pdim2, double* __restrict__ pest,
    const Levels& lv)
{
  const double ev = est[t];
  const std::uint8_t b = dim[t];
  // the row this region's bounds come from, and the axis its parent halves
  // (none for a flat list)
  const std::size_t h = n / 2;
  std::size_t row = t, stride = n;
  int axis = -1;
  bool right = false;
  if (pdim) {
    right = t >= h;
    row = right ? t - h : t;
    stride = h;
    axis = pdim[row];
  }
#pragma unroll
  for (int j = 0; j < D; ++j) {
    double l, w;
    int g;
    read_row(L, H, lv, static_cast<std::size_t>(j) * stride + row, j, l, w, g);
    if (j == axis) {
      const double half = w / 2;
      if (right) l = l + half;
      w = half;
      ++g;
    }
    const std::size_t o = static_cast<std::size_t>(j) * m + i;
    L2[o] = l;
    if (lv.on)
      reinterpret_cast<std::uint16_t*>(H2)[o] = static_cast<std::uint16_t>(g);
    else
      H2[o] = w;
  }
  pdim2[i] = b;
  pest[i] = ev;
}

}  // namespace phases
}  // namespace pagani

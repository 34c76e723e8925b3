// small_loop.hip -- the device-resident loop's iterations on short lists, in
// one workgroup of one launch.
//
// An iteration over a few hundred regions is 10 us of work, but as three
// launches (evaluation, k_step_dev, compaction) it took 50-60 us: launch
// gaps, empty workgroups of grids sized for the round's largest list (4-8 us
// each), the ticket of k_step_dev with its device-wide fences (17-45 us),
// queued launches after the loop had stopped, and a round trip per round.
// Measured per integral, as those launches -> here: 5D oscillatory at 1e-3
// (one iteration of 32 regions, eight waves on their one tile) 65 -> 48 us; 3D
// Gaussian at 1e-4 443 -> 267 us, 5D discontinuous at 1e-4 2.07 -> 1.36 ms (228
// us and 1.18 ms with the shorter k_step_dev on the lists past small_cap).
// Here one workgroup of 512 threads runs the whole loop: uniform barriers in
// place of launches, the loop's state and the sums in LDS, the lists in the
// workspace's own buffers (so the loop can stop at any iteration and the
// launches, or the host, go on from there).  Bound by the latency of its
// phases: one compute unit evaluates 1/256 of what the device does, so the
// rule (small_cap) takes the lists whose evaluation there stays below the
// launches' cost.
//
// Every value is formed as the launches form it -- the evaluation at the
// list's slice count, the refinement chunk by chunk with the chunks' own
// reduction trees, decide_step, the compaction in list order -- so results
// are the same bits whichever way an iteration runs.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>

#include "device_common.hpp"
#include "devloop_decide.hpp"
#include "genz_visit.hpp"
#include "pagani/eval_kernel.hpp"
#include "small_loop.hpp"

namespace pagani {
namespace internal {
namespace {

namespace ph = pagani::phases;
using ph::DD;

constexpr int kSmallThreads = 512;  // two chunks of ph::kThreads
constexpr int kSmallWaves = kSmallThreads / 64;
constexpr int kWavesPerChunk = ph::kThreads / 64;
constexpr int kChunks = kSmallThreads / ph::kThreads;
static_assert(kSmallMax == kChunks * ph::kChunk, "a thread group per chunk");
static_assert(kSmallWaves >= PAGANI_MAX_SLICES, "a tile's waves");
static_assert(kSmallMax <= 65536, "list positions are 16-bit");

struct SmallShared {
  DevLoop s;
  DD sums[4][kSmallWaves];
  std::uint32_t cnt[kChunks][ph::kPerThread][kWavesPerChunk];  // active regions, then offsets
  std::uint16_t src[kSmallMax];
};

template <int D, class F>
__global__ void __launch_bounds__(kSmallThreads)
    k_small_loop(F f, DevLoop* __restrict__ loop, int iterations, int split, const SmallBufs b,
                 const pagani_eval_consts C)
{
#pragma clang fp contract(off)
  constexpr bool kPairs = detail::has_pair_sums<F>::value;
  constexpr int kTab = detail::pair_table_size<D, F>();
  __shared__ SmallShared sh;
  __shared__ double tab[kTab > 0 ? kTab : 1];
  __shared__ double part[(PAGANI_MAX_SLICES - 1) * PAGANI_NRULES * 64];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  static_assert(sizeof(DevLoop) % 4 == 0, "copied by words");
  constexpr int kWords = sizeof(DevLoop) / 4;
  constexpr int kHead = offsetof(DevLoop, trace) / 4;  // the trace is written, not read
  for (int i = tid; i < kHead; i += kSmallThreads)
    reinterpret_cast<std::uint32_t*>(&sh.s)[i] = reinterpret_cast<const std::uint32_t*>(loop)[i];
  if constexpr (kTab > 0)
    if (C.levels) detail::fill_pair_tables<D>(f, C, tab, tid, kSmallThreads);
  __syncthreads();
  if (split) {
    // the run's first list, split^D equal regions, as k_uniform_split forms it
    const double len = 1. / static_cast<double>(split);
    const int n = static_cast<int>(sh.s.it.n), cur = sh.s.it.cur ? 1 : 0;
    for (int t = tid; t < n; t += kSmallThreads) {
      int q = t;
      for (int j = 0; j < D; ++j) {
        const int id = q % split;
        q /= split;
        const std::size_t o = static_cast<std::size_t>(j) * n + t;
        b.L[cur][o] = static_cast<double>(id) * len;
        if (C.levels)
          reinterpret_cast<std::uint16_t*>(b.H[cur])[o] = 0;
        else
          b.H[cur][o] = len;
      }
    }
    __syncthreads();
  }

  for (int iter = 0; iter < iterations && sh.s.it.run; ++iter) {
    const std::size_t n = sh.s.it.n;
    const int cur = sh.s.it.cur ? 1 : 0;
    const bool parents = sh.s.it.has_parents != 0;
    const int slices = static_cast<int>(sh.s.it.slices);
    const double* L = b.L[cur];
    const double* H = b.H[cur];
    const std::uint8_t* P = sh.s.it.split ? b.pdim[cur] : nullptr;

    // evaluation: kSmallWaves / slices tiles at a time
    {
      const LaunchList list{n, L, H, P, slices};
      const int tiles = static_cast<int>((n + 63) / 64), step = kSmallWaves / slices;
      const int group = wave / slices, sw = wave % slices;
      const double* t0 = kTab > 0 && C.levels ? tab : nullptr;
      for (int g = 0; g < tiles; g += step) {
        const int tile = g + group;
        std::size_t t;
        bool live;
        list.region(tile, lane, t, live);
        if (slices == 1) {
          if (tile < tiles) {
            detail::LoadedRow<kPairs ? D : 1> row(L, H, P, n, t, C);
            detail::eval_regions_wave<D, F, double, kPairs>(
                f, L, H, P, n, t, live, C.lows, C.range, C.jac, C, 1, 0, lane, nullptr, &row, t0,
                b.est, b.err0, b.dim);
          }
        } else {
          // slices divide the workgroup's waves (they are powers of two);
          // every wave passes the barrier inside, one with a tile past the
          // list too (its last region again, not stored)
          detail::eval_regions_wave<D, F, double, false>(
              f, L, H, P, n, t, live && tile < tiles, C.lows, C.range, C.jac, C, slices, sw, lane,
              part + group * (slices - 1) * PAGANI_NRULES * 64, nullptr, nullptr, b.est, b.err0,
              b.dim);
          __syncthreads();
        }
      }
    }
    __syncthreads();

    // refinement, relerr flags and the chunks' sums (refine_chunk)
    const int chunk = tid / ph::kThreads, ctid = tid % ph::kThreads;
    const int cwave = wave % kWavesPerChunk;
    const int nch = static_cast<int>(ph::num_chunks(n, parents));
    double* errs = parents ? b.err1 : b.err0;
    std::uint32_t flags = 0;  // of this thread's regions, bit k
    std::size_t base = 0, end = 0;
    if (chunk < nch) ph::chunk_range(chunk, n, parents, base, end);
    {
      const std::size_t h = n / 2;
      DD v[4] = {{0, 0}, {0, 0}, {0, 0}, {0, 0}};
      for (int k = 0; k < ph::kPerThread; ++k) {
        const std::size_t t = base + static_cast<std::size_t>(k) * ph::kThreads + ctid;
        bool a = false;
        if (t < end) {
          const double e = b.est[t];
          double r = b.err0[t];
          a = true;
          if (parents) {
            const bool right = t >= h;
            const std::size_t sib = right ? t - h : t + h;
            const std::size_t par = right ? t - h : t;
            ph::refine_region(e, r, b.est[sib], b.err0[sib], b.pest[par], sh.s.epsrel,
                              sh.s.relerr, r, a);
            errs[t] = r;
          }
          b.active[t] = a ? 1 : 0;
          v[0] = ph::dd_add(v[0], e);
          v[1] = ph::dd_add(v[1], r);
          if (a) {
            v[2] = ph::dd_add(v[2], e);
            v[3] = ph::dd_add(v[3], r);
            flags |= 1u << k;
          }
        }
        const std::uint32_t c = static_cast<std::uint32_t>(__popcll(__ballot(a)));
        if (lane == 0) sh.cnt[chunk][k][cwave] = c;
      }
      ph::wave_reduce4(v);
      if (lane == 0)
#pragma unroll
        for (int i = 0; i < 4; ++i) sh.sums[i][wave] = v[i];
    }
    __syncthreads();
    // the active regions' offsets in list order: wave 0 scans the counts
    static_assert(kChunks * ph::kPerThread * kWavesPerChunk == 2 * 64, "two counts per lane");
    if (wave == 0) {
      std::uint32_t* c = &sh.cnt[0][0][0];
      const std::uint32_t c0 = c[2 * lane], c1 = c[2 * lane + 1];
      std::uint32_t inc = c0 + c1;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const std::uint32_t y = __shfl_up(inc, o, 64);
        if (lane >= o) inc += y;
      }
      c[2 * lane] = inc - c0 - c1;
      c[2 * lane + 1] = inc - c1;
      const std::uint32_t total = __shfl(inc, 63, 64);
      // chunk 1's offset: what lies before its first count
      const std::uint32_t off1 = __shfl(inc - c0 - c1, 32, 64);
      if (lane == 0) {
        double sums[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          // the chunk records, their fold and the final sum, as refine_chunk,
          // fold_block and k_finalize form them (sums with zero records are
          // the sums)
          DD r[kChunks];
#pragma unroll
          for (int k = 0; k < kChunks; ++k) {
            r[k] = sh.sums[i][k * kWavesPerChunk];
#pragma unroll
            for (int w = 1; w < kWavesPerChunk; ++w)
              r[k] = ph::dd_add(r[k], sh.sums[i][k * kWavesPerChunk + w]);
          }
          DD x = ph::dd_add(r[0], nch > 1 ? r[1] : DD{0.0, 0.0});
          x = ph::dd_add(DD{0.0, 0.0}, x);
          sums[i] = x.hi + x.lo;
        }
        decide_step(&sh.s, sums[0], sums[1], sums[2], sums[3], total);
        if (sh.s.status == kDevHost) {
          // what the host needs to finish the iteration from its records
          for (int i = 0; i < 4; ++i) b.scal->sum[i] = sums[i];
          b.scal->mn = 0.0;
          b.scal->mx = 0.0;
          b.scal->count = total;
          b.scal->pad = 0;
          b.off[0] = 0;
          if (nch > 1) b.off[1] = off1;
          b.foff[0] = 0;
        }
      }
    }
    __syncthreads();
    if (!sh.s.cp.run) break;
    // filter + split: the kept regions become the next list's parents
    for (int k = 0; k < ph::kPerThread; ++k) {
      const bool a = (flags >> k) & 1u;
      const unsigned long long ballot = __ballot(a);
      const unsigned long long below = lane ? (ballot & ((1ull << lane) - 1ull)) : 0ull;
      if (a)
        sh.src[sh.cnt[chunk][k][cwave] + static_cast<std::uint32_t>(__popcll(below))] =
            static_cast<std::uint16_t>(base + static_cast<std::size_t>(k) * ph::kThreads + ctid);
    }
    __syncthreads();
    const std::size_t m = sh.s.cp.m;
    for (std::size_t q = tid; q < m; q += kSmallThreads)
      ph::move_region<D>(n, m, sh.src[q], q, L, H, P, b.est, b.dim, b.L[cur ^ 1], b.H[cur ^ 1],
                         b.pdim[cur ^ 1], b.pest, b.lv);
    __syncthreads();
  }
  __syncthreads();
  const int words = kHead + static_cast<int>(sh.s.ntrace * sizeof(TraceRec) / 4);
  for (int i = tid; i < (words < kWords ? words : kWords); i += kSmallThreads)
    reinterpret_cast<std::uint32_t*>(loop)[i] = reinterpret_cast<const std::uint32_t*>(&sh.s)[i];
}

// The dimensions whose kernels this part of the source holds (PAGANI_PART,
// see build.py).
constexpr int kPartFirst[] = {PAGANI_MIN_DIM, 5, 7, 9, PAGANI_GENZ_MAX_DIM + 1};

template <int D, class Fn>
int with_part_dim(int d, Fn&& fn)
{
  if constexpr (D >= kPartFirst[PAGANI_PART + 1]) {
    return PAGANI_EUNSUPPORTED;
  } else {
    if (d == D) return fn(std::integral_constant<int, D>{});
    return with_part_dim<D + 1>(d, fn);
  }
}

}  // namespace

template <int Part>
int launch_small_part(hipStream_t s, const pagani_genz& g, DevLoop* loop, int iterations,
                      int split, const SmallBufs& b, const pagani_eval_consts& C);

template <>
int launch_small_part<PAGANI_PART>(hipStream_t s, const pagani_genz& g, DevLoop* loop,
                                   int iterations, int split, const SmallBufs& b,
                                   const pagani_eval_consts& C)
{
  return with_part_dim<kPartFirst[PAGANI_PART]>(g.ndim, [&](auto D) {
    constexpr int Dv = decltype(D)::value;
    return visit_genz<double, Dv>(&g, [&](const auto& f) {
      using F = std::decay_t<decltype(f)>;
      hipLaunchKernelGGL((k_small_loop<Dv, F>), dim3(1), dim3(kSmallThreads), 0, s, f, loop,
                         iterations, split, b, C);
      return hipGetLastError() == hipSuccess ? PAGANI_OK : PAGANI_EHIP;
    });
  });
}

#if PAGANI_PART == 0
// One compute unit issues about one wave instruction per cycle, and at two
// waves per SIMD some 60 % of that: 40 000 instructions are 30 us, what an
// iteration's launches cost.  Instructions per tile of 64 regions: pair sums
// and cosine sums by axis, the corner peak in groups of points.
std::size_t small_cap(int family, int d)
{
  if (d < PAGANI_MIN_DIM || d > PAGANI_GENZ_MAX_DIM) return 0;
  const double points = 1 + 8 * d + 6 * d * (d - 1) + 4. * d * (d - 1) * (d - 2) / 3 +
                        std::ldexp(1.0, d);
  const double per_tile = family == PAGANI_GENZ_CORNER_PEAK ? 12 * points + 300 : 160. * d + 250;
  const double tiles = std::floor(40000 / per_tile);
  return std::min<std::size_t>(kSmallMax, 64 * static_cast<std::size_t>(std::max(tiles, 1.0)));
}

hipError_t launch_small_loop(hipStream_t s, const pagani_genz& g, DevLoop* loop, int iterations,
                             int split, const SmallBufs& b, const pagani_eval_consts& C)
{
  const int d = g.ndim;
  auto launch = d < kPartFirst[1]   ? &launch_small_part<0>
                : d < kPartFirst[2] ? &launch_small_part<1>
                : d < kPartFirst[3] ? &launch_small_part<2>
                                    : &launch_small_part<3>;
  return launch(s, g, loop, iterations, split, b, C) == PAGANI_OK ? hipSuccess : hipErrorLaunchFailure;
}
#endif

}  // namespace internal
}  // namespace pagani

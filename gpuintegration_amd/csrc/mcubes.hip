// mcubes.hip -- the m-Cubes driver (pagani_mc_* entry points).
//
// One vegas() run (cuda/mcubes/vegasT.cuh:640-1000): the run constants and
// the uniform grid on the host; per iteration one sampling launch over every
// cube (the integrand's kernel, behind a pagani_mc_sample_fn), one
// reduction launch that folds the workgroup partials in a fixed order, and
// one that combines the iteration into the running estimate, applies the
// stopping rule and, in adjusting iterations, refines the grid in place.  The
// host queues up to 16 iterations at a time.  5D, 10^6 samples, 10
// iterations: 771 -> 316 us against a round trip and a refinement on the host
// per iteration.  simple_integrate's retries with AdjustParams
// (vegasT.cuh:1082-1112) wrap the run.  All device memory is allocated at
// creation: the largest launch has kMaxGrid workgroups.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cstring>
#include <string>
#include <vector>

#include "device_common.hpp"
#include "genz_visit.hpp"
#include "mcubes_edge.hpp"
#include "mcubes_grid.hpp"
#include "pagani.h"
#include "pagani/mcubes_kernel.hpp"

namespace {

namespace ph = pagani::phases;
using pagani::mc::kBins;
using pagani::mc::kThreads;

constexpr std::uint32_t kMaxGrid = 1024;
constexpr int kOutDoubles = 2 + PAGANI_MC_MAX_DIM * kBins;

thread_local std::string g_mc_create_error;

// Iterations queued between two reads of the run's state at most: later ones
// become no-ops when the run ends.
constexpr int kQueue = 16;

// The run's state, doubles that follow the grid's ndim * (kBins + 1) entries.
enum : int {
  kEnded = 0,  // the run has ended (pagani_mc_args::ended)
  kLive,       // this iteration was sampled: k_mc_step's order to run
  kSi,
  kSchi,
  kSwgt,
  kEstimate,
  kChiSq,
  kErrorest,
  kStatus,
  kCount,  // iterations run of those queued together
  kTi,
  kTsi = kTi + kQueue,
  kStateDoubles = kTsi + kQueue
};

// Sums over the workgroups: out[0] = sum fb, out[1] = sum f2b, out[2 + i] =
// histogram entry i.  Workgroup b folds 64 entries: wave w of its 16 adds
// the partials of workgroups w, w + 16, ... in that order, then the wave
// sums are added in wave order -- a fixed order for any run.  Bound by the
// latency of that chain of loads (2 500 entries of 701 workgroups: 25 us one
// by one), so each wave has eight in flight.
constexpr int kRedWaves = 16;
constexpr std::uint32_t kRedDepth = 8;

__global__ void __launch_bounds__(64 * kRedWaves)
    k_mc_reduce(const double* __restrict__ part, const double* __restrict__ hist,
                std::uint32_t grid, std::uint32_t nhist, double* __restrict__ out,
                double* __restrict__ state)
{
  __shared__ double ws[kRedWaves][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const std::uint32_t t = blockIdx.x * 64 + lane;  // output entry
  const bool ended = state[kEnded] != 0.0;
  if (blockIdx.x == 0 && threadIdx.x == 0) state[kLive] = ended ? 0.0 : 1.0;
  if (ended) return;
  double s = 0.0;
  if (t < nhist + 2) {
    const double* p = t < 2 ? part + t : hist + (t - 2);
    const std::size_t step = t < 2 ? 2 : nhist;
    std::uint32_t g = wave;
    for (; g + (kRedDepth - 1) * kRedWaves < grid; g += kRedDepth * kRedWaves) {
      double v[kRedDepth];
#pragma unroll
      for (std::uint32_t k = 0; k < kRedDepth; ++k) v[k] = p[(g + k * kRedWaves) * step];
#pragma unroll
      for (std::uint32_t k = 0; k < kRedDepth; ++k) s += v[k];
    }
    for (; g < grid; g += kRedWaves) s += p[g * step];
  }
  ws[wave][lane] = s;
  __syncthreads();
  if (wave == 0 && t < nhist + 2) {
    double r = ws[0][lane];
#pragma unroll
    for (int w = 1; w < kRedWaves; ++w) r += ws[w][lane];
    out[t] = r;
  }
}

// What ends an iteration, one workgroup per adapted axis: its grid refined
// in place, and in the first one the iteration joined to the run's weighted
// mean and the stopping rule.  On the host these were a copy, a
// synchronisation, 2 500 powers and an upload, 100 us of an iteration of 130
// (5D, 10^6 samples).
constexpr int kStepThreads = 512;
constexpr double kAlpha = 1.5;  // Internal_Vegas_Params alph, vegas_utils.cuh:158
static_assert(kBins < kStepThreads, "a thread per bin, and one to spare");

// One iteration into the running weighted mean (vegasT.cuh:847-859,
// :968-980): the estimate, chi^2 per degree of freedom and standard
// deviation, then GetStatus (vegas_utils.cuh:233-254).
__device__ void combine(double* st, double ti, double tsi, int it, double epsrel, double epsabs)
{
#pragma clang fp contract(off)
  const double wgt = 1.0 / tsi;
  const double si = st[kSi] + wgt * ti;
  const double schi = st[kSchi] + wgt * ti * ti;
  const double swgt = st[kSwgt] + wgt;
  const double estimate = si / swgt;
  double chi_sq = (schi - si * estimate) / (static_cast<double>(it) - 0.9999);
  if (chi_sq < 0.0) chi_sq = 0.0;
  const double errorest = __builtin_sqrt(1.0 / swgt);
  st[kSi] = si;
  st[kSchi] = schi;
  st[kSwgt] = swgt;
  st[kEstimate] = estimate;
  st[kChiSq] = chi_sq;
  st[kErrorest] = errorest;
  const bool ok = fabs(errorest / estimate) <= epsrel || errorest <= epsabs;
  st[kStatus] = ok && it >= 5 ? 0.0 : 1.0;
  if (ok && it >= 5) st[kEnded] = 1.0;
}

// The refinement after an adjusting iteration (vegasT.cuh:880-925) of one
// axis: the smoothed bins' damped weights r, and rebin (vegasT.cuh:617-637):
// new right edges that put the weight rc in every bin, linear inside the old
// bins.  The reference walks the bins with a running remainder; here edge i
// lies where the weights' prefix sum C reaches i rc, found by a search, with
// C and i rc to twice the working precision, so no edge carries the rounding
// of the edges before it.
__device__ bool refine_axis(const double* __restrict__ hist, const double* xi, double& edge)
{
#pragma clang fp contract(off)
  __shared__ double h[kBins + 1], x[kBins + 1], r[kBins + 1];
  __shared__ ph::DD C[kBins + 1], wsum[kStepThreads / 64];
  const int i = threadIdx.x + 1, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (i <= kBins) {
    h[i] = hist[i - 1];
    x[i] = xi[i];
  }
  if (i == 1) x[0] = xi[0];
  __syncthreads();
  double s = 0.0;
  if (i == 1)
    s = (h[1] + h[2]) / 2.0;
  else if (i < kBins)
    s = (h[i - 1] + h[i] + h[i + 1]) / 3.0;
  else if (i == kBins)
    s = (h[kBins - 1] + h[kBins]) / 2.0;
  ph::DD t = ph::wave_reduce(ph::DD{s, 0.0});
  if (lane == 0) wsum[wave] = t;
  __syncthreads();
  t = wsum[0];
#pragma unroll
  for (int w = 1; w < kStepThreads / 64; ++w) t = ph::dd_add(t, wsum[w]);
  const double dt = t.hi + t.lo;
  if (!(dt > 0.0)) return false;
  const double ri = i <= kBins ? pow((1.0 - s / dt) / (log(dt) - log(s)), kAlpha) : 0.0;
  ph::DD c{ri, 0.0};
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    ph::DD y;
    y.hi = __shfl_up(c.hi, o, 64);
    y.lo = __shfl_up(c.lo, o, 64);
    if (lane >= o) c = ph::dd_add(y, c);
  }
  __syncthreads();  // wsum's first use is over
  if (lane == 63) wsum[wave] = c;
  __syncthreads();
  ph::DD before{0.0, 0.0}, total{0.0, 0.0};
#pragma unroll
  for (int w = 0; w < kStepThreads / 64; ++w) {
    if (w < wave) before = ph::dd_add(before, wsum[w]);
    total = ph::dd_add(total, wsum[w]);
  }
  if (i <= kBins) {
    C[i] = ph::dd_add(before, c);
    r[i] = ri;
  }
  __syncthreads();
  if (i > kBins) return false;
  edge = 1.0;
  if (i < kBins) {
    const double rc = (total.hi + total.lo) / static_cast<double>(kBins);
    const double th = i * rc, tl = __builtin_fma(static_cast<double>(i), rc, -th);
    edge = pagani::mc::rebin_edge(C, r, x, kBins, th, tl);
  }
  return true;
}

__global__ void __launch_bounds__(kStepThreads)
    k_mc_step(int d, int hist_dims, int it, int slot, int joins, double dv2g, double epsrel,
              double epsabs, const double* __restrict__ out, double* xi, double* state)
{
  if (state[kLive] == 0.0) return;
  if (blockIdx.x == 0 && threadIdx.x == blockDim.x - 1) {  // a thread without a bin
    const double ti = out[0], tsi = out[1] * dv2g;
    state[kTi + slot] = ti;
    state[kTsi + slot] = tsi;
    state[kCount] = slot + 1;
    if (joins) combine(state, ti, tsi, it, epsrel, epsabs);
  }
  if (!hist_dims) return;
  const int axis = blockIdx.x, i = threadIdx.x + 1;
  double edge = 0.0;
  if (refine_axis(out + 2 + axis * kBins, xi + axis * (kBins + 1), edge)) {
    // one adapted axis is every axis' grid (vegasT1D.cuh:606-636)
    const int last = hist_dims == 1 ? d : axis + 1;
    for (int j = axis; j < last; ++j) xi[j * (kBins + 1) + i] = edge;
  }
}

}  // namespace

struct pagani_mc {
  int ndim = 0;
  int device = 0;
  hipStream_t stream = nullptr;
  std::string error;
  double* d_xi = nullptr;   // the grid, then the run's state
  double* d_part = nullptr;
  double* d_hist = nullptr;
  double* d_out = nullptr;
  double* h_out = nullptr;  // pinned
  double* h_xi = nullptr;   // pinned, as d_xi
  std::vector<double> ti, tsi;
  std::vector<double> grid;  // last run's final grid
  bool timing = false;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  pagani_mc_stats stats{};
};

namespace {

std::size_t grid_size(const pagani_mc* mc)
{
  return static_cast<std::size_t>(mc->ndim) * (kBins + 1);
}

int fail(pagani_mc* mc, int code, const std::string& msg)
{
  if (mc) mc->error = msg;
  return code;
}

int hip_fail(pagani_mc* mc, hipError_t e, const char* where)
{
  (void)hipGetLastError();
  return fail(mc, PAGANI_EHIP, std::string(where) + ": " + hipGetErrorString(e));
}

#define MC_TRY(mc, expr)                                  \
  do {                                                    \
    const hipError_t e_ = (expr);                         \
    if (e_ != hipSuccess) return hip_fail(mc, e_, #expr); \
  } while (0)

struct Launch {
  std::uint32_t grid = 0, cpt = 0;
};

// cubes_per_thread so that at most kMaxGrid workgroups cover every cube
Launch shape(std::uint64_t ncubes)
{
  const std::uint64_t per_wg_max = static_cast<std::uint64_t>(kThreads) * kMaxGrid;
  Launch l;
  l.cpt = static_cast<std::uint32_t>(std::max<std::uint64_t>(1, (ncubes + per_wg_max - 1) / per_wg_max));
  const std::uint64_t per_wg = static_cast<std::uint64_t>(kThreads) * l.cpt;
  l.grid = static_cast<std::uint32_t>((ncubes + per_wg - 1) / per_wg);
  return l;
}

int check_setup(pagani_mc* mc, const pagani::mc::Setup& s)
{
  if (!(s.ng >= 1) || !(s.ncubes >= 1))
    return fail(mc, PAGANI_EBADARG, "ncall too small: no stratum per axis");
  if (s.ncubes >= 4294967296.0)
    return fail(mc, PAGANI_EUNSUPPORTED, "more than 2^32 cubes (the reference numbers cubes in 32 bits)");
  return PAGANI_OK;
}

void fill_args(pagani_mc* mc, const pagani::mc::Setup& s, const Launch& l, int generator,
               pagani_mc_args& a)
{
  std::memset(&a, 0, sizeof(a));
  a.xi = mc->d_xi;
  for (int j = 0; j < mc->ndim; ++j) {
    a.lo[j] = s.lo[j];
    a.dx[j] = s.dx[j];
  }
  a.xjac = s.xjac;
  a.dxg = s.dxg;
  a.xnd = s.xnd;
  a.ncubes = static_cast<std::uint32_t>(s.ncubes);
  a.ng = static_cast<std::uint32_t>(s.ng);
  a.npg = static_cast<std::uint32_t>(s.npg);
  a.cubes_per_thread = l.cpt;
  a.grid = l.grid;
  a.generator = generator;
  a.part = mc->d_part;
  a.hist = mc->d_hist;
  a.stream = mc->stream;
  a.ended = nullptr;
}

// One sampling launch and its reduction into d_out, queued.
int queue_pass(pagani_mc* mc, pagani_mc_sample_fn sample, void* ctx, pagani_mc_args& a)
{
  const std::uint32_t nhist = a.hist_dims * kBins;
  if (mc->timing) MC_TRY(mc, hipEventRecord(mc->ev0, mc->stream));
  const int rc = sample(ctx, &a);
  if (rc) return fail(mc, rc < 0 ? rc : PAGANI_EHIP, "sampling callback failed");
  if (mc->timing) MC_TRY(mc, hipEventRecord(mc->ev1, mc->stream));
  hipLaunchKernelGGL(k_mc_reduce, dim3((nhist + 2 + 63) / 64), dim3(64 * kRedWaves), 0,
                     mc->stream, mc->d_part, mc->d_hist, a.grid, nhist, mc->d_out,
                     mc->d_xi + grid_size(mc));
  MC_TRY(mc, hipGetLastError());
  return PAGANI_OK;
}

int add_sample_time(pagani_mc* mc)
{
  if (!mc->timing) return PAGANI_OK;
  float ms = 0;
  MC_TRY(mc, hipEventElapsedTime(&ms, mc->ev0, mc->ev1));
  mc->stats.sample_ms += ms;
  return PAGANI_OK;
}

// The grid and a run's fresh state.
int upload_grid(pagani_mc* mc, const double* xi, const pagani_mc_result* so_far)
{
  const std::size_t n = grid_size(mc);
  std::memcpy(mc->h_xi, xi, n * sizeof(double));
  double* st = mc->h_xi + n;
  std::fill(st, st + kStateDoubles, 0.0);
  st[kStatus] = 1.0;
  if (so_far) {
    st[kEstimate] = so_far->estimate;
    st[kChiSq] = so_far->chi_sq;
    st[kErrorest] = so_far->errorest;
  }
  MC_TRY(mc, hipMemcpyAsync(mc->d_xi, mc->h_xi, (n + kStateDoubles) * sizeof(double),
                            hipMemcpyHostToDevice, mc->stream));
  return PAGANI_OK;
}

// One vegas() run: adjust_iters iterations that refine the grid, then the
// others up to titer.  Chunks of `queue` iterations are queued, each three
// launches with no word from the host in between; when the stopping rule
// ends the run, the rest of the chunk does nothing.
int run(pagani_mc* mc, pagani_mc_sample_fn sample, void* ctx, int queue, double epsrel,
        double epsabs, const double* lows, const double* highs, const pagani_mc_params& p,
        double ncall, int titer, pagani_mc_result* out)
{
  const int d = mc->ndim;
  pagani::mc::Setup s;
  pagani::mc::setup(s, d, ncall, lows, highs);
  int rc = check_setup(mc, s);
  if (rc) return rc;
  const int hd = p.one_axis ? 1 : d;
  std::vector<double> xi(grid_size(mc));
  pagani::mc::grid_init(d, xi.data());
  const Launch l = shape(static_cast<std::uint64_t>(s.ncubes));
  pagani_mc_args a;
  fill_args(mc, s, l, p.generator, a);
  const std::uint64_t per_iter = static_cast<std::uint64_t>(s.calls);
  if ((rc = upload_grid(mc, xi.data(), out))) return rc;
  double* const state = mc->d_xi + xi.size();
  const double* const st = mc->h_xi + xi.size();
  if (queue > 1) a.ended = state + kEnded;
  const int last = std::max(p.adjust_iters, titer);
  for (int it = 1; it <= last && out->status;) {
    const int first = it, end = std::min(last, it + queue - 1);
    for (; it <= end; ++it) {
      const bool adjusts = it <= p.adjust_iters;
      a.hist_dims = adjusts ? static_cast<std::uint32_t>(hd) : 0;
      a.key = pagani::mc::iter_key(p.seed, it);
      if (!(rc = queue_pass(mc, sample, ctx, a))) {
        hipLaunchKernelGGL(k_mc_step, dim3(adjusts ? hd : 1), dim3(adjusts ? kStepThreads : 64), 0,
                           mc->stream, d, static_cast<int>(a.hist_dims), it, it - first,
                           !adjusts || it > p.skip_iters ? 1 : 0, s.dv2g, epsrel, epsabs,
                           mc->d_out, mc->d_xi, state);
        if (hipGetLastError() != hipSuccess) rc = fail(mc, PAGANI_EHIP, "k_mc_step launch failed");
      }
      if (rc) {
        (void)hipStreamSynchronize(mc->stream);  // h_xi is the next run's
        return rc;
      }
    }
    // the state, and with it the grid
    MC_TRY(mc, hipMemcpyAsync(mc->h_xi, mc->d_xi, (xi.size() + kStateDoubles) * sizeof(double),
                              hipMemcpyDeviceToHost, mc->stream));
    MC_TRY(mc, hipStreamSynchronize(mc->stream));
    if ((rc = add_sample_time(mc))) return rc;
    const int done = static_cast<int>(st[kCount]);
    for (int k = 0; k < done; ++k) {
      mc->ti.push_back(st[kTi + k]);
      mc->tsi.push_back(st[kTsi + k]);
    }
    out->iters += done;
    out->neval += per_iter * done;
    mc->stats.samples += per_iter * done;
    mc->stats.launches += done;
    out->estimate = st[kEstimate];
    out->chi_sq = st[kChiSq];
    out->errorest = st[kErrorest];
    out->status = st[kStatus] != 0.0 ? 1 : 0;
    std::copy(mc->h_xi, mc->h_xi + xi.size(), xi.begin());
  }
  mc->grid = xi;
  return PAGANI_OK;
}

int validate(pagani_mc* mc, const pagani_mc_params* p, const double* lows, const double* highs)
{
  if (!p) return fail(mc, PAGANI_EBADARG, "null params");
  if (!(p->ncall >= 1) || p->total_iters < 0 || p->adjust_iters < 0 || p->skip_iters < 0)
    return fail(mc, PAGANI_EBADARG, "bad m-Cubes parameters");
  if (p->generator != PAGANI_MC_RNG_DEFAULT && p->generator != PAGANI_MC_RNG_LCG)
    return fail(mc, PAGANI_EBADARG, "unknown generator");
  for (int j = 0; j < mc->ndim; ++j) {
    const double lo = lows ? lows[j] : 0.0, hi = highs ? highs[j] : 1.0;
    if (!(hi > lo)) return fail(mc, PAGANI_EBADARG, "empty integration box");
  }
  return PAGANI_OK;
}

template <int D>
int genz_sample(void* ctx, const pagani_mc_args* a)
{
  const pagani_genz* g = static_cast<const pagani_genz*>(ctx);
  return pagani::internal::visit_genz<double, D>(
      g, [&](const auto& f) { return pagani::mc::launch_any<D>(f, a); });
}

pagani_mc_sample_fn genz_sampler(int ndim)
{
  switch (ndim) {
    case 2: return &genz_sample<2>;
    case 3: return &genz_sample<3>;
    case 4: return &genz_sample<4>;
    case 5: return &genz_sample<5>;
    case 6: return &genz_sample<6>;
    case 7: return &genz_sample<7>;
    case 8: return &genz_sample<8>;
    default: return nullptr;
  }
}

int integrate(pagani_mc* mc, pagani_mc_sample_fn sample, void* ctx, int queue, double epsrel,
              double epsabs, const double* lows, const double* highs,
              const pagani_mc_params* params, pagani_mc_result* out)
{
  if (!mc) return PAGANI_EBADARG;
  if (!out || !sample) return fail(mc, PAGANI_EBADARG, "null argument");
  std::memset(out, 0, sizeof(*out));
  out->status = 1;
  int rc = validate(mc, params, lows, highs);
  if (rc) return rc;
  MC_TRY(mc, hipSetDevice(mc->device));
  const auto t0 = std::chrono::steady_clock::now();
  mc->ti.clear();
  mc->tsi.clear();
  double ncall = params->ncall;
  int titer = params->total_iters;
  do {
    out->runs++;
    out->ncall = ncall;
    rc = run(mc, sample, ctx, queue, epsrel, epsabs, lows, highs, *params, ncall, titer, out);
    if (rc) {
      out->status = 1;
      return rc;
    }
  } while (params->adjust_params && out->status == 1 && pagani::mc::adjust_params(ncall, titer));
  mc->stats.integrals++;
  mc->stats.wall_ms +=
      std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  return PAGANI_OK;
}

}  // namespace

extern "C" {

pagani_mc* pagani_mc_create(int ndim, int device)
{
  g_mc_create_error.clear();
  if (ndim < 1 || ndim > PAGANI_MC_MAX_DIM) {
    g_mc_create_error = "ndim outside [1, 16]";
    return nullptr;
  }
  int ndev = 0;
  hipError_t e = hipGetDeviceCount(&ndev);
  if (e != hipSuccess || ndev <= 0) {
    (void)hipGetLastError();
    g_mc_create_error = std::string("hipGetDeviceCount: ") + hipGetErrorString(e);
    return nullptr;
  }
  if (device < 0 && hipGetDevice(&device) != hipSuccess) {
    (void)hipGetLastError();
    g_mc_create_error = "hipGetDevice failed";
    return nullptr;
  }
  if (device >= ndev) {
    g_mc_create_error = "device index out of range";
    return nullptr;
  }
  if ((e = hipSetDevice(device)) != hipSuccess) {
    (void)hipGetLastError();
    g_mc_create_error = std::string("hipSetDevice: ") + hipGetErrorString(e);
    return nullptr;
  }
  pagani_mc* mc = new pagani_mc();
  mc->ndim = ndim;
  mc->device = device;
  const std::size_t nxi = grid_size(mc) + kStateDoubles;
  const std::size_t nhist = static_cast<std::size_t>(kMaxGrid) * ndim * kBins;
  bool ok = hipStreamCreateWithFlags(&mc->stream, hipStreamNonBlocking) == hipSuccess &&
            hipMalloc(&mc->d_xi, nxi * sizeof(double)) == hipSuccess &&
            hipMalloc(&mc->d_part, 2 * kMaxGrid * sizeof(double)) == hipSuccess &&
            hipMalloc(&mc->d_hist, nhist * sizeof(double)) == hipSuccess &&
            hipMalloc(&mc->d_out, kOutDoubles * sizeof(double)) == hipSuccess &&
            hipHostMalloc(&mc->h_out, kOutDoubles * sizeof(double), hipHostMallocDefault) ==
                hipSuccess &&
            hipHostMalloc(&mc->h_xi, nxi * sizeof(double), hipHostMallocDefault) == hipSuccess &&
            hipEventCreate(&mc->ev0) == hipSuccess && hipEventCreate(&mc->ev1) == hipSuccess;
  if (!ok) {
    (void)hipGetLastError();
    g_mc_create_error = "device allocation failed";
    pagani_mc_destroy(mc);
    return nullptr;
  }
  return mc;
}

void pagani_mc_destroy(pagani_mc* mc)
{
  if (!mc) return;
  (void)hipSetDevice(mc->device);
  if (mc->stream) (void)hipStreamSynchronize(mc->stream);
  if (mc->d_xi) (void)hipFree(mc->d_xi);
  if (mc->d_part) (void)hipFree(mc->d_part);
  if (mc->d_hist) (void)hipFree(mc->d_hist);
  if (mc->d_out) (void)hipFree(mc->d_out);
  if (mc->h_out) (void)hipHostFree(mc->h_out);
  if (mc->h_xi) (void)hipHostFree(mc->h_xi);
  if (mc->ev0) (void)hipEventDestroy(mc->ev0);
  if (mc->ev1) (void)hipEventDestroy(mc->ev1);
  if (mc->stream) (void)hipStreamDestroy(mc->stream);
  delete mc;
}

const char* pagani_mc_last_error(const pagani_mc* mc)
{
  return mc ? mc->error.c_str()
            : (g_mc_create_error.empty() ? "null m-Cubes handle" : g_mc_create_error.c_str());
}

int pagani_mc_set_timing(pagani_mc* mc, int enable)
{
  if (!mc) return PAGANI_EBADARG;
  mc->timing = enable != 0;
  return PAGANI_OK;
}

int pagani_mc_get_stats(const pagani_mc* mc, pagani_mc_stats* out)
{
  if (!mc || !out) return PAGANI_EBADARG;
  *out = mc->stats;
  return PAGANI_OK;
}

int pagani_mc_reset_stats(pagani_mc* mc)
{
  if (!mc) return PAGANI_EBADARG;
  mc->stats = pagani_mc_stats{};
  return PAGANI_OK;
}

int pagani_mc_integrate_cb(pagani_mc* mc, pagani_mc_sample_fn sample, void* ctx, double epsrel,
                           double epsabs, const double* lows, const double* highs,
                           const pagani_mc_params* params, pagani_mc_result* out)
{
  return integrate(mc, sample, ctx, 1, epsrel, epsabs, lows, highs, params, out);
}

int pagani_mc_integrate_queued(pagani_mc* mc, pagani_mc_sample_fn sample, void* ctx,
                               double epsrel, double epsabs, const double* lows,
                               const double* highs, const pagani_mc_params* params,
                               pagani_mc_result* out)
{
  // with timing on, an event pair around each iteration's sampling
  const int queue = mc && mc->timing ? 1 : kQueue;
  return integrate(mc, sample, ctx, queue, epsrel, epsabs, lows, highs, params, out);
}

int pagani_mc_integrate_genz(pagani_mc* mc, const pagani_genz* f, double epsrel,
                             double epsabs, const double* lows, const double* highs,
                             const pagani_mc_params* params, pagani_mc_result* out)
{
  if (!mc) return PAGANI_EBADARG;
  if (!f || !out) return fail(mc, PAGANI_EBADARG, "null argument");
  if (f->ndim != mc->ndim) return fail(mc, PAGANI_EBADARG, "descriptor ndim differs from the handle's");
  const pagani_mc_sample_fn fn = genz_sampler(f->ndim);
  if (!fn) return fail(mc, PAGANI_EUNSUPPORTED, "Genz descriptors cover ndim 2..8");
  if (f->family < PAGANI_GENZ_OSCILLATORY || f->family > PAGANI_GENZ_DISCONTINUOUS)
    return fail(mc, PAGANI_EBADARG, "unknown Genz family");
  pagani_genz g = *f;
  return pagani_mc_integrate_queued(mc, fn, &g, epsrel, epsabs, lows, highs, params, out);
}

int pagani_mc_trace(const pagani_mc* mc, double* ti, double* tsi, size_t cap, size_t* len)
{
  if (!mc) return PAGANI_EBADARG;
  const std::size_t n = mc->ti.size();
  for (std::size_t i = 0; i < n && i < cap; ++i) {
    if (ti) ti[i] = mc->ti[i];
    if (tsi) tsi[i] = mc->tsi[i];
  }
  if (len) *len = n;
  return PAGANI_OK;
}

int pagani_mc_grid(const pagani_mc* mc, double* xi)
{
  if (!mc || !xi) return PAGANI_EBADARG;
  if (mc->grid.empty()) return PAGANI_EBADARG;
  std::memcpy(xi, mc->grid.data(), mc->grid.size() * sizeof(double));
  return PAGANI_OK;
}

int pagani_mc_sample_genz(pagani_mc* mc, const pagani_genz* f, double ncall, const double* lows,
                          const double* highs, const double* xi, uint64_t key, int generator,
                          int hist_dims, double* ti, double* tsi, double* hist)
{
  if (!mc) return PAGANI_EBADARG;
  if (!f || !xi || !ti || !tsi || (hist_dims && !hist))
    return fail(mc, PAGANI_EBADARG, "null argument");
  if (f->ndim != mc->ndim) return fail(mc, PAGANI_EBADARG, "descriptor ndim differs from the handle's");
  if (hist_dims != 0 && hist_dims != 1 && hist_dims != mc->ndim)
    return fail(mc, PAGANI_EBADARG, "hist_dims must be 0, 1 or ndim");
  const pagani_mc_sample_fn fn = genz_sampler(f->ndim);
  if (!fn) return fail(mc, PAGANI_EUNSUPPORTED, "Genz descriptors cover ndim 2..8");
  pagani_mc_params p{};
  p.ncall = ncall;
  p.generator = generator;
  int rc = validate(mc, &p, lows, highs);
  if (rc) return rc;
  MC_TRY(mc, hipSetDevice(mc->device));
  pagani::mc::Setup s;
  pagani::mc::setup(s, mc->ndim, ncall, lows, highs);
  if ((rc = check_setup(mc, s))) return rc;
  if ((rc = upload_grid(mc, xi, nullptr))) return rc;
  const Launch l = shape(static_cast<std::uint64_t>(s.ncubes));
  pagani_mc_args a;
  fill_args(mc, s, l, generator, a);
  a.hist_dims = static_cast<std::uint32_t>(hist_dims);
  a.key = key;
  pagani_genz desc = *f;
  if ((rc = queue_pass(mc, fn, &desc, a))) return rc;
  MC_TRY(mc, hipMemcpyAsync(mc->h_out, mc->d_out, (hist_dims * kBins + 2) * sizeof(double),
                            hipMemcpyDeviceToHost, mc->stream));
  MC_TRY(mc, hipStreamSynchronize(mc->stream));
  if ((rc = add_sample_time(mc))) return rc;
  mc->stats.samples += static_cast<std::uint64_t>(s.calls);
  mc->stats.launches++;
  *ti = mc->h_out[0];
  *tsi = mc->h_out[1];
  if (hist_dims)
    std::memcpy(hist, mc->h_out + 2, static_cast<std::size_t>(hist_dims) * kBins * sizeof(double));
  return PAGANI_OK;
}

}  // extern "C"

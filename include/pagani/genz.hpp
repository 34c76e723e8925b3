// genz.hpp -- the six Genz test families as device functors.
//
// The reference's fixed-parameter functors F_1..F_6 (common/cuda/
// integrands.cuh:1303-1934) are instances of these families with given
// (a, u).  Real = double for the FP64 path, float for the mixed-precision
// path (FP32 integrand, FP64 accumulation).  Parameters are pre-processed on
// the host (a^2, 1/a^2, 2*pi*u_0) so the device does no divisions by a.
//
// The families that depend on x only through x - u (product peak, Gaussian,
// C0) also offer the "centred" form: origin(i) = u_i and centered(t...) =
// f(u + t).  The evaluation kernel then folds u into each region's centre
// once, so a rule point costs one FMA per axis fewer.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <type_traits>

#include "pagani.h"

namespace pagani {
namespace math {

// e^x for x <= 709 (the exponents of the Gaussian and C0 families are minus
// sums of non-negative terms, the discontinuous family's are bounded by
// sum a_i).  x = n ln2 + r with n the integer nearest x / ln2 and |r| <=
// ln2/2, r from a two-part ln2 (Cody-Waite); e^r by a degree-11 polynomial;
// 2^n by ldexp, which also rounds subnormal results, gives 0 below about
// -745.1 and infinity above about 709.78.  n comes from one FMA: adding
// 1.5 * 2^52 to x log2e (|x log2e| < 2^51) leaves a double whose unit is 1,
// so the sum is rounded to the nearest integer, which its low 32 bits hold
// in two's complement; subtracting the shift again gives n as a double (no
// separate multiply, round or conversion instruction).  The coefficients
// interpolate e^r at the 12 Chebyshev nodes of [-ln2/2, ln2/2] (computed in
// extended precision, then rounded to double; the check that recomputes
// them is in the tests): max polynomial error 0.14 ulp.  The range handling
// is one clamp, which also maps -inf to 0 (and NaN to 0: the families never
// produce NaN from finite input).
__device__ __forceinline__ double exp_bounded(double x)
{
  constexpr double kLog2e = 0x1.71547652b82fep+0;
  constexpr double kLn2Hi = 0x1.62e42fefa39efp-1;
  constexpr double kLn2Lo = 0x1.abc9e3b39803fp-56;
  constexpr double kShift = 0x1.8p+52;
  constexpr double c[12] = {
      0x1.0000000000000p+0,  0x1.0000000000000p+0,  0x1.0000000000011p-1, 0x1.555555555555fp-3,
      0x1.555555554f0c7p-5,  0x1.111111110e636p-7,  0x1.6c16c187face9p-10, 0x1.a01a01b4a99f9p-13,
      0x1.a01991b378c3ap-16, 0x1.71ddeea4df7bbp-19, 0x1.28b3fce70e98ep-22, 0x1.af6d18013a587p-26};
  x = __builtin_fmax(x, -1.0e4);
  const double t = __builtin_fma(x, kLog2e, kShift);
  const double n = t - kShift;
  double r = __builtin_fma(-n, kLn2Hi, x);
  r = __builtin_fma(-n, kLn2Lo, r);
  double p = c[11];
#pragma unroll
  for (int k = 10; k >= 0; --k) p = __builtin_fma(p, r, c[k]);
  return __builtin_ldexp(p, static_cast<int>(__builtin_bit_cast(unsigned long long, t)));
}
__device__ __forceinline__ double exp_neg(double x) { return exp_bounded(x); }
__device__ __forceinline__ float exp_neg(float x) { return ::expf(x); }
__device__ __forceinline__ float exp_bounded(float x) { return ::expf(x); }

__device__ __forceinline__ double exp_(double x) { return ::exp(x); }
__device__ __forceinline__ float exp_(float x) { return ::expf(x); }
__device__ __forceinline__ double cos_(double x) { return ::cos(x); }
__device__ __forceinline__ float cos_(float x) { return ::cosf(x); }
__device__ __forceinline__ double fabs_(double x) { return __builtin_fabs(x); }
__device__ __forceinline__ float fabs_(float x) { return __builtin_fabsf(x); }
__device__ __forceinline__ double fmax_(double x, double y) { return __builtin_fmax(x, y); }
__device__ __forceinline__ float fmax_(float x, float y) { return __builtin_fmaxf(x, y); }
// x y + z.  FP64: the contraction written out, so that every kernel an
// integrand is inlined into (the launches, the short-list loop, the segments)
// forms the same bits.  FP32 integrands run in the evaluation kernel alone,
// which contracts each place as it did before the others existed (the first
// two products either way round, by how often they are used): 1 ulp of an FP32
// value is 1e-3 of a small error estimate.
__device__ __forceinline__ double fma_(double x, double y, double z) { return __builtin_fma(x, y, z); }
__device__ __forceinline__ float fma_(float x, float y, float z) { return z + x * y; }
}  // namespace math

// The rule's generator magnitudes lambda1..lambda5 (rule.cpp's kLam): the
// points of one axis are c -+ lambda_i h.
constexpr double kLambda[5] = {.4779536579022695061928604197171830064732,
                               .2030285873691198677998034402373279133258,
                               .4476273546261781288207704806530998539285, .125,
                               .3430378987808781457001426145164678603407};
constexpr double lambda2(int i) { return kLambda[i] * kLambda[i]; }

// Truncated Taylor series and the rule's magnitudes, for the pair sums of the
// factored integrands (eval_kernel.hpp, has_pair_sums).
namespace series {
constexpr double factorial(int n)
{
  double f = 1.0;
  for (int k = 2; k <= n; ++k) f *= k;
  return f;
}
// The degree N in z of sum_k z^k / (Step k + Off)! whose first term left out
// is at most 2^-56 for 0 <= z <= zmax (the sums here are at least 1).
constexpr int degree(double zmax, int Step, int Off = 0)
{
  double p = zmax;
  for (int n = 0;; ++n, p *= zmax)
    if (p <= 0x1p-56 * factorial(Step * (n + 1) + Off)) return n;
}
// sum_{k <= N} z^k / (Step k + Off)!
template <int N, int Step, int Off>
__device__ __forceinline__ double sum(double z)
{
#pragma clang fp contract(off)
  double p = 1.0 / factorial(Step * N + Off);
#pragma unroll
  for (int k = N - 1; k >= 0; --k) p = __builtin_fma(p, z, 1.0 / factorial(Step * k + Off));
  return p;
}
// fn(std::integral_constant<int, i>) for the rule's five magnitudes
template <class Fn>
__device__ __forceinline__ void for_lambda(Fn&& fn)
{
  fn(std::integral_constant<int, 0>{});
  fn(std::integral_constant<int, 1>{});
  fn(std::integral_constant<int, 2>{});
  fn(std::integral_constant<int, 3>{});
  fn(std::integral_constant<int, 4>{});
}
}  // namespace series

// The largest centre sum s0 for which an exponential family evaluates a
// region as products: e^s0 and e^-s0 stay normal with room to spare (FP64
// 2^+-1022 is e^+-708; FP32 2^+-126 is e^+-87).
template <class Real>
constexpr double kFactorRange = sizeof(Real) == 8 ? 650.0 : 80.0;

namespace math {
// e^x (x <= 709) for the product forms of the exponential families: at
// the integrand's precision where it holds the value (FP32: |x| <= 80),
// else in FP64, so that an FP32 integrand's centre values and factors stay
// normal over the FP64 range of the products.
__device__ __forceinline__ double exp_factor(double x, double) { return exp_bounded(x); }

// 1 / x for finite, normal x: the hardware reciprocal refined by two
// Newton steps (each doubles the correct bits: r' = r + r (1 - x r)).
__device__ __forceinline__ double recip(double x)
{
  double r = __builtin_amdgcn_rcp(x);
  double e = __builtin_fma(-x, r, 1.0);
  r = __builtin_fma(r, e, r);
  e = __builtin_fma(-x, r, 1.0);
  return __builtin_fma(r, e, r);
}
// a / b for finite, normal b with a normal reciprocal: one Newton step (48
// bits), and the quotient corrected by its remainder.
__device__ __forceinline__ double quotient(double a, double b)
{
  double r = __builtin_amdgcn_rcp(b);
  r = __builtin_fma(r, __builtin_fma(-b, r, 1.0), r);
  const double q = a * r;
  return __builtin_fma(__builtin_fma(-q, b, a), r, q);
}
__device__ __forceinline__ double exp_factor(double x, float)
{
  return __builtin_fabs(x) <= 80.0 ? static_cast<double>(::expf(static_cast<float>(x)))
                                   : exp_bounded(x);
}
}  // namespace math

// 2 cosh(l_i n/2) and 2 l_i sinh(l_i n/2) for the rule's five magnitudes and
// n < kCoshSteps, [(5 n + i) 2], formed by the compiler: the powers of
// e^(+-l_i/2) in double-double arithmetic (two-sum, and Dekker's product).
constexpr int kCoshSteps = 201, kCoshLds = 51;
struct CoshTable {
  double v[kCoshSteps * 10];
};
namespace dd {
struct Num {
  double hi, lo;
};
constexpr Num norm(double a, double b)
{
  const double s = a + b, t = s - a;
  return {s, (a - (s - t)) + (b - t)};
}
constexpr Num add(Num a, Num b)
{
  const Num s = norm(a.hi, b.hi);
  return norm(s.hi, s.lo + a.lo + b.lo);
}
constexpr Num mul(Num a, Num b)
{
  constexpr double k = 134217729.0;  // 2^27 + 1
  const double ta = k * a.hi, ah = ta - (ta - a.hi), al = a.hi - ah;
  const double tb = k * b.hi, bh = tb - (tb - b.hi), bl = b.hi - bh;
  const double p = a.hi * b.hi;
  const double e = ((ah * bh - p) + ah * bl + al * bh) + al * bl;
  return norm(p, e + (a.hi * b.lo + a.lo * b.hi));
}
// e^x, |x| < 1/4: the Taylor series by Horner's rule, 1 + x/1 (1 + x/2 (...));
// the quotients x/k corrected by one residual
constexpr Num exp(double x)
{
  Num s{1.0, 0.0};
  for (int k = 26; k >= 1; --k) {
    const double q = x / k;
    const Num r = mul({q, 0.0}, {static_cast<double>(k), 0.0});
    s = add({1.0, 0.0}, mul(s, {q, ((x - r.hi) - r.lo) / k}));
  }
  return s;
}
}  // namespace dd
constexpr CoshTable make_cosh_table()
{
  CoshTable t{};
  for (int i = 0; i < 5; ++i) {
    const dd::Num up = dd::exp(.5 * kLambda[i]), down = dd::exp(-.5 * kLambda[i]);
    dd::Num p{1.0, 0.0}, q{1.0, 0.0};
    for (int n = 0; n < kCoshSteps; ++n) {
      t.v[2 * (5 * n + i)] = dd::add(p, q).hi;
      t.v[2 * (5 * n + i) + 1] = dd::mul(dd::add(p, {-q.hi, -q.lo}), {kLambda[i], 0.0}).hi;
      p = dd::mul(p, up);
      q = dd::mul(q, down);
    }
  }
  return t;
}
static __device__ const CoshTable kCoshTable = make_cosh_table();

// Marks a member as present for FP64 integrands only (an FP32 integrand
// keeps its FP32 functions).
template <class Real>
using if_double = std::enable_if_t<std::is_same_v<Real, double>, int>;

// cos(2 pi u_0 + sum a_i x_i)
template <class Real, int D>
struct Oscillatory {
  Real a[D];
  Real phase;  // 2 pi u_0
  template <class... X>
  __device__ Real operator()(X... xs) const
  {
    const Real x[D] = {static_cast<Real>(xs)...};
    Real s = phase;
#pragma unroll
    for (int i = 0; i < D; ++i) s += a[i] * x[i];
    return math::cos_(s);
  }
  // v = a x (origin 0): f = cos(phase + sum v), additively separable
  __device__ double origin(int) const { return 0.0; }
  __device__ double axis_scale(int i) const { return static_cast<double>(a[i]); }
  template <class... T>
  __device__ Real centered(T... vs) const
  {
    const Real v[D] = {static_cast<Real>(vs)...};
    Real s = phase;
#pragma unroll
    for (int i = 0; i < D; ++i) s += v[i];
    return math::cos_(s);
  }
  static constexpr bool heavy_outer = true;  // cos: argument reduction and two polynomials
  // f = cos(phase_angle() + sum_j v_j): the kernel sums each set's sign
  // combinations as cos of the centre's angle times per-axis cosines
  static constexpr bool cosine = true;
  __device__ double phase_angle() const { return static_cast<double>(phase); }
  __device__ double term(int, double v) const { return v; }
  __device__ double outer(double s) const
  {
    return static_cast<double>(math::cos_(static_cast<Real>(static_cast<double>(phase) + s)));
  }
};

// prod 1 / (a_i^-2 + (x_i - u_i)^2), evaluated as one division
template <class Real, int D>
struct ProductPeak {
  Real ia2[D];  // 1 / a_i^2
  Real u[D];
  Real a[D];
  double k2;    // prod a_i^2
  template <class... X>
  __device__ Real operator()(X... xs) const
  {
    const Real x[D] = {static_cast<Real>(xs)...};
    Real den = 1;
#pragma unroll
    for (int i = 0; i < D; ++i) {
      const Real t = x[i] - u[i];
      den *= ia2[i] + t * t;
    }
    return Real(1) / den;
  }
  // f(u + v / a) = prod a_i^2 / (1 + v_i^2): the kernel hands over
  // v = a (x - u); multiplicatively separable, term 1 / (1 + v^2)
  __device__ double origin(int i) const { return static_cast<double>(u[i]); }
  __device__ double axis_scale(int i) const { return static_cast<double>(a[i]); }
  template <class... T>
  __device__ Real centered(T... vs) const
  {
    const Real v[D] = {static_cast<Real>(vs)...};
    Real den = 1;
#pragma unroll
    for (int i = 0; i < D; ++i) den *= math::fma_(v[i], v[i], Real(1));
    return static_cast<Real>(k2) / den;
  }
  // With A = 1 + v^2, p = 1 + (v + l h)^2 and q = 1 + (v - l h)^2 the pair's
  // factors are A/p and A/q, their sum A (p + q) / (p q).  The five
  // reciprocals of an axis come from one (the product of the five p q, then
  // unwound), so an axis has one division where the factors one by one have
  // twenty.  The chain's rounding and that of A (p + q) is taken out of each
  // quotient by its remainder (not of lambda4's, which weighs in a null rule
  // only): the sum rounds as two factors one by one do.  Without it a region's
  // error is 1.1 to 1.2 times theirs, 2D to 5D; 8D, 10^6 regions: 54 -> 56 us,
  // one by one 110.  |v|, |h| <= 1e13 keeps that product (of twenty numbers
  // up to 1.5e13), and the centre's prod_j A (ten of 1e26), below 1e265.
  struct Centre {
    double den = 1.0, big = 0.0;
    __device__ void add(const ProductPeak&, int, double c, double h)
    {
      den *= __builtin_fma(c, c, 1.0);
      big = __builtin_fmax(big, __builtin_fmax(__builtin_fabs(c), __builtin_fabs(h)));
    }
    __device__ bool safe(const ProductPeak&) const { return big <= 1e13; }
    __device__ double value(const ProductPeak& f) const { return f.k2 / den; }
  };
  static constexpr int kWidthValues = 0, kTableSize = 0;
  template <class R = Real, if_double<R> = 0>
  __device__ void pair_sums(int, double v, double h, const double*, const double*,
                            double (&s)[5]) const
  {
#pragma clang fp contract(off)
    const double A = __builtin_fma(v, v, 1.0);
    double p[5], q[5], pq[5], left[5];  // the products p q, and the product of those before
    double run = 1.0;
#pragma unroll
    for (int i = 0; i < 5; ++i) {
      const double vp = __builtin_fma(kLambda[i], h, v), vm = __builtin_fma(-kLambda[i], h, v);
      p[i] = __builtin_fma(vp, vp, 1.0);
      q[i] = __builtin_fma(vm, vm, 1.0);
      pq[i] = p[i] * q[i];
      left[i] = run;
      run *= pq[i];
    }
    double r = __builtin_amdgcn_rcp(run);
    r = __builtin_fma(r, __builtin_fma(-run, r, 1.0), r);
#pragma unroll
    for (int i = 4; i >= 0; --i) {
      const double t = p[i] + q[i], num = A * t, ri = r * left[i], y = num * ri;
      const double rem = __builtin_fma(-y, pq[i], num) + __builtin_fma(A, t, -num);
      s[i] = i == 3 ? y : __builtin_fma(rem, ri, y);
      r *= pq[i];
    }
  }
  static constexpr bool multiplicative = true;
  static constexpr bool linear_outer = true;
  __device__ double term(int, double v) const { return 1.0 / (1.0 + v * v); }
  __device__ double outer(double p) const { return static_cast<double>(static_cast<Real>(k2 * p)); }
};

// (1 + sum a_i x_i)^-(d+1), the power by repeated multiplication
template <class Real, int D>
struct CornerPeak {
  Real a[D];
  template <class... X>
  __device__ Real operator()(X... xs) const
  {
    const Real x[D] = {static_cast<Real>(xs)...};
    Real s = 1;
#pragma unroll
    for (int i = 0; i < D; ++i) s += a[i] * x[i];
    return power(s);
  }
  static __device__ Real power(Real s)
  {
    Real p = s;
#pragma unroll
    for (int i = 0; i < D; ++i) p *= s;
    return Real(1) / p;
  }
  // v = a x (origin 0): f = (1 + sum v)^-(d+1), additively separable
  __device__ double origin(int) const { return 0.0; }
  __device__ double axis_scale(int i) const { return static_cast<double>(a[i]); }
  template <class... T>
  __device__ Real centered(T... vs) const
  {
    const Real v[D] = {static_cast<Real>(vs)...};
    Real s = 1;
#pragma unroll
    for (int i = 0; i < D; ++i) s += v[i];
    return power(s);
  }
  __device__ double term(int, double v) const { return v; }
  __device__ double outer(double s) const
  {
    return static_cast<double>(power(static_cast<Real>(1.0 + s)));
  }
  // outer summed over one, two and four points, FP64, by one reciprocal, that
  // of the product of the points' powers; a power takes log2(d) products, so
  // a point costs 8 instructions where a division and d products cost 27.
  // (The power of a reciprocal would multiply the reciprocal's error by d + 1:
  // a region's error 1.3 times that of single points at 2D and 3D, where this
  // has 0.95 and 0.84 of it.)  sum_safe bounds a region's
  // bases away from zero and infinity, so the products of four powers stay in
  // range (every offset of a rule point is below half the width).
  __device__ double base() const { return 1.0; }
  static constexpr double bound()
  {
    double b = 1.0;
    for (int i = 0; i < 240 / (D + 1); ++i) b *= 2.0;  // (b^(D + 1))^4 <= 2^960
    return b;
  }
  template <int N>
  static __device__ double power_of(double b)
  {
    if constexpr (N == 1)
      return b;
    else if constexpr (N % 2)
      return power_of<N - 1>(b) * b;
    else {
      const double t = power_of<N / 2>(b);
      return t * t;
    }
  }
  template <class R = Real, if_double<R> = 0>
  __device__ bool sum_safe(const double (&c)[D], const double (&h)[D]) const
  {
    double s = 1.0, w = 0.0;
#pragma unroll
    for (int j = 0; j < D; ++j) {
      s += c[j];
      w += __builtin_fabs(h[j]);
    }
    w *= .5;
    return s - w >= 1.0 / bound() && s + w <= bound();
  }
  template <class R = Real, if_double<R> = 0>
  __device__ double sum1(double b0) const
  {
    return math::quotient(1.0, power_of<D + 1>(b0));
  }
  template <class R = Real, if_double<R> = 0>
  __device__ double sum2(double b0, double b1) const
  {
#pragma clang fp contract(off)
    const double a = power_of<D + 1>(b0), b = power_of<D + 1>(b1);
    return math::quotient(a + b, a * b);
  }
  template <class R = Real, if_double<R> = 0>
  __device__ double sum4(double b0, double b1, double b2, double b3) const
  {
#pragma clang fp contract(off)
    const double a = power_of<D + 1>(b0), b = power_of<D + 1>(b1);
    const double c = power_of<D + 1>(b2), d = power_of<D + 1>(b3);
    const double ab = a * b, cd = c * d;
    return math::quotient(__builtin_fma(a + b, cd, (c + d) * ab), ab * cd);
  }
};

// exp(-sum a_i^2 (x_i - u_i)^2)
template <class Real, int D>
struct Gaussian {
  Real a[D];   // a_i
  Real a2[D];  // a_i^2
  Real u[D];
  template <class... X>
  __device__ Real operator()(X... xs) const
  {
    const Real x[D] = {static_cast<Real>(xs)...};
    const Real t0 = x[0] - u[0];
    Real s = a2[0] * (t0 * t0);
#pragma unroll
    for (int i = 1; i < D; ++i) {
      const Real t = x[i] - u[i];
      s += a2[i] * (t * t);
    }
    return math::exp_neg(-s);
  }
  // f(u + v / a): the evaluation kernel hands over v = a (x - u), the
  // region's centre and half-widths scaled by a once per region, so a point
  // costs one FMA per axis for v and one for the sum of squares
  __device__ double origin(int i) const { return static_cast<double>(u[i]); }
  __device__ double axis_scale(int i) const { return static_cast<double>(a[i]); }
  template <class... T>
  __device__ Real centered(T... vs) const
  {
    const Real v[D] = {static_cast<Real>(vs)...};
    Real s = v[0] * v[0];
#pragma unroll
    for (int i = 1; i < D; ++i) s = math::fma_(v[i], v[i], s);
    return math::exp_neg(-s);
  }
  // additively separable in v: f = outer(sum_j term(j, v_j)); the terms
  // and their sums in FP64, outer in the integrand's precision
  __device__ double term(int, double v) const { return v * v; }
  __device__ double outer(double s) const
  {
    return static_cast<double>(math::exp_neg(static_cast<Real>(-s)));
  }
  // outer(s + d) = outer(s) e^-d.  The terms are non-negative, so in a
  // region whose centre sums to s0 every factor is at most e^s0 and every
  // point's value at most 1: s0 bounded well inside the FP64 exponent range
  // keeps the centre's value, each factor and every partial product normal
  // (an FP32 integrand takes those FP32 cannot hold in FP64).
  static constexpr bool exponential = true;
  __device__ double factor(double d) const { return math::exp_factor(-d, Real()); }
  __device__ double centre_value(double s0) const { return math::exp_factor(-s0, Real()); }
  __device__ bool factor_safe(double s0) const { return s0 <= kFactorRange<double>; }
  // e^(v^2 - (v - l h)^2) + e^(v^2 - (v + l h)^2) = e^(-(l h)^2) 2 cosh(l y)
  // with y = 2 v h.  The first factor is a function of the width alone.  For
  // the second |y| = n/2 + r, |r| <= 1/4: cosh and sinh of l n/2 from a
  // table, those of l r from short series, so the pair costs 14
  // instructions where its two exponentials cost 38.  |y| > 100 takes the
  // exponentials.
  struct Centre {
    double sum = 0.0;
    __device__ void add(const Gaussian&, int, double c, double) { sum = __builtin_fma(c, c, sum); }
    __device__ bool safe(const Gaussian& f) const { return f.factor_safe(sum); }
    __device__ double value(const Gaussian&) const { return math::exp_bounded(-sum); }
  };
  static constexpr int kWidthValues = 5, kTableSize = kCoshLds * 10;
  __device__ double width_arg(int, double h) const { return h; }
  __device__ void width_values(double h, double (&w)[5]) const
  {
#pragma clang fp contract(off)
    const double X = h * h;
#pragma unroll
    for (int i = 0; i < 5; ++i) w[i] = math::exp_bounded(-(lambda2(i) * X));
  }
  __device__ static void fill_table(double* tab, int tid, int threads)
  {
    for (int e = tid; e < kTableSize / 2; e += threads) {
      const double c = kCoshTable.v[2 * e], s = kCoshTable.v[2 * e + 1];
      tab[2 * e] = c;
      tab[2 * e + 1] = s;
    }
  }
  template <class R = Real, if_double<R> = 0>
  __device__ void pair_sums(int, double v, double h, const double* w, const double* tab,
                            double (&s)[5]) const
  {
#pragma clang fp contract(off)
    const double y = __builtin_fabs((v + v) * h);
    if (y <= .5 * (kCoshSteps - 1)) {
      constexpr double kShift = 0x1.8p+52;
      const double t = __builtin_fma(y, 2.0, kShift);
      const int n = static_cast<int>(__builtin_bit_cast(unsigned long long, t));
      const double r = __builtin_fma(-.5, t - kShift, y), R2 = r * r;
      // the table's first rows are in LDS, all of it in memory
      double row[10];
      if (tab && n < kCoshLds) {
#pragma unroll
        for (int i = 0; i < 10; ++i) row[i] = tab[10 * n + i];
      } else {
#pragma unroll
        for (int i = 0; i < 10; ++i) row[i] = kCoshTable.v[10 * n + i];
      }
      series::for_lambda([&](auto i) {
        constexpr int I = decltype(i)::value;
        constexpr double zmax = lambda2(I) * .0625;
        const double z = lambda2(I) * R2;
        const double ch = series::sum<series::degree(zmax, 2), 2, 0>(z);
        const double sh = series::sum<series::degree(zmax, 2, 1), 2, 1>(z);
        s[I] = w[I] * __builtin_fma(row[2 * I], ch, (row[2 * I + 1] * r) * sh);
      });
    } else {
      const double t = v * v;
#pragma unroll 1
      for (int i = 0; i < 5; ++i) {
        const double l = i == 0 ? kLambda[0] : i == 1 ? kLambda[1] : i == 2 ? kLambda[2] : i == 3 ? kLambda[3] : kLambda[4];
        const double vm = __builtin_fma(-l, h, v), vp = __builtin_fma(l, h, v);
        const double e = math::exp_bounded(__builtin_fma(-vm, vm, t)) +
                         math::exp_bounded(__builtin_fma(-vp, vp, t));
#pragma unroll
        for (int k = 0; k < 5; ++k) s[k] = k == i ? e : s[k];
      }
    }
  }
};

// exp(-sum a_i |x_i - u_i|)
template <class Real, int D>
struct C0 {
  Real a[D];
  Real u[D];
  template <class... X>
  __device__ Real operator()(X... xs) const
  {
    const Real x[D] = {static_cast<Real>(xs)...};
    Real s = 0;
#pragma unroll
    for (int i = 0; i < D; ++i) s += a[i] * math::fabs_(x[i] - u[i]);
    return math::exp_neg(-s);
  }
  // f(u + v / a): the kernel hands over v = a (x - u) (see Gaussian)
  __device__ double origin(int i) const { return static_cast<double>(u[i]); }
  __device__ double axis_scale(int i) const { return static_cast<double>(a[i]); }
  template <class... T>
  __device__ Real centered(T... vs) const
  {
    const Real v[D] = {static_cast<Real>(vs)...};
    Real s = math::fabs_(v[0]);
#pragma unroll
    for (int i = 1; i < D; ++i) s += math::fabs_(v[i]);
    return math::exp_neg(-s);
  }
  __device__ double term(int, double v) const { return __builtin_fabs(v); }
  __device__ double outer(double s) const
  {
    return static_cast<double>(math::exp_neg(static_cast<Real>(-s)));
  }
  // The points v -+ l h of one axis change |v| by -+l|h| while they stay on
  // v's side of the kink: factors e^(l|h|) and e^(-l|h|), functions of the
  // width alone, so a region forms an exponential only for the axes that
  // reach the kink.  There (l|h| > |v|) the near point has e^(2|v| - l|h|) =
  // (e^(-l|h|) e^|v|) e^|v| (|v| <= 650 where the factored form is taken, so
  // e^|v| stays finite and the first product is at most 1).
  struct Centre {
    double sum = 0.0;
    __device__ void add(const C0&, int, double c, double) { sum += __builtin_fabs(c); }
    __device__ bool safe(const C0& f) const { return f.factor_safe(sum); }
    __device__ double value(const C0&) const { return math::exp_bounded(-sum); }
  };
  static constexpr int kWidthValues = 10, kTableSize = 0;
  __device__ double width_arg(int, double h) const { return h; }
  __device__ void width_values(double h, double (&w)[10]) const
  {
#pragma unroll
    for (int i = 0; i < 5; ++i) {
      w[2 * i] = math::exp_bounded(-(kLambda[i] * __builtin_fabs(h)));
      w[2 * i + 1] = math::recip(w[2 * i]);
    }
  }
  template <class R = Real, if_double<R> = 0>
  __device__ void pair_sums(int, double v, double h, const double* w, const double*,
                            double (&s)[5]) const
  {
#pragma clang fp contract(off)
    const double av = __builtin_fabs(v), ah = __builtin_fabs(h);
#pragma unroll
    for (int i = 0; i < 5; ++i) s[i] = w[2 * i] + w[2 * i + 1];
    if (kLambda[0] * ah > av) {  // lambda1 is the largest
      const double aux = math::exp_bounded(av);
#pragma unroll
      for (int i = 0; i < 5; ++i) {
        const double across = w[2 * i] + (w[2 * i] * aux) * aux;
        s[i] = kLambda[i] * ah > av ? across : s[i];
      }
    }
  }
  // outer(s + d) = outer(s) e^-d, non-negative terms (see Gaussian)
  static constexpr bool exponential = true;
  __device__ double factor(double d) const { return math::exp_factor(-d, Real()); }
  __device__ double centre_value(double s0) const { return math::exp_factor(-s0, Real()); }
  __device__ bool factor_safe(double s0) const { return s0 <= kFactorRange<double>; }
};

// 0 if any x_i > u_i, else exp(sum a_i x_i)
template <class Real, int D>
struct Discontinuous {
  Real a[D];
  Real u[D];
  double c;  // sum a_i u_i
  template <class... X>
  __device__ Real operator()(X... xs) const
  {
    const Real x[D] = {static_cast<Real>(xs)...};
    // "some x_i > u_i" as max_i (x_i - u_i) > 0: one compare instead of a
    // chain of lane masks
    Real m = x[0] - u[0];
    Real s = a[0] * x[0];
#pragma unroll
    for (int i = 1; i < D; ++i) {
      m = math::fmax_(m, x[i] - u[i]);
      s += a[i] * x[i];
    }
    const Real v = math::exp_(s);
    return m > Real(0) ? Real(0) : v;
  }
  // t = x - u (origin u, unit scale): f = [all t_i <= 0] exp(c + sum a_i t_i),
  // additively separable with a validity mask per axis
  __device__ double origin(int i) const { return static_cast<double>(u[i]); }
  __device__ double axis_scale(int) const { return 1.0; }
  template <class... T>
  __device__ Real centered(T... ts) const
  {
    const Real t[D] = {static_cast<Real>(ts)...};
    Real m = t[0];
    Real s = a[0] * t[0];
#pragma unroll
    for (int i = 1; i < D; ++i) {
      m = math::fmax_(m, t[i]);
      s = math::fma_(a[i], t[i], s);
    }
    const Real v = math::exp_bounded(static_cast<Real>(c) + s);
    return m > Real(0) ? Real(0) : v;
  }
  static constexpr bool masked = true;
  __device__ bool valid(int, double t) const { return t <= 0.0; }
  __device__ double term(int i, double t) const { return static_cast<double>(a[i]) * t; }
  __device__ double outer(double s) const
  {
    return static_cast<double>(math::exp_bounded(static_cast<Real>(c + s)));
  }
  // outer(s + d) = outer(s) e^d.  The centre's value e^(c + s0) is kept
  // well inside the exponent range; the factors are bounded by e^(a_j h_j)
  // (the kernel sends a region whose sums overflow anyway to the generic
  // loop).
  static constexpr bool exponential = true;
  __device__ double factor(double d) const
  {
    return static_cast<double>(math::exp_bounded(static_cast<Real>(d)));
  }
  // the points t -+ delta change a_j t by -+a_j delta: factors e^(-a_j
  // delta) and its reciprocal
  __device__ void factor_pair(int j, double, double delta, double, double& fm, double& fp) const
  {
    fm = factor(-static_cast<double>(a[j]) * delta);
    fp = math::recip(fm);
  }
  // the same two factors, functions of the width alone, summed over the valid
  // points
  struct Centre {
    double sum = 0.0;
    __device__ void add(const Discontinuous& f, int j, double t, double)
    {
      sum = __builtin_fma(static_cast<double>(f.a[j]), t, sum);
    }
    __device__ bool safe(const Discontinuous& f) const { return f.factor_safe(sum); }
    __device__ double value(const Discontinuous& f) const { return math::exp_bounded(f.c + sum); }
  };
  static constexpr int kWidthValues = 10, kTableSize = 0;
  __device__ double width_arg(int j, double h) const { return static_cast<double>(a[j]) * h; }
  __device__ void width_values(double ah, double (&w)[10]) const
  {
#pragma unroll
    for (int i = 0; i < 5; ++i) {
      w[2 * i] = math::exp_bounded(-(kLambda[i] * ah));
      w[2 * i + 1] = math::recip(w[2 * i]);
    }
  }
  template <class R = Real, if_double<R> = 0>
  __device__ void pair_sums(int j, double t, double h, const double* w, const double*,
                            double (&s)[5]) const
  {
#pragma clang fp contract(off)
#pragma unroll
    for (int i = 0; i < 5; ++i) {
      const bool m = valid(j, __builtin_fma(-kLambda[i], h, t));
      const bool p = valid(j, __builtin_fma(kLambda[i], h, t));
      s[i] = (m ? w[2 * i] : 0.0) + (p ? w[2 * i + 1] : 0.0);
    }
  }
  __device__ bool factor_safe(double s0) const
  {
    return __builtin_fabs(c + s0) <= kFactorRange<Real> - (sizeof(Real) == 8 ? 100.0 : 20.0);
  }
};

}  // namespace pagani

// Semi-analytic Heston European call prices on the device (FP64).
//
// The reference prices its Heston checks with a COS-method pricer
// (FiniteDifference/heston.py:490-693, used at rtol 1e-3 by
// FiniteDifference/tests/test_HestonOptionGPU.py:74-112).  This file prices
// the same call with Lewis's single-integral formula (Lewis 2001):
//
//   C = S - sqrt(S K) e^{-rT/2} / pi * int_0^inf Re[e^{iuk} phi(u - i/2)] / (u^2 + 1/4) du,
//   k = ln(S/K) + rT,
//
// where phi is the characteristic function of ln(S_T/S) - rT in the "little
// trap" form of Albrecher, Mayer, Schoutens and Tistaert (2007), which is
// continuous on the principal branch of the complex logarithm.  At
// u - i/2 the term u^2 + iu of the Riccati solution is the real u^2 + 1/4.
//
// Quadrature: Gauss-Legendre with kN1 nodes on [0, a] and kN2 nodes on the
// tail [a, inf) mapped by u = a / t, t in (0, 1].  The integrand decays like
// exp(-c u) / u^2 with c = sqrt(1 - rho^2) (v0 + kappa theta T) / sigma, and
// a = 20 / c (clamped to [10, 2e4]) puts the bulk of the oscillations on the
// first panel.  One 64-lane wave prices one option: each lane sums
// (kN1 + kN2) / 64 = 9 nodes and the wave reduces with cross-lane shuffles.
// Measured against adaptive quadrature of the same integral to infinity,
// the error over the surrogate's parameter box is below 3e-10.

#include "common.h"

#include <cmath>
#include <mutex>
#include <vector>

namespace {

constexpr int kN1 = 512;
constexpr int kN2 = 64;
constexpr int kRowLen = 9;  // S0, K, r, v0, T, kappa, theta, sigma, rho

__constant__ double c_x1[kN1];
__constant__ double c_w1[kN1];
__constant__ double c_x2[kN2];
__constant__ double c_w2[kN2];

struct cd {
  double re, im;
};

__device__ inline cd cadd(cd a, cd b) { return {a.re + b.re, a.im + b.im}; }
__device__ inline cd csub(cd a, cd b) { return {a.re - b.re, a.im - b.im}; }
__device__ inline cd cmul(cd a, cd b) {
  return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}
__device__ inline cd cscale(cd a, double s) { return {a.re * s, a.im * s}; }
__device__ inline cd cdiv(cd a, cd b) {
  // Smith's algorithm: no overflow from squaring |b|
  if (fabs(b.re) >= fabs(b.im)) {
    const double q = b.im / b.re, den = b.re + b.im * q;
    return {(a.re + a.im * q) / den, (a.im - a.re * q) / den};
  }
  const double q = b.re / b.im, den = b.re * q + b.im;
  return {(a.re * q + a.im) / den, (a.im * q - a.re) / den};
}
__device__ inline cd cexp_(cd a) {
  double s, c;
  sincos(a.im, &s, &c);
  const double m = exp(a.re);
  return {m * c, m * s};
}
__device__ inline cd clog_(cd a) { return {log(hypot(a.re, a.im)), atan2(a.im, a.re)}; }
// principal square root (real part >= 0)
__device__ inline cd csqrt_(cd a) {
  const double m = hypot(a.re, a.im);
  if (m == 0.0) return {0.0, 0.0};
  if (a.re >= 0.0) {
    const double s = sqrt(0.5 * (m + a.re));
    return {s, 0.5 * a.im / s};
  }
  const double t = copysign(sqrt(0.5 * (m - a.re)), a.im);
  return {0.5 * a.im / t, t};
}

// Re[e^{iuk} phi(u - i/2)] / (u^2 + 1/4)
__device__ inline double lewis_integrand(double u, double k, double v0, double T, double kappa,
                                         double theta, double sigma, double rho) {
  const double s2 = sigma * sigma;
  const double q = u * u + 0.25;
  const cd xi = {kappa - 0.5 * sigma * rho, -sigma * rho * u};
  const cd d = csqrt_(cadd(cmul(xi, xi), cd{s2 * q, 0.0}));
  const cd xm = csub(xi, d);
  const cd g = cdiv(xm, cadd(xi, d));
  const cd e = cexp_(cscale(d, -T));
  const cd one = {1.0, 0.0};
  const cd ge = csub(one, cmul(g, e));
  const cd lg = clog_(cdiv(ge, csub(one, g)));
  const cd A = cscale(csub(cscale(xm, T), cscale(lg, 2.0)), kappa * theta / s2);
  const cd B = cscale(cdiv(cmul(xm, csub(one, e)), ge), v0 / s2);
  const cd z = cadd(cadd(A, B), cd{0.0, u * k});
  double s, c;
  sincos(z.im, &s, &c);
  return exp(z.re) * c / q;
}

// ---- elementary functions ------------------------------------------------------
// For finite arguments of ordinary size only, which is what makes them half as
// long as the general ones: reductions by a multiple n of pi/2 or ln 2 taken
// out in two fused steps (exact to 1e-16 absolute while |n| < 2^51), then
// polynomials interpolated at Chebyshev nodes (relative error of each function
// below 3e-17 before rounding).

constexpr double kRound = 6755399441055744.0;  // 1.5 * 2^52: adding it rounds to an integer

template <int N>
__device__ inline double horner(double z, const double (&c)[N]) {
  double p = c[0];
#pragma unroll
  for (int k = 1; k < N; ++k) p = __builtin_fma(p, z, c[k]);
  return p;
}

// x = n pi/2 + r, |r| <= pi/4; n's last bits
__device__ inline double reduce_pi2(double x, int &n) {
  const double t = __builtin_fma(x, 0.6366197723675814, kRound), k = t - kRound;
  n = __double2loint(t);
  return __builtin_fma(-k, 6.123233995736766e-17, __builtin_fma(-k, 1.5707963267948966, x));
}
__device__ inline double sin_part(double r, double z) {
  constexpr double c[] = {1.5918122138279555e-10, -2.5051131745270944e-08, 2.7557316102054947e-06,
                          -0.00019841269836757503, 0.008333333333330948, -0.16666666666666666};
  return __builtin_fma(r * z, horner(z, c), r);
}
__device__ inline double cos_part(double z) {
  constexpr double c[] = {-1.1382626709737559e-11, 2.0876146199889678e-09, -2.755731727144046e-07,
                          2.4801587298765127e-05, -0.0013888888888887398, 0.041666666666666664};
  return __builtin_fma(z * z, horner(z, c), __builtin_fma(-0.5, z, 1.0));
}
__device__ inline double flip(double x, int bit1) {  // -x if bit 1 is set
  return __hiloint2double(__double2hiint(x) ^ ((bit1 & 2) << 30), __double2loint(x));
}
__device__ inline void sincos_(double x, double &s, double &c) {
  int n;
  const double r = reduce_pi2(x, n), z = r * r;
  const double sp = sin_part(r, z), cp = cos_part(z);
  s = flip(n & 1 ? cp : sp, n);
  c = flip(n & 1 ? sp : cp, n + 1);
}
__device__ inline double cos_(double x) {
  int n;
  const double r = reduce_pi2(x, n), z = r * r;
  const double sp = sin_part(r, z), cp = cos_part(z);
  return flip(n & 1 ? sp : cp, n + 1);
}
__device__ inline double exp_(double x) {
  constexpr double c[] = {2.5100397765153145e-08, 2.762008047483383e-07, 2.75572684189161e-06,
                          2.4801521312008337e-05, 0.00019841269863099656, 0.0013888888917204163,
                          0.008333333333330044, 0.04166666666662414, 0.16666666666666669,
                          0.5000000000000001};
  x = fmin(fmax(x, -2000.0), 2000.0);
  const double t = __builtin_fma(x, 1.4426950408889634, kRound), k = t - kRound;
  const double r =
      __builtin_fma(-k, 2.3190468138462996e-17, __builtin_fma(-k, 0.6931471805599453, x));
  return ldexp(1.0 + __builtin_fma(r * r, horner(r, c), r), __double2loint(t));
}

// 1 / x for a normal x of ordinary size, by two Newton steps (zeros, infinities
// and subnormal numbers are not looked after, as the pivots' recip does).
__device__ inline double recip_(double x) {
  double y = __builtin_amdgcn_rcp(x);
  y = __builtin_fma(y, __builtin_fma(-x, y, 1.0), y);
  return __builtin_fma(y, __builtin_fma(-x, y, 1.0), y);
}
__device__ inline double div_(double a, double b) {
  const double rb = recip_(b), q = a * rb;
  return __builtin_fma(__builtin_fma(-q, b, a), rb, q);
}
// log x = e ln 2 + 2 atanh((m - 1) / (m + 1)), x = 2^e m, m in [sqrt 1/2, sqrt 2)
__device__ inline double log_(double x) {
  constexpr double c[] = {0.14617034915312363, 0.1533167432387183, 0.18182890544058972,
                          0.222222111154066, 0.28571428626093204, 0.3999999999989925,
                          0.666666666666667};
  double m = __builtin_amdgcn_frexp_mant(x);
  int e = __builtin_amdgcn_frexp_exp(x);
  const bool low = m < 0.7071067811865476;
  m = low ? m + m : m;
  e = low ? e - 1 : e;
  const double s = div_(m - 1.0, m + 1.0), z = s * s, k = (double)e;
  const double l = __builtin_fma(s * z, horner(z, c), s + s);
  return __builtin_fma(k, 0.6931471805599453, __builtin_fma(k, 2.3190468138462996e-17, l));
}
// The angle of (x, y) != 0, by t = tan of it or of its distance from pi/4.
__device__ inline double atan2_(double y, double x) {
  constexpr double c[] = {-0.019176351702928952, 0.039231230934061674, -0.05085435366790903,
                          0.058581462656476686, -0.06664511156502541, 0.07692183171343514,
                          -0.09090904577342869, 0.11111111015238656, -0.1428571428466634,
                          0.19999999999995519, -0.3333333333333333};
  const double ay = fabs(y), ax = fabs(x), mx = fmax(ax, ay), mn = fmin(ax, ay);
  const bool far = mn > 0.41421356237309503 * mx;
  const double t = div_(far ? mn - mx : mn, far ? mn + mx : mx), z = t * t;
  double a = __builtin_fma(t * z, horner(z, c), t) + (far ? 0.7853981633974483 : 0.0);
  a = ay > ax ? 1.5707963267948966 - a : a;
  a = x < 0.0 ? 3.141592653589793 - a : a;
  return copysign(a, y);
}

// The same for parameters of ordinary size, with an option's constants formed
// once, and rearranged: with N = xp - xm e (xm, xp = xi -+ d),
//   (1 - g e) / (1 - g) = N / (2 d),   xm (1 - e) / (1 - g e) = -s2 q (1 - e) / N,
// so one reciprocal takes the place of three complex divisions, the logarithm
// is that of |N|^2 / (4 |d|^2), and the radicand's real part is a sum of squares
// (|rho| < 1): no branches, no scaling.  Bound by the FP64 units: some
// 310 instructions a node, five of them reciprocals, where the general form
// takes 900; 200,003 options in 1.13 ms instead of 2.30.
struct Lewis {
  double xr, xr2, sr, s2, s2r, c0, T, kts, v0, k;
};

// x > 0 (normal): its square root and the reciprocal of that, by two
// Goldschmidt steps from the hardware estimate and a correction of the root.
__device__ inline void sqrt_rsqrt(double x, double &s, double &rs) {
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  double e = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, e, g);
  h = __builtin_fma(h, e, h);
  e = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, e, g);
  h = __builtin_fma(h, e, h);
  s = __builtin_fma(__builtin_fma(-g, g, x), h, g);
  rs = h + h;
}

__device__ inline double lewis_integrand(double u, const Lewis &o) {
  const double q = u * u + 0.25, xi = o.sr * u;
  const double re = (o.s2r * u) * u + o.c0, im = o.xr2 * xi;
  double m, rm, dr, rdr;  // m = |d|^2
  sqrt_rsqrt(re * re + im * im, m, rm);
  sqrt_rsqrt(0.5 * (m + re), dr, rdr);
  const double di = 0.5 * im * rdr;
  // of xi +- d the one without cancellation (Re d > 0, and Im d has the sign of
  // xr times Im xi), and the other from their product -s2 q
  const double br = o.xr + (o.xr >= 0.0 ? dr : -dr), bi = xi + (o.xr >= 0.0 ? di : -di);
  const double p = -(o.s2 * q) * recip_(br * br + bi * bi), sr = p * br, si = -(p * bi);
  const double xpr = o.xr >= 0.0 ? br : sr, xpi = o.xr >= 0.0 ? bi : si;
  const double xmr = o.xr >= 0.0 ? sr : br, xmi = o.xr >= 0.0 ? si : bi;
  double s, c;
  sincos_(di * o.T, s, c);
  const double E = exp_(-(dr * o.T)), er = E * c, ei = -(E * s);
  const double Nr = xpr - (xmr * er - xmi * ei), Ni = xpi - (xmr * ei + xmi * er);
  const double nn = Nr * Nr + Ni * Ni;
  const double lr = log_(0.25 * (nn * rm));  // twice the logarithm's real part
  const double li = atan2_(Ni * dr - Nr * di, Nr * dr + Ni * di);
  const double rq = recip_(nn * q);  // 1 / nn = q rq, 1 / q = nn rq
  const double a1 = 1.0 - er, f = -(q * o.v0) * (q * rq);
  const double zr = o.kts * (xmr * o.T - lr) + f * (a1 * Nr - ei * Ni);
  const double zi = o.kts * (xmi * o.T - 2.0 * li) - f * (a1 * Ni + ei * Nr) + u * o.k;
  return exp_(zr) * cos_(zi) * (nn * rq);
}

__global__ __launch_bounds__(256, 3) void heston_cf_kernel(const double *__restrict__ rows,
                                                        int64_t n, double *__restrict__ out) {
  const int lane = threadIdx.x & 63;
  const int64_t opt = (int64_t)blockIdx.x * (blockDim.x / 64) + (threadIdx.x >> 6);
  if (opt >= n) return;  // uniform across the wave
  const double *p = rows + opt * kRowLen;
  const double S = p[0], K = p[1], r = p[2], v0 = p[3], T = p[4];
  const double kappa = p[5], theta = p[6], sigma = p[7], rho = p[8];
  if (!(S > 0.0 && K > 0.0 && T > 0.0 && sigma > 0.0 && v0 >= 0.0 && theta >= 0.0 &&
        fabs(rho) < 1.0)) {
    if (lane == 0) out[opt] = __builtin_nan("");
    return;
  }
  const double c = sqrt(1.0 - rho * rho) * (v0 + kappa * theta * T) / sigma;
  const double a = fmin(fmax(c > 0.0 ? 20.0 / c : 2e4, 10.0), 2e4);
  const double k = log(S / K) + r * T;
  Lewis o;
  o.xr = kappa - 0.5 * sigma * rho;
  o.xr2 = 2.0 * o.xr;
  o.sr = -sigma * rho;
  o.s2 = sigma * sigma;
  o.s2r = o.s2 * ((1.0 - rho) * (1.0 + rho));
  o.c0 = o.xr * o.xr + 0.25 * o.s2;
  o.T = T;
  o.kts = kappa * theta / o.s2;
  o.v0 = v0;
  o.k = k;
  // Nodes reach u = 2878 a.  Ordinary: every square stays far inside the
  // exponent range, the phases below 1e14, and sigma is not so small that
  // kappa theta / sigma^2 magnifies the roundings of the logarithm.
  const double um = 3e3 * a;
  const bool ordinary = sigma >= 1e-3 && sigma < 1e6 && fabs(o.xr) < 1e6 && T < 1e6 &&
                        (sigma * T * (1.0 + fabs(o.kts)) + v0 / sigma + fabs(k)) * um < 1e14;
  double sum = 0.0;
  auto integrate = [&](auto f) {
#pragma unroll 1
    for (int j = lane; j < kN1 + kN2; j += 64) {
      double u, w;
      if (j < kN1) {
        u = 0.5 * a * (c_x1[j] + 1.0);
        w = 0.5 * a * c_w1[j];
      } else {
        const double t = 0.5 * (c_x2[j - kN1] + 1.0);
        u = a / t;
        w = 0.5 * c_w2[j - kN1] * a / (t * t);
      }
      sum += w * f(u);
    }
  };
  if (ordinary)
    integrate([&](double u) { return lewis_integrand(u, o); });
  else
    integrate([&](double u) { return lewis_integrand(u, k, v0, T, kappa, theta, sigma, rho); });
  for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
  if (lane == 0) out[opt] = S - sqrt(S * K) * exp(-0.5 * r * T) / M_PI * sum;
}

// Gauss-Legendre nodes and weights on (-1, 1) by Newton iteration on P_n.
void gauss_legendre(int n, double *x, double *w) {
  for (int i = 0; i < (n + 1) / 2; ++i) {
    double z = cos(M_PI * (i + 0.75) / (n + 0.5)), dp = 0.0;
    for (int it = 0; it < 100; ++it) {
      double p0 = 1.0, p1 = z;
      for (int m = 2; m <= n; ++m) {
        const double p2 = ((2.0 * m - 1.0) * z * p1 - (m - 1.0) * p0) / m;
        p0 = p1;
        p1 = p2;
      }
      const double pn = n == 1 ? z : p1, pm = n == 1 ? 1.0 : p0;
      dp = n * (z * pn - pm) / (z * z - 1.0);
      const double dz = pn / dp;
      z -= dz;
      if (fabs(dz) < 1e-16) break;
    }
    double p0 = 1.0, p1 = z;
    for (int m = 2; m <= n; ++m) {
      const double p2 = ((2.0 * m - 1.0) * z * p1 - (m - 1.0) * p0) / m;
      p0 = p1;
      p1 = p2;
    }
    dp = n == 1 ? 1.0 : n * (z * p1 - p0) / (z * z - 1.0);
    const double wi = 2.0 / ((1.0 - z * z) * dp * dp);
    x[i] = -z;
    x[n - 1 - i] = z;
    w[i] = wi;
    w[n - 1 - i] = wi;
  }
}

std::mutex g_cf_mutex;
std::vector<bool> g_cf_ready;  // per device: node tables copied

int ensure_nodes() {
  int dev = 0;
  FDADI_TRY_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(g_cf_mutex);
  if ((int)g_cf_ready.size() <= dev) g_cf_ready.resize(dev + 1, false);
  if (g_cf_ready[dev]) return FDADI_OK;
  std::vector<double> x1(kN1), w1(kN1), x2(kN2), w2(kN2);
  gauss_legendre(kN1, x1.data(), w1.data());
  gauss_legendre(kN2, x2.data(), w2.data());
  FDADI_TRY_HIP(hipMemcpyToSymbol(HIP_SYMBOL(c_x1), x1.data(), sizeof(double) * kN1));
  FDADI_TRY_HIP(hipMemcpyToSymbol(HIP_SYMBOL(c_w1), w1.data(), sizeof(double) * kN1));
  FDADI_TRY_HIP(hipMemcpyToSymbol(HIP_SYMBOL(c_x2), x2.data(), sizeof(double) * kN2));
  FDADI_TRY_HIP(hipMemcpyToSymbol(HIP_SYMBOL(c_w2), w2.data(), sizeof(double) * kN2));
  g_cf_ready[dev] = true;
  return FDADI_OK;
}

}  // namespace

extern "C" {

int fdadi_gauss_legendre(int32_t n, double *x, double *w) {
  FDADI_REQUIRE(n >= 1 && n <= 4096, FDADI_ERR_ARG, "fdadi_gauss_legendre: n must be 1..4096");
  FDADI_REQUIRE(x && w, FDADI_ERR_ARG, "fdadi_gauss_legendre: null output");
  gauss_legendre(n, x, w);
  return FDADI_OK;
}

int fdadi_heston_cf_call(const double *d_rows, int64_t n, double *d_out, void *stream) {
  FDADI_REQUIRE(n >= 0, FDADI_ERR_ARG, "fdadi_heston_cf_call: negative count");
  if (n == 0) return FDADI_OK;
  FDADI_REQUIRE(d_rows && d_out, FDADI_ERR_ARG, "fdadi_heston_cf_call: null buffer");
  const int st = ensure_nodes();
  if (st != FDADI_OK) return st;
  constexpr int kBlock = 256;  // four options per work-group
  const int64_t groups = (n + 3) / 4;
  FDADI_REQUIRE(groups <= 0x7fffffff, FDADI_ERR_ARG, "fdadi_heston_cf_call: too many options");
  hipLaunchKernelGGL(heston_cf_kernel, dim3((unsigned)groups), dim3(kBlock), 0,
                     fdadi::as_stream(stream), d_rows, n, d_out);
  FDADI_CHECK_LAUNCH();
  return FDADI_OK;
}

}  // extern "C"

// device_common.hpp -- types and window arithmetic shared by the gfx950 kernels.
//
// Window and index rule follow the reference exactly:
//   phi(t) = (pi b)^-1/2 exp(-t^2 / b)                 src/cunfft_kernel.cu:162-166
//   u      = rint(n x) - signbit(x) - m  (half-even)   src/cunfft_kernel.cu:175-182
//   taps   l = u .. u + 2m + 1, wrapped mod n           src/cunfft_kernel.cu:528-531
// The split of n*x into integer cell and fraction is always done in FP64.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace cunfft {

template <typename T> struct cplx;
template <> struct cplx<float> { using type = float2; };
template <> struct cplx<double> { using type = double2; };
template <typename T> using cplx_t = typename cplx<T>::type;

// Windows: the reference's Gaussian, and NFFT3's Kaiser-Bessel and sinc power.
enum Window : int { WIN_GAUSSIAN = 0, WIN_KAISER_BESSEL = 1, WIN_SINC = 2 };

// Per-transform geometry passed by value to every gridding kernel.
struct Geom {
    int d;
    int m;
    int W;                // 2m + 2 taps per axis
    int win;              // Window
    int64_t N[3];
    int64_t n[3];
    int64_t M;
    double invb[3];       // Gaussian: 1 / b_t
    double nrm[3];        // Gaussian: (pi b_t)^-1/2
    double shp[3];        // Kaiser-Bessel: b_t = pi (2 - 1 / sigma_t); sinc: a_t (sinc_phi)
};

__host__ __device__ __forceinline__ int sign_bit(double x) { return __builtin_signbit(x) ? 1 : 0; }

// Index wrap onto [0, n) for any grid length n (the reference masks with
// n - 1, src/cunfft_kernel.cu:528-531, which needs a power of two).
// wrap_hi: a in [0, 2n) (a wrapped window start plus a tap offset < n).
__device__ __forceinline__ int64_t wrap_hi(int64_t a, int64_t n) { return a >= n ? a - n : a; }
__host__ __device__ __forceinline__ uint32_t wrap_hi32(uint32_t a, uint32_t n) { return a >= n ? a - n : a; }

// Floor modulo a mod n in [0, n) for any a; the division runs only outside
// [-n, n), i.e. for nodes outside [-1/2, 1/2).
__host__ __device__ __forceinline__ int64_t wrap_mod(int64_t a, int64_t n)
{
    if (a < -n || a >= n) a %= n;
    return a < 0 ? a + n : a;
}

// First window cell u mod n in [0, n) and the FP64 fraction c = n x - u for
// any node x.  For x in [-1/2, 1/2) this is the reference's rule exactly; for
// other finite x it is the reference's too, whose mask with n - 1
// (src/cunfft_kernel.cu:528-531) is u mod n for a power-of-two n.  A
// non-finite or huge n x (|rint(n x)| >= 2^52, where n x has no fraction
// left) is given the cell of x = 0 and keeps its non-finite fraction: its
// taps are NaN or zero, never an index outside the grid.  rint rounds half to
// even like the reference's llrint.
__host__ __device__ __forceinline__ int64_t window_cell(double x, int64_t n, int m, double &c)
{
    const double nx = (double)n * x;
    double r = rint(nx);
    r = fabs(r) < 0x1p52 ? r : 0.0;   // false for NaN as well
    const int64_t u = (int64_t)r - sign_bit(x) - m;
    c = nx - (double)u;
    return wrap_mod(u, n);
}

template <typename T> __device__ __forceinline__ T win_exp(T v);
template <> __device__ __forceinline__ float win_exp<float>(float v) { return expf(v); }
template <> __device__ __forceinline__ double win_exp<double>(double v) { return exp(v); }

// Kaiser-Bessel window in grid units (NFFT3's; the reference is
// Gaussian-only), shape b, support m, analytic continuation past |s| = m:
//   phi(s) = sinh(b r) / (pi r), r = sqrt(m^2 - s^2)        |s| < m
//          = sin(b r) / (pi r),  r = sqrt(s^2 - m^2)        |s| > m
// (b / pi at |s| = m).  With q = b^2 (m^2 - s^2) both are (b / pi) S(q),
//   S(q) = sum_j q^j / (2j+1)! = sinh(z) / z or sin(z) / z,  z = sqrt|q|,
// and phi' = -(b^3 s / pi) R(q), R(q) = 2 S'(q) = sum_j 2(j+1) q^j / (2j+3)!
//          = (cosh z - sinh(z) / z) / q  or  (cos z - sin(z) / z) / q.
// The weights of a node batch are one evaluation per lane on the way to every
// gridding loop, and the library's sinh and sin are long.  Here: Taylor sums up to
// z = 1, above it one exponential for both hyperbolic functions, and sin and cos from
// one reduction by multiples of pi (a node's taps have |s| <= m + 3/2, so z is at most
// 2 pi sqrt(3m + 9/4) there: 33 for m <= 8, 45 for m = 16).
// Nodes set, forward and adjoint of 50021 2D nodes, m = 3, FP32: 171 -> 146 us.
// A larger z comes only from a node without a position (window_cell): weight
// zero, or NaN for a non-finite one.
constexpr int kKbZMax = 256;

// sum_j q^j / (2j+1)! for |q| <= 1, to the last place (Horner, K terms).
template <typename T> __device__ __forceinline__ T kb_series(T q)
{
    constexpr int K = sizeof(T) == 4 ? 6 : 9;
    T p = (T)1;
#pragma unroll
    for (int k = K; k >= 1; --k) p = (T)1 + q * p * (T)(1.0 / (2 * k * (2 * k + 1)));
    return p;
}

// sinh(z) / z for 1 < z <= b m (b < 2 pi, m <= 16: below 101).  FP32: the hardware
// exp2 of the rounded z log2(e), times what the rounding left.
//  * exp(z) leaves the FP32 range at z = 88.7, sinh(z) at 89.4 (m = 15 and 16 at an
//    oversampling of 4.5 and more get there), so e is exp(z) / 2: hi - 1 is exact for
//    hi >= 1.44 (and must not be contracted with the product, of which lo is the rest).
//  * log2(e) is rounded down for hi, so lo is positive and what is past the range is
//    infinite, not NaN.
__device__ __forceinline__ float kb_sinhc(float z)
{
#pragma clang fp contract(off)
    const float hi = z * 1.44269490f;
    const float lo = fmaf(z, 1.92596299e-8f, fmaf(z, 1.44269504f, -hi));   // log2(e) in two parts
    const float x = __builtin_amdgcn_exp2f(hi - 1.f);
    const float e = fmaf(x, lo * 0.693147181f, x);
    return (e - 0.25f / e) / z;
}
__device__ __forceinline__ double kb_sinhc(double z)
{
    const double e = exp(z);
    return 0.5 * (e - 1.0 / e) / z;
}

__device__ __forceinline__ float kb_reduce(float z, float k)   // z - k pi, pi in two parts
{
    return fmaf(-k, -8.74227766e-8f, fmaf(-k, 3.14159274f, z));
}
__device__ __forceinline__ double kb_reduce(double z, double k)
{
    return fma(-k, 1.2246467991473532e-16, fma(-k, 3.141592653589793116, z));
}

// sin z and cos z for 0 <= z <= kKbZMax: z = k pi + r, Taylor sums on |r| <= pi/2.
template <typename T> __device__ __forceinline__ void kb_sincos(T z, T &s, T &c)
{
    constexpr int K = sizeof(T) == 4 ? 6 : 10;
    const T k = rint(z * (T)0.318309886183790671538);
    const T r = kb_reduce(z, k), r2 = -r * r;
    T ps = (T)1, pc = (T)1;
#pragma unroll
    for (int j = K; j >= 1; --j) ps = (T)1 + r2 * ps * (T)(1.0 / (2 * j * (2 * j + 1)));
#pragma unroll
    for (int j = K + 1; j >= 1; --j) pc = (T)1 + r2 * pc * (T)(1.0 / ((2 * j - 1) * (2 * j)));
    const bool odd = ((int)k & 1) != 0;
    s = odd ? -(r * ps) : r * ps;
    c = odd ? -pc : pc;
}

template <typename T> __device__ __forceinline__ T kb_phi(T s, T m, T b)
{
    const T d = m * m - s * s;
    const T z = b * sqrt(fabs(d));
    T v;
    if (z <= (T)1) {
        v = kb_series<T>(d > (T)0 ? z * z : -z * z);
    } else if (!(z <= (T)kKbZMax)) {
        v = z * (T)0;
    } else if (d > (T)0) {
        v = kb_sinhc(z);
    } else {
        T c;
        kb_sincos<T>(z, v, c);
        v /= z;
    }
    return b * (T)0.318309886183790671538 * v;
}

// phi for the FP32 node gradients: those are handed out as float64 values
// (autograd.py), so their bits are kept, and with them the weights' evaluation.
__device__ __forceinline__ float kb_phi_grad(float s, float m, float b)
{
    const float inv_pi = 0.318309886183790671538f;
    const float d = m * m - s * s;
    const float r = sqrtf(fabsf(d));
    if (r == 0.f) return b * inv_pi;
    return inv_pi * (d > 0.f ? sinhf(b * r) : sinf(b * r)) / r;
}
__device__ __forceinline__ double kb_phi_grad(double s, double m, double b) { return kb_phi<double>(s, m, b); }

// d phi / d s: FP32 as it was (see kb_phi_grad), with the series in d near |s| = m.
template <typename T> __device__ __forceinline__ T kb_dphi(T s, T m, T b);
template <> __device__ __forceinline__ float kb_dphi<float>(float s, float m, float b)
{
    const float inv_pi = 0.318309886183790671538f;
    const float d = m * m - s * s;
    if (fabsf(d) < 1e-2f) {
        const float b2 = b * b;
        const float g = b * b2 * (1.f / 6.f + b2 * d * (2.f / 120.f + b2 * d * (3.f / 5040.f + b2 * d * 4.f / 362880.f)));
        return -2.f * s * g * inv_pi;
    }
    const float r = sqrtf(fabsf(d));
    const float br = b * r;
    if (d > 0.f) return -s * (br * coshf(br) - sinhf(br)) * inv_pi / (r * r * r);
    return s * (br * cosf(br) - sinf(br)) * inv_pi / (r * r * r);
}
template <> __device__ __forceinline__ double kb_dphi<double>(double s, double m, double b)
{
    using T = double;
    const T d = m * m - s * s;
    const T z = b * sqrt(fabs(d));
    T v;
    if (z <= (T)1) {
        // 1/3 + q/30 + ...: the ratio of term k to term k - 1 is q (k+1) / (k (2k+2)(2k+3))
        constexpr int K = 9;
        const T q = d > (T)0 ? z * z : -z * z;
        T p = (T)1;
#pragma unroll
        for (int k = K; k >= 1; --k) p = (T)1 + q * p * (T)((k + 1.0) / (k * (2.0 * k + 2.0) * (2.0 * k + 3.0)));
        v = p * (T)(1.0 / 3.0);
    } else if (!(z <= (T)kKbZMax)) {
        v = z * (T)0;
    } else if (d > (T)0) {
        const T e = exp(z), i = (T)1 / e;
        v = ((T)0.5 * (e + i) - (T)0.5 * (e - i) / z) / (z * z);
    } else {
        T sn, cs;
        kb_sincos<T>(z, sn, cs);
        v = -(cs - sn / z) / (z * z);
    }
    return -s * (b * b * b * (T)0.318309886183790671538) * v;
}

// Sinc-power window in grid units (NFFT3's SINC_POWER; the reference is
// Gaussian-only):
//   phi(s) = a sinc(pi a s)^(2m),   sinc(u) = sin(u) / u,   a = (2 sigma - 1) / (2 sigma m),
// whose Fourier transform is the centred cardinal B-spline M_2m(nu / a) of
// order 2m, zero for |nu| >= m a = 1 - 1/(2 sigma): the oversampled grid's
// first alias of the band edge.  The roll-off divides by M_2m(k / (n a)).
template <typename T> __device__ __forceinline__ T sin_pi(T v);
template <> __device__ __forceinline__ float sin_pi<float>(float v) { return sinpif(v); }
template <> __device__ __forceinline__ double sin_pi<double>(double v) { return sinpi(v); }
template <typename T> __device__ __forceinline__ T cos_pi(T v);
template <> __device__ __forceinline__ float cos_pi<float>(float v) { return cospif(v); }
template <> __device__ __forceinline__ double cos_pi<double>(double v) { return cospi(v); }

// v^k for k >= 0 by squaring.
template <typename T> __device__ __forceinline__ T ipow(T v, int k)
{
    T r = (T)1;
    for (; k > 0; k >>= 1) {
        if (k & 1) r *= v;
        v *= v;
    }
    return r;
}

template <typename T> __device__ __forceinline__ T sinc_pi(T t)   // sin(pi t) / (pi t)
{
    return t == (T)0 ? (T)1 : sin_pi<T>(t) / ((T)3.14159265358979323846 * t);
}

template <typename T> __device__ __forceinline__ T sinc_phi(T s, int m, T a)
{
    return a * ipow<T>(sinc_pi<T>(a * s), 2 * m);
}

// d phi / d s = a 2m sinc^(2m-1)(u) pi a g(u), u = pi a s, g(u) = d sinc / du
// = (u cos u - sin u) / u^2, by its series -u/3 + u^3/30 - u^5/840 + u^7/45360
// for |u| < 0.1 (the closed form cancels there).
template <typename T> __device__ __forceinline__ T sinc_dphi(T s, int m, T a)
{
    const T pi = (T)3.14159265358979323846;
    const T t = a * s, u = pi * t;
    T g;
    if (fabs(u) < (T)0.1) {
        const T u2 = u * u;
        g = u * ((T)(-1.0 / 3.0) + u2 * ((T)(1.0 / 30.0) + u2 * ((T)(-1.0 / 840.0) + u2 * (T)(1.0 / 45360.0))));
    } else {
        g = (u * cos_pi<T>(t) - sin_pi<T>(t)) / (u * u);
    }
    return a * (T)(2 * m) * ipow<T>(sinc_pi<T>(t), 2 * m - 1) * pi * a * g;
}

// Window weight of tap offset s along axis t.
template <typename T> __device__ __forceinline__ T window_weight(T s, const Geom &ge, int t)
{
    if (ge.win == WIN_KAISER_BESSEL) return kb_phi<T>(s, (T)ge.m, (T)ge.shp[t]);
    if (ge.win == WIN_SINC) return sinc_phi<T>(s, ge.m, (T)ge.shp[t]);
    return win_exp<T>(-s * s * (T)ge.invb[t]) * (T)ge.nrm[t];
}

// d/dx phi(n x - l) = n phi'(s).
template <typename T>
__device__ __forceinline__ T window_weight_dx(T s, T p, const Geom &ge, int t)
{
    if (ge.win == WIN_KAISER_BESSEL) return (T)ge.n[t] * kb_dphi<T>(s, (T)ge.m, (T)ge.shp[t]);
    if (ge.win == WIN_SINC) return (T)ge.n[t] * sinc_dphi<T>(s, ge.m, (T)ge.shp[t]);
    return (T)ge.n[t] * ((T)-2.0 * s * (T)ge.invb[t]) * p;
}

// w[l] = phi(c - l) for l = 0..W-1 along axis t in precision T; the offset
// c - l is formed in FP64 and rounded once.
template <typename T, int W>
__device__ __forceinline__ void window_weights(double c, const Geom &ge, int t, T (&w)[W])
{
#pragma unroll
    for (int l = 0; l < W; ++l) w[l] = window_weight<T>((T)(c - (double)l), ge, t);
}

// Weights and their x-derivatives.
template <typename T, int W>
__device__ __forceinline__ void window_weights_dx(double c, const Geom &ge, int t, T (&w)[W],
                                                  T (&dw)[W])
{
#pragma unroll
    for (int l = 0; l < W; ++l) {
        const T s = (T)(c - (double)l);
        w[l] = ge.win == WIN_KAISER_BESSEL ? kb_phi_grad(s, (T)ge.m, (T)ge.shp[t]) : window_weight<T>(s, ge, t);
        dw[l] = window_weight_dx<T>(s, w[l], ge, t);
    }
}

template <typename T> __device__ __forceinline__ cplx_t<T> cmake(T a, T b)
{
    cplx_t<T> r;
    r.x = a;
    r.y = b;
    return r;
}

}  // namespace cunfft

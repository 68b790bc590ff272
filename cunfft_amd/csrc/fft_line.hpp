// fft_line.hpp -- register-resident FFT passes for gfx950 (fft_line_f32.hip and
// fft_line_f64.hip instantiate them; fft.hip holds the pass set-up and the
// generic pass for the line lengths not listed here).
//
// One pass transforms all lines of one axis.  The line length is a template
// argument: TPL = L / EPT threads share a line, thread t holding the elements
// t + TPL q (q < EPT) in registers.  Every Stockham stage reads its butterflies
// in exactly this order (input r of butterfly j sits at j + r L / R, and a
// thread's butterflies are j = t + TPL b), and so does the last stage write its
// results.  So the global loads go straight to registers, the results straight
// from registers to global memory, and LDS holds the data only between stages:
// a 256-point line takes one exchange (16 x 16) and one barrier.
//
// What bounds it: on small grids (a 2D transform of 512^2 .. 1024^2) the chain
// load -> stages -> store of one workgroup, on large ones HBM and the memory-side
// cache.  Mean time per pass, before (an LDS-resident pass: line positions by
// 64-bit divisions, the twiddle table staged in LDS, two exchanges more) -> now:
//   2D 1024^2 FP32, 512 of 1024 points kept   15.6 -> 9.0 us
//   2D 512^2 FP64                             12.2 -> 7.6 us
//   3D 256^3 FP32                             40 -> 27 us (4.2 TB/s; a copy: 4.7)
//   3D 256^3 FP64                             62 -> 47 us
//   1D 2^23 FP64, first / second half         288 / 179 -> 80 / 82 us: one column of
//     4096 points per workgroup (16-byte accesses) became two, and the second half
//     now writes its lines side by side instead of with a stride
//   1D 2048 FP64, one line                    12.1 -> 8.0 us
//
// Both transform directions run the forward kernel: DFT+ (x) = swap(DFT-
// (swap(x))) with swap exchanging real and imaginary part, applied where the
// elements are loaded and stored.
//
// Lines of 4 and 8 points, one thread each, are here for the same reason (forward /
// adjoint of a 8 x 64 x 512 grid FP64, generic pass for the first axis -> now:
// 48 / 70 -> 33 / 56 us; 8 x 256 x 256 58 / 87 -> 28 / 58).
#pragma once
#include "internal.hpp"

namespace cunfft {

// Radices of a line (product L) and elements per thread (a multiple of each).
template <int L> struct LinePlan {
    static constexpr int EPT = 0, NS = 0;
    static constexpr int R[4] = {1, 1, 1, 1};
};
#define CUNFFT_LINE(LEN, E, N, A, B, C_, D)                    \
    template <> struct LinePlan<LEN> {                         \
        static constexpr int EPT = E, NS = N;                  \
        static constexpr int R[4] = {A, B, C_, D};             \
    };
CUNFFT_LINE(4, 4, 1, 4, 1, 1, 1)
CUNFFT_LINE(8, 8, 1, 8, 1, 1, 1)
CUNFFT_LINE(16, 16, 1, 16, 1, 1, 1)
CUNFFT_LINE(32, 16, 2, 16, 2, 1, 1)
CUNFFT_LINE(64, 16, 2, 16, 4, 1, 1)
CUNFFT_LINE(128, 16, 2, 16, 8, 1, 1)
CUNFFT_LINE(256, 16, 2, 16, 16, 1, 1)
CUNFFT_LINE(512, 16, 3, 16, 16, 2, 1)
CUNFFT_LINE(1024, 16, 3, 16, 16, 4, 1)
CUNFFT_LINE(2048, 16, 3, 16, 16, 8, 1)
CUNFFT_LINE(4096, 16, 3, 16, 16, 16, 1)
CUNFFT_LINE(48, 24, 2, 8, 6, 1, 1)
CUNFFT_LINE(72, 24, 2, 12, 6, 1, 1)
CUNFFT_LINE(96, 24, 2, 12, 8, 1, 1)
CUNFFT_LINE(144, 24, 2, 12, 12, 1, 1)
CUNFFT_LINE(192, 24, 3, 12, 8, 2, 1)
CUNFFT_LINE(288, 24, 3, 12, 12, 2, 1)
CUNFFT_LINE(384, 24, 3, 8, 8, 6, 1)
CUNFFT_LINE(576, 24, 3, 12, 12, 4, 1)
CUNFFT_LINE(768, 24, 3, 12, 8, 8, 1)
CUNFFT_LINE(1152, 24, 3, 12, 12, 8, 1)
CUNFFT_LINE(1536, 24, 4, 8, 8, 8, 3)
#undef CUNFFT_LINE

#define CUNFFT_POW2_LINES(X) \
    X(4) X(8) X(16) X(32) X(64) X(128) X(256) X(512) X(1024) X(2048) X(4096)
#define CUNFFT_MIXED_LINES(X) \
    X(48) X(72) X(96) X(144) X(192) X(288) X(384) X(576) X(768) X(1152) X(1536)

// Lengths a split axis's two passes run here (other factors: the generic pass).
#define CUNFFT_SPLIT_LINES(X) \
    X(64) X(128) X(256) X(512) X(1024) X(2048) X(4096) X(96) X(192) X(384) X(768) X(1536)

template <int L> constexpr int line_threads_max() { return L >= 1024 ? 512 : 256; }
// wavefronts per SIMD the registers are budgeted for (24 FP32 elements and their
// FP64 roll-off factors spill at 4)
template <typename T, int EPT> constexpr int line_waves() { return sizeof(T) == 8 ? 2 : (EPT > 16 ? 3 : 4); }
// LDS elements of a line: one more every R[0] elements (the first stage writes
// with stride R[0]) and one per line.
template <int L> constexpr int line_pitch() { return L + L / LinePlan<L>::R[0] + 1; }

// ------------------------------------------------ forward DFTs in registers --
template <typename T> __device__ __forceinline__ cplx_t<T> cadd(cplx_t<T> a, cplx_t<T> b)
{
    return cmake<T>(a.x + b.x, a.y + b.y);
}
template <typename T> __device__ __forceinline__ cplx_t<T> csub(cplx_t<T> a, cplx_t<T> b)
{
    return cmake<T>(a.x - b.x, a.y - b.y);
}
__device__ __forceinline__ float fmadd(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fmadd(double a, double b, double c) { return __builtin_fma(a, b, c); }
// Products with their roundings written out, one product of each sum rounded and
// one fused, so the bits do not depend on what the compiler would contract.  Which
// one is fused (and the order in which a radix 8 is taken, below) keeps the bits
// of the LDS-resident pass that ran the power-of-two lines before: an FP32 node
// gradient, which the autograd wrapper hands out as float64, is the same number
// to the last of its 32 bits.
template <typename T> __device__ __forceinline__ cplx_t<T> cmulf(cplx_t<T> a, cplx_t<T> b)
{
    return cmake<T>(fmadd(a.x, b.x, -(a.y * b.y)), fmadd(a.y, b.x, a.x * b.y));
}
// z (c - i s) with c = cos, s = sin of the angle
template <typename T> __device__ __forceinline__ cplx_t<T> crot(cplx_t<T> z, T c, T s)
{
    return cmake<T>(fmadd(z.x, c, z.y * s), fmadd(z.y, c, -(z.x * s)));
}

template <typename T> __device__ __forceinline__ cplx_t<T> crot_x(cplx_t<T> z, T c, T s)
{
    return cmake<T>(fmadd(z.x, c, z.y * s), fmadd(z.x, -s, z.y * c));
}

template <typename T, int R> struct Dft;
template <typename T> struct Dft<T, 2> {
    __device__ __forceinline__ static void run(cplx_t<T> (&v)[2])
    {
        const cplx_t<T> a = v[0], b = v[1];
        v[0] = cadd<T>(a, b);
        v[1] = csub<T>(a, b);
    }
};
template <typename T> struct Dft<T, 3> {
    __device__ __forceinline__ static void run(cplx_t<T> (&v)[3])
    {
        const T h = (T)0.86602540378443864676;   // sqrt(3) / 2
        const cplx_t<T> a = v[0], s = cadd<T>(v[1], v[2]), d = csub<T>(v[1], v[2]);
        const T mx = a.x - (T)0.5 * s.x, my = a.y - (T)0.5 * s.y;
        v[0] = cadd<T>(a, s);
        v[1] = cmake<T>(mx + h * d.y, my - h * d.x);
        v[2] = cmake<T>(mx - h * d.y, my + h * d.x);
    }
};
template <typename T> struct Dft<T, 4> {
    __device__ __forceinline__ static void run(cplx_t<T> (&v)[4])
    {
        const cplx_t<T> a0 = cadd<T>(v[0], v[2]), a1 = csub<T>(v[0], v[2]);
        const cplx_t<T> a2 = cadd<T>(v[1], v[3]), a3 = csub<T>(v[1], v[3]);
        v[0] = cadd<T>(a0, a2);
        v[2] = csub<T>(a0, a2);
        v[1] = cmake<T>(a1.x + a3.y, a1.y - a3.x);
        v[3] = cmake<T>(a1.x - a3.y, a1.y + a3.x);
    }
};
// N = A B: with n = B n1 + n2 and k = k1 + A k2, B DFTs of A points, the
// twiddles exp(-2 pi i n2 k1 / N), then A DFTs of B points.
template <typename T, int A, int B, typename TW>
__device__ __forceinline__ void dft_ab(cplx_t<T> (&v)[A * B], TW twiddle)
{
    cplx_t<T> y[B][A];
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) {
        cplx_t<T> a[A];
#pragma unroll
        for (int n1 = 0; n1 < A; ++n1) a[n1] = v[B * n1 + n2];
        Dft<T, A>::run(a);
#pragma unroll
        for (int k1 = 0; k1 < A; ++k1) y[n2][k1] = a[k1];
    }
    twiddle(y);
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) {
        cplx_t<T> b[B];
#pragma unroll
        for (int n2 = 0; n2 < B; ++n2) b[n2] = y[n2][k1];
        Dft<T, B>::run(b);
#pragma unroll
        for (int k2 = 0; k2 < B; ++k2) v[k1 + A * k2] = b[k2];
    }
}
template <typename T> struct Dft<T, 6> {
    __device__ __forceinline__ static void run(cplx_t<T> (&v)[6])
    {
        const T h = (T)0.86602540378443864676;
        dft_ab<T, 3, 2>(v, [&](cplx_t<T>(&y)[2][3]) {
            y[1][1] = crot<T>(y[1][1], (T)0.5, h);    // 60 degrees
            y[1][2] = crot<T>(y[1][2], (T)-0.5, h);   // 120
        });
    }
};
template <typename T> struct Dft<T, 8> {
    __device__ __forceinline__ static void run(cplx_t<T> (&v)[8])
    {
        const T h = (T)0.70710678118654752440;   // sqrt(1/2)
        dft_ab<T, 4, 2>(v, [&](cplx_t<T>(&y)[2][4]) {
            y[1][1] = cmake<T>(h * (y[1][1].x + y[1][1].y), h * (y[1][1].y - y[1][1].x));
            y[1][2] = cmake<T>(y[1][2].y, -y[1][2].x);
            y[1][3] = cmake<T>(h * (y[1][3].y - y[1][3].x), -h * (y[1][3].x + y[1][3].y));
        });
    }
};
template <typename T> struct Dft<T, 12> {
    __device__ __forceinline__ static void run(cplx_t<T> (&v)[12])
    {
        const T h = (T)0.86602540378443864676;
        dft_ab<T, 4, 3>(v, [&](cplx_t<T>(&y)[3][4]) {
            y[1][1] = crot<T>(y[1][1], h, (T)0.5);            // 30 degrees
            y[1][2] = crot<T>(y[1][2], (T)0.5, h);            // 60
            y[1][3] = cmake<T>(y[1][3].y, -y[1][3].x);        // 90
            y[2][1] = crot<T>(y[2][1], (T)0.5, h);            // 60
            y[2][2] = crot<T>(y[2][2], (T)-0.5, h);           // 120
            y[2][3] = cmake<T>(-y[2][3].x, -y[2][3].y);       // 180
        });
    }
};
// XF: the terms with the other product fused (lines of 256 points and more).
template <typename T, bool XF> __device__ __forceinline__ void dft16(cplx_t<T> (&v)[16])
{
    const T c1 = (T)0.92387953251128675613;   // cos(pi/8)
    const T s1 = (T)0.38268343236508977173;   // sin(pi/8)
    const T h = (T)0.70710678118654752440;
    auto rx = [](cplx_t<T> z, T c, T s) { return XF ? crot_x<T>(z, c, s) : crot<T>(z, c, s); };
    dft_ab<T, 4, 4>(v, [&](cplx_t<T>(&y)[4][4]) {
        y[1][1] = crot<T>(y[1][1], c1, s1);
        y[1][2] = rx(y[1][2], h, h);
        y[1][3] = crot<T>(y[1][3], s1, c1);
        y[2][1] = crot<T>(y[2][1], h, h);
        y[2][2] = cmake<T>(y[2][2].y, -y[2][2].x);
        y[2][3] = rx(y[2][3], -h, h);
        y[3][1] = crot<T>(y[3][1], s1, c1);
        y[3][2] = rx(y[3][2], -h, h);
        y[3][3] = rx(y[3][3], -c1, -s1);
    });
}

// ----------------------------------------------------------- line addresses --
// Grid row, fhat row and roll-off factor of line pa (support index over the
// axes before t in FFT order, last axis fastest).  All counts fit 32 bits
// (line_tpl, fft.hip).
struct LineAt {
    int64_t gbase;
    int64_t fbase;
    double fac;
};
template <typename T> __device__ __forceinline__ LineAt line_at(const FftPass<T> &P, uint32_t pa)
{
    LineAt li;
    uint32_t a = 0, fq = 0;
    double fac = 1.0;
    if (P.t == 1) {
        const uint32_t N0 = (uint32_t)P.N[0], h0 = N0 >> 1;
        a = pa < h0 ? pa : pa + ((uint32_t)P.n[0] - N0);
        fq = pa < h0 ? pa + h0 : pa - h0;
        fac = P.roc[P.rocoff[0] + pa];
    } else if (P.t == 2) {
        const uint32_t N0 = (uint32_t)P.N[0], h0 = N0 >> 1, N1 = (uint32_t)P.N[1], h1 = N1 >> 1;
        const uint32_t p0 = pa / N1, p1 = pa - p0 * N1;
        const uint32_t i0 = p0 < h0 ? p0 : p0 + ((uint32_t)P.n[0] - N0);
        const uint32_t i1 = p1 < h1 ? p1 : p1 + ((uint32_t)P.n[1] - N1);
        a = i0 * (uint32_t)P.n[1] + i1;
        fq = (p0 < h0 ? p0 + h0 : p0 - h0) * N1 + (p1 < h1 ? p1 + h1 : p1 - h1);
        fac = P.roc[P.rocoff[1] + p1] * P.roc[P.rocoff[0] + p0];
    }
    li.gbase = (int64_t)a * P.Lf * P.So;
    li.fbase = (int64_t)fq * P.N[P.t == 0 ? 0 : (P.t == 1 ? 1 : 2)];
    li.fac = fac;
    return li;
}

// How the threads of a workgroup are spread over (line c, thread t of a line).
enum LineMap : int { MAP_ROWS = 0, MAP_COLS = 1 };

// MAPI / MAPO: thread spread of the loads and of the stores (rows: t fastest, a
// line is contiguous; columns: c fastest, C adjacent columns are contiguous).
// They differ for the second pass of a split axis, whose C lines are read as
// rows and written side by side.
template <typename T, int L, int MAPI, int MAPO, int SPLIT>
__device__ __forceinline__ void fft_line(const FftPass<T> &P, uint32_t blk, cplx_t<T> *buf)
{
    using C2 = cplx_t<T>;
    using PL = LinePlan<L>;
    constexpr int EPT = PL::EPT, NS = PL::NS, TPL = L / EPT, PITCH = line_pitch<L>(), R0 = PL::R[0];
    static_assert(EPT > 0 && L % EPT == 0, "a listed line length");
    const int tid = threadIdx.x, C = P.C, logC = P.logC;
    const bool active = tid < C * TPL;
    int c, t;
    auto spread = [&](int map) {
        if (map == MAP_COLS) {
            c = tid & (C - 1);
            t = tid >> logC;
        } else {
            c = tid / TPL;
            t = tid - c * TPL;
        }
    };
    // LDS cell of element o of line c
    auto cell = [&](int o) {
        const int p = o + o / R0;
        return MAPI == MAP_COLS ? (p << logC) + c : c * PITCH + p;
    };
    const int Nt = (int)P.N[P.t == 0 ? 0 : (P.t == 1 ? 1 : 2)], hN = Nt >> 1;
    const int Lf = (int)P.Lf, L1 = (int)P.L1;
    const double *__restrict__ roct = P.roc + P.rocoff[P.t == 0 ? 0 : (P.t == 1 ? 1 : 2)];
    const bool swp = P.sign > 0;
    spread(MAPI);

    // ---- the thread's line
    uint32_t pa = 0, s = 0;      // line index, column
    bool valid = active;
    if constexpr (MAPI == MAP_COLS) {
        const uint32_t nch = (uint32_t)(P.S >> logC);
        pa = blk / nch;                                   // uniform
        s = ((blk - pa * nch) << logC) + (uint32_t)c;
    } else {
        pa = (blk << logC) + (uint32_t)c;
        valid = active && pa < (uint32_t)P.n_pa;
        pa = valid ? pa : 0u;
    }
    uint32_t k2 = 0;
    LineAt li;
    auto locate = [&] {
        uint32_t pb = pa;
        if constexpr (SPLIT == SPLIT_B) {
            pb = pa / (uint32_t)P.L2;
            k2 = pa - pb * (uint32_t)P.L2;
        }
        li = line_at<T>(P, pb);
    };
    locate();
    const int i1 = SPLIT == SPLIT_A ? (int)(s / (uint32_t)P.So) : 0;
    auto full_in = [&](int i) { return SPLIT == SPLIT_A ? i1 + L1 * i : i; };

    // ---- loads (all in flight before the first use)
    C2 v[EPT];
    const bool from_fhat = SPLIT != SPLIT_B && (P.mode & FFT_FROM_FHAT);
    if (from_fhat) {
        double fr[EPT];
#pragma unroll
        for (int q = 0; q < EPT; ++q) {
            // the whole slice q outside the support (uniform): zero, nothing loaded
            const int lo = L1 * TPL * q;
            v[q] = cmake<T>(0, 0);
            fr[q] = 0.0;
            if (lo >= hN && lo + L1 * TPL <= Lf - hN) continue;
            const int ifl = full_in(t + TPL * q);
            const bool low = ifl < hN, in = valid && (low || ifl >= Lf - hN);
            const int p = low ? ifl : ifl - (Lf - Nt), qf = low ? ifl + hN : ifl - (Lf - hN);
            v[q] = P.fhat_in[li.fbase + (in ? qf : 0)];
            fr[q] = in ? roct[in ? p : 0] : 0.0;
        }
#pragma unroll
        for (int q = 0; q < EPT; ++q) {
            const double f = li.fac * fr[q];
            // a factor of zero marks an element outside the support
            v[q] = fr[q] != 0.0 ? cmake<T>((T)((double)v[q].x * f), (T)((double)v[q].y * f))
                                : cmake<T>(0, 0);
        }
    } else {
        const bool pruned = P.mode & FFT_IN_PRUNED;
        const int64_t base = li.gbase + (SPLIT == SPLIT_B ? (int64_t)k2 * P.L1 * P.So : 0) + s;
        const C2 *__restrict__ src = P.g + (valid ? base + (int64_t)t * P.S : 0);
        const int64_t step = valid ? (int64_t)TPL * P.S : 0;
#pragma unroll
        for (int q = 0; q < EPT; ++q) {
            const int lo = L1 * TPL * q;
            v[q] = cmake<T>(0, 0);
            if (SPLIT != SPLIT_B && pruned && lo >= hN && lo + L1 * TPL <= Lf - hN) continue;
            v[q] = src[q * step];
        }
        if (SPLIT != SPLIT_B && pruned) {
#pragma unroll
            for (int q = 0; q < EPT; ++q) {
                const int ifl = full_in(t + TPL * q);
                if (ifl >= hN && ifl < Lf - hN) v[q] = cmake<T>(0, 0);
            }
        }
    }
    if (swp) {
#pragma unroll
        for (int q = 0; q < EPT; ++q) v[q] = cmake<T>(v[q].y, v[q].x);
    }
    if constexpr (SPLIT == SPLIT_B) {
        // w_Lf^(-i k2); i k2 < L1 L2 = Lf
#pragma unroll
        for (int q = 0; q < EPT; ++q) {
            const uint32_t e = (uint32_t)(t + TPL * q) * k2;
            double sn, cs;
            sincospi(-2.0 * (double)e / (double)Lf, &sn, &cs);
            const double wr = (double)v[q].x, wi = (double)v[q].y;
            v[q] = cmake<T>((T)(wr * cs - wi * sn), (T)(wr * sn + wi * cs));
        }
    }

    // ---- stages
    const C2 *__restrict__ tw = P.tw;
    auto stage = [&](auto s_c, auto ns_c) {
        constexpr int SI = decltype(s_c)::value, Ns = decltype(ns_c)::value, R = PL::R[SI];
        constexpr int NBF = EPT / R;
        static_assert(EPT % R == 0 && L % (R * Ns) == 0, "whole butterflies per thread");
        // radix 8 of a power-of-two line: a radix-4 and a radix-2 stage back to back
        // (w[b][r]: r < 4 the radix-4 twiddles, r >= 4 the radix-2 ones)
        constexpr bool R42 = R == 8 && (L & (L - 1)) == 0;
        C2 w[NBF][R];
        if constexpr (SI > 0 || R42) {
#pragma unroll
            for (int b = 0; b < NBF; ++b) {
                const int jm = (t + b * TPL) % Ns;
                constexpr int u = L / (R * Ns);
                if constexpr (R42) {
#pragma unroll
                    for (int r = 1; r < 4; ++r) w[b][r] = tw[2 * r * jm * u];
#pragma unroll
                    for (int r = 0; r < 4; ++r) w[b][4 + r] = tw[(jm + Ns * r) * u];
                } else {
#pragma unroll
                    for (int r = 1; r < R; ++r) w[b][r] = tw[r * jm * u];
                }
            }
        }
        if constexpr (SI > 0) {
            __syncthreads();   // (the twiddle loads above are on their way meanwhile)
#pragma unroll
            for (int q = 0; q < EPT; ++q) v[q] = active ? buf[cell(t + TPL * q)] : cmake<T>(0, 0);
#pragma unroll
            for (int b = 0; b < NBF; ++b)
#pragma unroll
                for (int r = 1; r < R; ++r)
                    if (!R42 || r > 1)
                        v[b + r * NBF] = cmulf<T>(v[b + r * NBF], w[b][R42 ? r / 2 : r]);
        }
#pragma unroll
        for (int b = 0; b < NBF; ++b) {
            C2 a[R];
#pragma unroll
            for (int r = 0; r < R; ++r) a[r] = v[b + r * NBF];
            if constexpr (R42) {
                dft_ab<T, 4, 2>(a, [&](C2(&y)[2][4]) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) y[1][r] = cmulf<T>(y[1][r], w[b][4 + r]);
                });
            } else if constexpr (R == 16) {
                dft16<T, (L >= 256)>(a);
            } else {
                Dft<T, R>::run(a);
            }
#pragma unroll
            for (int r = 0; r < R; ++r) v[b + r * NBF] = a[r];
        }
        if constexpr (SI < NS - 1) {
            if constexpr (SI > 0) __syncthreads();   // every thread has read the previous exchange
            if (active) {
#pragma unroll
                for (int b = 0; b < NBF; ++b) {
                    const int j = t + b * TPL;
                    const int o = (j / Ns) * (Ns * R) + j % Ns;
#pragma unroll
                    for (int r = 0; r < R; ++r) buf[cell(o + r * Ns)] = v[b + r * NBF];
                }
            }
            if constexpr (SI == NS - 2 && MAPO != MAPI) spread(MAPO);
        }
    };
    using std::integral_constant;
    stage(integral_constant<int, 0>{}, integral_constant<int, 1>{});
    if constexpr (NS > 1) stage(integral_constant<int, 1>{}, integral_constant<int, PL::R[0]>{});
    if constexpr (NS > 2) stage(integral_constant<int, 2>{}, integral_constant<int, PL::R[0] * PL::R[1]>{});
    if constexpr (NS > 3)
        stage(integral_constant<int, 3>{}, integral_constant<int, PL::R[0] * PL::R[1] * PL::R[2]>{});

    // ---- stores
    if constexpr (MAPO != MAPI) {
        pa = (blk << logC) + (uint32_t)c;
        valid = active && pa < (uint32_t)P.n_pa;
        pa = valid ? pa : 0u;
        locate();
    }
    if (!valid) return;
    if (swp) {
#pragma unroll
        for (int q = 0; q < EPT; ++q) v[q] = cmake<T>(v[q].y, v[q].x);
    }
    if constexpr (SPLIT == SPLIT_A) {
        C2 *dst = P.g + li.gbase + s + (int64_t)t * P.S;
        const int64_t step = (int64_t)TPL * P.S;
#pragma unroll
        for (int q = 0; q < EPT; ++q) dst[q * step] = v[q];
    } else {
        // full output index of element i: i, or k2 + L2 i for the second half of a split axis
        const int L2 = SPLIT == SPLIT_B ? (int)P.L2 : 1;
        if (P.mode & FFT_TO_FHAT) {
            double fr[EPT];
#pragma unroll
            for (int q = 0; q < EPT; ++q) {
                const int kf = (SPLIT == SPLIT_B ? (int)k2 : 0) + L2 * (t + TPL * q);
                const bool in = kf < hN || kf >= Lf - hN;
                fr[q] = roct[in ? (kf < hN ? kf : kf - (Lf - Nt)) : 0];
            }
#pragma unroll
            for (int q = 0; q < EPT; ++q) {
                const int kf = (SPLIT == SPLIT_B ? (int)k2 : 0) + L2 * (t + TPL * q);
                const bool low = kf < hN;
                if (low || kf >= Lf - hN) {
                    const double f = li.fac * fr[q];
                    P.fhat_out[li.fbase + (low ? kf + hN : kf - (Lf - hN))] =
                        cmake<T>((T)((double)v[q].x * f), (T)((double)v[q].y * f));
                }
            }
        } else {
            const bool pruned = P.mode & FFT_OUT_PRUNED;
            const int64_t S = SPLIT == SPLIT_B ? P.So : P.S;
            C2 *out = SPLIT == SPLIT_B ? P.dst : P.g;
            C2 *dst = out + li.gbase + s + (int64_t)((SPLIT == SPLIT_B ? (int64_t)k2 : 0) + (int64_t)L2 * t) * S;
            const int64_t step = (int64_t)TPL * L2 * S;
#pragma unroll
            for (int q = 0; q < EPT; ++q) {
                const int kf = (SPLIT == SPLIT_B ? (int)k2 : 0) + L2 * (t + TPL * q);
                if (!pruned || kf < hN || kf >= Lf - hN) dst[q * step] = v[q];
            }
        }
    }
}

template <typename T, int L, int MAPI, int MAPO, int SPLIT>
__global__ __launch_bounds__(line_threads_max<L>(), (line_waves<T, LinePlan<L>::EPT>())) void k_fft_line(FftPass<T> P)
{
    extern __shared__ __align__(16) unsigned char line_lds[];
    uint32_t blk = blockIdx.x;
    if constexpr (MAPI == MAP_COLS) {
        // column groups narrower than a 128-byte line: neighbours, which share
        // lines, go to the same XCD (workgroups are dealt round-robin over 8)
        if (P.C * (int)sizeof(cplx_t<T>) < 128 && gridDim.x % 8 == 0)
            blk = (blk & 7u) * (gridDim.x >> 3) + (blk >> 3);
    }
    fft_line<T, L, MAPI, MAPO, SPLIT>(P, blk, reinterpret_cast<cplx_t<T> *>(line_lds));
}

// The passes of many transforms in one grid (the jobs' lengths differ; threads, 256 at
// most, and LDS for the largest workgroup among them).  Rows and columns apart.  Short
// lines need few threads, and idle wavefronts would hold the registers of others: six
// 3D problems of 64^3 grids x 2, FP64, 497 -> 309 us (forward), 256 x 8 lines of 1024
// points FP32 53 -> 36 us against 256 threads for all.
template <typename T, int MAP>
__global__ __launch_bounds__(256, (line_waves<T, 24>())) void k_fft_line_batch(const FftPass<T> *__restrict__ passes,
                                                        const BlockMap *__restrict__ map)
{
    extern __shared__ __align__(16) unsigned char line_lds[];
    const BlockMap bm = map[blockIdx.x];
    const FftPass<T> &P = passes[bm.job];
    cplx_t<T> *buf = reinterpret_cast<cplx_t<T> *>(line_lds);
    switch (P.L) {
#define CUNFFT_CASE(LEN) \
    case LEN: fft_line<T, LEN, MAP, MAP, SPLIT_NONE>(P, bm.blk, buf); break;
        CUNFFT_POW2_LINES(CUNFFT_CASE)
        CUNFFT_MIXED_LINES(CUNFFT_CASE)
#undef CUNFFT_CASE
    }
}

// ------------------------------------------------------------- dispatch --
template <typename T> void launch_fft_line(const FftPass<T> &P, int64_t blocks, size_t lds, hipStream_t s)
{
    const unsigned nt = (unsigned)((P.C * P.tpl + 63) / 64 * 64), nb = (unsigned)blocks;
    const bool rows = P.S == 1;
    if (P.split == SPLIT_NONE) {
        switch (P.L) {
#define CUNFFT_CASE(LEN)                                                                       \
    case LEN:                                                                                  \
        if (rows) k_fft_line<T, LEN, MAP_ROWS, MAP_ROWS, SPLIT_NONE><<<nb, nt, lds, s>>>(P);   \
        else k_fft_line<T, LEN, MAP_COLS, MAP_COLS, SPLIT_NONE><<<nb, nt, lds, s>>>(P);        \
        break;
            CUNFFT_POW2_LINES(CUNFFT_CASE)
            CUNFFT_MIXED_LINES(CUNFFT_CASE)
#undef CUNFFT_CASE
        default: throw Error(CUNFFT_ERR_UNSUPPORTED, "FFT line length");
        }
    } else {
        switch (P.L) {
#define CUNFFT_CASE(LEN)                                                                       \
    case LEN:                                                                                  \
        if (P.split == SPLIT_A)                                                                \
            k_fft_line<T, LEN, MAP_COLS, MAP_COLS, SPLIT_A><<<nb, nt, lds, s>>>(P);            \
        else if (rows)                                                                         \
            k_fft_line<T, LEN, MAP_ROWS, MAP_COLS, SPLIT_B><<<nb, nt, lds, s>>>(P);            \
        else                                                                                   \
            k_fft_line<T, LEN, MAP_COLS, MAP_COLS, SPLIT_B><<<nb, nt, lds, s>>>(P);            \
        break;
            CUNFFT_SPLIT_LINES(CUNFFT_CASE)
#undef CUNFFT_CASE
        default: throw Error(CUNFFT_ERR_UNSUPPORTED, "FFT line length");
        }
    }
    CUNFFT_HIP(hipGetLastError());
}

template <typename T>
void launch_fft_line_batch(const FftPass<T> *passes, const BlockMap *map, uint32_t nblk, bool rows,
                           int threads, size_t lds, hipStream_t s)
{
    if (rows) k_fft_line_batch<T, MAP_ROWS><<<nblk, threads, lds, s>>>(passes, map);
    else k_fft_line_batch<T, MAP_COLS><<<nblk, threads, lds, s>>>(passes, map);
    CUNFFT_HIP(hipGetLastError());
}

}  // namespace cunfft

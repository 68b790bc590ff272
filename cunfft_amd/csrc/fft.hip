// fft.hip -- LDS-resident Stockham FFT pass for gfx950 with fused roll-off.
//
// Replaces the three reference steps around the FFT:
//   forward  kernelRollOf_{1,2,3}d + memset  (src/cunfft_kernel.cu:240-412,
//            src/cunfft_wrapper.cu:32-75)  then cufftExec(.., CUFFT_FORWARD)
//   adjoint  cufftExec(.., CUFFT_INVERSE) then kernelRollOf_adjoint_{1,2,3}d
//            (src/cunfft_kernel.cu:264-467, src/cunfft_wrapper.cu:77-121)
// A d-dimensional transform is d passes, one per axis, each one HBM read and
// one write.  The forward passes skip lines that are still all zero and read
// only the N_t nonzero entries of each line; the first forward pass reads fhat
// and applies exp(fac k^2) on the way in.  The adjoint passes write only the
// N_t entries that survive the crop; the last one writes fhat with exp(fac k^2).
// Twiddles come from a per-length table computed in extended precision on the
// host.
//
// The usual line lengths (4 .. 4096 powers of two, 3 2^k and 9 2^k from 48 to 1536)
// run the register-resident pass of fft_line.hpp.  This file holds the set-up
// of the passes and the generic pass for the other lengths 2^a 3^b: each
// workgroup loads C whole lines into LDS, runs Stockham stages there and writes
// the lines back.
#include <algorithm>
#include <type_traits>

#include "fft_line.hpp"

namespace cunfft {

// (instantiated in fft_line_f32.hip and fft_line_f64.hip)
extern template void launch_fft_line<float>(const FftPass<float> &, int64_t, size_t, hipStream_t);
extern template void launch_fft_line<double>(const FftPass<double> &, int64_t, size_t, hipStream_t);

constexpr int kFftThreads = 256;
// Elements C * L per workgroup of the generic pass: up to kFftElems.
constexpr int kFftElems = 4096;
// global loads in flight per thread from fhat (FP64: fewer, the registers run
// short); loads from the grid, with no FP64 roll-off factor to hold, take twice
// as many (FP64 3D 256^3 passes 3% faster, FP32 unchanged)
template <typename T> constexpr int fft_load_batch() { return sizeof(T) == 4 ? 8 : 4; }
constexpr int kMaxRowsPerGroup = 64;
constexpr int kFftLineLds = 144 * 1024;   // LDS of a register-resident pass's lines, at most

template <typename T>
__device__ __forceinline__ cplx_t<T> cmul(const cplx_t<T> a, const cplx_t<T> b)
{
    return cmake<T>(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

template <typename T>
__device__ __forceinline__ cplx_t<T> twiddle(const cplx_t<T> *__restrict__ tw, int q, int sign)
{
    cplx_t<T> w = tw[q];
    if (sign > 0) w.y = -w.y;
    return w;
}

// 4-point DFT with kernel exp(sign 2 pi i r q / 4).
template <typename T> __device__ __forceinline__ void dft4(cplx_t<T> (&v)[4], int sign)
{
    const cplx_t<T> a0 = cmake<T>(v[0].x + v[2].x, v[0].y + v[2].y);
    const cplx_t<T> a1 = cmake<T>(v[0].x - v[2].x, v[0].y - v[2].y);
    const cplx_t<T> a2 = cmake<T>(v[1].x + v[3].x, v[1].y + v[3].y);
    const cplx_t<T> a3 = cmake<T>(v[1].x - v[3].x, v[1].y - v[3].y);
    // omega * a3 with omega = sign * i
    const T sr = sign > 0 ? -a3.y : a3.y;
    const T si = sign > 0 ? a3.x : -a3.x;
    v[0] = cmake<T>(a0.x + a2.x, a0.y + a2.y);
    v[2] = cmake<T>(a0.x - a2.x, a0.y - a2.y);
    v[1] = cmake<T>(a1.x + sr, a1.y + si);
    v[3] = cmake<T>(a1.x - sr, a1.y - si);
}

struct LineInfo {
    int64_t gbase;  // grid offset of the line's axis start (without the column)
    int64_t fbase;  // fhat offset of the row (passes on the last axis)
    double fac;     // product of roll-off factors of the axes before t
};

// Map the line index pa (support of the axes before t, FFT order, last axis
// fastest) to its grid row, its fhat row and its roll-off factor.
template <typename T>
__device__ LineInfo line_info(const FftPass<T> &P, int64_t pa)
{
    LineInfo li;
    int64_t rem = pa;
    int64_t a = 0, gmul = 1, fq = 0, fmul = 1;
    double fac = 1.0;
    // axes tt = t-1 .. 0, unrolled so the per-axis fields are read by constant
    // index (no private-memory copy of the descriptor)
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int tt = 1 - k;
        if (tt >= P.t) continue;
        const int64_t Nn = P.N[tt], hN = Nn >> 1;
        const int64_t p = rem % Nn;
        rem /= Nn;
        const int64_t i = p < hN ? p : p + (P.n[tt] - Nn);
        const int64_t q = p < hN ? p + hN : p - hN;
        a += i * gmul;
        gmul *= P.n[tt];
        fq += q * fmul;
        fmul *= Nn;
        fac *= P.roc[P.rocoff[tt] + p];
    }
    li.gbase = a * P.Lf * P.So;
    li.fbase = fq * (P.t == 0 ? P.N[0] : (P.t == 1 ? P.N[1] : P.N[2]));
    li.fac = fac;
    return li;
}

// a = q d + r for 0 <= a < 2^22 with rd = 1/d in FP32 (exact after one
// correction step)
__device__ __forceinline__ void divmod_small(int a, int d, float rd, int &q, int &r)
{
    q = (int)((float)a * rd);
    r = a - q * d;
    if (r < 0) {
        --q;
        r += d;
    } else if (r >= d) {
        ++q;
        r -= d;
    }
}

// R-point DFT with kernel exp(sign 2 pi i r q / R), R = 2, 3, 4.
template <typename T, int R> __device__ __forceinline__ void dft_r(cplx_t<T> (&v)[R], int sign)
{
    if constexpr (R == 2) {
        const cplx_t<T> a = v[0], b = v[1];
        v[0] = cmake<T>(a.x + b.x, a.y + b.y);
        v[1] = cmake<T>(a.x - b.x, a.y - b.y);
    } else if constexpr (R == 3) {
        // y1,2 = a - (b + c)/2 +- sign i (sqrt(3)/2)(b - c)
        const T h = (T)0.86602540378443864676;   // sqrt(3) / 2
        const cplx_t<T> a = v[0], b = v[1], c = v[2];
        const T sx = b.x + c.x, sy = b.y + c.y;
        const T dx = (T)sign * h * (b.x - c.x), dy = (T)sign * h * (b.y - c.y);
        const T mx = a.x - (T)0.5 * sx, my = a.y - (T)0.5 * sy;
        v[0] = cmake<T>(a.x + sx, a.y + sy);
        v[1] = cmake<T>(mx - dy, my + dx);
        v[2] = cmake<T>(mx + dy, my - dx);
    } else {
        dft4<T>(v, sign);
    }
}

// One Stockham stage of radix R for any L (stride Q = L/R, Ns = product of
// the radices before it): butterfly j of line c reads j + rQ, multiplies
// input r by exp(sign 2 pi i r (j mod Ns) / (R Ns)), and writes its R-point
// DFT to (j div Ns) R Ns + (j mod Ns) + r Ns.
template <typename T, int E, int R>
__device__ __forceinline__ void stage_any(cplx_t<T> *buf, const cplx_t<T> *__restrict__ tw, int L,
                                          int C, int ldsL, int Ns, int sign, int tid)
{
    const int Q = L / R;
    const int nb = C * Q;
    const int tws = L / (R * Ns);    // twiddle-table step of exp(2 pi i / (R Ns))
    const float rQ = 1.0f / (float)Q, rN = 1.0f / (float)Ns;
    constexpr int KB = (E / R + kFftThreads - 1) / kFftThreads;
    cplx_t<T> v[KB][R];
#pragma unroll
    for (int k = 0; k < KB; ++k) {
        const int b = tid + k * kFftThreads;
        if (b < nb) {
            int c, j, jq, jr;
            divmod_small(b, Q, rQ, c, j);
            divmod_small(j, Ns, rN, jq, jr);
            const cplx_t<T> *base = buf + c * ldsL + j;
#pragma unroll
            for (int r = 0; r < R; ++r) v[k][r] = base[r * Q];
#pragma unroll
            for (int r = 1; r < R; ++r) v[k][r] = cmul<T>(v[k][r], twiddle<T>(tw, r * jr * tws, sign));
            dft_r<T, R>(v[k], sign);
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < KB; ++k) {
        const int b = tid + k * kFftThreads;
        if (b < nb) {
            int c, j, jq, jr;
            divmod_small(b, Q, rQ, c, j);
            divmod_small(j, Ns, rN, jq, jr);
            cplx_t<T> *ob = buf + c * ldsL + jq * (R * Ns) + jr;
#pragma unroll
            for (int r = 0; r < R; ++r) ob[r * Ns] = v[k][r];
        }
    }
    __syncthreads();
}

template <typename T, int E, int SPLIT>
__device__ __forceinline__ void fft_pass(const FftPass<T> &P, int64_t blk)
{
    using C2 = cplx_t<T>;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    C2 *buf = reinterpret_cast<C2 *>(smem_raw);
    __shared__ int64_t s_gbase[kMaxRowsPerGroup];   // input offset of the line (column 0)
    __shared__ int64_t s_obase[kMaxRowsPerGroup];   // SPLIT_B: output offset of the line
    __shared__ int64_t s_fbase[kMaxRowsPerGroup];
    __shared__ double s_fac[kMaxRowsPerGroup];
    __shared__ int s_valid[kMaxRowsPerGroup];
    __shared__ int s_k2[kMaxRowsPerGroup];          // SPLIT_B: output index k2 of the line
    __shared__ int s_i1[kMaxRowsPerGroup];          // SPLIT_A: index i1 of the column

    const int tid = threadIdx.x;
    const int L = P.L, C = P.C, logC = P.logC, ldsL = P.ldsL;
    const bool rows = (P.S == 1);
    int64_t pa0, s0;
    if (rows) {
        pa0 = blk << logC;
        s0 = 0;
    } else {
        const int64_t nch = P.S >> logC;
        pa0 = blk / nch;
        s0 = (blk - pa0 * nch) << logC;
    }
    if (tid < (rows ? C : 1)) {
        const int64_t pa = pa0 + tid;
        const bool valid = pa < P.n_pa;
        int64_t pb = valid ? pa : 0, k2 = 0;
        if (SPLIT == SPLIT_B) {
            k2 = pb % P.L2;
            pb /= P.L2;
        }
        const LineInfo li = line_info<T>(P, pb);
        s_gbase[tid] = li.gbase + (SPLIT == SPLIT_B ? k2 * P.L1 * P.So : 0);
        s_obase[tid] = li.gbase;
        s_fbase[tid] = li.fbase;
        s_fac[tid] = li.fac;
        s_valid[tid] = valid;
        s_k2[tid] = (int)k2;
    }
    if (SPLIT == SPLIT_A && tid < C) s_i1[tid] = (int)((s0 + tid) / P.So);
    // the twiddle table of the axis, staged in LDS after the lines
    C2 *twl = buf + C * ldsL;
    for (int q = tid; q < L; q += kFftThreads) twl[q] = P.tw[q];
    __syncthreads();

    const float rL = 1.0f / (float)L;
    const int total = C * L;
    const int64_t Lf = P.Lf;
    const int Nt = (int)(P.t == 0 ? P.N[0] : (P.t == 1 ? P.N[1] : P.N[2]));
    const int hN = Nt >> 1;
    const double *roct =
        P.roc + (P.t == 0 ? P.rocoff[0] : (P.t == 1 ? P.rocoff[1] : P.rocoff[2]));
    // the full-axis index of element i of line / column c before the pass
    auto in_index = [&](int i, int c) -> int64_t {
        if constexpr (SPLIT == SPLIT_A) return (int64_t)s_i1[c] + P.L1 * (int64_t)i;
        return i;
    };

    // loads in batches of kFftLoadBatch per thread, all issued before the
    // first LDS store (a pass is bound by memory latency otherwise): every
    // lane loads, from a clamped address where it has nothing to load, and
    // the value is zeroed after
    auto stage_in = [&](auto from_fhat_tag) {
        constexpr bool FROM_FHAT = decltype(from_fhat_tag)::value;
        constexpr int kFftLoadBatch = fft_load_batch<T>() * (FROM_FHAT ? 1 : 2);
        const bool in_pruned = P.mode & FFT_IN_PRUNED;
        for (int e0 = tid; e0 < total; e0 += kFftLoadBatch * kFftThreads) {
            C2 v[kFftLoadBatch];
            double fr[kFftLoadBatch];   // roll-off factor of a load from fhat
            int at[kFftLoadBatch];
            bool ok[kFftLoadBatch];
#pragma unroll
            for (int u = 0; u < kFftLoadBatch; ++u) {
                const int e = e0 + u * kFftThreads;
                int c, i;
                if (rows) {
                    divmod_small(e, L, rL, c, i);
                } else {
                    c = e & (C - 1);
                    i = e >> logC;
                }
                const bool in = e < total;
                const int li = rows && in ? c : 0;
                at[u] = in ? c * ldsL + i : -1;
                const int64_t ifl = in_index(i, in ? c : 0);
                const bool insupp = (ifl < hN) || (ifl >= Lf - hN);
                if constexpr (FROM_FHAT) {
                    ok[u] = in && s_valid[li] && insupp;
                    const int p = (int)(ifl < hN ? ifl : ifl - (Lf - Nt));
                    const int q = p < hN ? p + hN : p - hN;
                    const int64_t fb = s_fbase[li];
                    const double fl = s_fac[li];
                    v[u] = P.fhat_in[ok[u] ? fb + q : 0];
                    fr[u] = fl * roct[ok[u] ? p : 0];
                } else {
                    ok[u] = in && s_valid[li] && (!in_pruned || insupp);
                    const int64_t gb = s_gbase[li];
                    v[u] = P.g[ok[u] ? gb + (int64_t)i * P.S + s0 + (rows ? 0 : c) : 0];
                }
            }
#pragma unroll
            for (int u = 0; u < kFftLoadBatch; ++u) {
                C2 w = ok[u] ? v[u] : cmake<T>(0, 0);
                if constexpr (FROM_FHAT)
                    w = cmake<T>((T)((double)w.x * fr[u]), (T)((double)w.y * fr[u]));
                if constexpr (SPLIT == SPLIT_B) {
                    // w_Lf^(sign i1 k2), the angle reduced mod Lf and taken in FP64
                    if (at[u] >= 0) {
                        const int c = at[u] / ldsL, i = at[u] - c * ldsL;
                        const int64_t q = ((int64_t)i * s_k2[rows ? c : 0]) % Lf;
                        double sn, cs;
                        sincospi((double)P.sign * 2.0 * (double)q / (double)Lf, &sn, &cs);
                        const double wr = (double)w.x, wi = (double)w.y;
                        w = cmake<T>((T)(wr * cs - wi * sn), (T)(wr * sn + wi * cs));
                    }
                }
                if (at[u] >= 0) buf[at[u]] = w;
            }
        }
    };
    if (P.mode & FFT_FROM_FHAT)
        stage_in(std::true_type{});
    else
        stage_in(std::false_type{});
    __syncthreads();

    // L = 2^a 3^b: radix 4 while the power-of-two part allows, one radix 2 if a
    // is odd, then b radix-3 stages
    int p2 = L;
    for (int k = 0; k < P.n3; ++k) p2 /= 3;
    int Ns = 1;
    while (Ns * 4 <= p2) {
        stage_any<T, E, 4>(buf, twl, L, C, ldsL, Ns, P.sign, tid);
        Ns *= 4;
    }
    if (Ns < p2) {
        stage_any<T, E, 2>(buf, twl, L, C, ldsL, Ns, P.sign, tid);
        Ns *= 2;
    }
    for (int k = 0; k < P.n3; ++k) {
        stage_any<T, E, 3>(buf, twl, L, C, ldsL, Ns, P.sign, tid);
        Ns *= 3;
    }

    for (int e = tid; e < total; e += kFftThreads) {
        int c, i;
        if (rows) {
            divmod_small(e, L, rL, c, i);
        } else {
            c = e & (C - 1);
            i = e >> logC;
        }
        const int li = rows ? c : 0;
        if (!s_valid[li]) continue;
        if constexpr (SPLIT == SPLIT_A) {
            // the first half of a split axis: back in place, nothing pruned
            P.g[s_gbase[li] + (int64_t)i * P.S + s0 + (rows ? 0 : c)] = buf[c * ldsL + i];
            continue;
        }
        // full output index: i, or k2 + L2 k1 for the second half of a split axis
        const int64_t kf = SPLIT == SPLIT_B ? s_k2[li] + P.L2 * (int64_t)i : (int64_t)i;
        const bool insupp = (kf < hN) || (kf >= Lf - hN);
        if (P.mode & FFT_TO_FHAT) {
            if (insupp) {
                const int p = (int)(kf < hN ? kf : kf - (Lf - Nt));
                const int q = p < hN ? p + hN : p - hN;
                const C2 v = buf[c * ldsL + i];
                const double f = s_fac[li] * roct[p];
                P.fhat_out[s_fbase[li] + q] = cmake<T>((T)((double)v.x * f), (T)((double)v.y * f));
            }
        } else if (!(P.mode & FFT_OUT_PRUNED) || insupp) {
            if constexpr (SPLIT == SPLIT_B)
                P.dst[s_obase[li] + kf * P.So + s0 + (rows ? 0 : c)] = buf[c * ldsL + i];
            else
                P.g[s_gbase[li] + (int64_t)i * P.S + s0 + (rows ? 0 : c)] = buf[c * ldsL + i];
        }
    }
}

template <typename T, int E, int SPLIT>
__global__ __launch_bounds__(kFftThreads) void k_fft_pass(FftPass<T> P)
{
    fft_pass<T, E, SPLIT>(P, blockIdx.x);
}

// Passes of many transforms in one grid (a batch's jobs; LDS sized for the
// largest).  Batches run unsplit axes only.
template <typename T, int E>
__global__ __launch_bounds__(kFftThreads) void k_fft_pass_batch(const FftPass<T> *__restrict__ passes,
                                                                const BlockMap *__restrict__ map)
{
    const BlockMap bm = map[blockIdx.x];
    fft_pass<T, E, SPLIT_NONE>(passes[bm.job], bm.blk);
}

template <typename T>
void launch_fft_pass(const FftPass<T> &p, int64_t blocks, size_t lds_bytes, hipStream_t s)
{
    if (blocks <= 0) return;
    if (blocks >= (int64_t(1) << 32) / kFftThreads)
        throw Error(CUNFFT_ERR_UNSUPPORTED, "FFT pass needs too many workgroups");
    if (p.tpl > 0) {
        launch_fft_line<T>(p, blocks, lds_bytes, s);
        return;
    }
    if (p.split == SPLIT_A)
        k_fft_pass<T, kFftElems, SPLIT_A><<<(unsigned)blocks, kFftThreads, lds_bytes, s>>>(p);
    else if (p.split == SPLIT_B)
        k_fft_pass<T, kFftElems, SPLIT_B><<<(unsigned)blocks, kFftThreads, lds_bytes, s>>>(p);
    else
        k_fft_pass<T, kFftElems, SPLIT_NONE><<<(unsigned)blocks, kFftThreads, lds_bytes, s>>>(p);
    CUNFFT_HIP(hipGetLastError());
}

template <typename T>
void launch_fft_batch(const FftPass<T> *passes, const BlockMap *map, uint32_t nblk,
                      size_t lds_bytes, hipStream_t s)
{
    if (nblk == 0) return;
    k_fft_pass_batch<T, kFftElems><<<nblk, kFftThreads, lds_bytes, s>>>(passes, map);
    CUNFFT_HIP(hipGetLastError());
}

static int ilog2_i(int64_t v)
{
    int l = 0;
    while ((int64_t(1) << l) < v) ++l;
    return l;
}

static int64_t prev_pow2_i(int64_t v)
{
    int64_t p = 1;
    while (2 * p <= v) p <<= 1;
    return p;
}

static int64_t next_pow2_i(int64_t v)
{
    int64_t p = 1;
    while (p < v) p <<= 1;
    return p;
}

// Threads per line of the register-resident pass for P, or 0: its line length
// is not listed, or its counts leave 32 bits.
template <typename T> static int line_tpl(const FftPass<T> &P)
{
    int64_t total = P.Lf * P.So;
    for (int q = 0; q < P.t; ++q) total *= P.n[q];
    if (total >= (int64_t(1) << 32) || P.n_pa >= (int64_t(1) << 31) || P.S >= (int64_t(1) << 31)) return 0;
    switch (P.L) {
#define CUNFFT_CASE(LEN) \
    case LEN: return LEN / LinePlan<LEN>::EPT;
        CUNFFT_POW2_LINES(CUNFFT_CASE)
        CUNFFT_MIXED_LINES(CUNFFT_CASE)
#undef CUNFFT_CASE
    }
    return 0;
}
template <typename T> static bool line_split_ok(const FftPass<T> &P)
{
    switch (P.L) {
#define CUNFFT_CASE(LEN) case LEN:
        CUNFFT_SPLIT_LINES(CUNFFT_CASE)
#undef CUNFFT_CASE
        return true;
    }
    return false;
}
static int line_pitch_of(int L)
{
    switch (L) {
#define CUNFFT_CASE(LEN) \
    case LEN: return line_pitch<LEN>();
        CUNFFT_POW2_LINES(CUNFFT_CASE)
        CUNFFT_MIXED_LINES(CUNFFT_CASE)
#undef CUNFFT_CASE
    }
    return L;
}

// Lines per workgroup (C, a power of two) with the launch's blocks and LDS, from
// P.L, P.S and P.n_pa.
//
// Register-resident pass: as many lines as fill 256 threads (512 from 1024
// points on, where 256 threads hold too few adjacent columns), columns at most
// one 128-byte line wide.  A small grid takes fewer lines per workgroup, down to
// one wavefront (rows) or 64 bytes of a row (columns), until 512 workgroups
// spread over the 256 CUs.  A batch's jobs are many and share a launch of at most 256
// threads per workgroup: always the full number of lines.
//
// Generic pass: rows are packed up to 2048 elements per workgroup; strided
// passes take adjacent columns up to kFftElems elements.
template <typename T> static void pass_shape(FftLaunch<T> &out, FftUse use)
{
    FftPass<T> &P = out.P;
    P.n3 = 0;
    for (int l = P.L; l % 3 == 0; l /= 3) ++P.n3;
    P.tpl = line_tpl<T>(P);
    if (P.split != SPLIT_NONE && !line_split_ok<T>(P)) P.tpl = 0;
    if (use == FFT_GRADIENT && sizeof(T) == 4 && P.n3 > 0) P.tpl = 0;
    const bool batch = use == FFT_BATCH;
    int64_t C;
    if (P.tpl > 0) {
        constexpr int cs = (int)sizeof(cplx_t<T>);
        const int64_t most = batch || P.L < 1024 ? 256 : 512;
        const int64_t wide = P.split == SPLIT_B && P.S == 1 ? P.L2 & -P.L2 : P.S & -P.S;
        const size_t line = (size_t)line_pitch_of(P.L) * cs;
        const bool rows = P.S == 1, side = !rows || P.split == SPLIT_B;   // side by side in memory
        C = std::max<int64_t>(1, prev_pow2_i(most / P.tpl));
        if (side) C = std::min<int64_t>(std::min<int64_t>(C, 128 / cs), wide);
        else C = std::min<int64_t>(C, next_pow2_i(P.n_pa));
        while (C > 1 && C * line > (size_t)kFftLineLds) C >>= 1;
        auto blocks = [&](int64_t c) { return rows ? (P.n_pa + c - 1) / c : P.n_pa * (P.S / c); };
        while (!batch && C > 1 && blocks(C) < 512 && (side ? C * cs > 64 : C * P.tpl > 64)) C >>= 1;
        out.blocks = blocks(C);
        P.ldsL = 0;
        out.lds = (size_t)C * line;
    } else if (P.S == 1) {
        const int64_t target = 2048;
        C = P.L >= target ? 1 : prev_pow2_i(target / P.L);
        C = std::min<int64_t>(C, 64);
        C = std::min<int64_t>(C, next_pow2_i(P.n_pa));
        out.blocks = (P.n_pa + C - 1) / C;
        P.ldsL = P.L;
    } else {
        // adjacent columns: C divides S (the largest power of two in S bounds it)
        const int64_t cdef = sizeof(T) == 8 ? 8 : 16;
        C = std::min<int64_t>(cdef, P.S & -P.S);
        C = std::min<int64_t>(C, std::max<int64_t>(1, prev_pow2_i(kFftElems / P.L)));
        out.blocks = P.n_pa * (P.S / C);
        P.ldsL = C > 1 ? P.L + 1 : P.L;
    }
    P.C = (int)C;
    P.logC = ilog2_i(C);
    // generic pass: lines + twiddles
    if (P.tpl == 0) out.lds = ((size_t)C * P.ldsL + P.L) * sizeof(cplx_t<T>);
}

template <typename T>
static FftPass<T> pass_common(const Geom &ge, const double *roc, const int64_t *rocoff, int t,
                              bool forward, const cplx_t<T> *fhat_in, cplx_t<T> *fhat_out,
                              cplx_t<T> *g)
{
    FftPass<T> P{};
    P.g = g;
    P.fhat_in = fhat_in;
    P.fhat_out = fhat_out;
    P.roc = roc;
    for (int q = 0; q < 3; ++q) {
        P.rocoff[q] = rocoff[q];
        P.n[q] = ge.n[q];
        P.N[q] = ge.N[q];
    }
    P.d = ge.d;
    P.t = t;
    P.Lf = ge.n[t];
    P.So = 1;
    for (int q = t + 1; q < ge.d; ++q) P.So *= ge.n[q];
    P.n_pa = 1;
    for (int q = 0; q < t; ++q) P.n_pa *= ge.N[q];
    P.sign = forward ? -1 : +1;
    P.split = SPLIT_NONE;
    P.dst = nullptr;
    return P;
}

template <typename T>
FftLaunch<T> fft_pass_setup(const Geom &ge, const cplx_t<T> *tw, const double *roc,
                            const int64_t *rocoff, int t, bool forward, const cplx_t<T> *fhat_in,
                            cplx_t<T> *fhat_out, cplx_t<T> *g, FftUse use)
{
    const int d = ge.d;
    FftLaunch<T> out{};
    FftPass<T> &P = out.P;
    P = pass_common<T>(ge, roc, rocoff, t, forward, fhat_in, fhat_out, g);
    P.tw = tw;
    P.L = (int)ge.n[t];
    P.S = P.So;
    P.L1 = 1;
    P.L2 = P.L;
    if (forward)
        P.mode = (t == d - 1) ? FFT_FROM_FHAT : FFT_IN_PRUNED;
    else
        P.mode = (t == d - 1) ? FFT_TO_FHAT : FFT_OUT_PRUNED;
    pass_shape<T>(out, use);
    return out;
}

template <typename T>
int fft_axis_setup(const Geom &ge, const cplx_t<T> *const *tw, const double *roc,
                   const int64_t *rocoff, int t, bool forward, const cplx_t<T> *fhat_in,
                   cplx_t<T> *fhat_out, cplx_t<T> **g, cplx_t<T> **g_other, FftLaunch<T> *out, FftUse use)
{
    const int d = ge.d;
    if (fft_line_ok(ge.n[t])) {
        out[0] = fft_pass_setup<T>(ge, tw[0], roc, rocoff, t, forward, fhat_in, fhat_out, *g, use);
        return 1;
    }
    int64_t L1, L2;
    if (!fft_split(ge.n[t], L1, L2)) throw Error(CUNFFT_ERR_UNSUPPORTED, "no FFT for this axis length");
    if (!*g_other) throw Error(CUNFFT_ERR_STATE, "a split FFT axis needs the second grid buffer");
    // A: the L2-point FFTs over i2 (stride L1 S), in place, with the input
    // pruning (and the roll-off from fhat) of the axis
    FftLaunch<T> &A = out[0];
    A.P = pass_common<T>(ge, roc, rocoff, t, forward, fhat_in, fhat_out, *g);
    A.P.split = SPLIT_A;
    A.P.tw = tw[1];
    A.P.L = (int)L2;
    A.P.S = L1 * A.P.So;
    A.P.L1 = L1;
    A.P.L2 = L2;
    A.P.mode = forward ? ((t == d - 1) ? FFT_FROM_FHAT : FFT_IN_PRUNED) : 0;
    pass_shape<T>(A, use);
    // B: per k2 the L1-point FFT over i1 with the w_Lf twiddles, to the other
    // grid in natural order (or to fhat with the crop and roll-off)
    FftLaunch<T> &B = out[1];
    B.P = pass_common<T>(ge, roc, rocoff, t, forward, fhat_in, fhat_out, *g);
    B.P.split = SPLIT_B;
    B.P.tw = tw[0];
    B.P.L = (int)L1;
    B.P.S = B.P.So;
    B.P.L1 = L1;
    B.P.L2 = L2;
    B.P.n_pa *= L2;
    B.P.mode = forward ? 0 : ((t == d - 1) ? FFT_TO_FHAT : FFT_OUT_PRUNED);
    B.P.dst = B.P.mode == FFT_TO_FHAT ? nullptr : *g_other;
    pass_shape<T>(B, use);
    if (B.P.mode != FFT_TO_FHAT) std::swap(*g, *g_other);
    return 2;
}

template void launch_fft_pass<float>(const FftPass<float> &, int64_t, size_t, hipStream_t);
template void launch_fft_pass<double>(const FftPass<double> &, int64_t, size_t, hipStream_t);
template void launch_fft_batch<float>(const FftPass<float> *, const BlockMap *, uint32_t, size_t,
                                      hipStream_t);
template void launch_fft_batch<double>(const FftPass<double> *, const BlockMap *, uint32_t, size_t,
                                       hipStream_t);
template FftLaunch<float> fft_pass_setup<float>(const Geom &, const float2 *, const double *,
                                                const int64_t *, int, bool, const float2 *,
                                                float2 *, float2 *, FftUse);
template FftLaunch<double> fft_pass_setup<double>(const Geom &, const double2 *, const double *,
                                                  const int64_t *, int, bool, const double2 *,
                                                  double2 *, double2 *, FftUse);
template int fft_axis_setup<float>(const Geom &, const float2 *const *, const double *,
                                   const int64_t *, int, bool, const float2 *, float2 *, float2 **,
                                   float2 **, FftLaunch<float> *, FftUse);
template int fft_axis_setup<double>(const Geom &, const double2 *const *, const double *,
                                    const int64_t *, int, bool, const double2 *, double2 *,
                                    double2 **, double2 **, FftLaunch<double> *, FftUse);

}  // namespace cunfft

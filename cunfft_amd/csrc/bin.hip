// bin.hip -- the node-per-lane tiled gridding kernels.
//
// The reference grids one node per thread straight from global memory: the
// forward through a texture copy of the grid (src/cunfft_kernel.cu:514-1093,
// 1408-1418), the adjoint with two CAS-loop atomics per tap into global memory
// (src/cunfft_kernel.cu:97-130, 608-1197).  Here nodes are first sorted by the
// grid tile holding their window start (binning.hip), and each workgroup then
// owns one tile.  For d >= 2 the plane-tiled kernels of grid_tile.hpp use the
// sorted order; this file holds the node-per-lane tiled kernels used for d = 1
// and under CUNFFT_NODE_LANES:
//   forward  the padded tile (T_t + 2m + 1 cells per axis) is staged in LDS
//            once, and every node of the tile reads its (2m+2)^d taps there;
//   adjoint  the node contributions accumulate in an LDS copy of the padded
//            tile with LDS atomics, and the tile is added to the global grid
//            once, with coalesced global atomics, skipping cells no node
//            reached; a 1D tile in one chunk stores the cells that are its alone.
// The weights, the window start and the FP64 index/fraction split are the ones
// of the node-parallel kernels, so both paths compute the same taps.
#include <hip/amd_detail/amd_hip_unsafe_atomics.h>

#include <algorithm>
#include <type_traits>

#include "bin.hpp"

namespace cunfft {

// Threads per workgroup: 256, and 64 where a 1D launch has very many chunks.  A 1D tile
// is 4 KB, so 32 one-wavefront workgroups fit a CU, and none of a chunk's wavefronts
// waits for another to stage or flush the tile; but a wavefront alone takes a chunk's 256
// nodes 64 after 64, so it needs enough workgroups beside it and few nodes per tile.
// Forward / adjoint in us, 64 against 256 threads (m = 4):
//   FP64, 32768 tiles of 128 nodes   gather 127 / 190, scatter with its clears 146 / 230
//   FP64, 8192 tiles   48 nodes a tile 53 / 55, 60 / 78    200 nodes 75 / 73, 84 / 91
//   FP64, 2048 tiles   48 nodes        32 / 32, 35 / 37   1000 nodes 64 / 63, 101 / 88
//   FP64,  512 tiles  200 nodes        26 / 21, 29 / 24   1000 nodes 35 / 31, 43 / 37
//   FP64,    4 tiles 4000 nodes        15 / 11, 18 / 14   (FP32 the same, smaller)
//   FP64,    8 tiles 125000 nodes      30 / 31, 87 / 99   32 tiles 33000 nodes 40 / 40, 79 / 82
// Hence 64 for plans from 2048 tiles on with at most 256 nodes each, and for the sums of
// very many chunks (2^19 nodes) into few tiles (2^15 nodes each).  A batch deals the
// chunks of all its jobs: 64 from 8192 chunks on (36900 chunks of 256 nodes FP32 94 / 111,
// 198 / 229; 8192 of 80 nodes 53 / 55, 70 / 77; 48 chunks 18 / 17, 23 / 21).
constexpr int kTileThreads = 256, kTileThreadsNarrow = 64;
static bool narrow_groups(const Binning &b)
{
    if (b.d != 1) return false;
    return b.ntiles >= 2048 ? b.M <= 256 * b.ntiles : b.M >= (int64_t(1) << 19) && b.M >= b.ntiles << 15;
}
static bool narrow_groups(int d, uint32_t batch_chunks) { return d == 1 && batch_chunks >= 8192; }
constexpr int kMaxTileBytes = 120 * 1024;

template <int D, int W> struct Pad {
    static constexpr int P0 = TileShape<D>::T[0] + W - 1;
    static constexpr int P1 = D >= 2 ? TileShape<D>::T[1] + W - 1 : 1;
    static constexpr int P2 = D >= 3 ? TileShape<D>::T[2] + W - 1 : 1;
    static constexpr int PT = P0 * P1 * P2;
};

template <typename T, int D, int W> constexpr bool tile_fits()
{
    return (size_t)Pad<D, W>::PT * 2 * sizeof(T) <= (size_t)kMaxTileBytes;
}

// ------------------------------------------------------ tile helpers ----
template <int D>
__device__ __forceinline__ void tile_origin(uint32_t tile, const BinGeom &bg, int64_t (&o)[3])
{
    uint32_t rem = tile;
#pragma unroll
    for (int t = D - 1; t >= 0; --t) {
        const uint32_t tc = rem % (uint32_t)bg.nt[t];
        rem /= (uint32_t)bg.nt[t];
        o[t] = (int64_t)tc << bg.logT[t];
    }
#pragma unroll
    for (int t = D; t < 3; ++t) o[t] = 0;
}

// Global grid offset of padded-tile cell idx.
template <int D, int W>
__device__ __forceinline__ int64_t tile_cell(int idx, const int64_t (&o)[3], const Geom &ge)
{
    using PD = Pad<D, W>;
    const int p0 = idx / (PD::P1 * PD::P2);
    const int r = idx - p0 * (PD::P1 * PD::P2);
    const int p1 = r / PD::P2;
    const int p2 = r - p1 * PD::P2;
    const int64_t c0 = wrap_hi(o[0] + p0, ge.n[0]);
    if constexpr (D == 1) return c0;
    const int64_t c1 = wrap_hi(o[1] + p1, ge.n[1]);
    if constexpr (D == 2) return c0 * ge.n[1] + c1;
    const int64_t c2 = wrap_hi(o[2] + p2, ge.n[2]);
    return (c0 * ge.n[1] + c1) * ge.n[2] + c2;
}

// Window weights of the node at sorted position s and its LDS base offset.
template <typename T, int D, int W>
__device__ __forceinline__ int node_local(const double *__restrict__ xs, uint32_t s,
                                          const int64_t (&o)[3], const Geom &ge, T (&w)[D][W])
{
    using PD = Pad<D, W>;
    constexpr int stride[3] = {PD::P1 * PD::P2, PD::P2, 1};
    int base = 0;
#pragma unroll
    for (int t = 0; t < D; ++t) {
        double c;
        int lo = (int)(window_cell(xs[(int64_t)s * D + t], ge.n[t], ge.m, c) - o[t]);
        lo = lo < 0 ? 0 : (lo >= TileShape<D>::T[t] ? TileShape<D>::T[t] - 1 : lo);
        window_weights<T, W>(c, ge, t, w[t]);
        base += lo * stride[t];
    }
    return base;
}

// --------------------------------------------------------- tiled gather --
template <typename T, int D, int W, int NT>
__device__ __forceinline__ void gather_tiled(const cplx_t<T> *__restrict__ g,
                                             const double *__restrict__ xs,
                                             const uint32_t *__restrict__ perm, const Chunk ch,
                                             cplx_t<T> *__restrict__ f, const Geom &ge,
                                             const BinGeom &bg)
{
    using PD = Pad<D, W>;
    __shared__ cplx_t<T> tile[PD::PT];
    int64_t o[3];
    tile_origin<D>(ch.tile, bg, o);
    // 8 loads in flight per thread before the LDS stores (unconditional: a
    // lane past the end rewrites the last cell with its own value)
    for (int i0 = threadIdx.x; i0 < PD::PT; i0 += 8 * NT) {
        cplx_t<T> v[8];
        int at[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            at[u] = i0 + u * NT < PD::PT ? i0 + u * NT : PD::PT - 1;
            v[u] = g[tile_cell<D, W>(at[u], o, ge)];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) tile[at[u]] = v[u];
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < ch.count; i += NT) {
        const uint32_t s = ch.start + i;
        T w[D][W];
        const int base = node_local<T, D, W>(xs, s, o, ge, w);
        const cplx_t<T> *tb = tile + base;
        T sr = 0, si = 0;
        if constexpr (D == 1) {
#pragma unroll
            for (int a = 0; a < W; ++a) {
                const cplx_t<T> v = tb[a];
                sr += v.x * w[0][a];
                si += v.y * w[0][a];
            }
        } else if constexpr (D == 2) {
#pragma unroll
            for (int a = 0; a < W; ++a) {
                T r1 = 0, i1 = 0;
#pragma unroll
                for (int c = 0; c < W; ++c) {
                    const cplx_t<T> v = tb[a * PD::P1 + c];
                    r1 += v.x * w[1][c];
                    i1 += v.y * w[1][c];
                }
                sr += r1 * w[0][a];
                si += i1 * w[0][a];
            }
        } else {
#pragma unroll
            for (int a = 0; a < W; ++a) {
                T r1 = 0, i1 = 0;
#pragma unroll
                for (int c = 0; c < W; ++c) {
                    T r2 = 0, i2 = 0;
#pragma unroll
                    for (int e = 0; e < W; ++e) {
                        const cplx_t<T> v = tb[(a * PD::P1 + c) * PD::P2 + e];
                        r2 += v.x * w[2][e];
                        i2 += v.y * w[2][e];
                    }
                    r1 += r2 * w[1][c];
                    i1 += i2 * w[1][c];
                }
                sr += r1 * w[0][a];
                si += i1 * w[0][a];
            }
        }
        f[perm[s]] = cmake<T>(sr, si);
    }
}

template <typename T, int D, int W, int NT>
__global__ __launch_bounds__(NT) void k_gather_tiled(
    const cplx_t<T> *__restrict__ g, const double *__restrict__ xs, const uint32_t *__restrict__ perm,
    const Chunk *__restrict__ chunks, const uint32_t *__restrict__ n_chunks, cplx_t<T> *__restrict__ f,
    Geom ge, BinGeom bg)
{
    if (blockIdx.x >= n_chunks[0]) return;
    gather_tiled<T, D, W, NT>(g, xs, perm, chunks[blockIdx.x], f, ge, bg);
}

template <typename T, int D, int W, int NT>
__global__ __launch_bounds__(NT) void k_gather_tiled_batch(
    const GridJob<T> *__restrict__ jobs, const BlockMap *__restrict__ map)
{
    const BlockMap bm = map[blockIdx.x];
    const GridJob<T> &J = jobs[bm.job];
    gather_tiled<T, D, W, NT>(J.g, J.xs, J.perm, J.chunks[bm.blk], J.f_out, J.ge, J.bg);
}

// -------------------------------------------------------- tiled scatter --
template <typename T>
__device__ __forceinline__ void lds_add(T *p, T v)
{
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

template <typename T, typename A, int D, int W, int NT>
__device__ __forceinline__ void scatter_tiled(const double *__restrict__ xs,
                                              const uint32_t *__restrict__ perm,
                                              const cplx_t<T> *__restrict__ f, const Chunk ch,
                                              cplx_t<T> *__restrict__ g, const Geom &ge,
                                              const BinGeom &bg, bool own = false)
{
    using PD = Pad<D, W>;
    __shared__ A acc_re[PD::PT];
    __shared__ A acc_im[PD::PT];
    int64_t o[3];
    tile_origin<D>(ch.tile, bg, o);
    for (int idx = threadIdx.x; idx < PD::PT; idx += NT) {
        acc_re[idx] = 0;
        acc_im[idx] = 0;
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < ch.count; i += NT) {
        const uint32_t s = ch.start + i;
        T w[D][W];
        const int base = node_local<T, D, W>(xs, s, o, ge, w);
        const cplx_t<T> fj = f[perm[s]];
        A *re = acc_re + base;
        A *im = acc_im + base;
        if constexpr (D == 1) {
#pragma unroll
            for (int a = 0; a < W; ++a) {
                lds_add<A>(re + a, (A)(fj.x * w[0][a]));
                lds_add<A>(im + a, (A)(fj.y * w[0][a]));
            }
        } else if constexpr (D == 2) {
#pragma unroll
            for (int a = 0; a < W; ++a) {
                const T fr = fj.x * w[0][a], fi = fj.y * w[0][a];
#pragma unroll
                for (int c = 0; c < W; ++c) {
                    lds_add<A>(re + a * PD::P1 + c, (A)(fr * w[1][c]));
                    lds_add<A>(im + a * PD::P1 + c, (A)(fi * w[1][c]));
                }
            }
        } else {
#pragma unroll
            for (int a = 0; a < W; ++a) {
                const T fr0 = fj.x * w[0][a], fi0 = fj.y * w[0][a];
#pragma unroll
                for (int c = 0; c < W; ++c) {
                    const T fr = fr0 * w[1][c], fi = fi0 * w[1][c];
#pragma unroll
                    for (int e = 0; e < W; ++e) {
                        const int off = (a * PD::P1 + c) * PD::P2 + e;
                        lds_add<A>(re + off, (A)(fr * w[2][e]));
                        lds_add<A>(im + off, (A)(fi * w[2][e]));
                    }
                }
            }
        }
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < PD::PT; idx += NT) {
        const A vr = acc_re[idx], vi = acc_im[idx];
        if (D == 1 && own && idx >= W - 1 && idx < TileShape<D>::T[0]) {
            g[o[0] + idx] = cmake<T>((T)vr, (T)vi);   // no other tile reaches these cells
        } else if (vr != (A)0 || vi != (A)0) {
            cplx_t<T> *p = g + tile_cell<D, W>(idx, o, ge);
            unsafeAtomicAdd(&p->x, (T)vr);
            unsafeAtomicAdd(&p->y, (T)vi);
        }
    }
}

template <typename T, typename A, int D, int W, int NT>
__global__ __launch_bounds__(NT) void k_scatter_tiled(
    const double *__restrict__ xs, const uint32_t *__restrict__ perm, const cplx_t<T> *__restrict__ f,
    const Chunk *__restrict__ chunks, const uint32_t *__restrict__ n_chunks,
    const uint32_t *__restrict__ tile_count, cplx_t<T> *__restrict__ g, Geom ge, BinGeom bg)
{
    if (blockIdx.x >= n_chunks[0]) return;
    const Chunk ch = chunks[blockIdx.x];
    scatter_tiled<T, A, D, W, NT>(xs, perm, f, ch, g, ge, bg,
                              D == 1 && chunks_of(tile_count[ch.tile], bg.chunk_base) == 1);
}

// What the 1D scatter adds to: of a tile whose nodes are one chunk the cells that the
// tile before it reaches too (the chunk's workgroup stores the others), of any other
// tile all cells.  One wavefront per tile.
template <typename T, int W>
__global__ __launch_bounds__(256) void k_zero_shared(const uint32_t *__restrict__ tile_count, BinGeom bg,
                                                     cplx_t<T> *__restrict__ g)
{
    const int64_t tile = (int64_t)blockIdx.x * 4 + threadIdx.x / 64;
    if (tile >= bg.ntiles) return;
    const int n = chunks_of(tile_count[tile], bg.chunk_base) == 1 ? W - 1 : TileShape<1>::T[0];
    for (int i = threadIdx.x & 63; i < n; i += 64) g[tile * TileShape<1>::T[0] + i] = cmake<T>(0, 0);
}

template <typename T, typename A, int D, int W, int NT>
__global__ __launch_bounds__(NT) void k_scatter_tiled_batch(
    const GridJob<T> *__restrict__ jobs, const BlockMap *__restrict__ map)
{
    const BlockMap bm = map[blockIdx.x];
    const GridJob<T> &J = jobs[bm.job];
    scatter_tiled<T, A, D, W, NT>(J.xs, J.perm, J.f_in, J.chunks[bm.blk], J.g, J.ge, J.bg);
}

// Grid <- 0 for the node-lane scatter of every job, 1024 cells per block.
template <typename T>
__global__ __launch_bounds__(256) void k_zero_batch(const GridJob<T> *__restrict__ jobs,
                                                    const BlockMap *__restrict__ map)
{
    const BlockMap bm = map[blockIdx.x];
    const GridJob<T> &J = jobs[bm.job];
    const int64_t c0 = (int64_t)bm.blk * 1024 + threadIdx.x;
#pragma unroll
    for (int k = 0; k < 4; ++k)
        if (c0 + 256 * k < J.n_total) J.g[c0 + 256 * k] = cmake<T>(0, 0);
}

// ------------------------------------------------------------ dispatch --
// go(threads per workgroup), the number as a constant
template <int D, typename F> static void lane_launch(bool narrow, F &go)
{
    if constexpr (D == 1)
        if (narrow) return go(std::integral_constant<int, kTileThreadsNarrow>{});
    go(std::integral_constant<int, kTileThreads>{});
}

template <typename T, int D, int W>
static void launch_gather_lanes(const Geom &ge, const Binning &b, const cplx_t<T> *g, cplx_t<T> *f,
                                hipStream_t s)
{
    if constexpr (tile_fits<T, D, W>()) {
        auto go = [&](auto nt) {
            constexpr int NT = decltype(nt)::value;
            k_gather_tiled<T, D, W, NT><<<(unsigned)b.max_chunks, NT, 0, s>>>(
                g, b.xs, b.perm, b.chunks, b.n_chunks, f, ge, bin_geom(b));
        };
        lane_launch<D>(narrow_groups(b), go);
    } else {
        throw Error(CUNFFT_ERR_UNSUPPORTED, "tile does not fit in LDS");
    }
}

template <typename T, int D, int W>
static void launch_scatter_lanes(const Geom &ge, const Binning &b, const cplx_t<T> *f,
                                 cplx_t<T> *g, hipStream_t s)
{
    if constexpr (tile_fits<T, D, W>()) {
        if constexpr (D == 1)
            k_zero_shared<T, W><<<(unsigned)((b.ntiles + 3) / 4), 256, 0, s>>>(b.tile_count, bin_geom(b), g);
        else
            launch_zero<T>(g, ge.n[0] * ge.n[1] * ge.n[2], s);
        auto go = [&](auto nt) {
            constexpr int NT = decltype(nt)::value;
            k_scatter_tiled<T, double, D, W, NT><<<(unsigned)b.max_chunks, NT, 0, s>>>(
                b.xs, b.perm, f, b.chunks, b.n_chunks, b.tile_count, g, ge, bin_geom(b));
        };
        lane_launch<D>(narrow_groups(b), go);
    } else {
        throw Error(CUNFFT_ERR_UNSUPPORTED, "tile does not fit in LDS");
    }
}

#define CUNFFT_TILED_W(FN, D)                                             \
    switch (ge.W) {                                                       \
    case 4: FN<T, D, 4>(ge, b, a0, a1, s); break;                         \
    case 6: FN<T, D, 6>(ge, b, a0, a1, s); break;                         \
    case 8: FN<T, D, 8>(ge, b, a0, a1, s); break;                         \
    case 10: FN<T, D, 10>(ge, b, a0, a1, s); break;                       \
    case 12: FN<T, D, 12>(ge, b, a0, a1, s); break;                       \
    case 14: FN<T, D, 14>(ge, b, a0, a1, s); break;                       \
    case 16: if constexpr (D < 3) FN<T, D, 16>(ge, b, a0, a1, s); break;  \
    case 18: if constexpr (D < 3) FN<T, D, 18>(ge, b, a0, a1, s); break;  \
    default: throw Error(CUNFFT_ERR_UNSUPPORTED, "tiled gridding needs m <= 8"); \
    }

template <typename T>
void launch_gather_binned(const Geom &ge, const Binning &b, const cplx_t<T> *g, const double *x,
                          cplx_t<T> *f, hipStream_t s)
{
    if (!b.usable || !b.built) {
        launch_gather_plain<T>(ge, g, x, f, s);
        return;
    }
    if (b.planes()) {
        launch_tile_gather<T>(ge, b, g, f, s);
        return;
    }
    const cplx_t<T> *a0 = g;
    cplx_t<T> *a1 = f;
    switch (ge.d) {
    case 1: CUNFFT_TILED_W(launch_gather_lanes, 1) break;
    case 2: CUNFFT_TILED_W(launch_gather_lanes, 2) break;
    default: CUNFFT_TILED_W(launch_gather_lanes, 3) break;
    }
    CUNFFT_HIP(hipGetLastError());
}

template <typename T>
bool launch_scatter_binned(const Geom &ge, const Binning &b, const double *x, const cplx_t<T> *f,
                           cplx_t<T> *g, hipStream_t s, hipEvent_t mid)
{
    const int64_t nt = ge.n[0] * ge.n[1] * ge.n[2];
    if (!b.usable || !b.built) {
        launch_zero<T>(g, nt, s);
        launch_scatter_atomic<T>(ge, x, f, g, s);
        return false;
    }
    if (b.planes()) {
        launch_tile_spread<T>(ge, b, f, g, s, mid);
        return mid != nullptr;
    }
    const cplx_t<T> *a0 = f;
    cplx_t<T> *a1 = g;
    switch (ge.d) {
    case 1: CUNFFT_TILED_W(launch_scatter_lanes, 1) break;
    case 2: CUNFFT_TILED_W(launch_scatter_lanes, 2) break;
    default: CUNFFT_TILED_W(launch_scatter_lanes, 3) break;
    }
    CUNFFT_HIP(hipGetLastError());
    return false;
}

// ------------------------------------------------------------ batches --
int64_t tile_fold_blocks(int d, int variant, int64_t ntiles, int elem_bytes)
{
    int64_t T[3];
    tile_shape(d, variant, T);
    if (d >= 2 && elem_bytes == 4) {   // column-segment fold: kFoldSegBytes of a core column per thread
        const int64_t tpt = T[0] * (d == 3 ? T[1] : 1) * (T[d - 1] * 2 * elem_bytes / kFoldSegBytes);
        return tpt <= 256 ? (ntiles + 256 / tpt - 1) / (256 / tpt) : ntiles * (tpt / 256);
    }
    const int64_t core = T[0] * T[1] * T[2];
    return ntiles * (core >= 512 ? core / 512 : 1);
}

template <typename T, int D, int W>
static void launch_lanes_batch(BatchStage st, const GridJob<T> *jobs, const BlockMap *map,
                               uint32_t nblk, hipStream_t s)
{
    if constexpr (tile_fits<T, D, W>()) {
        auto go = [&](auto nt) {
            constexpr int NT = decltype(nt)::value;
            if (st == BS_GATHER)
                k_gather_tiled_batch<T, D, W, NT><<<nblk, NT, 0, s>>>(jobs, map);
            else
                k_scatter_tiled_batch<T, double, D, W, NT><<<nblk, NT, 0, s>>>(jobs, map);
        };
        lane_launch<D>(narrow_groups(D, nblk), go);
    } else {
        throw Error(CUNFFT_ERR_UNSUPPORTED, "tile does not fit in LDS");
    }
}

template <typename T>
void launch_batch_stage(BatchStage st, const GridJob<T> *jobs, const BlockMap *map, uint32_t nblk,
                        int d, int W, int config, hipStream_t s)
{
    if (nblk == 0) return;
    if (st == BS_ZERO) {
        k_zero_batch<T><<<nblk, 256, 0, s>>>(jobs, map);
    } else if ((st == BS_GATHER && (d == 1 || config == kTileVariants)) || st == BS_SCATTER_LANES) {
        const BatchStage a0 = st;
        const BlockMap *a1 = map;
#define CUNFFT_LANES_W(D)                                                            \
    switch (W) {                                                                     \
    case 4: launch_lanes_batch<T, D, 4>(a0, jobs, a1, nblk, s); break;               \
    case 6: launch_lanes_batch<T, D, 6>(a0, jobs, a1, nblk, s); break;               \
    case 8: launch_lanes_batch<T, D, 8>(a0, jobs, a1, nblk, s); break;               \
    case 10: launch_lanes_batch<T, D, 10>(a0, jobs, a1, nblk, s); break;             \
    case 12: launch_lanes_batch<T, D, 12>(a0, jobs, a1, nblk, s); break;             \
    case 14: launch_lanes_batch<T, D, 14>(a0, jobs, a1, nblk, s); break;             \
    case 16: if constexpr (D < 3) launch_lanes_batch<T, D, 16>(a0, jobs, a1, nblk, s); break; \
    case 18: if constexpr (D < 3) launch_lanes_batch<T, D, 18>(a0, jobs, a1, nblk, s); break; \
    default: throw Error(CUNFFT_ERR_UNSUPPORTED, "tiled gridding needs m <= 8");     \
    }
        switch (d) {
        case 1: CUNFFT_LANES_W(1) break;
        case 2: CUNFFT_LANES_W(2) break;
        default: CUNFFT_LANES_W(3) break;
        }
#undef CUNFFT_LANES_W
    } else {
        launch_tile_batch<T>(st, jobs, map, nblk, d, W, config, s);
        return;
    }
    CUNFFT_HIP(hipGetLastError());
}

template void launch_batch_stage<float>(BatchStage, const GridJob<float> *, const BlockMap *,
                                        uint32_t, int, int, int, hipStream_t);
template void launch_batch_stage<double>(BatchStage, const GridJob<double> *, const BlockMap *,
                                         uint32_t, int, int, int, hipStream_t);

template void launch_gather_binned<float>(const Geom &, const Binning &, const float2 *,
                                          const double *, float2 *, hipStream_t);
template void launch_gather_binned<double>(const Geom &, const Binning &, const double2 *,
                                           const double *, double2 *, hipStream_t);
template bool launch_scatter_binned<float>(const Geom &, const Binning &, const double *,
                                           const float2 *, float2 *, hipStream_t, hipEvent_t);
template bool launch_scatter_binned<double>(const Geom &, const Binning &, const double *,
                                            const double2 *, double2 *, hipStream_t, hipEvent_t);

}  // namespace cunfft

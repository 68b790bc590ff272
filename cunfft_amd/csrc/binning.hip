// binning.hip -- nodes sorted by grid tile on the device.
//
// The reference grids its nodes in the caller's order (one thread per node,
// src/cunfft_kernel.cu:514-1197).  Here they are first sorted by the grid tile
// that holds their window start, so that one workgroup can grid a tile's nodes
// against LDS.  A binning is a short sequence of small kernels: with 10^4 .. 10^5
// nodes every one of them costs its launch and one or two memory round trips, not
// its bytes.  So the passes are few and no thread waits for one load before it
// asks for the next:
//
//   k_bin_keys     sort key and window descriptor per node, and the first radix
//                  digit's counts per block
//   k_rs_scatter   stable radix pass; the block sums the digit counts of the
//                  blocks before it itself (up to kRsDirect blocks, else
//                  k_rs_scan has done it), and holds its items in registers
//   k_rs_hist      digit counts for each further pass
//   k_bin_place    sorted descriptors; first position of every tile
//   k_bin_chunks   tile counts and the chunk list; the blocks sum the chunk
//                  counts before them (up to kChunkDirect blocks, else
//                  k_bin_chunk_part has done it)
//
// 8 launches for 65536 nodes in 2D where separate scans, a fill and two boundary
// kernels took 21.  Measured, before -> now: 2D, 65536 nodes FP64 131 -> 38 us; 2D,
// 2^18 nodes 130 -> 53 us; 3D, 400009 nodes FP32 130 -> 68 us; 3D, 2^21 nodes FP32
// 276 -> 222 us (three passes over the pairs: the scattered 4-byte writes).
#include <algorithm>

#include "bin.hpp"

namespace cunfft {

constexpr int kLaneTileBytes = 120 * 1024;   // LDS tile of the node-lane kernels, at most

BinGeom bin_geom(const Binning &b)
{
    BinGeom g{};
    g.d = b.d;
    for (int t = 0; t < 3; ++t) {
        int l = 0;
        while ((int64_t(1) << l) < b.T[t]) ++l;
        g.logT[t] = l;
        g.nt[t] = b.nt[t];
    }
    g.ntiles = b.ntiles;
    g.sub_shift = b.elem_bytes == 4 ? 1 : 0;
    g.sub_sort = b.sub_sort;
    g.chunk_base = b.chunk_base;
    g.seg_shift = b.seg_shift;
    return g;
}

// ----------------------------------------------------------- block helpers --
// Exclusive scan of one value per thread over a workgroup of NT threads; the
// total in every thread.  ws: NT / 64 words of LDS, free again after the call's
// second barrier at the next call's first.
template <int NT>
__device__ __forceinline__ uint32_t block_exscan(uint32_t v, uint32_t *ws, uint32_t &total)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t a = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t u = __shfl_up(a, off, 64);
        if (lane >= off) a += u;
    }
    if (lane == 63) ws[wave] = a;
    __syncthreads();
    uint32_t before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) {
        const uint32_t s = ws[w];
        before += w < wave ? s : 0u;
        all += s;
    }
    __syncthreads();
    total = all;
    return before + a - v;
}

// ------------------------------------------------------------- radix sort --
// Stable LSD radix sort of (composite key, node index) pairs.  Block b holds the
// items [b IB, (b + 1) IB), IB = 256 IPT; hist row b its digit counts.  No atomic
// decides a position, so the result is the same on every run.
constexpr int kRsThreads = 256;
constexpr int kRsDigits = 256;
constexpr int kRsDirect = 64;      // hist rows a scatter block sums itself
// Items per thread: 4 keep 2^16 nodes within kRsDirect blocks and spread up to
// 2^20 over the CUs (2^18 nodes in 64 blocks of 16 items per thread: the key pass
// and each scatter took 14 us, in 256 blocks 6 us and 5 us more for k_rs_scan);
// past that 16, which halve the counts' traffic.
static int rs_ipt(int64_t M) { return M <= (int64_t(1) << 20) ? 4 : 16; }
static int64_t rs_blocks(int64_t M)
{
    const int64_t ib = (int64_t)kRsThreads * rs_ipt(M);
    return (M + ib - 1) / ib;
}

// What the key kernel needs of the geometry.
struct KeyGeom {
    int64_t n[3];
    uint32_t nt[3];
    int logT[3];
    int m;
    int sub_shift;
    uint32_t sub_range;   // 1: the tile alone
};

// Composite key of every node (its tile times sub_range plus its sub_key within
// the tile), its window descriptor by node index (plane-tiled kernels; desc_j
// NULL otherwise) and the block's counts of digit key & mask.  The descriptor is
// the FP64 index/fraction split of window_cell with lo_t the window start
// relative to the tile origin, in [0, T_t) by construction of the key.
template <typename T, int D, int IPT>
__global__ __launch_bounds__(kRsThreads) void k_bin_keys(const double *__restrict__ x,
                                                         uint32_t *__restrict__ keys,
                                                         NodeDesc<T> *__restrict__ desc_j, int64_t M,
                                                         KeyGeom kg, uint32_t mask,
                                                         uint32_t *__restrict__ hist)
{
    __shared__ uint32_t h[kRsDigits];
    const int tid = threadIdx.x;
    h[tid] = 0;
    __syncthreads();
    const int64_t i0 = (int64_t)blockIdx.x * (kRsThreads * IPT) + tid;
    constexpr int U = IPT < 4 ? IPT : 4;
    for (int k0 = 0; k0 < IPT; k0 += U) {
        double xv[U][D];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t j = i0 + (int64_t)(k0 + u) * kRsThreads;
            const double *p = x + (j < M ? j : 0) * D;
#pragma unroll
            for (int t = 0; t < D; ++t) xv[u][t] = p[t];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t j = i0 + (int64_t)(k0 + u) * kRsThreads;
            uint32_t tile = 0, loc = 0, lo[3] = {0, 0, 0};
            NodeDesc<T> nd{};
#pragma unroll
            for (int t = 0; t < D; ++t) {
                double c;
                const int64_t w = window_cell(xv[u][t], kg.n[t], kg.m, c);
                const uint32_t w32 = (uint32_t)w, tc = w32 >> kg.logT[t];   // w < n_t <= 2^24
                lo[t] = w32 - (tc << kg.logT[t]);
                loc |= lo[t] << (8 * t);
                nd.f[t] = (T)(c - (double)kg.m);
                tile = tile * kg.nt[t] + tc;
            }
            const uint32_t key =
                kg.sub_range > 1 ? tile * kg.sub_range + sub_key(D, lo, kg.logT, kg.sub_shift) : tile;
            if (j < M) {
                keys[j] = key;
                if (desc_j) {
                    nd.loc = loc;
                    desc_j[j] = nd;
                }
                atomicAdd(&h[key & mask], 1u);
            }
        }
    }
    __syncthreads();
    hist[(size_t)blockIdx.x * kRsDigits + tid] = h[tid];
}

template <int IPT>
__global__ __launch_bounds__(kRsThreads) void k_rs_hist(const uint32_t *__restrict__ keys, int64_t M,
                                                        int shift, uint32_t mask,
                                                        uint32_t *__restrict__ hist)
{
    __shared__ uint32_t h[kRsDigits];
    const int tid = threadIdx.x;
    h[tid] = 0;
    const int64_t i0 = (int64_t)blockIdx.x * (kRsThreads * IPT) + tid;
    uint32_t key[IPT];
#pragma unroll
    for (int k = 0; k < IPT; ++k) {
        const int64_t i = i0 + (int64_t)k * kRsThreads;
        key[k] = keys[i < M ? i : M - 1];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < IPT; ++k)
        if (i0 + (int64_t)k * kRsThreads < M) atomicAdd(&h[(key[k] >> shift) & mask], 1u);
    __syncthreads();
    hist[(size_t)blockIdx.x * kRsDigits + tid] = h[tid];
}

// More than kRsDirect blocks: the counts of each digit become their exclusive
// prefix over the blocks, and the digit's total goes to tot.  16 digits per
// workgroup, 64 runs of rows each.
__global__ __launch_bounds__(1024) void k_rs_scan(uint32_t *__restrict__ hist, uint32_t nblk,
                                                  uint32_t *__restrict__ tot)
{
    __shared__ uint32_t part[64][17];
    const int dl = threadIdx.x & 15, run = threadIdx.x >> 4;
    const uint32_t per = (nblk + 63) / 64;
    const uint32_t r0 = run * per, r1 = r0 + per < nblk ? r0 + per : nblk;
    uint32_t *p = hist + blockIdx.x * 16 + dl;
    uint32_t sum = 0;
#pragma unroll 8
    for (uint32_t r = r0; r < r1; ++r) sum += p[(size_t)r * kRsDigits];
    part[run][dl] = sum;
    __syncthreads();
    uint32_t before = 0;
    for (int k = 0; k < run; ++k) before += part[k][dl];
    if (run == 63) tot[blockIdx.x * 16 + dl] = before + sum;
    for (uint32_t r = r0; r < r1; ++r) {
        const uint32_t v = p[(size_t)r * kRsDigits];
        p[(size_t)r * kRsDigits] = before;
        before += v;
    }
}

// One radix pass.  Wavefront w takes the items [w 64 IPT, (w + 1) 64 IPT) of the
// block, 64 at a time; an item's rank among the earlier ones of its digit is its
// wavefront's running count plus the number of lower lanes holding the digit
// (ballots on the digit's bits).  vals_in NULL: the values are the item indices.
// DIRECT: hist holds the counts, else k_rs_scan's prefixes with the totals in tot.
template <int IPT, bool DIRECT>
__global__ __launch_bounds__(kRsThreads) void k_rs_scatter(
    const uint32_t *__restrict__ keys_in, const uint32_t *__restrict__ vals_in, int64_t M, int shift,
    int bits, const uint32_t *__restrict__ hist, const uint32_t *__restrict__ tot, uint32_t nblk,
    uint32_t *__restrict__ keys_out, uint32_t *__restrict__ vals_out)
{
    constexpr int NWV = kRsThreads / 64;
    __shared__ uint32_t cnt[NWV][kRsDigits];
    __shared__ uint32_t ws[NWV];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t mask = (1u << bits) - 1u;
    const int64_t i0 = (int64_t)blockIdx.x * (kRsThreads * IPT) + wave * (64 * IPT) + lane;
    uint32_t key[IPT], val[IPT], rank[IPT];
#pragma unroll
    for (int k = 0; k < IPT; ++k) {
        const int64_t i = i0 + 64 * k;
        key[k] = keys_in[i < M ? i : M - 1];
        val[k] = vals_in ? vals_in[i < M ? i : M - 1] : (uint32_t)i;
    }
    // digit tid: items in the blocks before this one, and in all
    uint32_t mine = 0, total = 0;
    if constexpr (DIRECT) {
#pragma unroll 16
        for (uint32_t r = 0; r < nblk; ++r) {
            const uint32_t v = hist[(size_t)r * kRsDigits + tid];
            total += v;
            mine += r < blockIdx.x ? v : 0u;
        }
    } else {
        mine = hist[(size_t)blockIdx.x * kRsDigits + tid];
        total = tot[tid];
    }
#pragma unroll
    for (int w = 0; w < NWV; ++w) cnt[w][tid] = 0;
    uint32_t all;
    const uint32_t base = block_exscan<kRsThreads>(total, ws, all) + mine;   // (barriers inside)
    const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
    for (int k = 0; k < IPT; ++k) {
        const bool valid = i0 + 64 * k < M;
        const uint32_t dg = (key[k] >> shift) & mask;
        uint64_t peers = __ballot(valid);
        for (int bit = 0; bit < bits; ++bit) {
            const uint64_t ones = __ballot((dg >> bit) & 1u);
            peers &= ((dg >> bit) & 1u) ? ones : ~ones;
        }
        const uint32_t lower = (uint32_t)__popcll(peers & below);
        const uint32_t run = cnt[wave][dg];
        rank[k] = run + lower;
        // the digit's first lane moves the wavefront's running count on; a
        // wavefront's LDS accesses execute in order (compiler barriers only)
        __asm__ volatile("" ::: "memory");
        if (valid && lower == 0) cnt[wave][dg] = run + (uint32_t)__popcll(peers);
        __asm__ volatile("" ::: "memory");
    }
    __syncthreads();
    uint32_t at = base;
#pragma unroll
    for (int w = 0; w < NWV; ++w) {
        const uint32_t c = cnt[w][tid];
        cnt[w][tid] = at;
        at += c;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < IPT; ++k) {
        if (i0 + 64 * k >= M) continue;
        const uint32_t pos = cnt[wave][(key[k] >> shift) & mask] + rank[k];
        keys_out[pos] = key[k];
        vals_out[pos] = val[k];
    }
}

// ---------------------------------------------------------- tiles, chunks --
// Sorted position s: the node's descriptor (or coordinates), and the first
// sorted position of its tile and of the empty tiles before it (after it, at the
// last position).  Long runs of empty tiles are filled by the whole wavefront.
template <typename T>
__global__ __launch_bounds__(256) void k_bin_place(const uint32_t *__restrict__ skeys,
                                                   const uint32_t *__restrict__ perm, int64_t M,
                                                   int sub_bits, uint32_t ntiles,
                                                   const NodeDesc<T> *__restrict__ desc_j,
                                                   NodeDesc<T> *__restrict__ desc,
                                                   const double *__restrict__ x, double *__restrict__ xs,
                                                   int d, uint32_t *__restrict__ first)
{
    const int64_t s = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int lane = threadIdx.x & 63;
    // empty run [u0, u1) in front of (and with) the tile of s, its first position
    uint32_t u0 = 0, u1 = 0;
    if (s < M) {
        const uint32_t t = skeys[s] >> sub_bits;
        u0 = s == 0 ? 0u : (skeys[s - 1] >> sub_bits) + 1u;
        u1 = t + 1u;
        const int64_t j = perm[s];
        if (desc_j) {
            desc[s] = desc_j[j];
        } else {
            for (int q = 0; q < d; ++q) xs[s * d + q] = x[j * d + q];
        }
        for (uint32_t u = u0; u < u1 && u < u0 + 4u; ++u) first[u] = (uint32_t)s;
        u0 += 4u;
    }
    auto fill = [&](bool on, uint32_t a, uint32_t b, uint32_t v) {
        for (uint64_t m = __ballot(on); m; m &= m - 1) {
            const int src = __ffsll((unsigned long long)m) - 1;
            const uint32_t a0 = __shfl(a, src), b0 = __shfl(b, src), v0 = __shfl(v, src);
            for (uint32_t u = a0 + lane; u < b0; u += 64) first[u] = v0;
        }
    };
    fill(s < M && u0 < u1, u0, u1, (uint32_t)s);
    fill(s == M - 1, u1, ntiles, (uint32_t)M);
}

constexpr int kTileBlock = 1024;   // tiles per workgroup of the chunk kernels
constexpr int kChunkDirect = 64;   // workgroups that sum the chunk counts before them

__device__ __forceinline__ uint32_t tile_nodes(const uint32_t *__restrict__ first, int64_t t,
                                               int64_t ntiles, uint32_t M)
{
    return (t + 1 < ntiles ? first[t + 1] : M) - first[t];
}

// part[b] = chunks of the tiles of workgroup b (more than kChunkDirect of them).
__global__ __launch_bounds__(kTileBlock) void k_bin_chunk_part(const uint32_t *__restrict__ first,
                                                               int64_t ntiles, uint32_t M, int base,
                                                               uint32_t *__restrict__ part)
{
    __shared__ uint32_t ws[kTileBlock / 64];
    const int64_t t = (int64_t)blockIdx.x * kTileBlock + threadIdx.x;
    uint32_t all;
    (void)block_exscan<kTileBlock>(t < ntiles ? chunks_of(tile_nodes(first, t, ntiles, M), base) : 0u, ws, all);
    if (threadIdx.x == 0) part[blockIdx.x] = all;
}

// Tile counts, the first chunk of every tile, the chunk list and its length.
// part NULL: the chunks of the tiles before the workgroup's are counted here.
__global__ __launch_bounds__(kTileBlock) void k_bin_chunks(const uint32_t *__restrict__ first,
                                                           int64_t ntiles, uint32_t M, int base,
                                                           const uint32_t *__restrict__ part,
                                                           uint32_t *__restrict__ count,
                                                           uint32_t *__restrict__ chunk_start,
                                                           Chunk *__restrict__ chunks,
                                                           uint32_t *__restrict__ n_chunks)
{
    __shared__ uint32_t ws[kTileBlock / 64];
    const int tid = threadIdx.x;
    const int64_t t0 = (int64_t)blockIdx.x * kTileBlock, t = t0 + tid;
    uint32_t sum = 0;
    if (part) {
        for (int64_t b = tid; b < (int64_t)blockIdx.x; b += kTileBlock) sum += part[b];
    } else {
#pragma unroll 4
        for (int64_t u = tid; u < t0; u += kTileBlock) sum += chunks_of(tile_nodes(first, u, ntiles, M), base);
    }
    uint32_t before, all;
    (void)block_exscan<kTileBlock>(sum, ws, before);
    const uint32_t c = t < ntiles ? tile_nodes(first, t, ntiles, M) : 0u;
    const uint32_t o0 = before + block_exscan<kTileBlock>(chunks_of(c, base), ws, all);
    if (t < ntiles) {
        count[t] = c;
        chunk_start[t] = o0;
        const uint32_t s0 = first[t];
        uint32_t o = o0;
        const uint32_t len = 1u << chunk_shift(c, base);
        for (uint32_t s = 0; s < c; s += len, ++o)
            chunks[o] = Chunk{(uint32_t)t, s0 + s, c - s < len ? c - s : len, 0u};
    }
    if (t == ntiles - 1) n_chunks[0] = o0 + chunks_of(c, base);
}

// ------------------------------------------------------------------ host --
// log2 of the nodes per chunk of a plan of M nodes.  A wavefront walks its chunk's
// nodes one after the other, each a chain of LDS round trips, so with few nodes the
// longest chunk sets the time and most CUs idle; a chunk costs the staging or the slot
// of its padded tile, so with many nodes longer ones win.  Forward + adjoint in us at
// 256 / 128 / 64 / 32 nodes per chunk:
//   2D     4097 nodes  126 /  82 /  59 /  51       3D   30001 nodes  143 /  131 /  138 /  159
//   2D    50021 nodes  332 / 218 / 172 / 164       3D   60001 nodes  510 /  423 /  437 /  471
//   2D   100800 nodes  220 / 220 / 242 / 242       3D  400009 nodes 1090 / 1029 / 1062 / 1169
//   2D   262144 nodes  182 / 188 / 211 / 222       3D  262145 nodes  646 /  643 /  705 /  797
// Hence about 1024 chunks at most from splitting in 2D (50021 nodes, which that gives 64
// per chunk, would gain 5% more with 32; a line that lets them have 32 costs 100800
// radial nodes 10%), and 128 nodes or more in 3D, whose slots are larger: there only
// where no evenly filled tile is split (at 123 nodes per tile, where a third would be,
// 342 us instead of 293).  A batch has its problems to fill the GPU: the longest chunks.
// 1D, a node per lane; the line is flat (m = 4, FP64):
//   2^16 cells, 32768 nodes   40 /  40 /  41 /  46   clustered     40 /  40 /  41 /  42
//   2^16 cells, 65536 nodes   42 /  43 /  47 /  53   clustered     41 /  42 /  44 /  49
//   2^20 cells, 40000 nodes   74 /  74 /  74 /  74   clustered     84 /  81 /  79 /  80
//   2^20 cells, 90000 nodes   75 /  74 /  75 /  79   clustered     90 /  83 /  82 /  86
// 64 nodes while that is at most 512 chunks, 128 up to as many, then 256.
static int plan_chunk_base(int d, int64_t M, int64_t ntiles)
{
    if (d == 1) return M <= 32768 ? 6 : M <= 65536 ? 7 : kChunkShift;
    if (d == 3) return M <= 80 * ntiles && (M >> 7) <= 4096 ? 7 : kChunkShift;
    int s = kChunkShiftMin;
    while (s < kChunkShift && (M >> s) > 1024) ++s;
    return s;
}

// log2 of the chunks per chain of the 3D matrix-core spread, at most (chain_shift, by the
// chunks there are, may take none).  A chain of k tiles writes
// (9 k + 8) / (17 k) of the slots that single chunks write (W = 10) and is one
// workgroup's work in one piece.  Forward + adjoint (the adjoint at m = 6) in us for
// chains of 1 / 2 / 4 / 8 chunks:
//   FP32 256^3 grid, 2^21 nodes     1645 / 1549 / 1570 / 1675
//   FP32  64^3 grid,  30001 nodes    133 /  125 /  141 /  173
//   FP64 256^3 grid, 2^21 nodes     4390 / 4149 / 4051 / 4119
//   FP64 128^3 grid, 262145 nodes    661 /  622 /  643 /  671
//   FP64 128^3 grid, 2^18, m = 6     559 /  533 /  527 /  655
//   FP64  64^3 grid,  60001, m = 6   317 /  319 /  397 /  494
//   FP32 / FP64 128 x 64 x 64 grid, 122881 nodes, m = 4   93 / 117, 100 / 134, 115 / 157
//   FP64 256 x 64 x 64 grid, 245761 nodes, m = 3         133 /  138 /  153
// So two from 4096 tiles on (8 chains and more per resident FP64 workgroup), four for
// FP64 from 16384; below, the chains leave workgroups idle at the end in most cases (the
// FP32 64^3 grid alone would gain: its 700 chunks are fewer than the resident workgroups).
static int plan_seg_shift(int elem_bytes, int64_t ntiles)
{
    return ntiles < 4096 ? 0 : elem_bytes == 8 && ntiles >= 16384 ? 2 : 1;
}

bool Binning::plan(const Geom &ge, int elem_bytes_, int kernel_variant, int tile_variant_)
{
    variant = kernel_variant;
    tile_variant = tile_variant_;
    elem_bytes = elem_bytes_;
    d = ge.d;
    usable = 0;
    const int W = ge.W;
    if (W > 18 || ge.M >= (int64_t(1) << 31)) return false;
    int64_t shape[3];
    tile_shape(d, planes() ? tile_variant : 0, shape);
    int64_t bytes = 2 * elem_bytes;
    ntiles = 1;
    int64_t ncells = 1;
    for (int t = 0; t < 3; ++t) {
        T[t] = t < d ? shape[t] : 1;
        if (t < d && (ge.n[t] < T[t] || ge.n[t] % T[t] != 0)) return false;
        nt[t] = t < d ? ge.n[t] / T[t] : 1;
        ntiles *= nt[t];
        ncells *= t < d ? ge.n[t] : 1;
        if (t < d) bytes *= T[t] + W - 1;
    }
    if (ntiles >= (int64_t(1) << 31)) return false;
    chunk_base = own_scratch && (planes() || d == 1) ? plan_chunk_base(d, ge.M, ntiles) : kChunkShift;
    seg_shift = planes() && own_scratch ? plan_seg_shift(elem_bytes, ntiles) : 0;
    if (planes()) {
        // plane-tiled kernels: 32-bit grid offsets and the LDS tile must fit
        if (ncells > (int64_t(1) << 32)) return false;
        const bool fits = elem_bytes == 4 ? tile_kernels_fit<float>(ge, tile_variant, compensated)
                                          : tile_kernels_fit<double>(ge, tile_variant, false);
        if (!fits) return false;
        slot_cells = elem_bytes == 4 ? tile_slot_cells<float>(ge, tile_variant)
                                     : tile_slot_cells<double>(ge, tile_variant);
    } else {
        if (bytes > kLaneTileBytes) return false;
        if (d == 3 && W > 14) return false;
    }
    // the composite sort key must fit 32 bits
    sub_sort = true;
    if (planes() && (uint64_t)ntiles * sub_range(bin_geom(*this)) > (uint64_t(1) << 32)) return false;
    // a run of nodes is only kept in registers by the 3D VALU spread: not on the matrix
    // cores (8^3 tiles, W <= 14, a plan's own binning; a batch's 3D spread is the VALU's)
    sub_sort = d == 3 && !(tile_variant == 0 && W <= 14 && own_scratch);
    const uint64_t kmax = (uint64_t)ntiles * (planes() ? sub_range(bin_geom(*this)) : 1u);
    int bits = 1;
    while ((uint64_t(1) << bits) < kmax) ++bits;
    key_bits = bits;
    sort_passes = (bits + 7) / 8;
    usable = 1;
    return true;
}

static size_t align256(size_t v) { return (v + 255) & ~size_t(255); }

// Offsets of the buffers in the binning's device block (base non-NULL: set the
// pointers from it).  Sizes:
//   keys, keys2, perm, perm2    M u32 each
//   scan_part                   256 digit totals, or the chunk sums of the tile blocks
//   tile_count/_start, chunk_start  ntiles u32 each; n_chunks 2 (count, work counter)
//   chunks                      max_chunks
//   plane-tiled: desc, desc2    M descriptors each; slots, fs (own scratch)
//   node-lane:   xs             M d doubles
//   rs_hist                     256 u32 per radix block: in fs or xs, which are
//                               written after the sort (both hold 8 bytes per node,
//                               a radix block at least 1024 nodes), or on its own
static size_t bin_layout(Binning &b, int64_t M, char *base)
{
    const int64_t nblk = rs_blocks(M);
    const int64_t max_chunks = b.ntiles + ((M + (int64_t(1) << b.chunk_base) - 1) >> b.chunk_base);
    const int64_t nparts = (b.ntiles + kTileBlock - 1) / kTileBlock;
    const size_t db = b.elem_bytes == 4 ? sizeof(NodeDesc<float>) : sizeof(NodeDesc<double>);
    size_t off = 0;
    auto take = [&](size_t bytes) {
        char *p = base ? base + off : nullptr;
        off += align256(bytes ? bytes : 16);
        return p;
    };
    uint32_t *keys = (uint32_t *)take(4 * (size_t)M), *keys2 = (uint32_t *)take(4 * (size_t)M);
    uint32_t *perm = (uint32_t *)take(4 * (size_t)M), *perm2 = (uint32_t *)take(4 * (size_t)M);
    uint32_t *scan_part = (uint32_t *)take(4 * (size_t)std::max<int64_t>(kRsDigits, nparts));
    uint32_t *tile_count = (uint32_t *)take(4 * (size_t)b.ntiles);
    uint32_t *tile_start = (uint32_t *)take(4 * (size_t)b.ntiles);
    uint32_t *chunk_start = (uint32_t *)take(4 * (size_t)b.ntiles);
    uint32_t *n_chunks = (uint32_t *)take(8);   // chunk count, then the spread's work counter
    Chunk *chunks = (Chunk *)take(sizeof(Chunk) * (size_t)max_chunks);
    const size_t hist_bytes = 4 * (size_t)kRsDigits * nblk;
    void *desc = nullptr, *desc2 = nullptr, *slots = nullptr, *fs = nullptr;
    uint32_t *rs_hist = nullptr;
    double *xs = nullptr;
    if (b.planes()) {
        desc = take((size_t)M * db);
        desc2 = take((size_t)M * db);
        if (b.own_scratch) {
            slots = take((size_t)max_chunks * b.slot_cells * 2 * b.elem_bytes);
            fs = take(std::max((size_t)M * 2 * b.elem_bytes, hist_bytes));
            rs_hist = (uint32_t *)fs;
        } else {
            rs_hist = (uint32_t *)take(hist_bytes);
        }
    } else {
        xs = (double *)take(std::max(sizeof(double) * (size_t)M * b.d, hist_bytes));
        rs_hist = (uint32_t *)xs;
    }
    if (base) {
        b.keys = keys;
        b.keys2 = keys2;
        b.perm = perm;
        b.perm2 = perm2;
        b.rs_hist = rs_hist;
        b.scan_part = scan_part;
        b.tile_count = tile_count;
        b.tile_start = tile_start;
        b.chunk_start = chunk_start;
        b.n_chunks = n_chunks;
        b.chunks = chunks;
        b.desc = desc;
        b.desc2 = desc2;
        b.slots = slots;
        b.fs = fs;
        b.xs = xs;
        b.max_chunks = max_chunks;
        b.M = M;
    }
    return off;
}

size_t Binning::bytes_for(int64_t M_) const { return bin_layout(const_cast<Binning &>(*this), M_, nullptr); }

void Binning::carve(char *base, int64_t M_) { bin_layout(*this, M_, base); }

bool Binning::bind(void *base, size_t bytes, int64_t M_)
{
    if (!usable || bytes < bytes_for(M_)) return false;
    release();
    block = base;
    own_block = false;
    carve(static_cast<char *>(base), M_);
    return true;
}

template <typename T, int IPT>
static void launch_keys(const Binning &b, const KeyGeom &kg, uint32_t mask, const double *x,
                        NodeDesc<T> *dj, int64_t nblk, hipStream_t s)
{
    const unsigned nb = (unsigned)nblk;
    switch (b.d) {
    case 1: k_bin_keys<T, 1, IPT><<<nb, kRsThreads, 0, s>>>(x, b.keys, dj, b.M, kg, mask, b.rs_hist); break;
    case 2: k_bin_keys<T, 2, IPT><<<nb, kRsThreads, 0, s>>>(x, b.keys, dj, b.M, kg, mask, b.rs_hist); break;
    default: k_bin_keys<T, 3, IPT><<<nb, kRsThreads, 0, s>>>(x, b.keys, dj, b.M, kg, mask, b.rs_hist); break;
    }
}

// The radix passes; returns the sorted keys.  Pass p reads (kin, vin) and writes
// (kout, vout); the values alternate so that the last pass writes perm.
template <int IPT> static uint32_t *launch_sort(const Binning &b, int64_t nblk, hipStream_t s)
{
    const unsigned nb = (unsigned)nblk;
    const int P = b.sort_passes, bits = (b.key_bits + P - 1) / P;   // digits of equal width
    const uint32_t mask = (1u << bits) - 1u;
    uint32_t *kin = b.keys, *kout = b.keys2;
    for (int p = 0; p < P; ++p) {
        uint32_t *vout = (P - 1 - p) % 2 == 0 ? b.perm : b.perm2;
        const uint32_t *vin = p == 0 ? nullptr : (vout == b.perm ? b.perm2 : b.perm);
        if (p > 0) k_rs_hist<IPT><<<nb, kRsThreads, 0, s>>>(kin, b.M, bits * p, mask, b.rs_hist);
        if (nblk <= kRsDirect) {
            k_rs_scatter<IPT, true><<<nb, kRsThreads, 0, s>>>(kin, vin, b.M, bits * p, bits, b.rs_hist,
                                                              nullptr, nb, kout, vout);
        } else {
            k_rs_scan<<<kRsDigits / 16, 1024, 0, s>>>(b.rs_hist, nb, b.scan_part);
            k_rs_scatter<IPT, false><<<nb, kRsThreads, 0, s>>>(kin, vin, b.M, bits * p, bits, b.rs_hist,
                                                               b.scan_part, nb, kout, vout);
        }
        std::swap(kin, kout);
    }
    return kin;
}

template <typename T> void Binning::run_build(const Geom &ge, const BinGeom &bg, const double *x,
                                              hipStream_t s)
{
    NodeDesc<T> *dj = planes() ? static_cast<NodeDesc<T> *>(desc2) : nullptr;   // by node
    KeyGeom kg{};
    for (int t = 0; t < 3; ++t) {
        kg.n[t] = ge.n[t];
        kg.nt[t] = (uint32_t)bg.nt[t];
        kg.logT[t] = bg.logT[t];
    }
    kg.m = ge.m;
    kg.sub_shift = bg.sub_shift;
    kg.sub_range = planes() ? sub_range(bg) : 1u;
    int sub_bits = 0;   // tile extents are powers of two, and so is sub_range
    while ((1u << sub_bits) < kg.sub_range) ++sub_bits;
    const int64_t nblk = rs_blocks(M);
    const int bits = (key_bits + sort_passes - 1) / sort_passes;
    const uint32_t mask = (1u << bits) - 1u;
    uint32_t *skeys;
    if (rs_ipt(M) == 4) {
        launch_keys<T, 4>(*this, kg, mask, x, dj, nblk, s);
        skeys = launch_sort<4>(*this, nblk, s);
    } else {
        launch_keys<T, 16>(*this, kg, mask, x, dj, nblk, s);
        skeys = launch_sort<16>(*this, nblk, s);
    }
    k_bin_place<T><<<(unsigned)((M + 255) / 256), 256, 0, s>>>(
        skeys, perm, M, sub_bits, (uint32_t)ntiles, dj, static_cast<NodeDesc<T> *>(desc), x, xs, d, tile_start);
    const int64_t nparts = (ntiles + kTileBlock - 1) / kTileBlock;
    if (nparts > kChunkDirect)
        k_bin_chunk_part<<<(unsigned)nparts, kTileBlock, 0, s>>>(tile_start, ntiles, (uint32_t)M, chunk_base,
                                                                     scan_part);
    k_bin_chunks<<<(unsigned)nparts, kTileBlock, 0, s>>>(tile_start, ntiles, (uint32_t)M, chunk_base,
                                                         nparts > kChunkDirect ? scan_part : nullptr,
                                                         tile_count, chunk_start, chunks, n_chunks);
}

void Binning::build(const Geom &ge, const double *x, hipStream_t s)
{
    if (!usable) return;
    if (!block || M != ge.M) {
        if (block && !own_block)
            throw Error(CUNFFT_ERR_STATE, "bound binning memory is sized for another node count");
        release();
        const size_t bytes = bytes_for(ge.M);
        void *p = nullptr;
        CUNFFT_HIP(hipMalloc(&p, bytes));
        block = p;
        own_block = true;
        carve(static_cast<char *>(p), ge.M);
    }
    const BinGeom bg = bin_geom(*this);
    if (elem_bytes == 4) run_build<float>(ge, bg, x, s);
    else run_build<double>(ge, bg, x, s);
    CUNFFT_HIP(hipGetLastError());
    built = 1;
}

void Binning::release()
{
    if (block && own_block) (void)hipFree(block);
    block = nullptr;
    own_block = false;
    keys = keys2 = perm = perm2 = rs_hist = scan_part = nullptr;
    tile_count = tile_start = chunk_start = n_chunks = nullptr;
    chunks = nullptr;
    xs = nullptr;
    desc = desc2 = slots = fs = nullptr;
    built = 0;
    M = 0;
}

}  // namespace cunfft

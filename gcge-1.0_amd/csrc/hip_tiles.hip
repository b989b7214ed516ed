// hip_tiles.hip -- Gram products G = V^T W and block linear combinations
// Y = beta Y + alpha X C on the gfx950 matrix cores.
//
// Both work on column-major multivectors (leading dimension a multiple of
// 256 elements, so every column is 2 KiB / 1 KiB aligned) and use the
// 16x16x4 MFMA shapes: v_mfma_f64_16x16x4f64 for FP64 data and
// v_mfma_f32_16x16x4f32 for FP32 data (FP32 accumulation).  Lane layout of
// these instructions, lane l = 0..63 of a wavefront:
//   A operand (16 x 4):  A[l % 16][l / 16]
//   B operand (4 x 16):  B[l / 16][l % 16]
//   D (16 x 16), slot t of lane l:  FP32  D[4 (l / 16) + t][l % 16]
//                                   FP64  D[4 t + l / 16][l % 16]
// (the FP64 result rows are interleaved; checked on the device).
//
// Gram: the n rows are cut into chunks; a workgroup owns one chunk and one
// output block, and the reduction index k of the MFMA runs over rows.  Partial
// blocks go to a per-chunk buffer that a second kernel sums in a fixed order.
// Few columns (k_gram_mfma): each lane loads R consecutive rows of one column
// as one aligned vector (32 bytes), so a superstep of the wavefront covers 4 R
// rows and MFMA step t takes row  base + 4 R s + (l / 16) R + t  for both
// operands.  Otherwise (k_gram_slab) V and W go through LDS.
// Very thin products (p <= 4, q <= 8 or the transpose) take a vector kernel
// that keeps the whole p x q block in registers and reads V and W once.
//
// LinComb: a wavefront owns 16, 32 or (FP32) 64 rows of Y, as leave workgroups
// enough, and all its columns up to 128; X supplies the A operand straight from HBM, C the B
// operand from a copy packed on the host in operand order and staged through
// LDS for the workgroup.  Thin combinations (p, q <= 8) take a vector kernel
// with C in the kernel arguments and 16-byte row vectors.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <type_traits>
#include <vector>

#include "gram_shape.h"
#include "hip_common.h"

namespace gh {

namespace {

constexpr int kThreads = 256;       // 4 wavefronts per workgroup
constexpr int kGramTargetWG = 2048; // workgroups a Gram launch aims for
constexpr double kRowsBytes = 200e6;  // X and Y of k_lincomb_rows at most
constexpr int kSlabThreads = 512;   // slab Gram: 8 wavefronts per workgroup

typedef double dx4 __attribute__((ext_vector_type(4)));
typedef float fx4 __attribute__((ext_vector_type(4)));
typedef float fx8 __attribute__((ext_vector_type(8)));

template <typename T>
struct MT;

template <>
struct MT<double> {
    using acc_t = dx4;
    using vec_t = dx4;              // R rows of one column
    static constexpr int R = 4;
    __device__ static __forceinline__ acc_t mma(double a, double b, acc_t c)
    {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    // result row of slot t in lane group g = l / 16
    __device__ static __forceinline__ int drow(int g, int t) { return 4 * t + g; }
    // order of the 16 rows of an operand so that, slot by slot, the lane
    // groups hold neighbouring result rows: operand row i is row spread(i)
    __device__ static __forceinline__ int spread(int i) { return i; }
};

template <>
struct MT<float> {
    using acc_t = fx4;
    using vec_t = fx8;
    static constexpr int R = 8;
    __device__ static __forceinline__ acc_t mma(float a, float b, acc_t c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    __device__ static __forceinline__ int drow(int g, int t) { return 4 * g + t; }
    __device__ static __forceinline__ int spread(int i) { return 4 * (i & 3) + (i >> 2); }
};

// R consecutive rows [row, row + R) of one column, zero past `end`
template <typename T>
__device__ __forceinline__ void load_rows(const T *__restrict__ col, int64_t row, int64_t end,
                                          T (&v)[MT<T>::R])
{
    constexpr int R = MT<T>::R;
    if (row + R <= end) {
        const typename MT<T>::vec_t x = *reinterpret_cast<const typename MT<T>::vec_t *>(col + row);
#pragma unroll
        for (int t = 0; t < R; t++) v[t] = x[t];
    } else {
#pragma unroll
        for (int t = 0; t < R; t++) v[t] = (row + t < end) ? col[row + t] : T(0);
    }
}

__device__ __forceinline__ double wave_sum(double v)
{
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    return v;
}

// Workgroups are dealt round-robin to the 8 XCDs; this renumbering gives
// each XCD a contiguous range of logical blocks, so the tiles of one row
// chunk run together on one XCD and share its L2.
__device__ __forceinline__ int xcd_logical_block()
{
    const int per = (int)(gridDim.x >> 3);
    return (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
}

// ---------------------------------------------------------------- Gram (MFMA)
// Workgroup tile TP x TQ = (GP WP 16) x (GQ WQ 16); its 4 wavefronts are
// arranged GP x GQ over the tile and GK = 4 / (GP GQ) ways over the rows.
// partial[chunk][j * p + i] = sum over the chunk's rows of V(r, i) W(r, j).
template <typename T, int WP, int WQ, int GP, int GQ>
__global__ __launch_bounds__(kThreads) void k_gram_mfma(int64_t n, const T *__restrict__ V, int64_t ldv, int p,
                                                        const T *__restrict__ W, int64_t ldw, int q, int tiles_p,
                                                        int tiles_q, int nchunk, int64_t rows_per_chunk,
                                                        int upper_only, double *__restrict__ partial)
{
    constexpr int GK = 4 / (GP * GQ);
    constexpr int R = MT<T>::R;
    constexpr int S = 4 * R;  // rows per wavefront superstep
    constexpr int TP = GP * WP * 16, TQ = GQ * WQ * 16;
    using acc_t = typename MT<T>::acc_t;
    __shared__ double red[GK > 1 ? (GK - 1) * GP * GQ * WP * WQ * 4 * 64 : 1];

    const int ntile = tiles_p * tiles_q;
    const int logical = xcd_logical_block();
    if (logical >= ntile * nchunk) return;
    const int chunk = logical / ntile, tile = logical % ntile;
    const int i0t = (tile % tiles_p) * TP, j0t = (tile / tiles_p) * TQ;
    if (upper_only && i0t > j0t + TQ - 1) return;  // tile entirely below the diagonal

    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int wp = wave % GP, wq = (wave / GP) % GQ, wk = wave / (GP * GQ);
    const int i0 = i0t + wp * WP * 16, j0 = j0t + wq * WQ * 16;
    const int m = lane & 15, kk = lane >> 4;
    const int64_t rb = (int64_t)chunk * rows_per_chunk;
    const int64_t re = min(n, rb + rows_per_chunk);

    // Columns past p (q) are clamped to the last one: they feed only result
    // rows (columns) >= p (q), which are never stored, so no lane branches.
    const T *vc[WP];
    const T *wc[WQ];
#pragma unroll
    for (int x = 0; x < WP; x++) vc[x] = V + (int64_t)min(i0 + x * 16 + m, p - 1) * ldv;
#pragma unroll
    for (int y = 0; y < WQ; y++) wc[y] = W + (int64_t)min(j0 + y * 16 + m, q - 1) * ldw;

    acc_t acc[WP][WQ];
#pragma unroll
    for (int x = 0; x < WP; x++)
#pragma unroll
        for (int y = 0; y < WQ; y++) acc[x][y] = acc_t{};

    // full supersteps (every row below re): unguarded vector loads, the next
    // superstep's operands loaded before this one's MFMAs are issued
    using vec_t = typename MT<T>::vec_t;
    const int64_t step = (int64_t)GK * S;
    const int64_t full_end = rb + ((re - rb) / S) * S;
    int64_t s = rb + (int64_t)wk * S;
    if (s < full_end) {
        auto load = [&](int64_t ss, vec_t (&aa)[WP], vec_t (&bb)[WQ]) {
#pragma unroll
            for (int x = 0; x < WP; x++) aa[x] = *reinterpret_cast<const vec_t *>(vc[x] + ss + (int64_t)kk * R);
#pragma unroll
            for (int y = 0; y < WQ; y++) bb[y] = *reinterpret_cast<const vec_t *>(wc[y] + ss + (int64_t)kk * R);
        };
        auto mma = [&](const vec_t (&aa)[WP], const vec_t (&bb)[WQ]) {
#pragma unroll
            for (int t = 0; t < R; t++)
#pragma unroll
                for (int x = 0; x < WP; x++)
#pragma unroll
                    for (int y = 0; y < WQ; y++) acc[x][y] = MT<T>::mma(aa[x][t], bb[y][t], acc[x][y]);
        };
        if constexpr (GP * GQ == 4) {
            // 64 x 64 tiles: one operand buffer (register budget for four
            // wavefronts per SIMD); latency is hidden by occupancy
            for (; s < full_end; s += step) {
                vec_t a0[WP], b0[WQ];
                load(s, a0, b0);
                mma(a0, b0);
            }
        } else {
            // supersteps in pairs with two operand buffers (loads of one in
            // flight while the MFMAs of the other are issued)
            vec_t a0[WP], b0[WQ], a1[WP], b1[WQ];
            // the last full superstep of this wavefront
            const int64_t last_full = s + ((full_end - 1 - s) / step) * step;
            load(s, a0, b0);
            for (; s + step < full_end; s += 2 * step) {
                load(s + step, a1, b1);
                mma(a0, b0);
                // unconditional (clamped to a full superstep) so the wait
                // before the next MFMAs covers only the older loads
                load(min(s + 2 * step, last_full), a0, b0);
                mma(a1, b1);
            }
            if (s < full_end) {
                mma(a0, b0);
                s += step;
            }
        }
    }
    // the partial superstep at the end of the chunk (rows past re read as 0)
    if (s < re) {
        const int64_t row = s + (int64_t)kk * R;
        T a[WP][R], b[WQ][R];
#pragma unroll
        for (int x = 0; x < WP; x++) load_rows<T>(vc[x], row, re, a[x]);
#pragma unroll
        for (int y = 0; y < WQ; y++) load_rows<T>(wc[y], row, re, b[y]);
#pragma unroll
        for (int t = 0; t < R; t++)
#pragma unroll
            for (int x = 0; x < WP; x++)
#pragma unroll
                for (int y = 0; y < WQ; y++) acc[x][y] = MT<T>::mma(a[x][t], b[y][t], acc[x][y]);
    }

    // sum the GK row-split partial tiles in wavefront order: the wavefronts
    // of row slice wk > 0 park their tiles in red[((wk - 1) GP GQ + wpq) SLOTS
    // + slot][lane], wpq = wp + GP wq, and slice 0 adds them
    const int wpq = wp + GP * wq;
    if constexpr (GK > 1) {
        constexpr int SLOTS = WP * WQ * 4;
        if (wk > 0) {
#pragma unroll
            for (int x = 0; x < WP; x++)
#pragma unroll
                for (int y = 0; y < WQ; y++)
#pragma unroll
                    for (int t = 0; t < 4; t++)
                        red[(((size_t)(wk - 1) * GP * GQ + wpq) * SLOTS + (x * WQ + y) * 4 + t) * 64 + lane] =
                            (double)acc[x][y][t];
        }
        __syncthreads();
        if (wk > 0) return;
    }

    double *out = partial + (int64_t)chunk * p * q;
#pragma unroll
    for (int x = 0; x < WP; x++)
#pragma unroll
        for (int y = 0; y < WQ; y++)
#pragma unroll
            for (int t = 0; t < 4; t++) {
                double v = (double)acc[x][y][t];
                if constexpr (GK > 1) {
                    constexpr int SLOTS = WP * WQ * 4;
#pragma unroll
                    for (int w = 0; w < GK - 1; w++)
                        v += red[(((size_t)w * GP * GQ + wpq) * SLOTS + (x * WQ + y) * 4 + t) * 64 + lane];
                }
                const int i = i0 + x * 16 + MT<T>::drow(kk, t), j = j0 + y * 16 + m;
                if (i < p && j < q) out[(int64_t)j * p + i] = v;
            }
}

// ---------------------------------------------------------------- Gram (LDS slabs)
// Workgroup output block of MB x NB 16 x 16 tiles over one row chunk, eight
// wavefronts.  Every SLAB rows (128 bytes of each column) the threads copy the
// block's columns of V and W into LDS (column-major, 16-byte pad per column:
// 144-byte column stride, so neither the 16-byte copies nor the operand
// reads of 16 consecutive columns meet a bank twice), two buffers
// deep.  The block's tiles, column by column, without those below the diagonal
// when upper_only, are dealt out in equal runs of at most NT per wavefront,
// whatever MB and NB: every SIMD has the same number of products.
// UPT: 16-byte units that a thread copies per slab, at least (MB + NB) / 4.
// Product t = 0 .. E - 1 of step 0 or 1, E = 16 / sizeof(T), takes row
// 4 E step + 4 t + l / 16  of the slab for both operands, or with RUN
// 2 E (l / 16) + E step + t, which a lane reads at once: 4 - 8 % faster at every
// size.  The two add the rows in different orders.  From 65 to 256 columns the
// slower one stays: with up to 128 columns on one side its sums keep the bits
// they had before this kernel, and with them the course of solves whose pairs lie
// at the tolerance (the other order moved residuals of a power-law graph's locked
// pairs to 1.04e-8, above their 1e-8).  Up to 64 columns k_gram_mfma's order is
// RUN's; with more than 128 on both sides, and past 256, the chunks changed
// anyway.
// Bound by memory for few columns (4.0 - 4.6 TB/s: each visit of a column
// reads 128 bytes of another page), by the matrix cores for many (67 TF in
// FP64 and 153 in FP32 for a large library product here; 46 and 84 reached, 53
// and 97 with the tiles' padding).  4.1M rows, ms, before (blocks of up to 8 x
// 8 tiles dealt out by column, 4 wavefronts, loads and LDS reads waited for
// one by one) and now, FP64 / FP32: 300 x 100 7.05 / 3.97 -> 5.31 / 2.91; 200
// x 100 4.80 / 2.74 -> 4.20 / 2.33; 100 x 100, upper 1.87 / 1.12 -> 1.63 /
// 0.86; 100 x 50 1.87 / 1.15 -> 1.73 / 0.90; 64 x 64 1.42 / 0.91 -> 1.06 /
// 0.45 (without LDS).
template <typename T, int NT, int UPT, bool RUN>
__global__ __launch_bounds__(kSlabThreads, (UPT <= 4 ? 4 : 2)) void k_gram_slab(
    int64_t n, const T *__restrict__ V, int64_t ldv, int p, const T *__restrict__ W, int64_t ldw, int q, int MB,
    int NB, int blocks_p, int blocks_q, int nchunk, int64_t rows_per_chunk, int upper_only,
    double *__restrict__ partial)
{
    constexpr int E = 16 / (int)sizeof(T);     // elements of a 16-byte unit
    constexpr int SLAB = 8 * E;                // rows per stage
    constexpr int LD = SLAB + E;               // LDS column stride (elements)
    constexpr int READS = RUN ? 2 : E;         // LDS reads of a tile's operands (two rows each unless RUN)
    using acc_t = typename MT<T>::acc_t;
    typedef T u16 __attribute__((ext_vector_type(E)));
    extern __shared__ __attribute__((aligned(16))) unsigned char slab_smem[];
    T *sbuf = reinterpret_cast<T *>(slab_smem);  // [2][(MB + NB) * 16 * LD]

    const int nblock = blocks_p * blocks_q;
    const int logical = xcd_logical_block();
    if (logical >= nblock * nchunk) return;
    const int chunk = logical / nblock, blk = logical % nblock;
    const int i0 = (blk % blocks_p) * MB * 16, j0 = (blk / blocks_p) * NB * 16;
    const int64_t rb = (int64_t)chunk * rows_per_chunk;
    const int64_t re = min(n, rb + rows_per_chunk);
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int m = lane & 15, kk = lane >> 4;
    const int units = (MB + NB) * 128, bufsize = (MB + NB) * 16 * LD;

    // tiles of column y that are computed: x = 0 .. rows_of(y) - 1 (those that
    // reach the matrix and, with upper_only, its diagonal)
    const int xall = min(MB, (p - i0 + 15) / 16), yall = min(NB, (q - j0 + 15) / 16);
    auto rows_of = [&](int y) { return upper_only ? max(0, min(xall, (j0 - i0) / 16 + y + 1)) : xall; };
    int live = 0;
    for (int y = 0; y < yall; y++) live += rows_of(y);
    if (live == 0) return;  // a block below the diagonal
    const int share = (live + 7) / 8, first = wave * share, mine = max(0, min(share, live - first));
    // its i-th tile (uniform; the slots past `mine` repeat the last one and are
    // not stored)
    auto walk = [&](auto &&f) {
        int y = 0, x = min(first, live - 1);
        while (x >= rows_of(y)) x -= rows_of(y++);
#pragma unroll
        for (int i = 0; i < NT; i++) {
            f(i, x, y);
            if (i + 1 < mine && ++x >= rows_of(y)) {
                x = 0;
                do y++;
                while (rows_of(y) == 0);
            }
        }
    };
    int ao[NT], bo[NT];  // LDS offsets of the tiles' operands
    walk([&](int i, int x, int y) {
        ao[i] = x * 16 * LD;
        bo[i] = (MB + y) * 16 * LD;
    });

    // this thread's copy units: column c (V for c < 16 MB, else W), 16 bytes
    // at row offset E * seg of the slab; columns past p (q) repeat the last
    // one and feed only result entries that are never stored
    const int seg = threadIdx.x & 7;
    const T *src[UPT];
#pragma unroll
    for (int u = 0; u < UPT; u++) {
        const int c = min((int)threadIdx.x + u * kSlabThreads, units - 1) >> 3;
        src[u] = (c < MB * 16 ? V + (int64_t)min(i0 + c, p - 1) * ldv
                              : W + (int64_t)min(j0 + c - MB * 16, q - 1) * ldw) + seg * E;
    }
    u16 reg[UPT];
    auto park = [&](T *buf) {
#pragma unroll
        for (int u = 0; u < UPT; u++) {
            const int unit = threadIdx.x + u * kSlabThreads;
            if (unit < units) *reinterpret_cast<u16 *>(buf + (unit >> 3) * LD + seg * E) = reg[u];
        }
    };

    acc_t acc[NT];
#pragma unroll
    for (int i = 0; i < NT; i++) acc[i] = acc_t{};
    // Products of a parked slab, each tile's operands read while the products
    // of the one before are issued (otherwise every read is waited for); with
    // MORE, the slab at row `next` is loaded into the registers meanwhile, one
    // load at a time among the first half of the products: a wavefront's loads
    // meet 8 columns, thus 8 pages, each, and block its issue when they come
    // together.  No branches: where paths meet, loads would be waited for.
    auto products = [&](const T *buf, int64_t next, auto more) {
        constexpr bool MORE = decltype(more)::value;
        const T *s = buf + m * LD + kk * (RUN ? 2 * E : 1);
        u16 a[2], b[2];
        auto rows = [&](const T *c, int step) {
            u16 v;
            if constexpr (RUN) {
                v = *reinterpret_cast<const u16 *>(c + step * E);
            } else {
#pragma unroll
                for (int t = 0; t < E; t++) v[t] = c[step * 4 * E + 4 * t];
            }
            return v;
        };
        auto read = [&](int j) {
            a[j & 1] = rows(s + ao[j % NT], j / NT);
            b[j & 1] = rows(s + bo[j % NT], j / NT);
        };
        read(0);
#pragma unroll
        for (int j = 0; j < 2 * NT; j++) {
            if (MORE && j < NT) {
#pragma unroll
                for (int u = j * UPT / NT; u < (j + 1) * UPT / NT; u++)
                    reg[u] = *reinterpret_cast<const u16 *>(src[u] + next);
            }
            if (j + 1 < 2 * NT) read(j + 1);
#pragma unroll
            for (int t = 0; t < E; t++) acc[j % NT] = MT<T>::mma(a[j & 1][t], b[j & 1][t], acc[j % NT]);
        }
        __builtin_amdgcn_sched_group_barrier(0x100, READS, 0);  // LDS reads of the first tile
#pragma unroll
        for (int j = 0; j < 2 * NT; j++) {
            if (MORE && j < NT) {
#pragma unroll
                for (int u = j * UPT / NT; u < (j + 1) * UPT / NT; u++)
                    __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // load
            }
            if (j + 1 < 2 * NT) __builtin_amdgcn_sched_group_barrier(0x100, READS, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, E, 0);  // products
        }
    };
    const int nslab = (int)((re - rb) / SLAB);
    const int64_t tail = rb + (int64_t)nslab * SLAB;
    if (nslab > 0) {
#pragma unroll
        for (int u = 0; u < UPT; u++) reg[u] = *reinterpret_cast<const u16 *>(src[u] + rb);
        park(sbuf);
        __syncthreads();
        for (int sl = 0; sl < nslab; sl++) {
            // the last slab is loaded and parked once more
            products(sbuf + (sl & 1) * bufsize, rb + (int64_t)min(sl + 1, nslab - 1) * SLAB, std::true_type{});
            park(sbuf + ((sl + 1) & 1) * bufsize);
            __syncthreads();
        }
    }
    if (tail < re) {  // the chunk's partial slab, zero past its end
        const int64_t r0 = tail + seg * E;
#pragma unroll
        for (int u = 0; u < UPT; u++)
#pragma unroll
            for (int e = 0; e < E; e++) reg[u][e] = (r0 + e < re) ? src[u][tail + e] : T(0);
        park(sbuf);
        __syncthreads();
        products(sbuf, tail, std::false_type{});
    }

    double *out = partial + (int64_t)chunk * p * q;
    walk([&](int i, int x, int y) {
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const int r = i0 + x * 16 + MT<T>::drow(kk, t), j = j0 + y * 16 + m;
            if (i < mine && r < p && j < q) out[(int64_t)j * p + r] = (double)acc[i][t];
        }
    });
}

// ---------------------------------------------------------------- Gram (thin)
// p <= PM, q <= QM; every thread keeps the PM x QM block of its rows in
// registers.  partial[block][o] with o = j * ldo + i, or i * ldo + j when
// transpose is set (the caller swapped V and W).
template <typename T, int PM, int QM>
__global__ __launch_bounds__(kThreads) void k_gram_thin(int64_t n, const T *__restrict__ V, int64_t ldv, int p,
                                                        const T *__restrict__ W, int64_t ldw, int q, int transpose,
                                                        int ldo, double *__restrict__ partial)
{
    __shared__ double sh[4][PM * QM];
    double acc[PM][QM];
#pragma unroll
    for (int a = 0; a < PM; a++)
#pragma unroll
        for (int b = 0; b < QM; b++) acc[a][b] = 0.0;
    const int64_t stride = (int64_t)gridDim.x * kThreads;
#pragma unroll 2
    for (int64_t r = (int64_t)blockIdx.x * kThreads + threadIdx.x; r < n; r += stride) {
        double v[PM], w[QM];
#pragma unroll
        for (int a = 0; a < PM; a++) v[a] = (a < p) ? (double)V[(int64_t)a * ldv + r] : 0.0;
#pragma unroll
        for (int b = 0; b < QM; b++) w[b] = (b < q) ? (double)W[(int64_t)b * ldw + r] : 0.0;
#pragma unroll
        for (int a = 0; a < PM; a++)
#pragma unroll
            for (int b = 0; b < QM; b++) acc[a][b] = fma(v[a], w[b], acc[a][b]);
    }
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
    for (int a = 0; a < PM; a++)
#pragma unroll
        for (int b = 0; b < QM; b++) {
            const double s = wave_sum(acc[a][b]);
            if (lane == 0) sh[wave][a * QM + b] = s;
        }
    __syncthreads();
    const int pq = p * q;
    for (int e = threadIdx.x; e < PM * QM; e += kThreads) {
        const int a = e / QM, b = e % QM;
        if (a < p && b < q) {
            const double s = (sh[0][e] + sh[1][e]) + (sh[2][e] + sh[3][e]);
            const int o = transpose ? a * ldo + b : b * ldo + a;
            partial[(int64_t)blockIdx.x * pq + o] = s;
        }
    }
}

// G[e] = sum_c partial[c][e] into host memory: 64 entries per workgroup, the 4
// wavefronts take every 4th chunk, 8 loads in flight (a wavefront has up to
// 128 chunks; one load at a time took 38 us on average in a mixed solve of
// the 64^3 generalized problem, this 9), combined in a fixed order; then the
// launch's number in seqs[workgroup].
// With upper_only, entries below the diagonal (i > j, e = j * p + i) are
// skipped.
__global__ __launch_bounds__(kThreads) void k_sum_chunks(const double *__restrict__ partial, int nchunk, int p,
                                                         int64_t pq, int upper_only, double *__restrict__ G,
                                                         unsigned long long *__restrict__ seqs,
                                                         unsigned long long seq)
{
    __shared__ double sh[4][64];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int64_t e = (int64_t)blockIdx.x * 64 + lane;
    bool live = e < pq;
    if (live && upper_only) live = (e % p) <= (e / p);
    double acc = 0.0;
    if (live) {
        int c = wave;
        for (; c + 28 < nchunk; c += 32) {
            double v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = partial[(int64_t)(c + 4 * u) * pq + e];
#pragma unroll
            for (int u = 0; u < 8; u++) acc += v[u];
        }
        for (; c < nchunk; c += 4) acc += partial[(int64_t)c * pq + e];
    }
    sh[wave][lane] = acc;
    __syncthreads();
    if (wave == 0 && e < pq) G[e] = live ? (sh[0][lane] + sh[1][lane]) + (sh[2][lane] + sh[3][lane]) : 0.0;
    __syncthreads();
    if (threadIdx.x == 0)
        __hip_atomic_store(seqs + blockIdx.x, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ---------------------------------------------------------------- LinComb (MFMA)
// Cp[((kb * nqb) + jb) * 64 + l] = C(4 kb + l / 16, 16 jb + l % 16), zero
// past p and q.  A wavefront owns RB blocks of 16 rows, row i of block h being
// row RB spread(i) + h of its 16 RB: a lane's A operands of the RB blocks are
// RB consecutive rows of one column of X, one vector load, and slot t of the
// lane groups 0 .. 3 are 4 RB consecutive rows of Y, 64 bytes for RB = 2 in
// FP64 and 4 in FP32.  It forms RN blocks of 16
// columns (all of them up to 128 columns, so X leaves memory once), RN fitted
// to q: 100 columns are 7 blocks, not 8.  The four wavefronts share C, staged
// in LDS in panels of 4 k blocks two deep (each reads 512 bytes per k block and
// column block; from L2 these reads cost as much as the products); X is
// loaded one panel ahead into registers.  Bound by the matrix cores for large
// p and q (a large library product reaches 67 TF here in FP64, 153 in FP32).
// Over 4.1M rows, ms, C from L2 at first, then from LDS, then with the panels'
// order pinned and Y's old values loaded ahead: FP32 300 x 100 3.44, 2.76, 2.58
// (95 TF); 100 x 100 1.45, 1.28, 0.98; 200 x 100 added to Y 2.24 -> 1.97; 300 x
// 130 (two passes of 5 blocks) 6.5, 3.8, 3.5; FP64 300 x 100 6.73, 5.19, 5.18
// (47 TF, 53 with the padding); 100 x 100 2.86, 2.11, 2.00; 300 x 130 12.5, 7.2,
// 7.0.  Every sum runs over k in ascending
// blocks of 4, whatever RB and RN.

// A wavefront's results to Y: slot t of lane group kk is operand row
// drow(kk, t), column block r column 16 (g0 + r) + m.  Where all rows exist,
// the old values of a column block are loaded before the block in front of it
// is stored: one access at a time, 28 of them in turn cost more than the
// products.
template <typename T, int RN, int RB>
__device__ __forceinline__ void store_tile(const typename MT<T>::acc_t (&acc)[RB][RN], T *__restrict__ Y,
                                           int64_t ldy, int g0, int q, int64_t rw, int64_t n, T al, T be)
{
    typedef T vec __attribute__((ext_vector_type(RB)));
    const int m = threadIdx.x & 15, kk = (threadIdx.x & 63) >> 4;
    if (rw + 16 * RB <= n) {
        auto at = [&](int r, int t) {
            const int j = min((g0 + r) * 16 + m, q - 1);
            return reinterpret_cast<vec *>(Y + (int64_t)j * ldy + rw + MT<T>::spread(MT<T>::drow(kk, t)) * RB);
        };
        if (be == T(0)) {
#pragma unroll
            for (int r = 0; r < RN; r++)
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    vec v;
#pragma unroll
                    for (int h = 0; h < RB; h++) v[h] = (al == T(1)) ? (T)acc[h][r][t] : al * (T)acc[h][r][t];
                    if ((g0 + r) * 16 + m < q) *at(r, t) = v;
                }
        } else {
            vec old[2][4];
#pragma unroll
            for (int t = 0; t < 4; t++) old[0][t] = *at(0, t);
#pragma unroll
            for (int r = 0; r < RN; r++) {
                if (r + 1 < RN) {
#pragma unroll
                    for (int t = 0; t < 4; t++) old[(r + 1) & 1][t] = *at(r + 1, t);
                }
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    vec v;
#pragma unroll
                    for (int h = 0; h < RB; h++) v[h] = be * old[r & 1][t][h] + al * (T)acc[h][r][t];
                    if ((g0 + r) * 16 + m < q) *at(r, t) = v;
                }
            }
        }
        return;
    }
#pragma unroll
    for (int r = 0; r < RN; r++) {
        const int j = (g0 + r) * 16 + m;
        if (j >= q) continue;
        T *yj = Y + (int64_t)j * ldy;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const int64_t row = rw + MT<T>::spread(MT<T>::drow(kk, t)) * RB;
#pragma unroll
            for (int h = 0; h < RB; h++) {
                const T v = (T)acc[h][r][t];
                if (row + h < n)
                    yj[row + h] = (be == T(0)) ? ((al == T(1)) ? v : al * v) : be * yj[row + h] + al * v;
            }
        }
    }
}

template <typename T, int RN, int RB>
__global__ __launch_bounds__(kThreads, RN <= 2 ? 4 : RN <= 4 ? 3 : 2) void k_lincomb_mfma(int64_t n, const T *__restrict__ X, int64_t ldx, int p,
                                                              T *__restrict__ Y, int64_t ldy, int q,
                                                              const T *__restrict__ Cp, int nkb, int nqb,
                                                              double alpha, double beta)
{
    using acc_t = typename MT<T>::acc_t;
    constexpr int KP = RB == 1 ? 8 : 4;          // k blocks per panel
    constexpr int E = 16 / (int)sizeof(T);       // elements of a 16-byte copy unit
    constexpr int UNITS = KP * RN * 64 / E;
    constexpr int UPT = (UNITS + kThreads - 1) / kThreads;
    // The order of a panel's loads, LDS reads and products is pinned: left to
    // the compiler the loads of X sink to the panel's end, where they are
    // waited for.  FP64 of up to 4 column blocks has three wavefronts per SIMD
    // to cover them and loses 4 - 6 % by it (100 x 50: 1.15 against 1.18 ms).
    constexpr bool PIN = sizeof(T) == 4 || RN > 4;
    constexpr int READS = (RN + 1) / 2;          // LDS reads of a k block's operands, two at a time
    typedef T u16 __attribute__((ext_vector_type(E)));
    struct alignas(RB * sizeof(T)) Rows {
        T e[RB];
    };
    __shared__ __attribute__((aligned(16))) T sc[2][UPT * kThreads * E];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int m = lane & 15, kk = lane >> 4;
    // rows past n up to the next multiple of 64 RB <= 256 lie in the columns'
    // padding: they feed only result rows that are not stored
    const int64_t rw = ((int64_t)blockIdx.x * 4 + wave) * 16 * RB;
    const T *xr = X + rw + MT<T>::spread(m) * RB;
    const T al = (T)alpha, be = (T)beta;
    const int npan = (nkb + KP - 1) / KP;
    for (int g0 = 0; g0 < nqb; g0 += RN) {
        u16 creg[UPT];
        Rows a[KP], an[KP];
        auto fetch = [&](int pan) {
#pragma unroll
            for (int i = 0; i < KP; i++) {
                const int c = (pan * KP + i) * 4 + kk;
                an[i] = *reinterpret_cast<const Rows *>(xr + (int64_t)min(c, p - 1) * ldx);
            }
#pragma unroll
            for (int u = 0; u < UPT; u++) {
                const int unit = min((int)threadIdx.x + u * kThreads, UNITS - 1);
                const int kl = unit * E / (RN * 64), off = unit * E % (RN * 64);
                const int kb = min(pan * KP + kl, nkb - 1);
                creg[u] = *reinterpret_cast<const u16 *>(Cp + ((int64_t)kb * nqb + g0) * 64 + off);
            }
        };
        // the fetched panel becomes the current one (here, not in fetch, is X
        // looked at: its loads are in flight during the panel before)
        auto park = [&](int pan) {
#pragma unroll
            for (int u = 0; u < UPT; u++) {
                // units past UNITS fill the buffer's end: no branch, in which
                // the load would be waited for
                *reinterpret_cast<u16 *>(&sc[pan & 1][(threadIdx.x + u * kThreads) * E]) = creg[u];
            }
            const bool whole = (pan + 1) * KP * 4 <= p;
#pragma unroll
            for (int i = 0; i < KP; i++)
#pragma unroll
                for (int h = 0; h < RB; h++)
                    a[i].e[h] = (whole || (pan * KP + i) * 4 + kk < p) ? an[i].e[h] : T(0);
        };
        acc_t acc[RB][RN];
#pragma unroll
        for (int h = 0; h < RB; h++)
#pragma unroll
            for (int r = 0; r < RN; r++) acc[h][r] = acc_t{};
        auto products = [&](int i, const T (&bb)[RN]) {
#pragma unroll
            for (int r = 0; r < RN; r++)
#pragma unroll
                for (int h = 0; h < RB; h++) acc[h][r] = MT<T>::mma(a[i].e[h], bb[r], acc[h][r]);
        };
        auto read = [&](int i, const T *c, T (&bb)[RN]) {
#pragma unroll
            for (int r = 0; r < RN; r++) bb[r] = c[(i * RN + r) * 64 + lane];
        };
        fetch(0);
        park(0);
        __syncthreads();
        for (int pan = 0; pan + 1 < npan; pan++) {
            fetch(pan + 1);
            if constexpr (!PIN) {
#pragma unroll
                for (int i = 0; i < KP; i++) {
                    T bb[RN];
                    read(i, sc[pan & 1], bb);
                    products(i, bb);
                }
            } else {
                __builtin_amdgcn_sched_barrier(0);  // issued before the products, not where they are used
                T bb[2][RN];
                read(0, sc[pan & 1], bb[0]);
#pragma unroll
                for (int i = 0; i < KP; i++) {
                    if (i + 1 < KP) read(i + 1, sc[pan & 1], bb[(i + 1) & 1]);
                    products(i, bb[i & 1]);
                }
                // C's operands one k block ahead of the products
                __builtin_amdgcn_sched_group_barrier(0x100, READS, 0);
#pragma unroll
                for (int i = 0; i < KP; i++) {
                    if (i + 1 < KP) __builtin_amdgcn_sched_group_barrier(0x100, READS, 0);
                    __builtin_amdgcn_sched_group_barrier(0x008, RN * RB, 0);
                }
                __builtin_amdgcn_sched_barrier(0);  // the loads are looked at after the products
            }
            park(pan + 1);
            __syncthreads();
        }
        // the last panel: 1 .. KP k blocks
#pragma unroll
        for (int i = 0; i < KP; i++)
            if ((npan - 1) * KP + i < nkb) {
                T bb[RN];
                read(i, sc[(npan - 1) & 1], bb);
                products(i, bb);
            }
        __syncthreads();  // the next pass overwrites sc
        store_tile<T, RN, RB>(acc, Y, ldy, g0, q, rw, n, al, be);
    }
}

// Result rows of one lane after regrouping: lane (g = l / 16, m) returns
// rows 4 g .. 4 g + 3 of column m of the 16 x 16 block.  For FP32 these are
// already its four slots; for FP64 (slot t holds row 4 t + g) the four lanes
// of a column exchange values in four rounds: in round k, lane g reads the
// slot g of lane (g + k) mod 4.
template <typename T>
__device__ __forceinline__ typename MT<T>::acc_t rows4(typename MT<T>::acc_t v, int g);

template <>
__device__ __forceinline__ fx4 rows4<float>(fx4 v, int)
{
    return v;
}

template <>
__device__ __forceinline__ dx4 rows4<double>(dx4 v, int g)
{
    const int lane = threadIdx.x & 63, m = lane & 15;
    dx4 w;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int src = (g + k) & 3;             // lane group this lane reads
        const int give = (g - k) & 3;            // slot this lane sends: the reader's g
        double send = v[0];
        send = give == 1 ? v[1] : send;
        send = give == 2 ? v[2] : send;
        send = give == 3 ? v[3] : send;
        const double got = __shfl(send, m + 16 * src, 64);
        w[0] = src == 0 ? got : w[0];
        w[1] = src == 1 ? got : w[1];
        w[2] = src == 2 ? got : w[2];
        w[3] = src == 3 ? got : w[3];
    }
    return w;
}

// y[0..3] = beta y + alpha v with the branch rules of y = a x + b y, as one
// 16- (FP32) or 32-byte (FP64) access; y is 4-element aligned
template <typename T>
__device__ __forceinline__ void store_rows4(T *y, typename MT<T>::acc_t v, T al, T be)
{
    typedef T v4 __attribute__((ext_vector_type(4)));
    v4 out;
    if (be == T(0)) {
#pragma unroll
        for (int t = 0; t < 4; t++) out[t] = (al == T(1)) ? (T)v[t] : al * (T)v[t];
    } else {
        const v4 old = *reinterpret_cast<const v4 *>(y);
#pragma unroll
        for (int t = 0; t < 4; t++) out[t] = be * old[t] + al * (T)v[t];
    }
    *reinterpret_cast<v4 *>(y) = out;
}

// The products of k_lincomb_mfma for few columns of few rows: a wavefront owns
// rows [rb, rb + 32) as two 16-row blocks (slot t of lane l holds row drow(l /
// 16, t) of its block and column l % 16), walks the output in groups of RN
// 16-column blocks and reads C from the caches; no LDS and no barriers, so more
// wavefronts are in flight, which is what a memory-bound product needs while X
// and Y fit the 256 MB cache (kRowsBytes, below it because other data is there
// too).  This kernel against k_lincomb_mfma, us: FP32 20 x 20, 512,000 rows (82
// MB) 21.5 against 25.0, 884,736 (142 MB) 32.1 against 37.7, 4.1M (655 MB) 159
// against 147; 40 x 40, 262,144 rows (84 MB) 26.7 against 26.9, 884,736 (283 MB)
// 91 against 72, 4.1M 374 against 285; FP64 20 x 20, 512,000 rows (164 MB) 37.4
// against 40.7, 884,736 (283 MB) 71.0 against 69.8.  Where q or p are larger it
// is the slower one at any size: FP32 150 x 50 over 4.1M rows 1.087 against
// 0.999 ms, 300 x 100 over 16,384 30.1 against 29.1 us (but 200 x 100 23.5
// against 25.5); FP64 50 x 50 over 4.1M rows 1.080 against 0.840.
template <typename T, int RN, int WC>
__global__ __launch_bounds__(kThreads) void k_lincomb_rows(int64_t n, const T *__restrict__ X, int64_t ldx, int p,
                                                           T *__restrict__ Y, int64_t ldy, int q,
                                                           const T *__restrict__ Cp, int nkb, int nqb, double alpha,
                                                           double beta)
{
    using acc_t = typename MT<T>::acc_t;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int m = lane & 15, kk = lane >> 4;
    // WC wavefronts share one 32-row block and split its column groups
    const int64_t rb = ((int64_t)blockIdx.x * (4 / WC) + wave / WC) * 32;
    const int wcol = wave % WC;
    if (rb >= n) return;  // no workgroup barrier in this kernel
    // Rows past n are clamped to the last row: they feed only result rows
    // >= n, which are never stored.  nqb is a multiple of RN (Cp is padded
    // with zero blocks), and only the last k block can be partial.
    const int64_t ra0 = min(rb + m, n - 1), ra1 = min(rb + 16 + m, n - 1);
    const int nkb_full = p / 4;
    const T al = (T)alpha, be = (T)beta;
    for (int jb0 = wcol * RN; jb0 < nqb; jb0 += WC * RN) {
        acc_t acc0[RN], acc1[RN];
#pragma unroll
        for (int r = 0; r < RN; r++) {
            acc0[r] = acc_t{};
            acc1[r] = acc_t{};
        }
        if (nkb_full > 0) {
            // k blocks in pairs with two operand buffers: the loads of one
            // block are in flight while the MFMAs of the other are issued
            const T *xk = X + (int64_t)kk * ldx;
            const T *cb = Cp + (int64_t)jb0 * 64 + lane;
            const int64_t xs = (int64_t)4 * ldx, cs = (int64_t)nqb * 64;
            T a0[2], a1[2], b0[RN], b1[RN];
            auto load = [&](int kb, T (&aa)[2], T (&bb)[RN]) {
                const T *x = xk + (int64_t)kb * xs;
                const T *c = cb + (int64_t)kb * cs;
                aa[0] = x[ra0];
                aa[1] = x[ra1];
#pragma unroll
                for (int r = 0; r < RN; r++) bb[r] = c[r * 64];
            };
            auto mma = [&](const T (&aa)[2], const T (&bb)[RN]) {
#pragma unroll
                for (int r = 0; r < RN; r++) {
                    acc0[r] = MT<T>::mma(aa[0], bb[r], acc0[r]);
                    acc1[r] = MT<T>::mma(aa[1], bb[r], acc1[r]);
                }
            };
            load(0, a0, b0);
            int kb = 0;
            for (; kb + 1 < nkb_full; kb += 2) {
                load(kb + 1, a1, b1);
                mma(a0, b0);
                // unconditional (clamped) so the wait before the next MFMAs
                // covers only the older loads
                load(min(kb + 2, nkb_full - 1), a0, b0);
                mma(a1, b1);
            }
            if (kb < nkb_full) mma(a0, b0);
        }
        if (nkb_full < nkb) {
            // partial last k block: columns past p read as 0
            const int k = nkb_full * 4 + kk;
            const bool kok = k < p;
            const T *xk = X + (int64_t)(kok ? k : 0) * ldx;
            const T a0 = kok ? xk[ra0] : T(0);
            const T a1 = kok ? xk[ra1] : T(0);
            const T *cb = Cp + ((int64_t)nkb_full * nqb + jb0) * 64 + lane;
#pragma unroll
            for (int r = 0; r < RN; r++) {
                const T bb = cb[r * 64];
                acc0[r] = MT<T>::mma(a0, bb, acc0[r]);
                acc1[r] = MT<T>::mma(a1, bb, acc1[r]);
            }
        }
        // epilogue: lane (kk, m) ends with rows rb + 16 h + 4 kk .. + 3 of
        // column m in registers (the FP64 result rows are regrouped across
        // the four lanes of a column first), written as one vector
#pragma unroll
        for (int r = 0; r < RN; r++) {
            const int j = (jb0 + r) * 16 + m;
            T *yj = Y + (int64_t)min(j, q - 1) * ldy;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const acc_t v = rows4<T>(h == 0 ? acc0[r] : acc1[r], kk);
                const int64_t row = rb + 16 * h + 4 * kk;
                if (j >= q) continue;
                if (row + 4 <= n) {
                    store_rows4<T>(yj + row, v, al, be);
                } else {
#pragma unroll
                    for (int t = 0; t < 4; t++)
                        if (row + t < n) {
                            const T vt = (T)v[t];
                            yj[row + t] = (be == T(0)) ? ((al == T(1)) ? vt : al * vt) : be * yj[row + t] + al * vt;
                        }
                }
            }
        }
    }
}

template <typename T, int RB>
void launch_lincomb_mfma(int rn, int64_t n, const void *X, int64_t ldx, int p, void *Y, int64_t ldy, int q,
                         const void *Cp, int nkb, int nqb, double alpha, double beta)
{
    const int grid = (int)((n + 64 * RB - 1) / (64 * RB));
#define GH_LC(RN_)                                                                                             \
    if (rn == RN_) {                                                                                            \
        k_lincomb_mfma<T, RN_, RB><<<grid, kThreads, 0, ctx().stream>>>(                                        \
            n, (const T *)X, ldx, p, (T *)Y, ldy, q, (const T *)Cp, nkb, nqb, alpha, beta);                     \
        return;                                                                                                 \
    }
    GH_LC(1) GH_LC(2) GH_LC(3) GH_LC(4) GH_LC(5) GH_LC(6) GH_LC(7) GH_LC(8)
#undef GH_LC
}

// ---------------------------------------------------------------- LinComb (thin)
// p <= PM, q <= QM: C travels in the kernel arguments; each thread owns VR
// consecutive rows (one 16-byte vector per column) and forms
// y_j = beta y_j + alpha sum_i x_i C(i, j), the sum as fma from zero in i order.
struct ThinCoef {
    double c[64];  // C(i, j) at j * p + i
};

template <typename T, int PM, int QM>
__global__ __launch_bounds__(kThreads) void k_lincomb_thin(int64_t n, const T *__restrict__ X, int64_t ldx, int p,
                                                           T *__restrict__ Y, int64_t ldy, int q, ThinCoef cf,
                                                           double alpha, double beta)
{
    constexpr int VR = 16 / sizeof(T);
    typedef T vec_t __attribute__((ext_vector_type(VR)));
    T c[PM][QM];
#pragma unroll
    for (int i = 0; i < PM; i++)
#pragma unroll
        for (int j = 0; j < QM; j++) c[i][j] = (i < p && j < q) ? (T)cf.c[j * p + i] : T(0);
    const T al = (T)alpha, be = (T)beta;
    const int64_t stride = (int64_t)gridDim.x * kThreads * VR;
    for (int64_t r = ((int64_t)blockIdx.x * kThreads + threadIdx.x) * VR; r < n; r += stride) {
        T x[PM][VR];
        const bool full = r + VR <= n;
#pragma unroll
        for (int i = 0; i < PM; i++) {
            if (i < p) {
                const T *xi = X + (int64_t)i * ldx + r;
                if (full) {
                    const vec_t v = *reinterpret_cast<const vec_t *>(xi);
#pragma unroll
                    for (int t = 0; t < VR; t++) x[i][t] = v[t];
                } else {
#pragma unroll
                    for (int t = 0; t < VR; t++) x[i][t] = (r + t < n) ? xi[t] : T(0);
                }
            }
        }
#pragma unroll
        for (int j = 0; j < QM; j++) {
            if (j >= q) break;
            T *yj = Y + (int64_t)j * ldy + r;
            T out[VR];
#pragma unroll
            for (int t = 0; t < VR; t++) {
                T acc = T(0);
#pragma unroll
                for (int i = 0; i < PM; i++)
                    if (i < p) acc = fma(x[i][t], c[i][j], acc);
                out[t] = acc;
            }
            if (full) {
                vec_t y;
                if (be != T(0)) y = *reinterpret_cast<const vec_t *>(yj);
#pragma unroll
                for (int t = 0; t < VR; t++)
                    y[t] = (be == T(0)) ? ((al == T(1)) ? out[t] : al * out[t]) : be * y[t] + al * out[t];
                *reinterpret_cast<vec_t *>(yj) = y;
            } else {
#pragma unroll
                for (int t = 0; t < VR; t++)
                    if (r + t < n)
                        yj[t] = (be == T(0)) ? ((al == T(1)) ? out[t] : al * out[t]) : be * yj[t] + al * out[t];
            }
        }
    }
}

template <typename T>
void launch_lincomb_thin(int64_t n, const void *X, int64_t ldx, int p, void *Y, int64_t ldy, int q,
                         const ThinCoef &cf, double alpha, double beta)
{
    constexpr int VR = 16 / sizeof(T);
    const int64_t threads = (n + VR - 1) / VR;
    const int grid = (int)std::min<int64_t>(8192, std::max<int64_t>(1, (threads + kThreads - 1) / kThreads));
    const int pm = p <= 1 ? 1 : p <= 2 ? 2 : p <= 4 ? 4 : 8;
    const int qm = q <= 1 ? 1 : q <= 2 ? 2 : q <= 4 ? 4 : 8;
#define GH_LT(P_, Q_)                                                                                          \
    if (pm == P_ && qm == Q_) {                                                                                 \
        k_lincomb_thin<T, P_, Q_><<<grid, kThreads, 0, ctx().stream>>>(n, (const T *)X, ldx, p, (T *)Y, ldy, q, \
                                                                       cf, alpha, beta);                        \
        return;                                                                                                 \
    }
    GH_LT(1, 1) GH_LT(1, 2) GH_LT(1, 4) GH_LT(1, 8)
    GH_LT(2, 1) GH_LT(2, 2) GH_LT(2, 4) GH_LT(2, 8)
    GH_LT(4, 1) GH_LT(4, 2) GH_LT(4, 4) GH_LT(4, 8)
    GH_LT(8, 1) GH_LT(8, 2) GH_LT(8, 4) GH_LT(8, 8)
#undef GH_LT
}

template <typename T, int PM, int QM>
void launch_thin(int grid, int64_t n, const void *V, int64_t ldv, int p, const void *W, int64_t ldw, int q,
                 int transpose, int ldo, double *partial)
{
    k_gram_thin<T, PM, QM><<<grid, kThreads, 0, ctx().stream>>>(n, (const T *)V, ldv, p, (const T *)W, ldw, q,
                                                                transpose, ldo, partial);
}

template <typename T>
void launch_thin_sized(int grid, int64_t n, const void *V, int64_t ldv, int p, const void *W, int64_t ldw, int q,
                       int transpose, int ldo, double *partial)
{
    const int pm = p <= 1 ? 1 : p <= 2 ? 2 : 4;
    const int qm = q <= 1 ? 1 : q <= 2 ? 2 : q <= 4 ? 4 : 8;
#define GH_THIN(P_, Q_) \
    if (pm == P_ && qm == Q_) return launch_thin<T, P_, Q_>(grid, n, V, ldv, p, W, ldw, q, transpose, ldo, partial);
    GH_THIN(1, 1) GH_THIN(1, 2) GH_THIN(1, 4) GH_THIN(1, 8)
    GH_THIN(2, 1) GH_THIN(2, 2) GH_THIN(2, 4) GH_THIN(2, 8)
    GH_THIN(4, 1) GH_THIN(4, 2) GH_THIN(4, 4) GH_THIN(4, 8)
#undef GH_THIN
}

struct GramShape {
    int WP, WQ, GP, GQ;
};

GramShape gram_shape(int p, int q)
{
    if (p <= 16 && q <= 16) return {1, 1, 1, 1};  // 16 x 16 tiles, rows split 4 ways
    if (p <= 32 && q <= 32) return {2, 2, 1, 1};  // 32 x 32, rows split 4 ways
    if (q <= 16) return {2, 1, 2, 1};             // 64 x 16, rows split 2 ways
    if (p <= 16) return {1, 2, 1, 2};             // 16 x 64, rows split 2 ways
    return {2, 2, 2, 2};                          // 64 x 64
}

template <typename T>
void launch_gram_mfma(const GramShape &g, int grid, int64_t n, const void *V, int64_t ldv, int p, const void *W,
                      int64_t ldw, int q, int tp, int tq, int nchunk, int64_t rpc, int upper, double *partial)
{
#define GH_GRAM(WP_, WQ_, GP_, GQ_)                                                                             \
    if (g.WP == WP_ && g.WQ == WQ_ && g.GP == GP_ && g.GQ == GQ_) {                                             \
        k_gram_mfma<T, WP_, WQ_, GP_, GQ_><<<grid, kThreads, 0, ctx().stream>>>(                                \
            n, (const T *)V, ldv, p, (const T *)W, ldw, q, tp, tq, nchunk, rpc, upper, partial);                \
        return;                                                                                                 \
    }
    GH_GRAM(1, 1, 1, 1)
    GH_GRAM(2, 2, 1, 1)
    GH_GRAM(2, 1, 2, 1)
    GH_GRAM(1, 2, 1, 2)
    GH_GRAM(2, 2, 2, 2)
#undef GH_GRAM
}

// Blocks of up to 16 columns of tiles (74 KiB of LDS, at most 8 tiles per
// wavefront, 128 registers): two workgroups per CU
bool slab_narrow(const SlabShape &s) { return s.MB + s.NB <= 16; }

size_t slab_lds(const SlabShape &s) { return (size_t)(s.MB + s.NB) * 16 * 144 * 2; }

template <typename T>
void launch_gram_slab(const SlabShape &s, int grid, int64_t n, const void *V, int64_t ldv, int p, const void *W,
                      int64_t ldw, int q, int nchunk, int64_t rpc, int upper, double *partial)
{
    // run: by the bits to keep, not by speed (k_gram_slab)
    const bool small = p <= 64 && q <= 64, run = small || ((p > 256 || q > 256) && !slab_narrow(s));
    const int upt = small ? 2 : slab_narrow(s) ? 4 : 7;
#define GH_SLAB(NT_, UPT_, RUN_)                                                                                \
    if (s.NT <= NT_ && upt == UPT_ && run == RUN_) {                                                            \
        k_gram_slab<T, NT_, UPT_, RUN_><<<grid, kSlabThreads, slab_lds(s), ctx().stream>>>(                     \
            n, (const T *)V, ldv, p, (const T *)W, ldw, q, s.MB, s.NB, s.bp, s.bq, nchunk, rpc, upper, partial); \
        return;                                                                                                 \
    }
    GH_SLAB(1, 2, true) GH_SLAB(2, 2, true)
    GH_SLAB(1, 4, false) GH_SLAB(2, 4, false) GH_SLAB(3, 4, false) GH_SLAB(4, 4, false) GH_SLAB(5, 4, false)
    GH_SLAB(6, 4, false) GH_SLAB(7, 4, false) GH_SLAB(8, 4, false)
    GH_SLAB(2, 7, false) GH_SLAB(4, 7, false) GH_SLAB(6, 7, false) GH_SLAB(8, 7, false) GH_SLAB(10, 7, false)
    GH_SLAB(12, 7, false) GH_SLAB(14, 7, false) GH_SLAB(17, 7, false)
    GH_SLAB(3, 7, true) GH_SLAB(6, 7, true) GH_SLAB(10, 7, true) GH_SLAB(14, 7, true) GH_SLAB(17, 7, true)
#undef GH_SLAB
}

bool aligned32(const void *p) { return ((uintptr_t)p & 31u) == 0; }

}  // namespace

bool gram(int prec, int64_t n, const void *V, int64_t ldv, int p, const void *W, int64_t ldw, int q, double *G,
          int ldg, bool upper_only)
{
    if (p <= 0 || q <= 0) return true;
    if (failed()) return false;
    const size_t es = elem_size(prec);
    const int64_t pq = (int64_t)p * q;
    const bool thin = (p <= 4 && q <= 8) || (q <= 4 && p <= 8);
    // launch geometry and scratch first: growing the scratch synchronizes the
    // stream, which must not happen inside a profiled launch
    int nchunk = 0;
    int64_t rpc = 0;
    int tp = 1, tq = 1;
    GramShape g{1, 1, 1, 1};
    // slab kernel from 6 tiles of columns of V and W together; below, the
    // kernel without LDS, with more workgroups in flight, moves the data
    // faster.  4.1M rows, that one against the slabs, us: 60 x 16 FP64 556
    // against 635 and FP32 292 against 321, 32 x 32 438 against 623 and 261
    // against 318, but 40 x 40 1036 against 848 and 627 against 403
    const bool slab = !thin && (p + 15) / 16 + (q + 15) / 16 >= 6;
    SlabShape slab_sh{0, 0, 0, 0, 0};
    if (thin) {
        nchunk = (int)std::min<int64_t>(1024, std::max<int64_t>(1, (n + kThreads - 1) / kThreads));
    } else if (slab) {
        if (!aligned32(V) || !aligned32(W) || (ldv * es) % 32 || (ldw * es) % 32) {
            latch(170, "gram: operands are not 32-byte aligned");
            return false;
        }
        slab_sh = slab_shape((p + 15) / 16, (q + 15) / 16, upper_only);
        tp = slab_sh.bp;
        tq = slab_sh.bq;
        const int64_t slab_rows = 128 / (int64_t)es;
        const int64_t max_chunks = std::max<int64_t>(1, (n + slab_rows - 1) / slab_rows);
        // Chunks: 512 for up to 128 x 128 columns, in inverse proportion
        // beyond, but a workgroup for every CU (300 x 100, one block: 256
        // chunks and not 170) and whole rounds of them where there are several
        const int blocks = tp * tq;
        nchunk = 512 / (((p + 127) / 128) * ((q + 127) / 128));
        if (nchunk < 256) nchunk = (nchunk * blocks + 255) / 256 * 256 / blocks;
        nchunk = (int)std::min<int64_t>({(int64_t)kMaxChunks, max_chunks, std::max(1, nchunk)});
        rpc = (n + nchunk - 1) / nchunk;
        rpc = ((rpc + slab_rows - 1) / slab_rows) * slab_rows;
        nchunk = (int)((n + rpc - 1) / rpc);
    } else {
        if (!aligned32(V) || !aligned32(W) || (ldv * es) % 32 || (ldw * es) % 32) {
            latch(170, "gram: operands are not 32-byte aligned");
            return false;
        }
        g = gram_shape(p, q);
        const int TP = g.GP * g.WP * 16, TQ = g.GQ * g.WQ * 16;
        const int GK = 4 / (g.GP * g.GQ);
        const int R = prec == GCGE_HIP_FP64 ? 4 : 8;
        tp = (p + TP - 1) / TP;
        tq = (q + TQ - 1) / TQ;
        const int64_t unit = (int64_t)4 * R * GK;  // rows one workgroup step covers
        const int64_t max_chunks = std::max<int64_t>(1, (n + unit - 1) / unit);
        nchunk = (int)std::min<int64_t>({(int64_t)kMaxChunks, max_chunks,
                                         std::max<int64_t>(1, (kGramTargetWG + tp * tq - 1) / (tp * tq))});
        rpc = (n + nchunk - 1) / nchunk;
        rpc = ((rpc + unit - 1) / unit) * unit;
        nchunk = (int)((n + rpc - 1) / rpc);
    }
    double *partial = (double *)scratch(sizeof(double) * (size_t)nchunk * pq);
    if (!partial) return false;
    {
        ProfScope ps(thin ? K_GRAM_THIN : (prec == GCGE_HIP_FP64 ? K_GRAM_MFMA_F64 : K_GRAM_MFMA_F32),
                     (double)n * (p + q) * es + 8.0 * pq, 2.0 * (double)n * pq);
        if (thin) {
            // the kernel wants p <= 4: swap the operands and transpose the output otherwise
            const bool swap = p > 4;
            if (prec == GCGE_HIP_FP64) {
                if (!swap) launch_thin_sized<double>(nchunk, n, V, ldv, p, W, ldw, q, 0, p, partial);
                else launch_thin_sized<double>(nchunk, n, W, ldw, q, V, ldv, p, 1, p, partial);
            } else {
                if (!swap) launch_thin_sized<float>(nchunk, n, V, ldv, p, W, ldw, q, 0, p, partial);
                else launch_thin_sized<float>(nchunk, n, W, ldw, q, V, ldv, p, 1, p, partial);
            }
        } else if (slab) {
            const int64_t blocks = (int64_t)tp * tq * nchunk;
            const int grid = (int)(((blocks + 7) / 8) * 8);
            if (prec == GCGE_HIP_FP64)
                launch_gram_slab<double>(slab_sh, grid, n, V, ldv, p, W, ldw, q, nchunk, rpc, upper_only ? 1 : 0,
                                         partial);
            else
                launch_gram_slab<float>(slab_sh, grid, n, V, ldv, p, W, ldw, q, nchunk, rpc, upper_only ? 1 : 0,
                                        partial);
        } else {
            const int64_t blocks = (int64_t)tp * tq * nchunk;
            const int grid = (int)(((blocks + 7) / 8) * 8);
            if (prec == GCGE_HIP_FP64)
                launch_gram_mfma<double>(g, grid, n, V, ldv, p, W, ldw, q, tp, tq, nchunk, rpc, upper_only ? 1 : 0,
                                         partial);
            else
                launch_gram_mfma<float>(g, grid, n, V, ldv, p, W, ldw, q, tp, tq, nchunk, rpc, upper_only ? 1 : 0,
                                        partial);
        }
    }
    if (!check(hipGetLastError(), "k_gram")) return false;
    // the thin kernel writes every entry, so upper_only only prunes MFMA tiles
    const int up = (!thin && upper_only) ? 1 : 0;
    const int sums = (int)((pq + 63) / 64);
    unsigned long long seq = 0, *seqs = host_seq(sums, &seq);
    double *h = host_buf((size_t)pq);
    if (!h || !seqs) return false;
    k_sum_chunks<<<sums, kThreads, 0, ctx().stream>>>(partial, nchunk, p, pq, up, h, seqs, seq);
    if (!check(hipGetLastError(), "k_sum_chunks")) return false;
    if (!wait_seq(sums, seq)) return false;
    for (int j = 0; j < q; j++) std::memcpy(G + (int64_t)j * ldg, h + (int64_t)j * p, sizeof(double) * p);
    return true;
}

// Whether k_lincomb_rows is the faster kernel while X and Y fit the cache
// (blocks: the column blocks that k_lincomb_mfma multiplies).  Few input columns
// make a product of stores, which its many small wavefronts keep in flight;
// against it stand the blocks that it multiplies for nothing, as it takes 4 or 8
// at a time.  k_lincomb_mfma has enough workgroups from 65,536 rows on in FP64
// (16,384 rows are one per CU) and from 262,144 in FP32.  us, this kernel / that
// one:
//   FP32, 110,592 rows: 3 x 200 20.1 / 34.6, 20 x 128 19.2 / 29.4, 20 x 65 15.7 /
//   19.2, 64 x 65 29.0 / 27.7; 262,144: 12 x 128 31.1 / 31.6, 32 x 128 39.6 / 42.0
//   FP64, 65,025 rows: 3 x 300 34.1 / 50.8, 48 x 64 18.3 / 23.0, 20 x 65 19.3 /
//   19.8, 48 x 65 28.2 / 25.7; 16,384: 3 x 200 12.7 / 14.9, 48 x 48 12.3 / 11.6;
//   125,316: 12 x 65 27.2 / 21.6
static bool lincomb_by_rows(int prec, int64_t n, int p, int q, int blocks)
{
    const int nqb = (q + 15) / 16, mine = nqb <= 2 ? nqb : nqb <= 4 ? 4 : (nqb + 7) / 8 * 8;
    const double pad = (double)mine / blocks, weight = p * pad * pad;
    if (prec == GCGE_HIP_FP64)
        return q <= 32 ? p <= 64 : n < 65536 && (n >= 24576 || q > 96) && weight < 64;
    if (q <= 64) return p < 128 || weight <= 128;
    return n < 262144 && weight < (n < 65536 ? 256 : 100);
}

bool lincomb(int prec, int64_t n, const void *X, int64_t ldx, int p, void *Y, int64_t ldy, int q, const double *C,
             int ldc, double alpha, double beta)
{
    if (q <= 0 || n <= 0) return true;
    if (failed()) return false;
    if (p <= 0) {
        // empty sum: Y = beta Y
        std::vector<double> b(kMaxCols, beta), a(kMaxCols, 0.0);
        for (int c0 = 0; c0 < q; c0 += kMaxCols)
            launch_axpby(prec, n, Y, ldy, (char *)Y + (size_t)c0 * ldy * elem_size(prec), ldy,
                         std::min(kMaxCols, q - c0), a.data(), b.data(), nullptr);
        return !failed();
    }
    if (p <= 8 && q <= 8) {
        if (((uintptr_t)X & 15u) || ((uintptr_t)Y & 15u) || (ldx * elem_size(prec)) % 16 ||
            (ldy * elem_size(prec)) % 16) {
            latch(171, "lincomb: operands are not 16-byte aligned");
            return false;
        }
        ThinCoef cf;
        for (int j = 0; j < q; j++)
            for (int i = 0; i < p; i++) cf.c[j * p + i] = C[(int64_t)j * ldc + i];
        ProfScope ps(K_LINCOMB_THIN, (double)n * (p + q + (beta != 0.0 ? q : 0)) * elem_size(prec),
                     2.0 * (double)n * p * q);
        if (prec == GCGE_HIP_FP64) launch_lincomb_thin<double>(n, X, ldx, p, Y, ldy, q, cf, alpha, beta);
        else launch_lincomb_thin<float>(n, X, ldx, p, Y, ldy, q, cf, alpha, beta);
        return check(hipGetLastError(), "k_lincomb_thin");
    }
    if (((uintptr_t)X & 15u) || (ldx * elem_size(prec)) % 16 || ((uintptr_t)Y & 31u) ||
        (ldy * elem_size(prec)) % 32 || ldx < (n + 255) / 256 * 256) {
        latch(171, "lincomb: operands are not aligned or padded");
        return false;
    }
    const size_t es = elem_size(prec);
    // column blocks per pass (RN, at most 8) so that the passes are equal;
    // k_lincomb_rows: 1, 2 or 4, beyond 4 by two wavefronts (WC)
    const int nkb = (p + 3) / 4, nqb0 = (q + 15) / 16;
    const int groups = (nqb0 + 7) / 8, even = (nqb0 + groups - 1) / groups;
    const bool rows = (double)n * (p + q) * es <= kRowsBytes && lincomb_by_rows(prec, n, p, q, even * groups);
    const int wc = rows && nqb0 > 4 ? 2 : 1;
    const int rn = rows ? (nqb0 <= 2 ? nqb0 : 4) : even;
    const int nqb = ((nqb0 + rn * wc - 1) / (rn * wc)) * rn * wc;  // zero blocks pad the last pass
    const size_t ncp = (size_t)nkb * nqb * 64;
    const void *dC = nullptr;
    if (prec == GCGE_HIP_FP64) {
        std::vector<double> cp(ncp, 0.0);
        for (int kb = 0; kb < nkb; kb++)
            for (int jb = 0; jb < nqb; jb++)
                for (int l = 0; l < 64; l++) {
                    const int k = 4 * kb + l / 16, j = 16 * jb + l % 16;
                    if (k < p && j < q) cp[((size_t)kb * nqb + jb) * 64 + l] = C[(int64_t)j * ldc + k];
                }
        dC = stage_to_device(cp.data(), sizeof(double) * ncp);
    } else {
        std::vector<float> cp(ncp, 0.0f);
        for (int kb = 0; kb < nkb; kb++)
            for (int jb = 0; jb < nqb; jb++)
                for (int l = 0; l < 64; l++) {
                    const int k = 4 * kb + l / 16, j = 16 * jb + l % 16;
                    if (k < p && j < q) cp[((size_t)kb * nqb + jb) * 64 + l] = (float)C[(int64_t)j * ldc + k];
                }
        dC = stage_to_device(cp.data(), sizeof(float) * ncp);
    }
    if (!dC) return false;
    {
        ProfScope ps(prec == GCGE_HIP_FP64 ? K_LINCOMB_MFMA_F64 : K_LINCOMB_MFMA_F32,
                     (double)n * (p + q + (beta != 0.0 ? q : 0)) * elem_size(prec), 2.0 * (double)n * p * q);
#define GH_LR(T_, RN_, WC_)                                                                                    \
    k_lincomb_rows<T_, RN_, WC_><<<(int)((n + 128 / WC_ - 1) / (128 / WC_)), kThreads, 0, ctx().stream>>>(      \
        n, (const T_ *)X, ldx, p, (T_ *)Y, ldy, q, (const T_ *)dC, nkb, nqb, alpha, beta)
        // k_lincomb_mfma: as many 16-row blocks per wavefront as leave 512 workgroups
        const int want = (int)std::min<int64_t>(4, n / (64 * 512));
        if (rows && prec == GCGE_HIP_FP64) {
            if (wc == 2) GH_LR(double, 4, 2);
            else if (rn == 1) GH_LR(double, 1, 1);
            else if (rn == 2) GH_LR(double, 2, 1);
            else GH_LR(double, 4, 1);
        } else if (rows) {
            if (wc == 2) GH_LR(float, 4, 2);
            else if (rn == 1) GH_LR(float, 1, 1);
            else if (rn == 2) GH_LR(float, 2, 1);
            else GH_LR(float, 4, 1);
        } else if (prec == GCGE_HIP_FP64) {
            if (want >= 2) launch_lincomb_mfma<double, 2>(rn, n, X, ldx, p, Y, ldy, q, dC, nkb, nqb, alpha, beta);
            else launch_lincomb_mfma<double, 1>(rn, n, X, ldx, p, Y, ldy, q, dC, nkb, nqb, alpha, beta);
        } else {
            if (want >= 4) launch_lincomb_mfma<float, 4>(rn, n, X, ldx, p, Y, ldy, q, dC, nkb, nqb, alpha, beta);
            else if (want >= 2) launch_lincomb_mfma<float, 2>(rn, n, X, ldx, p, Y, ldy, q, dC, nkb, nqb, alpha, beta);
            else launch_lincomb_mfma<float, 1>(rn, n, X, ldx, p, Y, ldy, q, dC, nkb, nqb, alpha, beta);
        }
#undef GH_LR
    }
    return check(hipGetLastError(), "k_lincomb");
}

}  // namespace gh

// hip_kernels.hip -- device kernels of the gfx950 GCGE backend.
//
// Compiled with -ffp-contract=off: element-wise kernels (SpMM, axpby, CG
// update, residual) round every product and sum separately, in the order of
// the reference's CPU loops (CSR_MatDotVec and CSR_VecAxpby,
// app/csr/gcge_app_csr.c:297-365), so a row of A x or an axpby is
// bit-identical to the CPU result.  Reductions (dots, Gram) use explicit
// fma and a fixed two-stage order: deterministic run to run, but not the
// CPU's sequential summation order.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <climits>
#include <type_traits>
#include <vector>

#include "hip_common.h"

namespace gh {

namespace {

constexpr int kBlock = 256;
constexpr int kSpmmRows = 256;   // rows per SpMM workgroup (one row per thread)
constexpr int kSpmmCap = 2048;   // staged nonzeros per SpMM workgroup

struct ColScalars {
    double a[kMaxCols];
    double b[kMaxCols];
    int idx[kMaxCols];
    int use_idx;
};

// y = a x + b y with the branch rules of CSR_VecAxpby (gcge_app_csr.c:330-365)
template <typename T>
__device__ __forceinline__ T axpby_el(T a, T x, T b, T y)
{
    if (a == T(0)) return b * y;
    if (b == T(0)) return (a == T(1)) ? x : a * x;
    return a * x + b * y;
}

__device__ __forceinline__ double wave_sum(double v)
{
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    return v;
}

// sum over a 256-thread block; result valid in thread 0
__device__ __forceinline__ double block_sum(double v, double *sh)
{
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0) sh[wid] = v;
    __syncthreads();
    double r = 0.0;
    if (threadIdx.x == 0) r = (sh[0] + sh[1]) + (sh[2] + sh[3]);
    __syncthreads();
    return r;
}

int grid_1d(int64_t n, int cap)
{
    int64_t b = (n + kBlock - 1) / kBlock;
    if (b > cap) b = cap;
    if (b < 1) b = 1;
    return (int)b;
}

// ------------------------------------------------ element-wise streams
// Kernels that read and write whole columns are bound by memory.  Two things
// decide what they reach there (48 columns of 4.1M rows in FP32, 16 MB each,
// GB/s): accesses of 16 bytes per lane, one per thread (copy 5230 with 4-byte
// accesses, 6236), and, for blocks that no cache holds, loads and stores that
// bypass them (copy 6794, search update 5390 -> 6380, residual update 5300 ->
// 6540).  Blocks that the 256 MB cache holds are read back from it by the next
// kernel: 252 MB of a search update take 53 us through it and 64 around it, 865
// MB 263 and 244; kStreamBytes lies between.
constexpr double kStreamBytes = 384e6;

template <typename T>
constexpr int kWide = 16 / (int)sizeof(T);  // elements of a 16-byte access

template <bool NT, typename V>
__device__ __forceinline__ V load_as(const V *p)
{
    if constexpr (NT) return __builtin_nontemporal_load(p);
    else return *p;
}

template <bool NT, typename V>
__device__ __forceinline__ void store_as(V *p, V v)
{
    if constexpr (NT) __builtin_nontemporal_store(v, p);
    else *p = v;
}

// V consecutive rows of a column from row i < n on.  Those past n lie in the
// column's padding (mat_dinv's too) and feed nothing that is stored: without a
// branch for them several runs are loaded at a time; where paths meet, each
// would be waited for (search update with the diagonal, FP32, 10 columns of 1.03M
// rows from the cache: 37.2 us with the branches, 35.3 without).
template <typename T, int V, bool NT>
__device__ __forceinline__ void load_run(const T *c, int64_t i, T (&v)[V])
{
    typedef T vec __attribute__((ext_vector_type(V)));
    const vec x = load_as<NT>(reinterpret_cast<const vec *>(c + i));
#pragma unroll
    for (int t = 0; t < V; t++) v[t] = x[t];
}

template <typename T, int V, bool NT>
__device__ __forceinline__ void store_run(T *__restrict__ c, int64_t i, int64_t n, const T (&v)[V])
{
    typedef T vec __attribute__((ext_vector_type(V)));
    if (i + V <= n) {
        vec x;
#pragma unroll
        for (int t = 0; t < V; t++) x[t] = v[t];
        store_as<NT>(reinterpret_cast<vec *>(c + i), x);
    } else {
#pragma unroll
        for (int t = 0; t < V; t++)
            if (i + t < n) c[i + t] = v[t];
    }
}

// Row of this thread's run; the grid covers the n rows
template <int V>
__device__ __forceinline__ int64_t run_row()
{
    return ((int64_t)blockIdx.x * kBlock + threadIdx.x) * V;
}

// ---------------------------------------------------------------- axpby
template <typename T, int V, bool NT>
__global__ __launch_bounds__(kBlock) void k_axpby(int64_t n, const T *x, int64_t ldx, T *y, int64_t ldy,
                                                  ColScalars s)
{
    const int j = blockIdx.y;
    const int64_t i = run_row<V>();
    if (i >= n) return;
    const T *xj = x + (s.use_idx ? (int64_t)s.idx[j] : (int64_t)j) * ldx;
    T *yj = y + (int64_t)j * ldy;
    const T a = (T)s.a[j], b = (T)s.b[j];
    T xv[V], yv[V];
    const auto put = [&] {
#pragma unroll
        for (int t = 0; t < V; t++) yv[t] = axpby_el<T>(a, xv[t], b, yv[t]);
        store_run<T, V, NT>(yj, i, n, yv);
    };
    if (a == T(0)) {
        load_run<T, V, NT>(yj, i, yv);
        put();
    } else if (b == T(0)) {
        load_run<T, V, NT>(xj, i, xv);
        put();
    } else {
        load_run<T, V, NT>(xj, i, xv);
        load_run<T, V, NT>(yj, i, yv);
        put();
    }
}

// ---------------------------------------------------------------- dots
// Thread t of block b adds the rows 256 b + t + 256 gridDim.x m, m = 0, 1, ...
// in turn, U of them loaded at a time (the order of the sums does not depend
// on U); f(row, loaded) for each.
template <int U, typename LD, typename F>
__device__ __forceinline__ void strided_rows(int64_t n, LD load, F f)
{
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if constexpr (U > 1) {
        for (; i + (U - 1) * stride < n; i += U * stride) {
            decltype(load(i)) v[U];
#pragma unroll
            for (int u = 0; u < U; u++) v[u] = load(i + u * stride);
#pragma unroll
            for (int u = 0; u < U; u++) f(i + u * stride, v[u]);
        }
    }
    for (; i < n; i += stride) f(i, load(i));
}

template <typename T>
struct Pair {
    T a, b;
};

template <typename T, int U, bool NT>
__global__ __launch_bounds__(kBlock) void k_dots(int64_t n, const T *__restrict__ x, int64_t ldx,
                                                 const T *__restrict__ y, int64_t ldy,
                                                 double *__restrict__ partial)
{
    __shared__ double sh[4];
    const int j = blockIdx.y;
    const T *xj = x + (int64_t)j * ldx;
    const T *yj = y + (int64_t)j * ldy;
    double acc = 0.0;
    strided_rows<U>(
        n, [&](int64_t i) { return Pair<T>{load_as<NT>(xj + i), load_as<NT>(yj + i)}; },
        [&](int64_t, const Pair<T> &v) { acc = fma((double)v.a, (double)v.b, acc); });
    const double s = block_sum(acc, sh);
    if (threadIdx.x == 0) partial[(int64_t)j * gridDim.x + blockIdx.x] = s;
}

// sum_b partial[j * nb + b] for j = blockIdx.x, fixed order: thread t adds the
// partials t, t + 256, ... in turn (loaded 8 at a time: 16,000 partials, as of
// a 160^3 grid's SpMM, are 63 dependent round trips per thread otherwise: 15
// us for 48 columns, 8 so)
__device__ __forceinline__ double sum_row(const double *__restrict__ partial, int nb, double *sh)
{
    const double *row = partial + (int64_t)blockIdx.x * nb;
    double acc = 0.0;
    int b = threadIdx.x;
    for (; b + 7 * kBlock < nb; b += 8 * kBlock) {
        double v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = row[b + u * kBlock];
#pragma unroll
        for (int u = 0; u < 8; u++) acc += v[u];
    }
    for (; b < nb; b += kBlock) acc += row[b];
    return block_sum(acc, sh);
}

// out[j] = the sum, in device memory
__global__ __launch_bounds__(kBlock) void k_reduce_rows(const double *__restrict__ partial, int nb,
                                                        double *__restrict__ out)
{
    __shared__ double sh[4];
    const double s = sum_row(partial, nb, sh);
    if (threadIdx.x == 0) out[blockIdx.x] = s;
}

// out[j] = the sum and seqs[j] = the launch's number, in host memory
__global__ __launch_bounds__(kBlock) void k_reduce_rows_host(const double *__restrict__ partial, int nb,
                                                             double *__restrict__ out,
                                                             unsigned long long *__restrict__ seqs,
                                                             unsigned long long seq)
{
    __shared__ double sh[4];
    const double s = sum_row(partial, nb, sh);
    if (threadIdx.x == 0) {
        out[blockIdx.x] = s;
        __hip_atomic_store(seqs + blockIdx.x, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// ---------------------------------------------------------------- copy / swap / rows
template <typename TX, typename TY, int V, bool NT>
__global__ __launch_bounds__(kBlock) void k_copy(int64_t n, const TX *__restrict__ x, int64_t ldx,
                                                 TY *__restrict__ y, int64_t ldy)
{
    const int64_t i = run_row<V>();
    if (i >= n) return;
    TX xv[V];
    TY yv[V];
    load_run<TX, V, NT>(x + (int64_t)blockIdx.y * ldx, i, xv);
#pragma unroll
    for (int t = 0; t < V; t++) yv[t] = (TY)xv[t];
    store_run<TY, V, NT>(y + (int64_t)blockIdx.y * ldy, i, n, yv);
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_swap(int64_t n, T *__restrict__ x, int64_t ldx,
                                                 T *__restrict__ y, int64_t ldy)
{
    const int j = blockIdx.y;
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += stride) {
        T t = x[(int64_t)j * ldx + i];
        x[(int64_t)j * ldx + i] = y[(int64_t)j * ldy + i];
        y[(int64_t)j * ldy + i] = t;
    }
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_zero_rows(int64_t n, T *__restrict__ x, int64_t ldx,
                                                      const unsigned char *__restrict__ mask)
{
    const int j = blockIdx.y;
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += stride)
        if (mask[i]) x[(int64_t)j * ldx + i] = T(0);
}

// ---------------------------------------------------------------- SpMM
// Column sums of d[0..KC) over a wavefront by recursive halving: at level j
// (partner lane ^ (32 >> j)) each lane keeps half of its columns (the upper
// half if its bit is set) and adds the partner's copy of them; after log2 KC
// levels it holds one column, lane >> (6 - log2 KC), which the remaining
// levels sum over the lanes that share it.  7 exchanges for 4 columns, 10 for
// 8, instead of 6 per column; the order is fixed, so the sums are
// reproducible.
template <int KC>
__device__ __forceinline__ double wave_colsum(double (&d)[KC], int lane)
{
    static_assert(KC >= 1 && KC <= 64 && (KC & (KC - 1)) == 0, "KC is a power of two");
    int m = KC;
#pragma unroll
    for (int mask = 32; mask >= 1; mask >>= 1) {
        if (m > 1) {
            const bool hi = (lane & mask) != 0;
            const int h = m / 2;
#pragma unroll
            for (int i = 0; i < KC / 2; i++) {
                if (i < h) {
                    const double send = hi ? d[i] : d[i + h];
                    const double keep = hi ? d[i + h] : d[i];
                    d[i] = keep + __shfl_xor(send, mask, 64);
                }
            }
            m = h;
        } else {
            d[0] = d[0] + __shfl_xor(d[0], mask, 64);
        }
    }
    return d[0];
}

// One thread per row; the workgroup's nonzeros are staged in LDS when they
// fit; columns are processed KC at a time.  Each row sum starts at 0 and
// adds val*x in CSR order, as CSR_MatDotVec does; the nonzeros go in batches
// of kSpmmBatch whose column indices, values and X gathers are all issued
// before the first product is added, so a row costs one memory round trip
// per batch rather than one per nonzero.  With DOT, the workgroup also
// writes partial[j * nblk + blk] = sum_r X(r,j) Y(r,j) (wavefront sums by
// wave_colsum, combined in LDS in a fixed order) at partial[j * pstride +
// blk].  Rows with more than long_thr entries are left to k_spmm_long.
// STREAM (used for FP32): row blocks are renumbered so that each XCD walks a
// contiguous range of rows (the plane neighbours of a stencil stay in its
// L2), and the matrix and Y, each touched once, bypass the caches
// (non-temporal) to leave L2 to X.
constexpr int kSpmmBatch = 4;

template <typename T, bool DOT, int KC, bool STREAM>
__global__ __launch_bounds__(kSpmmRows) void k_spmm(int n, const int *__restrict__ rowptr,
                                                    const int *__restrict__ col,
                                                    const T *__restrict__ val,
                                                    const T *__restrict__ X, int64_t ldx,
                                                    T *__restrict__ Y, int64_t ldy, int k,
                                                    ColScalars g, double *__restrict__ partial, int nblk,
                                                    int long_thr, int pstride)
{
    __shared__ int s_col[kSpmmCap];
    __shared__ T s_val[kSpmmCap];
    __shared__ double sdot[DOT ? kMaxCols : 1][4];
    int blk = blockIdx.x;
    if (STREAM) {
        const int per = (int)(gridDim.x >> 3);
        blk = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    }
    if (blk >= nblk) return;  // uniform per workgroup (grid rounded up to 8)
    const int r0 = blk * kSpmmRows;
    const int r = r0 + threadIdx.x;
    const int rend = min(r0 + kSpmmRows, n);
    const int e0 = rowptr[r0];
    const int e1 = rowptr[rend];
    const bool staged = (e1 - e0) <= kSpmmCap;
    if (staged) {
        for (int e = e0 + threadIdx.x; e < e1; e += kSpmmRows) {
            if (STREAM) {
                s_col[e - e0] = __builtin_nontemporal_load(col + e);
                s_val[e - e0] = __builtin_nontemporal_load(val + e);
            } else {
                s_col[e - e0] = col[e];
                s_val[e - e0] = val[e];
            }
        }
    }
    __syncthreads();
    int s = 0, t = 0;
    if (r < n) {
        s = rowptr[r];
        t = rowptr[r + 1];
    }
    const bool active = r < n && t - s <= long_thr;  // long rows: k_spmm_long
    if (!active) t = s;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int rs = r < n ? r : 0;  // a row index that is safe to gather
    for (int c0 = 0; c0 < k; c0 += KC) {
        const T *xb[KC];
#pragma unroll
        for (int kk = 0; kk < KC; kk++) {
            int c = min(c0 + kk, k - 1);
            int64_t xc = g.use_idx ? (int64_t)g.idx[c] : (int64_t)c;
            xb[kk] = X + xc * ldx;
        }
        T acc[KC];
#pragma unroll
        for (int kk = 0; kk < KC; kk++) acc[kk] = T(0);
        for (int e = s; e < t; e += kSpmmBatch) {
            const int cnt = t - e;  // > 0; the batch holds min(cnt, kSpmmBatch)
            int cj[kSpmmBatch];
            T v[kSpmmBatch];
#pragma unroll
            for (int u = 0; u < kSpmmBatch; u++) {
                if (u < cnt) {
                    if (staged) {
                        cj[u] = s_col[e + u - e0];
                        v[u] = s_val[e + u - e0];
                    } else if (STREAM) {
                        cj[u] = __builtin_nontemporal_load(col + e + u);
                        v[u] = __builtin_nontemporal_load(val + e + u);
                    } else {
                        cj[u] = col[e + u];
                        v[u] = val[e + u];
                    }
                } else {
                    cj[u] = rs;
                    v[u] = T(0);
                }
            }
            T xv[kSpmmBatch][KC];
#pragma unroll
            for (int u = 0; u < kSpmmBatch; u++)
#pragma unroll
                for (int kk = 0; kk < KC; kk++) xv[u][kk] = (u < cnt) ? xb[kk][cj[u]] : T(0);
#pragma unroll
            for (int u = 0; u < kSpmmBatch; u++)
                if (u < cnt) {
#pragma unroll
                    for (int kk = 0; kk < KC; kk++) acc[kk] = acc[kk] + v[u] * xv[u][kk];
                }
        }
        double d[KC];
#pragma unroll
        for (int kk = 0; kk < KC; kk++) {
            const int c = c0 + kk;
            if (active && c < k) {
                if (STREAM) __builtin_nontemporal_store(acc[kk], Y + (int64_t)c * ldy + r);
                else Y[(int64_t)c * ldy + r] = acc[kk];
            }
            if (DOT) d[kk] = (active && c < k) ? (double)xb[kk][r] * (double)acc[kk] : 0.0;
        }
        if (DOT) {
            const double colsum = wave_colsum<KC>(d, lane);
            constexpr int L = KC == 1 ? 0 : KC == 2 ? 1 : KC == 4 ? 2 : KC == 8 ? 3 : KC == 16 ? 4 : 5;
            const int c = c0 + (lane >> (6 - L));
            if ((lane & ((64 >> L) - 1)) == 0 && c < k) sdot[c][wid] = colsum;
        }
    }
    if (DOT) {
        __syncthreads();
        for (int c = threadIdx.x; c < k; c += kSpmmRows)
            partial[(int64_t)c * pstride + blk] = (sdot[c][0] + sdot[c][1]) + (sdot[c][2] + sdot[c][3]);
    }
}

// The rows longer than kLongRow: one wavefront per row (four per workgroup),
// lane l taking column c0 + l, so every column's sum runs over the row in CSR
// order from 0, as in k_spmm (bit-exact); the row's entries go in batches of
// kLongBatch whose column indices and values are read once for the
// wavefront and whose X gathers are all issued before the first product is
// added.  With DOT, the row's X(r,j) Y(r,j) goes to partial[j * pstride +
// pbase + li].
constexpr int kLongBatch = 8;

template <typename T, bool DOT>
__global__ __launch_bounds__(kSpmmRows) void k_spmm_long(const int *__restrict__ rowptr, const int *__restrict__ col,
                                                         const T *__restrict__ val, const T *__restrict__ X,
                                                         int64_t ldx, T *__restrict__ Y, int64_t ldy, int k,
                                                         ColScalars g, const int *__restrict__ long_rows, int nlong,
                                                         double *__restrict__ partial, int pstride, int pbase)
{
    const int lane = threadIdx.x & 63;
    const int li = blockIdx.x * (kSpmmRows / 64) + (threadIdx.x >> 6);
    if (li >= nlong) return;  // uniform per wavefront; no workgroup barrier here
    const int r = long_rows[li];
    const int s = rowptr[r], t = rowptr[r + 1];
    for (int c0 = 0; c0 < k; c0 += 64) {
        const int c = c0 + lane;
        const bool live = c < k;
        const int cc = live ? c : k - 1;
        const T *xc = X + (g.use_idx ? (int64_t)g.idx[cc] : (int64_t)cc) * ldx;
        T acc = T(0);
        for (int e = s; e < t; e += kLongBatch) {
            const int cnt = t - e;
            int cj[kLongBatch];
            T v[kLongBatch], xv[kLongBatch];
#pragma unroll
            for (int u = 0; u < kLongBatch; u++) {
                cj[u] = u < cnt ? col[e + u] : r;
                v[u] = u < cnt ? val[e + u] : T(0);
            }
#pragma unroll
            for (int u = 0; u < kLongBatch; u++) xv[u] = xc[cj[u]];
#pragma unroll
            for (int u = 0; u < kLongBatch; u++)
                if (u < cnt) acc = acc + v[u] * xv[u];
        }
        if (live) {
            Y[(int64_t)c * ldy + r] = acc;
            if (DOT) partial[(int64_t)c * pstride + pbase + li] = (double)xc[r] * (double)acc;
        }
    }
}

// ------------------------------------------------- SpMM, staged row blocks
// The column-gather kernel above reads, for every stored entry and column,
// X(col, j) straight from memory; on a stencil the seven gathers of a row hit
// the same few cache lines, but the L1 keeps almost none of them, so each
// column costs about eight times its own bytes in L2 requests.  Here a row
// block's workgroup first copies every X row its entries read -- its own 256
// rows, then the other rows its entries reference ("extras", listed once per
// block at matrix creation, sorted) -- for KC columns into LDS, with
// coalesced loads, and the rows then read their entries' values from LDS
// through 16-bit local column indices (also built at creation).  Each row's
// first ME entries (local indices in pairs, and values) stay in registers for
// all columns: 8 for stencils of up to 8 entries per row, 28 for the 27-point
// matrices, whose products are then bound by LDS reads (27 x 8 bytes per row
// and column) and not by re-reading 10 bytes per entry and pass.  With 28 in
// FP64 the compiler's own choice is 207 registers and two wavefronts per
// SIMD; three are asked for.  27-point matrix of a 96^3 grid, 50 columns:
// 0.45 ms in FP64 and 0.25 in FP32, against 2.09 and 0.93 gathered from a
// row-major copy of X (k_spmm_rows).  Y bypasses the caches at every size, which
// leaves them to X's faces (us, FP32 48 columns of 160^3 502 -> 481, FP64 40
// columns of a 1024^2 grid 168 -> 156, FP32 60 columns of 700^2 53 -> 45; the
// matrix that way: 160^3 502 -> 557, its lines serve several loads).  Every sum
// still runs over the row in CSR order from 0, so Y is bit-identical to
// k_spmm's.  Rows longer than long_thr are left to k_spmm_long.  Row blocks
// are numbered so that each XCD walks a contiguous range of rows (a stencil's
// plane neighbours stay in its L2).

// A slot holds KC consecutive columns of one X row.  Slots lie in planes of
// 16 bytes (plane h: columns h * E .. h * E + E - 1 of every slot), so the
// lanes of a wavefront that read neighbouring slots read consecutive 16-byte
// words: with a slot's 32 bytes (FP64, KC = 4) side by side the 16-byte reads
// step over every second word and each meets a bank twice.
template <typename T, int KC>
struct Slots {
    static constexpr int NP = KC * (int)sizeof(T) > 16 ? KC * (int)sizeof(T) / 16 : 1;
    static constexpr int E = KC / NP;
    struct alignas(E * sizeof(T)) Part {
        T v[E];
    };
    struct Row {
        T v[KC];
    };
    __device__ static __forceinline__ Row get(const Part *s, int cap, int slot)
    {
        Row x;
#pragma unroll
        for (int h = 0; h < NP; h++) {
            const Part p = s[h * cap + slot];
#pragma unroll
            for (int e = 0; e < E; e++) x.v[h * E + e] = p.v[e];
        }
        return x;
    }
    __device__ static __forceinline__ void put(Part *s, int cap, int slot, const Row &x)
    {
#pragma unroll
        for (int h = 0; h < NP; h++) {
            Part p;
#pragma unroll
            for (int e = 0; e < E; e++) p.v[e] = x.v[h * E + e];
            s[h * cap + slot] = p;
        }
    }
};

// The first ME entries of one row in registers: slots in pairs, values.
template <typename T, int ME>
struct RowHead {
    unsigned lc[ME / 2];
    T v[ME];
    __device__ __forceinline__ void load(const unsigned short *__restrict__ lcol, const T *__restrict__ val, int s,
                                         int cnt)
    {
#pragma unroll
        for (int u = 0; u < ME; u += 2) {
            const unsigned a = u < cnt ? lcol[s + u] : 0, b = u + 1 < cnt ? lcol[s + u + 1] : 0;
            lc[u / 2] = a | (b << 16);
            v[u] = u < cnt ? val[s + u] : T(0);
            v[u + 1] = u + 1 < cnt ? val[s + u + 1] : T(0);
        }
    }
    __device__ __forceinline__ int slot(int u) const
    {
        return (int)((u & 1) ? lc[u / 2] >> 16 : lc[u / 2] & 0xffffu);
    }
};

// Extras of a block that each thread holds in registers one pass ahead; the
// others load when their pass begins.
template <int ME>
constexpr int halo_prefetch = ME > 8 ? 2 : 1;

template <typename T, bool DOT, int KC, int ME>
__global__ __launch_bounds__(kSpmmRows, ME > 8 ? 3 : 1) void k_spmm_halo(int n, const int *__restrict__ rowptr,
                                                         const unsigned short *__restrict__ lcol,
                                                         const T *__restrict__ val, const int *__restrict__ brows,
                                                         const int *__restrict__ hptr, const int *__restrict__ hcol,
                                                         const T *__restrict__ X, int64_t ldx, T *__restrict__ Y,
                                                         int64_t ldy, int ktot, int kper, ColScalars g,
                                                         double *__restrict__ partial, int nblk, int long_thr,
                                                         int pstride, int hcap)
{
    using S = Slots<T, KC>;
    using Row = typename S::Row;
    constexpr int NE = halo_prefetch<ME>;
    extern __shared__ __align__(16) unsigned char halo_smem[];
    typename S::Part *sx = reinterpret_cast<typename S::Part *>(halo_smem);  // [NP][hcap]
    __shared__ double sdot[DOT ? kMaxCols : 1][4];
    const int per = (int)(gridDim.x >> 3);
    const int blk = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if (blk >= nblk) return;  // uniform per workgroup (grid rounded up to 8)
    const int k0 = blockIdx.y * kper, k = min(ktot, k0 + kper);  // this workgroup's columns
    const int tid = threadIdx.x, p = blk * kSpmmRows + tid;
    const int r = brows ? brows[p] : p < n ? p : -1;
    const int h0 = hptr[blk], nh = hptr[blk + 1] - h0;
    const int *hc = hcol + h0;
    int s = 0, t = 0;
    if (r >= 0) {
        s = rowptr[r];
        t = rowptr[r + 1];
    }
    const bool active = r >= 0 && t - s <= long_thr;  // long rows: k_spmm_long
    const int cnt = active ? t - s : 0;
    RowHead<T, ME> row;
    row.load(lcol, val, s, cnt);
    const int lane = tid & 63, wid = tid >> 6;
    // the own row and the first NE extras of this thread for the next KC
    // columns are loaded into registers while the current columns are
    // multiplied, so that a workgroup's loads overlap its own work
    int erow[NE];
#pragma unroll
    for (int i = 0; i < NE; i++) erow[i] = tid + i * kSpmmRows < nh ? hc[tid + i * kSpmmRows] : 0;
    Row pown, pext[NE];
    auto xcols = [&](int c0, const T *(&xc)[KC]) {
#pragma unroll
        for (int cc = 0; cc < KC; cc++) {
            const int c = min(c0 + cc, k - 1);
            xc[cc] = X + (g.use_idx ? (int64_t)g.idx[c] : (int64_t)c) * ldx;
        }
    };
    auto prefetch = [&](int c0) {
        const T *xc[KC];
        xcols(c0, xc);
        if (r >= 0) {
#pragma unroll
            for (int cc = 0; cc < KC; cc++) pown.v[cc] = xc[cc][r];
        }
#pragma unroll
        for (int i = 0; i < NE; i++)
            if (tid + i * kSpmmRows < nh) {
#pragma unroll
                for (int cc = 0; cc < KC; cc++) pext[i].v[cc] = xc[cc][erow[i]];
            }
    };
    prefetch(k0);
    for (int c0 = k0; c0 < k; c0 += KC) {
        if (r >= 0) S::put(sx, hcap, tid, pown);
#pragma unroll
        for (int i = 0; i < NE; i++)
            if (tid + i * kSpmmRows < nh) S::put(sx, hcap, kSpmmRows + tid + i * kSpmmRows, pext[i]);
        if (nh > NE * kSpmmRows) {
            const T *xc[KC];
            xcols(c0, xc);
            for (int j = tid + NE * kSpmmRows; j < nh; j += kSpmmRows) {
                const int er = hc[j];
                Row w;
#pragma unroll
                for (int cc = 0; cc < KC; cc++) w.v[cc] = xc[cc][er];
                S::put(sx, hcap, kSpmmRows + j, w);
            }
        }
        const Row xo = pown;
        __syncthreads();
        if (c0 + KC < k) prefetch(c0 + KC);
        T acc[KC];
#pragma unroll
        for (int cc = 0; cc < KC; cc++) acc[cc] = T(0);
#pragma unroll
        for (int u = 0; u < ME; u++)
            if (u < cnt) {
                const Row x = S::get(sx, hcap, row.slot(u));
#pragma unroll
                for (int cc = 0; cc < KC; cc++) acc[cc] = acc[cc] + row.v[u] * x.v[cc];
            }
        for (int e = s + ME; e < s + cnt; e++) {
            const Row x = S::get(sx, hcap, lcol[e]);
            const T ve = val[e];
#pragma unroll
            for (int cc = 0; cc < KC; cc++) acc[cc] = acc[cc] + ve * x.v[cc];
        }
        double d[KC];
#pragma unroll
        for (int cc = 0; cc < KC; cc++) {
            const int c = c0 + cc;
            if (active && c < k) store_as<true>(Y + (int64_t)c * ldy + r, acc[cc]);
            if (DOT) d[cc] = (active && c < k) ? (double)xo.v[cc] * (double)acc[cc] : 0.0;
        }
        if (DOT) {
            const double colsum = wave_colsum<KC>(d, lane);
            constexpr int L = KC == 1 ? 0 : KC == 2 ? 1 : KC == 4 ? 2 : KC == 8 ? 3 : KC == 16 ? 4 : 5;
            const int c = c0 + (lane >> (6 - L));
            if ((lane & ((64 >> L) - 1)) == 0 && c < k) sdot[c][wid] = colsum;
        }
        __syncthreads();  // the next chunk overwrites sx
    }
    if (DOT) {
        for (int c = k0 + tid; c < k; c += kSpmmRows)
            partial[(int64_t)c * pstride + blk] = (sdot[c][0] + sdot[c][1]) + (sdot[c][2] + sdot[c][3]);
    }
}

// ------------------------------------------------- SpMM, row-major gather
// Matrices whose column indices scatter (random graphs) make the column-major
// gather of k_spmm touch one cache line per stored entry and column, and
// matrices whose rows average more than 8 entries overflow its LDS stage, so
// that each thread reads its own row's indices and values.  For both
// (HIP_MAT::gather_rows, chosen at creation) the k columns are first copied into a
// row-major staging block Xt, row r holding X(r, 0..kp) (kp: k rounded up to
// the lane group G), and k_spmm_rows gathers whole row segments: G lanes of a
// wavefront take G consecutive columns of one row, so a stored entry costs
// one contiguous G * sizeof(T) read.  Every sum still runs over its row in
// CSR order from 0, so Y is bit-identical to the column-major path.

// Xt(r, c) = X(:, c)(r) (c < k; 0 for k <= c < kp): 64 x 64 tiles through LDS.
template <typename T>
__global__ __launch_bounds__(256) void k_rows_from_cols(int n, const T *__restrict__ X, int64_t ldx, int k,
                                                        ColScalars g, int kp, T *__restrict__ Xt)
{
    __shared__ T tile[64][65];
    const int r0 = blockIdx.x * 64, cb = blockIdx.y * 64;
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    for (int cc = ty; cc < 64; cc += 4) {
        const int c = cb + cc, r = r0 + tx;
        T v = T(0);
        if (c < k && r < n) v = X[(g.use_idx ? (int64_t)g.idx[c] : (int64_t)c) * ldx + r];
        tile[cc][tx] = v;
    }
    __syncthreads();
    const int kpe = min(64, kp - cb), rows = min(64, n - r0);
    for (int q = threadIdx.x; q < rows * kpe; q += 256) {
        const int rr = q / kpe, cc = q - rr * kpe;
        Xt[(int64_t)(r0 + rr) * kp + cb + cc] = tile[cc][rr];
    }
}

__device__ __forceinline__ float lane_bcast(float v, int src)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), src));
}

__device__ __forceinline__ double lane_bcast(double v, int src)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, src);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), src);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

constexpr int kRowsBatch = 8;       // gathers in flight per lane, short rows
constexpr int kLongRowsBatch = 32;  // gathers in flight per lane, long rows

// Sum over the CSR row [s, t) of val(e) * Xt(col(e), cc), in CSR order from
// 0, for a whole wavefront (lane = column): the row's column indices and
// values are read 64 at a time and broadcast from the lane holding them
// (readlane), so the gathers have uniform row addresses and kLongRowsBatch
// of them are in flight.  TA is the accumulation type (T for the SpMM, FP64
// for the residual check); rfill is a valid row for the idle slots.  Called
// by all 64 lanes together.
template <typename TA, typename TV, typename TX>
__device__ __forceinline__ TA wave_row_sum(const int *__restrict__ col, const TV *__restrict__ val, int s, int t,
                                           const TX *__restrict__ Xt, int kp, int cc, int rfill, int lane)
{
    TA acc = TA(0);
    for (int e = s; e < t; e += 64) {
        const int cnt = min(64, t - e);
        const int cv = lane < cnt ? col[e + lane] : rfill;
        const TV vv = lane < cnt ? val[e + lane] : TV(0);
#pragma unroll
        for (int h = 0; h < 64; h += kLongRowsBatch) {
            if (h < cnt) {
                TX xv[kLongRowsBatch];
#pragma unroll
                for (int u = 0; u < kLongRowsBatch; u++) {
                    const int cj = __builtin_amdgcn_readlane(cv, h + u);
                    xv[u] = Xt[(int64_t)cj * kp + cc];
                }
#pragma unroll
                for (int u = 0; u < kLongRowsBatch; u++)
                    if (h + u < cnt) acc = acc + lane_bcast(vv, h + u) * (TA)xv[u];
            }
        }
    }
    return acc;
}

// The same sum for one lane (row) of a lane group: kRowsBatch entries'
// gathers in flight; rfill is a valid row for the idle slots.
template <typename TA, typename TV, typename TX>
__device__ __forceinline__ TA lane_row_sum(const int *__restrict__ col, const TV *__restrict__ val, int s, int t,
                                           const TX *__restrict__ Xt, int kp, int c, int rfill)
{
    TA acc = TA(0);
    for (int e = s; e < t; e += kRowsBatch) {
        const int cnt = t - e;
        int cj[kRowsBatch];
        TV v[kRowsBatch];
        TX xv[kRowsBatch];
#pragma unroll
        for (int u = 0; u < kRowsBatch; u++) {
            cj[u] = u < cnt ? col[e + u] : rfill;
            v[u] = u < cnt ? val[e + u] : TV(0);
        }
#pragma unroll
        for (int u = 0; u < kRowsBatch; u++) xv[u] = Xt[(int64_t)cj[u] * kp + c];
#pragma unroll
        for (int u = 0; u < kRowsBatch; u++)
            if (u < cnt) acc = acc + v[u] * (TA)xv[u];
    }
    return acc;
}

// Rows handled by one workgroup of k_spmm_rows<G>: four wavefronts of
// max(16, 64 / G) rows each.
__host__ __device__ constexpr int rows_per_wg(int G) { return 4 * (64 / G > 16 ? 64 / G : 16); }

// Y(:, c0 + 0..G) = A X from the staging block Xt (grid.y: chunks of 64
// columns when G = 64).  Workgroups below nlb take the rows longer than
// long_thr, one wavefront per row with lane l on column c0 + l; the row's
// column indices and values are read 64 at a time and broadcast from the
// lane holding them (readlane), so the gathers have uniform row addresses
// and kLongRowsBatch of them are in flight.  The other workgroups take
// rows_per_wg(G) consecutive rows: lane l works on column c0 + l % G of row
// l / G (64 / G rows in flight per wavefront), the sums land in LDS and
// leave as contiguous column segments.  With DOT, sum_r X(r,c) Y(r,c) goes
// to partial[c * pstride + blk] per row workgroup and to
// partial[c * pstride + nblk + li] per long row.
template <typename T, bool DOT, int G>
__global__ __launch_bounds__(256) void k_spmm_rows(int n, const int *__restrict__ rowptr,
                                                   const int *__restrict__ col, const T *__restrict__ val,
                                                   const T *__restrict__ Xt, int kp, T *__restrict__ Y,
                                                   int64_t ldy, int k, const int *__restrict__ long_rows,
                                                   int nlong, int nlb, int long_thr,
                                                   double *__restrict__ partial, int pstride, int nblk)
{
    static_assert(G >= 2 && G <= 64 && (G & (G - 1)) == 0, "G is a power of two");
    constexpr int SG = 64 / G;
    constexpr int RWG = rows_per_wg(G);
    constexpr int RPW = RWG / 4;
    __shared__ T sY[G][RWG + 1];
    __shared__ unsigned char skip[RWG];
    __shared__ double sdot[DOT ? 4 : 1][G];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int c0 = blockIdx.y * 64;
    if ((int)blockIdx.x < nlb) {
        const int li = blockIdx.x * 4 + wid;
        if (li >= nlong) return;  // uniform per wavefront; this branch has no barrier
        const int r = long_rows[li];
        const int s = rowptr[r], t = rowptr[r + 1];
        const int c = c0 + lane;
        const bool live = c < k;
        const int cc = min(c, kp - 1);
        const T acc = wave_row_sum<T, T, T>(col, val, s, t, Xt, kp, cc, r, lane);
        if (live) {
            Y[(int64_t)c * ldy + r] = acc;
            if (DOT) partial[(int64_t)c * pstride + nblk + li] = (double)Xt[(int64_t)r * kp + cc] * (double)acc;
        }
        return;
    }
    const int blk = blockIdx.x - nlb;
    const int r0 = blk * RWG;
    const int cl = lane % G, sg = lane / G;
    const int c = c0 + cl;  // < kp: kp = G, or a multiple of 64 when G = 64
    const bool live = c < k;
    double dsum = 0.0;
    for (int i = sg; i < RPW; i += SG) {
        const int rl = wid * RPW + i, r = r0 + rl;
        int s = 0, t = 0;
        if (r < n) {
            s = rowptr[r];
            t = rowptr[r + 1];
        }
        const bool act = r < n && t - s <= long_thr;
        if (!act) t = s;
        const int rs = r < n ? r : 0;
        const T acc = lane_row_sum<T, T, T>(col, val, s, t, Xt, kp, c, rs);
        if (cl == 0) skip[rl] = act ? 0 : 1;
        sY[cl][rl] = acc;
        if (DOT && act && live) dsum += (double)Xt[(int64_t)r * kp + c] * (double)acc;
    }
    if (DOT) {
#pragma unroll
        for (int m = G; m < 64; m <<= 1) dsum += __shfl_xor(dsum, m, 64);
        if (sg == 0) sdot[wid][cl] = dsum;
    }
    __syncthreads();
    const int ncol = min(G, k - c0);
    for (int q = threadIdx.x; q < ncol * RWG; q += 256) {
        const int cc = q / RWG, rr = q - cc * RWG;
        const int r = r0 + rr;
        if (r < n && !skip[rr]) Y[(int64_t)(c0 + cc) * ldy + r] = sY[cc][rr];
    }
    if (DOT && (int)threadIdx.x < ncol)
        partial[(int64_t)(c0 + threadIdx.x) * pstride + blk] =
            (sdot[0][threadIdx.x] + sdot[1][threadIdx.x]) + (sdot[2][threadIdx.x] + sdot[3][threadIdx.x]);
}

// ---------------------------------------------------------------- residual
// r = A x - lambda B x (x when B is absent), in FP64 arithmetic whatever the
// storage precision of x, rounded as VecAxpby(-lambda, Bx, 1.0, Ax)
// (gcge_eigsol.c:579-588); partial sums of r.r, x.x and Bx.Bx per column.
template <typename TX, bool HASB>
__global__ __launch_bounds__(kSpmmRows) void k_residual(int n, const int *__restrict__ arp,
                                                        const int *__restrict__ acol,
                                                        const double *__restrict__ aval,
                                                        const int *__restrict__ brp,
                                                        const int *__restrict__ bcol,
                                                        const double *__restrict__ bval,
                                                        const TX *__restrict__ X, int64_t ldx, int k,
                                                        ColScalars g, double *__restrict__ partial)
{
    // The workgroup's rows of A are staged in LDS once and serve every
    // column; columns go in chunks of kResKC, each thread one row, and the
    // three sums of every column are reduced per wavefront into LDS and
    // combined after the last chunk (same order as block_sum).
    constexpr int kResKC = 4;
    __shared__ int s_col[kSpmmCap];
    __shared__ double s_val[kSpmmCap];
    __shared__ double sred[3 * kMaxCols][4];
    const int blk = blockIdx.x;
    const int r0 = blk * kSpmmRows;
    const int r = r0 + threadIdx.x;
    const int rend = min(r0 + kSpmmRows, n);
    const int e0 = arp[r0];
    const int e1 = arp[rend];
    const bool staged = (e1 - e0) <= kSpmmCap;
    if (staged) {
        for (int e = e0 + threadIdx.x; e < e1; e += kSpmmRows) {
            s_col[e - e0] = acol[e];
            s_val[e - e0] = aval[e];
        }
    }
    __syncthreads();
    const bool active = r < n;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    int s = 0, t = 0;
    if (active) {
        s = arp[r];
        t = arp[r + 1];
    }
    for (int c0 = 0; c0 < k; c0 += kResKC) {
        const TX *xj[kResKC];
#pragma unroll
        for (int kk = 0; kk < kResKC; kk++) xj[kk] = X + (int64_t)g.idx[min(c0 + kk, k - 1)] * ldx;
        double ax[kResKC];
#pragma unroll
        for (int kk = 0; kk < kResKC; kk++) ax[kk] = 0.0;
        if (active) {
            if (staged) {
                for (int e = s; e < t; e++) {
                    const int cj = s_col[e - e0];
                    const double v = s_val[e - e0];
#pragma unroll
                    for (int kk = 0; kk < kResKC; kk++) ax[kk] = ax[kk] + v * (double)xj[kk][cj];
                }
            } else {
                for (int e = s; e < t; e++) {
                    const int cj = acol[e];
                    const double v = aval[e];
#pragma unroll
                    for (int kk = 0; kk < kResKC; kk++) ax[kk] = ax[kk] + v * (double)xj[kk][cj];
                }
            }
        }
#pragma unroll
        for (int kk = 0; kk < kResKC; kk++) {
            const int c = c0 + kk;
            if (c >= k) break;
            double rr = 0.0, xx = 0.0, bb = 0.0;
            if (active) {
                const double xr = (double)xj[kk][r];
                double bx;
                if (HASB) {
                    bx = 0.0;
                    for (int e = brp[r]; e < brp[r + 1]; e++) bx = bx + bval[e] * (double)xj[kk][bcol[e]];
                } else {
                    bx = xr;
                }
                const double res = axpby_el<double>(-g.a[c], bx, 1.0, ax[kk]);
                rr = res * res;
                xx = xr * xr;
                bb = bx * bx;
            }
            rr = wave_sum(rr);
            xx = wave_sum(xx);
            bb = wave_sum(bb);
            if (lane == 0) {
                sred[3 * c + 0][wid] = rr;
                sred[3 * c + 1][wid] = xx;
                sred[3 * c + 2][wid] = bb;
            }
        }
    }
    __syncthreads();
    const int nb = gridDim.x;
    for (int q = threadIdx.x; q < 3 * k; q += kSpmmRows)
        partial[(int64_t)q * nb + blk] = (sred[q][0] + sred[q][1]) + (sred[q][2] + sred[q][3]);
}

// r = A x - lambda B x (Bx = x when B is absent) for matrices in staged row
// blocks: the X rows a 256-row block reads go through LDS as in k_spmm_halo
// -- own rows, A's extras, then B's extras -- for KC columns at a time, and
// both row sums are formed in FP64 from the staged values in CSR order from
// 0, as in k_residual.  One pass over X and the matrices; as in k_spmm_halo
// LDS reads and the staging of other rows bound it.  FP64, measured: 7-point
// 160^3, B = I, 100 columns 1.37 ms (k_residual 2.97, X read once 0.55); 96^3
// with the 27-point B, 50 columns 0.59 ms (k_residual_rows 2.69).
template <typename TX, bool HASB, int KC, int MEA, int MEB>
__global__ __launch_bounds__(kSpmmRows, HASB ? 2 : 3) void k_residual_halo(
    int n, const int *__restrict__ arp, const unsigned short *__restrict__ alcol, const double *__restrict__ aval,
    const int *__restrict__ brows, const int *__restrict__ ahptr, const int *__restrict__ ahcol,
    const int *__restrict__ brp,
    const unsigned short *__restrict__ blcol, const double *__restrict__ bval, const int *__restrict__ bhptr,
    const int *__restrict__ bhcol, const TX *__restrict__ X, int64_t ldx, int ktot, int kper,
    ColScalars g, double *__restrict__ partial, int nblk, int cap)
{
    using S = Slots<TX, KC>;
    using Row = typename S::Row;
    extern __shared__ __align__(16) unsigned char halo_smem[];
    typename S::Part *sx = reinterpret_cast<typename S::Part *>(halo_smem);  // [NP][cap]
    __shared__ double sred[3 * kMaxCols][4];
    const int per = (int)(gridDim.x >> 3);
    const int blk = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if (blk >= nblk) return;  // uniform per workgroup (grid rounded up to 8)
    const int k0 = blockIdx.y * kper, k = min(ktot, k0 + kper);  // this workgroup's columns
    const int tid = threadIdx.x, p = blk * kSpmmRows + tid;
    const int r = brows ? brows[p] : p < n ? p : -1;
    const int lane = tid & 63, wid = tid >> 6;
    const bool active = r >= 0;
    const int nha = ahptr[blk + 1] - ahptr[blk];
    const int nhb = HASB ? bhptr[blk + 1] - bhptr[blk] : 0;
    const int *hca = ahcol + ahptr[blk];
    const int *hcb = HASB ? bhcol + bhptr[blk] : nullptr;
    int as = 0, acnt = 0, bs = 0, bcnt = 0;
    if (active) {
        as = arp[r];
        acnt = arp[r + 1] - as;
        if (HASB) {
            bs = brp[r];
            bcnt = brp[r + 1] - bs;
        }
    }
    RowHead<double, MEA> ra;
    RowHead<double, HASB ? MEB : 2> rb;
    ra.load(alcol, aval, as, acnt);
    if (HASB) rb.load(blcol, bval, bs, bcnt);
    // slot of a B entry: its extras follow A's
    auto bslot = [&](int sl) { return sl < kSpmmRows ? sl : sl + nha; };
    auto rowof = [&](int j) { return j < nha ? hca[j] : hcb[j - nha]; };
    const int nh = nha + nhb;
    constexpr int NE = HASB ? halo_prefetch<MEB> + 1 : halo_prefetch<MEA>;
    int erow[NE];
#pragma unroll
    for (int i = 0; i < NE; i++) erow[i] = tid + i * kSpmmRows < nh ? rowof(tid + i * kSpmmRows) : 0;
    Row pown, pext[NE];
    auto xcols = [&](int c0, const TX *(&xc)[KC]) {
#pragma unroll
        for (int cc = 0; cc < KC; cc++) xc[cc] = X + (int64_t)g.idx[min(c0 + cc, k - 1)] * ldx;
    };
    auto prefetch = [&](int c0) {
        const TX *xc[KC];
        xcols(c0, xc);
        if (active) {
#pragma unroll
            for (int cc = 0; cc < KC; cc++) pown.v[cc] = xc[cc][r];
        }
#pragma unroll
        for (int i = 0; i < NE; i++)
            if (tid + i * kSpmmRows < nh) {
#pragma unroll
                for (int cc = 0; cc < KC; cc++) pext[i].v[cc] = xc[cc][erow[i]];
            }
    };
    prefetch(k0);
    for (int c0 = k0; c0 < k; c0 += KC) {
        if (active) S::put(sx, cap, tid, pown);
#pragma unroll
        for (int i = 0; i < NE; i++)
            if (tid + i * kSpmmRows < nh) S::put(sx, cap, kSpmmRows + tid + i * kSpmmRows, pext[i]);
        if (nh > NE * kSpmmRows) {
            const TX *xc[KC];
            xcols(c0, xc);
            for (int j = tid + NE * kSpmmRows; j < nh; j += kSpmmRows) {
                const int er = rowof(j);
                Row w;
#pragma unroll
                for (int cc = 0; cc < KC; cc++) w.v[cc] = xc[cc][er];
                S::put(sx, cap, kSpmmRows + j, w);
            }
        }
        const Row xo = pown;
        __syncthreads();
        if (c0 + KC < k) prefetch(c0 + KC);
        double ax[KC], bx[KC];
#pragma unroll
        for (int cc = 0; cc < KC; cc++) ax[cc] = bx[cc] = 0.0;
#pragma unroll
        for (int u = 0; u < MEA; u++)
            if (u < acnt) {
                const Row x = S::get(sx, cap, ra.slot(u));
#pragma unroll
                for (int cc = 0; cc < KC; cc++) ax[cc] = ax[cc] + ra.v[u] * (double)x.v[cc];
            }
        for (int e = as + MEA; e < as + acnt; e++) {
            const Row x = S::get(sx, cap, alcol[e]);
            const double ve = aval[e];
#pragma unroll
            for (int cc = 0; cc < KC; cc++) ax[cc] = ax[cc] + ve * (double)x.v[cc];
        }
        if (HASB) {
#pragma unroll
            for (int u = 0; u < MEB; u++)
                if (u < bcnt) {
                    const Row x = S::get(sx, cap, bslot(rb.slot(u)));
#pragma unroll
                    for (int cc = 0; cc < KC; cc++) bx[cc] = bx[cc] + rb.v[u] * (double)x.v[cc];
                }
            for (int e = bs + MEB; e < bs + bcnt; e++) {
                const Row x = S::get(sx, cap, bslot(blcol[e]));
                const double ve = bval[e];
#pragma unroll
                for (int cc = 0; cc < KC; cc++) bx[cc] = bx[cc] + ve * (double)x.v[cc];
            }
        }
        double drr[KC], dxx[KC], dbb[KC];
#pragma unroll
        for (int cc = 0; cc < KC; cc++) {
            const int c = c0 + cc;
            const bool live = active && c < k;
            const double xr = live ? (double)xo.v[cc] : 0.0;
            const double b = HASB ? bx[cc] : xr;
            const double res = live ? axpby_el<double>(-g.a[min(c, k - 1)], b, 1.0, ax[cc]) : 0.0;
            drr[cc] = res * res;
            dxx[cc] = xr * xr;
            dbb[cc] = live ? b * b : 0.0;
        }
        constexpr int L = KC == 1 ? 0 : KC == 2 ? 1 : 2;
        const double srr = wave_colsum<KC>(drr, lane), sxx = wave_colsum<KC>(dxx, lane);
        const double sbb = HASB ? wave_colsum<KC>(dbb, lane) : sxx;
        const int c = c0 + (lane >> (6 - L));
        if ((lane & ((64 >> L) - 1)) == 0 && c < k) {
            sred[3 * c + 0][wid] = srr;
            sred[3 * c + 1][wid] = sxx;
            sred[3 * c + 2][wid] = sbb;
        }
        __syncthreads();  // the next chunk overwrites sx
    }
    for (int q = 3 * k0 + tid; q < 3 * k; q += kSpmmRows)
        partial[(int64_t)q * nblk + blk] = (sred[q][0] + sred[q][1]) + (sred[q][2] + sred[q][3]);
}

// r = A x - lambda B x (Bx = x when B is absent) on the row-major gather
// path: the FP64 row sums of k_residual (CSR order from 0, x converted to
// FP64 per entry) gathered from the staged rows Xt, in the workgroup layout
// of k_spmm_rows (A's long rows one wavefront each; B has no row longer than
// long_thr).  The sums r.r, x.x and Bx.Bx of column c go to
// partial[(3c + q) * pstride + blk] per row workgroup and to
// partial[(3c + q) * pstride + nblk + li] per long row.
template <typename TX, int G, bool HASB>
__global__ __launch_bounds__(256) void k_residual_rows(int n, const int *__restrict__ rowptr,
                                                       const int *__restrict__ col, const double *__restrict__ val,
                                                       const int *__restrict__ brp, const int *__restrict__ bcol,
                                                       const double *__restrict__ bval, const TX *__restrict__ Xt,
                                                       int kp, int k, ColScalars g,
                                                       const int *__restrict__ long_rows, int nlong, int nlb,
                                                       int long_thr, double *__restrict__ partial, int pstride,
                                                       int nblk)
{
    constexpr int SG = 64 / G;
    constexpr int RWG = rows_per_wg(G);
    constexpr int RPW = RWG / 4;
    __shared__ double sred[4][G][3];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int c0 = blockIdx.y * 64;
    if ((int)blockIdx.x < nlb) {
        const int li = blockIdx.x * 4 + wid;
        if (li >= nlong) return;  // uniform per wavefront; this branch has no barrier
        const int r = long_rows[li];
        const int c = c0 + lane;
        const int cc = min(c, kp - 1);
        const double ax = wave_row_sum<double, double, TX>(col, val, rowptr[r], rowptr[r + 1], Xt, kp, cc, r, lane);
        const double xr = (double)Xt[(int64_t)r * kp + cc];
        const double bx =
            HASB ? wave_row_sum<double, double, TX>(bcol, bval, brp[r], brp[r + 1], Xt, kp, cc, r, lane) : xr;
        if (c < k) {
            const double res = axpby_el<double>(-g.a[c], bx, 1.0, ax);
            partial[(int64_t)(3 * c + 0) * pstride + nblk + li] = res * res;
            partial[(int64_t)(3 * c + 1) * pstride + nblk + li] = xr * xr;
            partial[(int64_t)(3 * c + 2) * pstride + nblk + li] = bx * bx;
        }
        return;
    }
    const int blk = blockIdx.x - nlb;
    const int r0 = blk * RWG;
    const int cl = lane % G, sg = lane / G;
    const int c = c0 + cl;  // < kp
    const bool live = c < k;
    double srr = 0.0, sxx = 0.0, sbb = 0.0;
    for (int i = sg; i < RPW; i += SG) {
        const int r = r0 + wid * RPW + i;
        int s = 0, t = 0, bs = 0, bt = 0;
        if (r < n) {
            s = rowptr[r];
            t = rowptr[r + 1];
            if (HASB) {
                bs = brp[r];
                bt = brp[r + 1];
            }
        }
        const bool act = r < n && t - s <= long_thr;
        if (!act) t = s, bt = bs;
        const int rs = r < n ? r : 0;
        const double ax = lane_row_sum<double, double, TX>(col, val, s, t, Xt, kp, c, rs);
        const double bx0 = HASB ? lane_row_sum<double, double, TX>(bcol, bval, bs, bt, Xt, kp, c, rs) : 0.0;
        if (act && live) {
            const double xr = (double)Xt[(int64_t)r * kp + c];
            const double bx = HASB ? bx0 : xr;
            const double res = axpby_el<double>(-g.a[c], bx, 1.0, ax);
            srr += res * res;
            sxx += xr * xr;
            sbb += bx * bx;
        }
    }
#pragma unroll
    for (int m = G; m < 64; m <<= 1) {
        srr += __shfl_xor(srr, m, 64);
        sxx += __shfl_xor(sxx, m, 64);
        sbb += __shfl_xor(sbb, m, 64);
    }
    if (sg == 0) {
        sred[wid][cl][0] = srr;
        sred[wid][cl][1] = sxx;
        sred[wid][cl][2] = sbb;
    }
    __syncthreads();
    const int q = threadIdx.x;
    if (q < min(G, k - c0)) {
        const int cq = c0 + q;
#pragma unroll
        for (int j = 0; j < 3; j++)
            partial[(int64_t)(3 * cq + j) * pstride + blk] =
                (sred[0][q][j] + sred[1][q][j]) + (sred[2][q][j] + sred[3][q][j]);
    }
}

// ---------------------------------------------------------------- CG update
// x += alpha p (VecAxpby(alpha, p, 1.0, x)); r -= alpha w
// (VecAxpby(-alpha, w, 1.0, r)); partial r.r  (gcge_cg.c:250-276)
template <typename T>
__global__ __launch_bounds__(kBlock) void k_cg_update(int64_t n, T *__restrict__ x, int64_t ldx,
                                                      const T *__restrict__ p, int64_t ldp,
                                                      const T *__restrict__ w, int64_t ldw,
                                                      T *__restrict__ r, int64_t ldr, ColScalars s,
                                                      double *__restrict__ partial)
{
    __shared__ double sh[4];
    const int j = blockIdx.y;
    const T al = (T)s.a[j];
    T *xj = x + (int64_t)j * ldx;
    const T *pj = p + (int64_t)j * ldp;
    const T *wj = w + (int64_t)j * ldw;
    T *rj = r + (int64_t)j * ldr;
    double acc = 0.0;
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += stride) {
        xj[i] = axpby_el<T>(al, pj[i], T(1), xj[i]);
        const T rn = axpby_el<T>(-al, wj[i], T(1), rj[i]);
        rj[i] = rn;
        acc = fma((double)rn, (double)rn, acc);
    }
    const double bs = block_sum(acc, sh);
    if (threadIdx.x == 0) partial[(int64_t)j * gridDim.x + blockIdx.x] = bs;
}

// ---------------------------------------------------------------- split CG steps
// r -= alpha w (VecAxpby(-alpha, w, 1.0, r)); partial r.r  (gcge_cg.c:250-276)
template <typename T, int U, bool NT>
__global__ __launch_bounds__(kBlock) void k_cg_resid(int64_t n, const T *__restrict__ w, int64_t ldw,
                                                     T *__restrict__ r, int64_t ldr, ColScalars s,
                                                     double *__restrict__ partial)
{
    __shared__ double sh[4];
    const int j = blockIdx.y;
    const T al = (T)s.a[j];
    const T *wj = w + (int64_t)j * ldw;
    T *rj = r + (int64_t)j * ldr;
    double acc = 0.0;
    strided_rows<U>(
        n, [&](int64_t i) { return Pair<T>{load_as<NT>(wj + i), load_as<NT>(rj + i)}; },
        [&](int64_t i, const Pair<T> &v) {
            const T rn = axpby_el<T>(-al, v.a, T(1), v.b);
            store_as<NT>(rj + i, rn);
            acc = fma((double)rn, (double)rn, acc);
        });
    const double bs = block_sum(acc, sh);
    if (threadIdx.x == 0) partial[(int64_t)j * gridDim.x + blockIdx.x] = bs;
}

// Jacobi-preconditioned residual step: r -= alpha w (same rounding as
// k_cg_resid), partial r.z (row 2j) and r.r (row 2j + 1) with z = dinv .* r
// rounded as k_cg_search<T, true> forms it
template <typename T>
struct Triple {
    T a, b, c;
};

template <typename T, int U, bool NT>
__global__ __launch_bounds__(kBlock) void k_pcg_resid(int64_t n, const T *__restrict__ w, int64_t ldw,
                                                      T *__restrict__ r, int64_t ldr, const T *__restrict__ dinv,
                                                      ColScalars s, double *__restrict__ partial)
{
    __shared__ double sh[4];
    const int j = blockIdx.y;
    const T al = (T)s.a[j];
    const T *wj = w + (int64_t)j * ldw;
    T *rj = r + (int64_t)j * ldr;
    double arz = 0.0, arr = 0.0;
    strided_rows<U>(
        n, [&](int64_t i) { return Triple<T>{load_as<NT>(wj + i), load_as<NT>(rj + i), dinv[i]}; },
        [&](int64_t i, const Triple<T> &v) {
            const T rn = axpby_el<T>(-al, v.a, T(1), v.b);
            const T zn = rn * v.c;
            store_as<NT>(rj + i, rn);
            arz = fma((double)rn, (double)zn, arz);
            arr = fma((double)rn, (double)rn, arr);
        });
    const double brz = block_sum(arz, sh);
    const double brr = block_sum(arr, sh);
    if (threadIdx.x == 0) {
        partial[(int64_t)(2 * j) * gridDim.x + blockIdx.x] = brz;
        partial[(int64_t)(2 * j + 1) * gridDim.x + blockIdx.x] = brr;
    }
}

// dinv[i] = 1 / a_ii; rows without a nonzero diagonal entry get 1 (no scaling)
__global__ __launch_bounds__(kBlock) void k_diag_inv(int n, const int *__restrict__ rowptr,
                                                     const int *__restrict__ col, const double *__restrict__ val,
                                                     double *__restrict__ d64, float *__restrict__ d32)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    double d = 0.0;
    for (int e = rowptr[i]; e < rowptr[i + 1]; e++)
        if (col[e] == i) d = d + val[e];
    const double inv = (d != 0.0) ? 1.0 / d : 1.0;
    d64[i] = inv;
    d32[i] = (float)inv;
}

// x += alpha p (VecAxpby(alpha, p, 1.0, x)) for the columns j < kx; then
// p = r + beta p (MultiVecAxpbyDiag(1, r, beta, p)) for the columns j < kp
// With PRE, the search direction is built from z = dinv .* r (the Jacobi-
// preconditioned residual, formed here rather than stored).
constexpr int kLoadsDone = 0x0f70;  // s_waitcnt vmcnt(0), nothing else

template <typename T, bool PRE, int V, bool NT>
__global__ __launch_bounds__(kBlock) void k_cg_search(int64_t n, T *__restrict__ x, int64_t ldx,
                                                      T *__restrict__ p, int64_t ldp, const T *__restrict__ r,
                                                      int64_t ldr, int kx, int kp, ColScalars s,
                                                      const T *__restrict__ dinv)
{
    const int j = blockIdx.y;
    const int64_t i = run_row<V>();
    if (i >= n) return;
    const T al = (T)s.a[j], be = (T)s.b[j];
    T *xj = x + (int64_t)j * ldx;
    T *pj = p + (int64_t)j * ldp;
    const T *rj = r + (int64_t)j * ldr;
    T pv[V], xv[V], rv[V], dv[V];
    const auto load_r = [&] {
        load_run<T, V, NT>(rj, i, rv);
        if (PRE) load_run<T, V, false>(dinv, i, dv);
    };
    const auto put_x = [&] {
#pragma unroll
        for (int t = 0; t < V; t++) xv[t] = axpby_el<T>(al, pv[t], T(1), xv[t]);
        store_run<T, V, NT>(xj, i, n, xv);
    };
    const auto put_p = [&] {
#pragma unroll
        for (int t = 0; t < V; t++) pv[t] = axpby_el<T>(T(1), PRE ? rv[t] * dv[t] : rv[t], be, pv[t]);
        store_run<T, V, NT>(pj, i, n, pv);
    };
    if (j < kx && j < kp) {
        // Past the caches the three streams are better read one after the other
        // (40 columns of 4.1M rows, us, together / in turn: FP32 528 / 515, FP64 1052
        // / 1017; with the diagonal FP32 513 / 517, 24 columns 311 / 305, FP64 1102 /
        // 1085, where the last wait gains nothing)
        load_run<T, V, NT>(pj, i, pv);
        if constexpr (NT) __builtin_amdgcn_s_waitcnt(kLoadsDone);
        load_run<T, V, NT>(xj, i, xv);
        if constexpr (NT) __builtin_amdgcn_s_waitcnt(kLoadsDone);
        load_r();
        if constexpr (NT && !PRE) __builtin_amdgcn_s_waitcnt(kLoadsDone);
        put_x();
        if constexpr (NT) __builtin_amdgcn_s_waitcnt(kLoadsDone);
        put_p();
    } else if (j < kx) {
        load_run<T, V, NT>(pj, i, pv);
        load_run<T, V, NT>(xj, i, xv);
        put_x();
    } else {
        load_run<T, V, NT>(pj, i, pv);
        load_r();
        put_p();
    }
}

// ---------------------------------------------------------------- gradient
// g_e = sum_i w_i x_i[row_e] x_i[col_e], one thread per stored entry
template <typename T>
__global__ __launch_bounds__(kBlock) void k_sampled_outer(int nnz, const int *__restrict__ rowidx,
                                                          const int *__restrict__ col,
                                                          const T *__restrict__ X, int64_t ldx,
                                                          int k, ColScalars s, double *__restrict__ g)
{
    const int e = blockIdx.x * kBlock + threadIdx.x;
    if (e >= nnz) return;
    const int r = rowidx[e], c = col[e];
    double acc = 0.0;
    for (int i = 0; i < k; i++) {
        const T *xi = X + (int64_t)i * ldx;
        acc = fma(s.a[i], (double)xi[r] * (double)xi[c], acc);
    }
    g[e] += acc;
}

__global__ __launch_bounds__(kBlock) void k_csr_gather_sum(int nparam, const int *__restrict__ jrp,
                                                           const int *__restrict__ jnz,
                                                           const double *__restrict__ jval,
                                                           const int *__restrict__ map, int nnz,
                                                           const double *__restrict__ g,
                                                           double *__restrict__ grad, double scale, int accumulate,
                                                           double *__restrict__ bad)
{
    const int p = blockIdx.x * kBlock + threadIdx.x;
    if (p >= nparam) return;
    double acc = 0.0;
    bool out = false;
    for (int t = jrp[p]; t < jrp[p + 1]; t++) {
        const int e = jnz[t];
        if (e < 0 || e >= nnz) {
            out = true;
            continue;
        }
        acc = fma(jval[t], g[map ? map[e] : e], acc);
    }
    if (out) *bad = 1.0;
    grad[p] = accumulate ? fma(scale, acc, grad[p]) : scale * acc;
}

// Host columns, as they lie in the staging buffer, into a multivector's row
// order and precision, and back: bound by the host link.  The upload of 16 FP64
// columns of 262,144 rows into an ordered matrix's block takes 1.18 ms, 2.97 with
// the permutation on the host; the download 2.18 and 5.1.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_rows_in(int64_t n, const double *__restrict__ x, int64_t ldx,
                                                    const int *__restrict__ perm, T *__restrict__ y, int64_t ldy)
{
    const int64_t i = run_row<1>();
    if (i < n) y[(int64_t)blockIdx.y * ldy + i] = (T)x[(int64_t)blockIdx.y * ldx + (perm ? (int64_t)perm[i] : i)];
}

// 16-byte units over the host link: as many reads in flight as there are
__global__ __launch_bounds__(kBlock) void k_fetch(const int4 *__restrict__ host, int4 *__restrict__ dev, size_t units)
{
    const size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (i < units) dev[i] = host[i];
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_rows_out(int64_t n, double *__restrict__ x, int64_t ldx,
                                                     const int *__restrict__ perm, const T *__restrict__ y,
                                                     int64_t ldy)
{
    const int64_t i = run_row<1>();
    if (i < n) x[(int64_t)blockIdx.y * ldx + (perm ? (int64_t)perm[i] : i)] = (double)y[(int64_t)blockIdx.y * ldy + i];
}

__global__ __launch_bounds__(kBlock) void k_rowidx(int n, const int *__restrict__ rowptr,
                                                   int *__restrict__ rowidx)
{
    const int r = blockIdx.x * kBlock + threadIdx.x;
    if (r >= n) return;
    for (int e = rowptr[r]; e < rowptr[r + 1]; e++) rowidx[e] = r;
}

__global__ __launch_bounds__(kBlock) void k_to_f32(int64_t n, const double *__restrict__ a,
                                                   float *__restrict__ b)
{
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i < n) b[i] = (float)a[i];
}

}  // namespace

// ======================================================================
// launchers
// ======================================================================

static ColScalars make_scalars(int k, const double *a, const double *b, const int *idx)
{
    ColScalars s;
    std::memset(&s, 0, sizeof(s));
    for (int j = 0; j < k; j++) {
        s.a[j] = a ? a[j] : 0.0;
        s.b[j] = b ? b[j] : 0.0;
        s.idx[j] = idx ? idx[j] : j;
    }
    s.use_idx = idx ? 1 : 0;
    return s;
}

// Grid of an element-wise kernel: every thread one run of V rows.  A multiple of
// 8 workgroups per column: workgroups are dealt out to the 8 XCDs in turn, so the
// same rows of every column meet on one XCD, whose L2 then holds what the columns
// share (the diagonal in k_cg_search: 10 FP32 columns of 1.03M rows 35.3 -> 29.8
// us, 64 228 -> 201).
static dim3 run_grid(int64_t n, int V, int k)
{
    const int64_t b = (n + (int64_t)kBlock * V - 1) / (kBlock * V);
    return dim3((unsigned)((b + 7) / 8 * 8), k);
}

// Calls f(V, NT) with constants: 16-byte accesses (a multivector's columns
// start on 1 KiB or 2 KiB boundaries), past the caches where more than
// kStreamBytes are touched
template <typename T, typename F>
static void run_variant(double held, F f)
{
    using W = std::integral_constant<int, kWide<T>>;
    if (held > kStreamBytes) f(W{}, std::true_type{});
    else f(W{}, std::false_type{});
}

// Calls f(U, NT) for the strided sums: 8 rows at a time past the caches; 4 at a
// time where threads have many (2 columns of 4.1M rows in FP32, residual update
// 23.9 -> 16.4 us), else one (16,384 rows, 20 columns: 2.7 us, 3.2 with 4)
template <typename F>
static void sum_variant(int64_t n, double bytes, F f)
{
    if (bytes > kStreamBytes) f(std::integral_constant<int, 8>{}, std::true_type{});
    else if (n >= 1 << 20) f(std::integral_constant<int, 4>{}, std::false_type{});
    else f(std::integral_constant<int, 1>{}, std::false_type{});
}

template <typename T>
static void axpby_t(int64_t n, const void *x, int64_t ldx, void *y, int64_t ldy, int k, const ColScalars &s,
                    double held)
{
    run_variant<T>(held, [&](auto V, auto NT) {
        k_axpby<T, V(), NT()><<<run_grid(n, V(), k), kBlock, 0, ctx().stream>>>(n, (const T *)x, ldx, (T *)y, ldy, s);
    });
}

void launch_axpby(int prec, int64_t n, const void *x, int64_t ldx, void *y, int64_t ldy, int k,
                  const double *a, const double *b, const int *xidx)
{
    if (k <= 0 || n <= 0 || failed()) return;
    ColScalars s = make_scalars(k, a, b, xidx);
    double bytes = 0.0, held = 0.0;  // moved; y is read and written but held once
    for (int j = 0; j < k; j++) {
        bytes += (double)n * elem_size(prec) * ((s.a[j] == 0.0 || s.b[j] == 0.0) ? 2 : 3);
        held += (double)n * elem_size(prec) * (s.a[j] == 0.0 ? 1 : 2);
    }
    ProfScope ps(K_AXPBY, bytes, 0.0);
    if (prec == GCGE_HIP_FP64) axpby_t<double>(n, x, ldx, y, ldy, k, s, held);
    else axpby_t<float>(n, x, ldx, y, ldy, k, s, held);
    check(hipGetLastError(), "k_axpby");
}

// Where a launch leaves rows x nb partial sums.  Few of them go straight to
// host memory, where the host adds them in k_reduce_rows_host's order: a launch
// less and its wait.  us a call, FP64 dots of 1 column of 16,384 rows (64
// partial sums) 14.6 -> 11.1, of 20 columns (1280) 15.9 -> 14.7, of 8 columns of
// 90,000 rows (2048) 15.8 -> 15.6, where the line is drawn.  Not where the launch
// also writes columns that are to be seen everywhere when the call returns: the
// host would have the sums while stores of the same launch may still lie in one
// XCD's L2, out of sight of other streams.  The launch that reduces comes after
// those stores (residual update of 1 column of
// 16,384 rows 16.6 us, 12.6 without; of 20 columns 18.1 and 16.0; with a
// system-scope release by every workgroup instead 29).
static double *partial_buf(size_t rows, size_t nb, Seen seen)
{
    return seen == Seen::in_stream && rows * nb <= kHostPartials ? host_partials(rows * nb)
                                                                 : (double *)scratch(sizeof(double) * rows * nb);
}

// sum_row and block_sum on the host
static double host_sum_row(const double *row, int nb)
{
    double v[kBlock];
    for (int t = 0; t < kBlock; t++) v[t] = 0.0;
    for (int b = 0; b < nb; b += kBlock)
        for (int t = 0; t < std::min(kBlock, nb - b); t++) v[t] += row[b + t];
    for (int w = 0; w < kBlock; w += 64)
        for (int off = 32; off > 0; off >>= 1)
            for (int l = 0; l < off; l++) v[w + l] += v[w + l + off];
    return (v[0] + v[64]) + (v[128] + v[192]);
}

static bool reduce_to_host(const double *partial, int rows, int nb, double *out)
{
    if (partial == ctx().hpart) {
        if (!wait_partials((size_t)rows * nb)) return false;
        for (int j = 0; j < rows; j++) out[j] = host_sum_row(partial + (size_t)j * nb, nb);
        return true;
    }
    unsigned long long seq = 0, *seqs = host_seq(rows, &seq);
    double *h = host_buf(rows);
    if (!h || !seqs) return false;
    k_reduce_rows_host<<<rows, kBlock, 0, ctx().stream>>>(partial, nb, h, seqs, seq);
    if (!check(hipGetLastError(), "k_reduce_rows_host") || !wait_seq(rows, seq)) return false;
    std::memcpy(out, h, sizeof(double) * rows);
    return true;
}

int dots_blocks(int64_t n) { return grid_1d(n, 256); }

static void launch_dots(int prec, int64_t n, const void *x, int64_t ldx, const void *y, int64_t ldy, int k,
                        double *partial, int nb)
{
    const dim3 grid(nb, k);
    sum_variant(n, 2.0 * k * (double)n * elem_size(prec), [&](auto U, auto NT) {
        if (prec == GCGE_HIP_FP64)
            k_dots<double, U(), NT()><<<grid, kBlock, 0, ctx().stream>>>(n, (const double *)x, ldx,
                                                                         (const double *)y, ldy, partial);
        else
            k_dots<float, U(), NT()><<<grid, kBlock, 0, ctx().stream>>>(n, (const float *)x, ldx, (const float *)y,
                                                                        ldy, partial);
    });
}

bool dots(int prec, int64_t n, const void *x, int64_t ldx, const void *y, int64_t ldy, int k,
          double *out)
{
    if (k <= 0) return true;
    if (failed()) return false;
    const int nb = dots_blocks(n);
    double *partial = partial_buf((size_t)k, nb, Seen::in_stream);
    if (!partial) return false;
    {
        ProfScope ps(K_DOTS, 2.0 * k * (double)n * elem_size(prec), 2.0 * k * (double)n);
        launch_dots(prec, n, x, ldx, y, ldy, k, partial, nb);
    }
    if (!check(hipGetLastError(), "k_dots")) return false;
    return reduce_to_host(partial, k, nb, out);
}

// The same dots with the partial sums in a caller-provided device buffer of
// at least k * dots_blocks(n) + k doubles and the sums copied on the backend
// stream into host memory out (pinned or not); no allocation, no profiler.
bool dots_with(int prec, int64_t n, const void *x, int64_t ldx, const void *y, int64_t ldy, int k, double *partial,
               double *out)
{
    if (k <= 0) return true;
    if (failed()) return false;
    const int nb = dots_blocks(n);
    launch_dots(prec, n, x, ldx, y, ldy, k, partial, nb);
    if (!check(hipGetLastError(), "k_dots")) return false;
    double *dres = partial + (int64_t)k * nb;
    k_reduce_rows<<<k, kBlock, 0, ctx().stream>>>(partial, nb, dres);
    if (!check(hipGetLastError(), "k_reduce_rows")) return false;
    if (!check(hipMemcpyAsync(out, dres, sizeof(double) * k, hipMemcpyDeviceToHost, ctx().stream), "D2H dots"))
        return false;
    return check(hipStreamSynchronize(ctx().stream), "hipStreamSynchronize");
}

template <typename TX, typename TY>
static void copy_t(int64_t n, const void *x, int64_t ldx, void *y, int64_t ldy, int k, double bytes)
{
    // stores of 16 bytes: with 32 per thread each store of a wavefront would leave
    // every second 16 bytes out (40 columns of 4.1M rows from FP32 to FP64 497 us,
    // 298 with 16); loads of 32 bytes, from FP64 to FP32, cost nothing
    run_variant<TY>(bytes, [&](auto V, auto NT) {
        k_copy<TX, TY, V(), NT()><<<run_grid(n, V(), k), kBlock, 0, ctx().stream>>>(n, (const TX *)x, ldx, (TY *)y,
                                                                                    ldy);
    });
}

void launch_copy(int xprec, const void *x, int64_t ldx, int yprec, void *y, int64_t ldy, int64_t n, int k)
{
    if (k <= 0 || n <= 0 || failed()) return;
    const double bytes = (double)k * n * (elem_size(xprec) + elem_size(yprec));
    ProfScope ps(K_COPY, bytes, 0.0);
    if (xprec == GCGE_HIP_FP64 && yprec == GCGE_HIP_FP64) copy_t<double, double>(n, x, ldx, y, ldy, k, bytes);
    else if (xprec == GCGE_HIP_FP64) copy_t<double, float>(n, x, ldx, y, ldy, k, bytes);
    else if (yprec == GCGE_HIP_FP64) copy_t<float, double>(n, x, ldx, y, ldy, k, bytes);
    else copy_t<float, float>(n, x, ldx, y, ldy, k, bytes);
    check(hipGetLastError(), "k_copy");
}

void launch_swap(int prec, void *x, int64_t ldx, void *y, int64_t ldy, int64_t n, int k)
{
    if (k <= 0 || n <= 0 || failed()) return;
    dim3 grid(grid_1d(n, 1024), k);
    ProfScope ps(K_SWAP, 4.0 * k * (double)n * elem_size(prec), 0.0);
    if (prec == GCGE_HIP_FP64)
        k_swap<double><<<grid, kBlock, 0, ctx().stream>>>(n, (double *)x, ldx, (double *)y, ldy);
    else
        k_swap<float><<<grid, kBlock, 0, ctx().stream>>>(n, (float *)x, ldx, (float *)y, ldy);
    check(hipGetLastError(), "k_swap");
}

void launch_zero_rows(int prec, void *x, int64_t ldx, int64_t n, int k, const unsigned char *mask)
{
    if (k <= 0 || n <= 0 || failed()) return;
    dim3 grid(grid_1d(n, 1024), k);
    if (prec == GCGE_HIP_FP64)
        k_zero_rows<double><<<grid, kBlock, 0, ctx().stream>>>(n, (double *)x, ldx, mask);
    else
        k_zero_rows<float><<<grid, kBlock, 0, ctx().stream>>>(n, (float *)x, ldx, mask);
    check(hipGetLastError(), "k_zero_rows");
}

template <typename T>
static const T *mat_vals(HIP_MAT *A);
template <>
const double *mat_vals<double>(HIP_MAT *A) { return A->val64; }
template <>
const float *mat_vals<float>(HIP_MAT *A) { return mat_val32(A); }

// Row-major gather path (see k_spmm_rows) for kc <= kMaxCols columns.
template <typename T, bool DOT, int G>
static bool spmm_rows_g(HIP_MAT *A, const T *val, const T *Xc, int64_t ldx, ColScalars g, T *Yc, int64_t ldy,
                        int kc, double *out, Seen seen)
{
    const int n = A->n, kp = G < 64 ? G : ((kc + 63) / 64) * 64;
    T *Xt = (T *)row_stage(sizeof(T) * (size_t)n * kp);
    if (!Xt) return false;
    const int RWG = rows_per_wg(G);
    const int nblk = (n + RWG - 1) / RWG, nlong = A->nlong, nlb = (nlong + 3) / 4;
    const int pstride = nblk + (DOT ? nlong : 0);
    double *partial = nullptr;
    if (DOT) {
        partial = partial_buf((size_t)kc, pstride, seen);
        if (!partial) return false;
    }
    {
        const double bytes = (sizeof(T) + 4.0) * A->nnz + 4.0 * (n + 1) + 2.0 * kc * (double)n * sizeof(T);
        const bool f64 = sizeof(T) == 8;
        ProfScope ps(DOT ? (f64 ? K_SPMM_DOT_F64 : K_SPMM_DOT_F32) : (f64 ? K_SPMM_F64 : K_SPMM_F32), bytes,
                     2.0 * kc * (double)A->nnz);
        k_rows_from_cols<T><<<dim3((n + 63) / 64, (kp + 63) / 64), 256, 0, ctx().stream>>>(n, Xc, ldx, kc, g, kp,
                                                                                            Xt);
        k_spmm_rows<T, DOT, G><<<dim3(nlb + nblk, G < 64 ? 1 : kp / 64), 256, 0, ctx().stream>>>(
            n, A->rowptr, A->col, val, Xt, kp, Yc, ldy, kc, A->long_rows, nlong, nlb,
            nlong > 0 ? kLongRow : INT_MAX, partial, pstride, nblk);
    }
    if (!check(hipGetLastError(), "k_spmm_rows")) return false;
    return !DOT || reduce_to_host(partial, kc, pstride, out);
}

template <typename T, bool DOT>
static bool spmm_rows(HIP_MAT *A, const T *val, const T *Xc, int64_t ldx, ColScalars g, T *Yc, int64_t ldy,
                      int kc, double *out, Seen seen)
{
    if (kc > 32) return spmm_rows_g<T, DOT, 64>(A, val, Xc, ldx, g, Yc, ldy, kc, out, seen);
    if (kc > 16) return spmm_rows_g<T, DOT, 32>(A, val, Xc, ldx, g, Yc, ldy, kc, out, seen);
    if (kc > 8) return spmm_rows_g<T, DOT, 16>(A, val, Xc, ldx, g, Yc, ldy, kc, out, seen);
    if (kc > 4) return spmm_rows_g<T, DOT, 8>(A, val, Xc, ldx, g, Yc, ldy, kc, out, seen);
    if (kc > 2) return spmm_rows_g<T, DOT, 4>(A, val, Xc, ldx, g, Yc, ldy, kc, out, seen);
    return spmm_rows_g<T, DOT, 2>(A, val, Xc, ldx, g, Yc, ldy, kc, out, seen);
}

// Columns per LDS pass of k_spmm_halo: 4, or GCGE_HIP_HALO_KC (1, 2, 4 or
// 8), halved while the staged rows exceed the byte budget
// (GCGE_HIP_HALO_LDS, default 40 KiB).
static int halo_kc(const HIP_MAT *A, size_t elem)
{
    const char *e = getenv("GCGE_HIP_HALO_KC");
    const int env_kc = e ? atoi(e) : 0;
    const char *l = getenv("GCGE_HIP_HALO_LDS");
    const long env_lds = l ? atol(l) : 40960;
    // default: 4 columns per pass in both precisions (measured on 3-D and
    // 2-D grids in tile order: 8 FP32 columns were 5-10 % slower, 2 were
    // 10-25 % slower), halved while over the budget
    int kc = (env_kc == 1 || env_kc == 2 || env_kc == 4 || env_kc == 8) ? env_kc : 4;
    if (env_kc != kc)
        while (kc > 1 && (size_t)kc * A->halo_cap * elem > (size_t)env_lds) kc /= 2;
    // never beyond 56 KiB of dynamic LDS (the kernel adds 4 KiB of its own)
    while (kc > 1 && (size_t)kc * A->halo_cap * elem > (size_t)56 * 1024) kc /= 2;
    return kc;
}

// More than 8 entries per row on average: 28 of them held in registers by
// the staged kernels, 8 otherwise.
static bool long_average(const HIP_MAT *A) { return A->nnz > 8.0 * A->n; }

// Columns per workgroup of the staged kernels: all k where the row blocks fill
// the chip, else a share of them (a multiple of KC), so that 1,024 workgroups
// (four per CU) are in flight; a block's entries are then read once per share.
// 64 blocks (128^2 grid), FP64 with dots: 20 columns 11.7 -> 8.0 us.
static int staged_columns(int nblk, int k, int KC)
{
    const int passes = (k + KC - 1) / KC, shares = std::min(passes, std::max(1, 1024 / nblk));
    return (passes + shares - 1) / shares * KC;
}

template <typename T, bool DOT, int KC>
static void spmm_halo_kc(HIP_MAT *A, const T *val, const T *Xc, int64_t ldx, ColScalars g, T *Yc, int64_t ldy,
                         int kc, double *partial, int nblk, int long_thr, int pstride)
{
    const size_t lds = (size_t)KC * A->halo_cap * sizeof(T);
    const int kper = staged_columns(nblk, kc, KC);
    const dim3 grid(((nblk + 7) / 8) * 8, (kc + kper - 1) / kper);
    if (long_average(A))
        k_spmm_halo<T, DOT, KC, 28><<<grid, kSpmmRows, lds, ctx().stream>>>(
            A->n, A->rowptr, A->lcol, val, A->brick_rows, A->halo_ptr, A->halo_col, Xc, ldx, Yc, ldy, kc, kper, g,
            partial, nblk, long_thr, pstride, A->halo_cap);
    else
        k_spmm_halo<T, DOT, KC, 8><<<grid, kSpmmRows, lds, ctx().stream>>>(
            A->n, A->rowptr, A->lcol, val, A->brick_rows, A->halo_ptr, A->halo_col, Xc, ldx, Yc, ldy, kc, kper, g,
            partial, nblk, long_thr, pstride, A->halo_cap);
}

template <typename T, bool DOT>
static bool spmm_halo(HIP_MAT *A, const T *val, const T *Xc, int64_t ldx, ColScalars g, T *Yc, int64_t ldy,
                      int kc, double *out, Seen seen)
{
    const int nblk = A->halo_blocks;
    const int nlong = A->nlong, long_thr = nlong > 0 ? kLongRow : INT_MAX;
    const int pstride = nblk + (DOT ? nlong : 0);
    double *partial = nullptr;
    if (DOT) {
        partial = partial_buf((size_t)kc, pstride, seen);
        if (!partial) return false;
    }
    {
        const double bytes = (sizeof(T) + 4.0) * A->nnz + 4.0 * (A->n + 1) + 2.0 * kc * (double)A->n * sizeof(T);
        const bool f64 = sizeof(T) == 8;
        ProfScope ps(DOT ? (f64 ? K_SPMM_DOT_F64 : K_SPMM_DOT_F32) : (f64 ? K_SPMM_F64 : K_SPMM_F32), bytes,
                     2.0 * kc * (double)A->nnz);
        switch (halo_kc(A, sizeof(T))) {
        case 8: spmm_halo_kc<T, DOT, 8>(A, val, Xc, ldx, g, Yc, ldy, kc, partial, nblk, long_thr, pstride); break;
        case 4: spmm_halo_kc<T, DOT, 4>(A, val, Xc, ldx, g, Yc, ldy, kc, partial, nblk, long_thr, pstride); break;
        case 2: spmm_halo_kc<T, DOT, 2>(A, val, Xc, ldx, g, Yc, ldy, kc, partial, nblk, long_thr, pstride); break;
        default: spmm_halo_kc<T, DOT, 1>(A, val, Xc, ldx, g, Yc, ldy, kc, partial, nblk, long_thr, pstride); break;
        }
        if (nlong > 0)
            k_spmm_long<T, DOT><<<(nlong + kSpmmRows / 64 - 1) / (kSpmmRows / 64), kSpmmRows, 0, ctx().stream>>>(
                A->rowptr, A->col, val, Xc, ldx, Yc, ldy, kc, g, A->long_rows, nlong, partial, pstride, nblk);
    }
    if (!check(hipGetLastError(), "k_spmm_halo")) return false;
    return !DOT || reduce_to_host(partial, kc, pstride, out);
}

template <typename T, bool DOT>
static bool spmm_t(HIP_MAT *A, const void *X, int64_t ldx, void *Y, int64_t ldy, int k, const int *xidx,
                   double *out, Seen seen)
{
    const int nblk = (A->n + kSpmmRows - 1) / kSpmmRows;
    const T *val = mat_vals<T>(A);
    if (!val) return false;
    for (int c0 = 0; c0 < k; c0 += kMaxCols) {
        const int kc = std::min(kMaxCols, k - c0);
        ColScalars g = make_scalars(kc, nullptr, nullptr, xidx ? xidx + c0 : nullptr);
        const T *Xc = (const T *)X + (xidx ? 0 : (int64_t)c0 * ldx);
        T *Yc = (T *)Y + (int64_t)c0 * ldy;
        if (A->gather_rows && kc >= 2) {  // one column gathers a line per entry either way
            if (!spmm_rows<T, DOT>(A, val, Xc, ldx, g, Yc, ldy, kc, DOT ? out + c0 : nullptr, seen)) return false;
            continue;
        }
        if (A->halo && (sizeof(T) == 8 || A->halo_f32)) {
            if (!spmm_halo<T, DOT>(A, val, Xc, ldx, g, Yc, ldy, kc, DOT ? out + c0 : nullptr, seen)) return false;
            continue;
        }
        // long rows (power-law graphs) go to k_spmm_long; their dot partials
        // follow the workgroups' in each column
        const int nlong = A->nlong, long_thr = nlong > 0 ? kLongRow : INT_MAX;
        const int pstride = nblk + (DOT ? nlong : 0);
        double *partial = nullptr;
        if (DOT) {
            partial = partial_buf((size_t)kc, pstride, seen);
            if (!partial) return false;
        }
        {
            const double bytes = (sizeof(T) + 4.0) * A->nnz + 4.0 * (A->n + 1) + 2.0 * kc * (double)A->n * sizeof(T);
            const bool f64 = sizeof(T) == 8;
            ProfScope ps(DOT ? (f64 ? K_SPMM_DOT_F64 : K_SPMM_DOT_F32) : (f64 ? K_SPMM_F64 : K_SPMM_F32), bytes,
                         2.0 * kc * (double)A->nnz);
            if (f64)
                k_spmm<T, DOT, 4, false><<<nblk, kSpmmRows, 0, ctx().stream>>>(
                    A->n, A->rowptr, A->col, val, Xc, ldx, Yc, ldy, kc, g, partial, nblk, long_thr, pstride);
            else if (DOT)
                k_spmm<T, DOT, 4, true><<<((nblk + 7) / 8) * 8, kSpmmRows, 0, ctx().stream>>>(
                    A->n, A->rowptr, A->col, val, Xc, ldx, Yc, ldy, kc, g, partial, nblk, long_thr, pstride);
            else
                k_spmm<T, DOT, 8, true><<<((nblk + 7) / 8) * 8, kSpmmRows, 0, ctx().stream>>>(
                    A->n, A->rowptr, A->col, val, Xc, ldx, Yc, ldy, kc, g, partial, nblk, long_thr, pstride);
            if (nlong > 0)
                k_spmm_long<T, DOT><<<(nlong + kSpmmRows / 64 - 1) / (kSpmmRows / 64), kSpmmRows, 0,
                                      ctx().stream>>>(A->rowptr, A->col, val, Xc, ldx, Yc, ldy, kc, g, A->long_rows,
                                                      nlong, partial, pstride, nblk);
        }
        if (!check(hipGetLastError(), "k_spmm")) return false;
        if (DOT && !reduce_to_host(partial, kc, pstride, out + c0)) return false;
    }
    return true;
}

void launch_spmm(int prec, HIP_MAT *A, const void *X, int64_t ldx, void *Y, int64_t ldy, int k, const int *xidx)
{
    if (k <= 0 || failed()) return;
    if (prec == GCGE_HIP_FP64) spmm_t<double, false>(A, X, ldx, Y, ldy, k, xidx, nullptr, Seen::in_stream);
    else spmm_t<float, false>(A, X, ldx, Y, ldy, k, xidx, nullptr, Seen::in_stream);
}

bool spmm_dot(int prec, HIP_MAT *A, const void *X, int64_t ldx, void *Y, int64_t ldy, int k, double *out, Seen seen)
{
    if (k <= 0) return true;
    if (failed()) return false;
    if (prec == GCGE_HIP_FP64) return spmm_t<double, true>(A, X, ldx, Y, ldy, k, nullptr, out, seen);
    return spmm_t<float, true>(A, X, ldx, Y, ldy, k, nullptr, out, seen);
}

// Residual sums of kc <= kMaxCols columns on the row-major gather path;
// out[3j + q]: r.r, x.x, Bx.Bx of column j.  B, when given, has no row longer
// than kLongRow.
template <typename T, int G>
static bool residual_rows_g(HIP_MAT *A, HIP_MAT *B, const T *X, int64_t ldx, ColScalars g, int kc, double *out)
{
    const int n = A->n, kp = G < 64 ? G : ((kc + 63) / 64) * 64;
    T *Xt = (T *)row_stage(sizeof(T) * (size_t)n * kp);
    if (!Xt) return false;
    const int RWG = rows_per_wg(G);
    const int nblk = (n + RWG - 1) / RWG, nlong = A->nlong, nlb = (nlong + 3) / 4;
    const int pstride = nblk + nlong;
    double *partial = partial_buf((size_t)3 * kc, pstride, Seen::in_stream);
    if (!partial) return false;
    {
        ProfScope ps(K_RESIDUAL,
                     12.0 * A->nnz + 4.0 * (n + 1) + (B ? 12.0 * B->nnz + 4.0 * (n + 1) : 0.0) +
                         (double)kc * n * sizeof(T),
                     2.0 * kc * (double)(A->nnz + (B ? B->nnz : 0)));
        k_rows_from_cols<T><<<dim3((n + 63) / 64, (kp + 63) / 64), 256, 0, ctx().stream>>>(n, X, ldx, kc, g, kp,
                                                                                           Xt);
        const dim3 grid(nlb + nblk, G < 64 ? 1 : kp / 64);
        const int lthr = nlong > 0 ? kLongRow : INT_MAX;
        if (B)
            k_residual_rows<T, G, true><<<grid, 256, 0, ctx().stream>>>(
                n, A->rowptr, A->col, A->val64, B->rowptr, B->col, B->val64, Xt, kp, kc, g, A->long_rows, nlong,
                nlb, lthr, partial, pstride, nblk);
        else
            k_residual_rows<T, G, false><<<grid, 256, 0, ctx().stream>>>(
                n, A->rowptr, A->col, A->val64, nullptr, nullptr, nullptr, Xt, kp, kc, g, A->long_rows, nlong, nlb,
                lthr, partial, pstride, nblk);
    }
    if (!check(hipGetLastError(), "k_residual_rows")) return false;
    return reduce_to_host(partial, 3 * kc, pstride, out);
}

template <typename T>
static bool residual_rows(HIP_MAT *A, HIP_MAT *B, const T *X, int64_t ldx, ColScalars g, int kc, double *out)
{
    if (kc > 32) return residual_rows_g<T, 64>(A, B, X, ldx, g, kc, out);
    if (kc > 16) return residual_rows_g<T, 32>(A, B, X, ldx, g, kc, out);
    if (kc > 8) return residual_rows_g<T, 16>(A, B, X, ldx, g, kc, out);
    if (kc > 4) return residual_rows_g<T, 8>(A, B, X, ldx, g, kc, out);
    if (kc > 2) return residual_rows_g<T, 4>(A, B, X, ldx, g, kc, out);
    return residual_rows_g<T, 2>(A, B, X, ldx, g, kc, out);
}

// Slots per column of k_residual_halo for A and B (or A alone), and columns
// per pass: 4, or 2 where the slots would exceed 56 KiB of LDS (the kernel
// adds 12).  0 when that kernel does not take them: both in staged blocks of
// the same rows, no row for k_spmm_long, the slots within the 56 KiB.
static int residual_halo_cap(const HIP_MAT *A, const HIP_MAT *B, size_t elem, int *kc)
{
    if (!A->halo || A->nlong > 0 || (B && (!B->halo || B->nlong > 0))) return 0;
    if (B && (!A->brick_rows != !B->brick_rows ||
              (A->brick_rows && !std::equal(A->brick_dims, A->brick_dims + 3, B->brick_dims))))
        return 0;
    const int cap = A->halo_cap + (B ? B->halo_cap - kSpmmRows : 0);
    const size_t room = (size_t)56 * 1024;
    *kc = cap * 4 * elem <= room ? 4 : 2;
    return cap * 2 * elem <= room ? cap : 0;
}

template <typename T, bool HASB, int MEA, int MEB>
static void residual_halo_launch(HIP_MAT *A, HIP_MAT *B, const T *X, int64_t ldx, int k, const ColScalars &g,
                                 double *partial, int cap, int kc)
{
    const int nblk = A->halo_blocks, kper = staged_columns(nblk, k, kc);
    const dim3 grid(((nblk + 7) / 8) * 8, (k + kper - 1) / kper);
    const size_t lds = (size_t)cap * kc * sizeof(T);
#define GH_RES(KC_)                                                                                             \
    k_residual_halo<T, HASB, KC_, MEA, MEB><<<grid, kSpmmRows, lds, ctx().stream>>>(                            \
        A->n, A->rowptr, A->lcol, A->val64, A->brick_rows, A->halo_ptr, A->halo_col,                            \
        HASB ? B->rowptr : nullptr, HASB ? B->lcol : nullptr, HASB ? B->val64 : nullptr,                        \
        HASB ? B->halo_ptr : nullptr, HASB ? B->halo_col : nullptr, X, ldx, k, kper, g, partial, nblk,  \
        cap)
    if (kc == 4) GH_RES(4);
    else GH_RES(2);
#undef GH_RES
}

template <typename T>
static void residual_halo(HIP_MAT *A, HIP_MAT *B, const T *X, int64_t ldx, int k, const ColScalars &g,
                          double *partial, int cap, int kc)
{
    const bool a28 = long_average(A), b28 = B && long_average(B);
    if (!B && !a28) residual_halo_launch<T, false, 8, 8>(A, B, X, ldx, k, g, partial, cap, kc);
    else if (!B) residual_halo_launch<T, false, 28, 8>(A, B, X, ldx, k, g, partial, cap, kc);
    else if (!a28 && !b28) residual_halo_launch<T, true, 8, 8>(A, B, X, ldx, k, g, partial, cap, kc);
    else if (!a28) residual_halo_launch<T, true, 8, 28>(A, B, X, ldx, k, g, partial, cap, kc);
    else if (!b28) residual_halo_launch<T, true, 28, 8>(A, B, X, ldx, k, g, partial, cap, kc);
    else residual_halo_launch<T, true, 28, 28>(A, B, X, ldx, k, g, partial, cap, kc);
}

template <typename T>
static bool residual_t(HIP_MAT *A, HIP_MAT *B, const void *X, int64_t ldx, const int *idx, int k,
                       const double *lambda, double *rnorm, double *xnorm, double *bxnorm)
{
    std::vector<double> tmp(3 * kMaxCols);
    int hkc = 4;
    const int cap = residual_halo_cap(A, B, sizeof(T), &hkc);
    const int nblk = cap ? A->halo_blocks : (A->n + kSpmmRows - 1) / kSpmmRows;
    for (int c0 = 0; c0 < k; c0 += kMaxCols) {
        const int kc = std::min(kMaxCols, k - c0);
        ColScalars g = make_scalars(kc, lambda + c0, nullptr, idx + c0);
        // row gather for scattered rows, and for long ones staged for SpMM but
        // not here (B's rows must all be short); a matrix with neither was
        // created with the direct gather asked for
        const auto by_rows = [](const HIP_MAT *M) { return M->gather_rows || (M->halo && long_average(M)); };
        const bool rows = by_rows(A) || (B && by_rows(B));
        if (!cap && rows && (!B || B->nlong == 0) && kc >= 2) {
            if (!residual_rows<T>(A, B, (const T *)X, ldx, g, kc, tmp.data())) return false;
            for (int j = 0; j < kc; j++) {
                rnorm[c0 + j] = std::sqrt(tmp[3 * j + 0]);
                xnorm[c0 + j] = std::sqrt(tmp[3 * j + 1]);
                if (bxnorm) bxnorm[c0 + j] = std::sqrt(tmp[3 * j + 2]);
            }
            continue;
        }
        double *partial = partial_buf((size_t)3 * kc, nblk, Seen::in_stream);
        if (!partial) return false;
        const double rbytes = 12.0 * A->nnz + 4.0 * (A->n + 1) + (B ? 12.0 * B->nnz + 4.0 * (B->n + 1) : 0.0) +
                              (double)kc * A->n * sizeof(T);
        {
            ProfScope ps(K_RESIDUAL, rbytes, 2.0 * kc * (double)(A->nnz + (B ? B->nnz : 0)));
            if (cap)
                residual_halo<T>(A, B, (const T *)X, ldx, kc, g, partial, cap, hkc);
            else if (B)
                k_residual<T, true><<<nblk, kSpmmRows, 0, ctx().stream>>>(
                    A->n, A->rowptr, A->col, A->val64, B->rowptr, B->col, B->val64, (const T *)X, ldx, kc, g,
                    partial);
            else
                k_residual<T, false><<<nblk, kSpmmRows, 0, ctx().stream>>>(
                    A->n, A->rowptr, A->col, A->val64, nullptr, nullptr, nullptr, (const T *)X, ldx, kc, g,
                    partial);
        }
        if (!check(hipGetLastError(), "k_residual")) return false;
        if (!reduce_to_host(partial, 3 * kc, nblk, tmp.data())) return false;
        for (int j = 0; j < kc; j++) {
            rnorm[c0 + j] = std::sqrt(tmp[3 * j + 0]);
            xnorm[c0 + j] = std::sqrt(tmp[3 * j + 1]);
            if (bxnorm) bxnorm[c0 + j] = std::sqrt(tmp[3 * j + 2]);
        }
    }
    return true;
}

bool residual_norms(int prec, HIP_MAT *A, HIP_MAT *B, const void *X, int64_t ldx, const int *idx, int k,
                    const double *lambda, double *rnorm, double *xnorm, double *bxnorm)
{
    if (k <= 0) return true;
    if (failed()) return false;
    if (prec == GCGE_HIP_FP64) return residual_t<double>(A, B, X, ldx, idx, k, lambda, rnorm, xnorm, bxnorm);
    return residual_t<float>(A, B, X, ldx, idx, k, lambda, rnorm, xnorm, bxnorm);
}

bool cg_update(int prec, int64_t n, void *x, int64_t ldx, const void *p, int64_t ldp, const void *w,
               int64_t ldw, void *r, int64_t ldr, int k, const double *alpha, double *rr)
{
    if (k <= 0) return true;
    if (failed()) return false;
    const int nb = grid_1d(n, 256);
    for (int c0 = 0; c0 < k; c0 += kMaxCols) {
        const int kc = std::min(kMaxCols, k - c0);
        ColScalars s = make_scalars(kc, alpha + c0, nullptr, nullptr);
        double *partial = partial_buf((size_t)kc, nb, Seen::everywhere);
        if (!partial) return false;
        dim3 grid(nb, kc);
        {
            ProfScope ps(prec == GCGE_HIP_FP64 ? K_CG_UPDATE_F64 : K_CG_UPDATE_F32,
                         6.0 * kc * (double)n * elem_size(prec), 6.0 * kc * (double)n);
            if (prec == GCGE_HIP_FP64)
                k_cg_update<double><<<grid, kBlock, 0, ctx().stream>>>(
                    n, (double *)x + (int64_t)c0 * ldx, ldx, (const double *)p + (int64_t)c0 * ldp, ldp,
                    (const double *)w + (int64_t)c0 * ldw, ldw, (double *)r + (int64_t)c0 * ldr, ldr, s, partial);
            else
                k_cg_update<float><<<grid, kBlock, 0, ctx().stream>>>(
                    n, (float *)x + (int64_t)c0 * ldx, ldx, (const float *)p + (int64_t)c0 * ldp, ldp,
                    (const float *)w + (int64_t)c0 * ldw, ldw, (float *)r + (int64_t)c0 * ldr, ldr, s, partial);
        }
        if (!check(hipGetLastError(), "k_cg_update")) return false;
        if (!reduce_to_host(partial, kc, nb, rr + c0)) return false;
    }
    return true;
}

bool cg_resid(int prec, int64_t n, const void *w, int64_t ldw, void *r, int64_t ldr, int k, const double *alpha,
              double *rr, Seen seen)
{
    if (k <= 0) return true;
    if (failed()) return false;
    const int nb = grid_1d(n, 256);
    for (int c0 = 0; c0 < k; c0 += kMaxCols) {
        const int kc = std::min(kMaxCols, k - c0);
        ColScalars s = make_scalars(kc, alpha + c0, nullptr, nullptr);
        double *partial = partial_buf((size_t)kc, nb, seen);
        if (!partial) return false;
        dim3 grid(nb, kc);
        {
            ProfScope ps(prec == GCGE_HIP_FP64 ? K_CG_UPDATE_F64 : K_CG_UPDATE_F32,
                         3.0 * kc * (double)n * elem_size(prec), 4.0 * kc * (double)n);
            sum_variant(n, 2.0 * kc * (double)n * elem_size(prec), [&](auto U, auto NT) {
                if (prec == GCGE_HIP_FP64)
                    k_cg_resid<double, U(), NT()><<<grid, kBlock, 0, ctx().stream>>>(
                        n, (const double *)w + (int64_t)c0 * ldw, ldw, (double *)r + (int64_t)c0 * ldr, ldr, s,
                        partial);
                else
                    k_cg_resid<float, U(), NT()><<<grid, kBlock, 0, ctx().stream>>>(
                        n, (const float *)w + (int64_t)c0 * ldw, ldw, (float *)r + (int64_t)c0 * ldr, ldr, s,
                        partial);
            });
        }
        if (!check(hipGetLastError(), "k_cg_resid")) return false;
        if (!reduce_to_host(partial, kc, nb, rr + c0)) return false;
    }
    return true;
}

bool pcg_resid(int prec, int64_t n, const void *w, int64_t ldw, void *r, int64_t ldr, const void *dinv, int k,
               const double *alpha, double *rz, double *rr, Seen seen)
{
    if (k <= 0) return true;
    if (failed()) return false;
    const int nb = grid_1d(n, 256);
    std::vector<double> tmp(2 * kMaxCols);
    for (int c0 = 0; c0 < k; c0 += kMaxCols) {
        const int kc = std::min(kMaxCols, k - c0);
        ColScalars s = make_scalars(kc, alpha + c0, nullptr, nullptr);
        double *partial = partial_buf((size_t)2 * kc, nb, seen);
        if (!partial) return false;
        dim3 grid(nb, kc);
        {
            ProfScope ps(prec == GCGE_HIP_FP64 ? K_CG_UPDATE_F64 : K_CG_UPDATE_F32,
                         3.0 * kc * (double)n * elem_size(prec) + (double)n * elem_size(prec), 6.0 * kc * (double)n);
            sum_variant(n, 2.0 * kc * (double)n * elem_size(prec), [&](auto U, auto NT) {
                if (prec == GCGE_HIP_FP64)
                    k_pcg_resid<double, U(), NT()><<<grid, kBlock, 0, ctx().stream>>>(
                        n, (const double *)w + (int64_t)c0 * ldw, ldw, (double *)r + (int64_t)c0 * ldr, ldr,
                        (const double *)dinv, s, partial);
                else
                    k_pcg_resid<float, U(), NT()><<<grid, kBlock, 0, ctx().stream>>>(
                        n, (const float *)w + (int64_t)c0 * ldw, ldw, (float *)r + (int64_t)c0 * ldr, ldr,
                        (const float *)dinv, s, partial);
            });
        }
        if (!check(hipGetLastError(), "k_pcg_resid")) return false;
        if (!reduce_to_host(partial, 2 * kc, nb, tmp.data())) return false;
        for (int j = 0; j < kc; j++) {
            rz[c0 + j] = tmp[2 * j];
            rr[c0 + j] = tmp[2 * j + 1];
        }
    }
    return true;
}

void launch_diag_inv(HIP_MAT *A)
{
    k_diag_inv<<<(A->n + kBlock - 1) / kBlock, kBlock, 0, ctx().stream>>>(A->n, A->rowptr, A->col, A->val64,
                                                                         A->dinv64, A->dinv32);
    check(hipGetLastError(), "k_diag_inv");
}

void launch_cg_search(int prec, int64_t n, void *x, int64_t ldx, void *p, int64_t ldp, const void *r, int64_t ldr,
                      int kx, int kp, const double *alpha, const double *beta, const void *dinv)
{
    const int k = std::max(kx, kp);
    if (k <= 0 || failed()) return;
    for (int c0 = 0; c0 < k; c0 += kMaxCols) {
        const int kc = std::min(kMaxCols, k - c0);
        const int kxc = std::max(0, std::min(kc, kx - c0)), kpc = std::max(0, std::min(kc, kp - c0));
        std::vector<double> aa(kc, 0.0), bb(kc, 0.0);
        for (int j = 0; j < kxc; j++) aa[j] = alpha[c0 + j];
        for (int j = 0; j < kpc; j++) bb[j] = beta[c0 + j];
        ColScalars s = make_scalars(kc, aa.data(), bb.data(), nullptr);
        {
            ProfScope ps(prec == GCGE_HIP_FP64 ? K_CG_SEARCH_F64 : K_CG_SEARCH_F32,
                         (3.0 * kxc + 3.0 * kpc - 1.0 * std::min(kxc, kpc)) * (double)n * elem_size(prec) +
                             (dinv && kpc > 0 ? (double)n * elem_size(prec) : 0.0),
                         0.0);
            const double held = (1.0 * kxc + kpc + kc) * (double)n * elem_size(prec);  // x, r and p
#define GH_SEARCH(T_, PRE_)                                                                                     \
    run_variant<T_>(held, [&](auto V, auto NT) {                                                          \
        k_cg_search<T_, PRE_, V(), NT()><<<run_grid(n, V(), kc), kBlock, 0, ctx().stream>>>(                    \
            n, (T_ *)x + (int64_t)c0 * ldx, ldx, (T_ *)p + (int64_t)c0 * ldp, ldp,                              \
            (const T_ *)r + (int64_t)c0 * ldr, ldr, kxc, kpc, s, (const T_ *)dinv);                             \
    })
            if (prec == GCGE_HIP_FP64) {
                if (dinv) GH_SEARCH(double, true);
                else GH_SEARCH(double, false);
            } else {
                if (dinv) GH_SEARCH(float, true);
                else GH_SEARCH(float, false);
            }
#undef GH_SEARCH
        }
        if (!check(hipGetLastError(), "k_cg_search")) return;
    }
}

bool sampled_outer(int prec, HIP_MAT *A, const void *X, int64_t ldx, int k, const double *w, double *g_dev)
{
    if (failed()) return false;
    const int *rowidx = mat_rowidx(A);
    if (!rowidx) return false;
    if (!check(hipMemsetAsync(g_dev, 0, sizeof(double) * A->nnz, ctx().stream), "memset g")) return false;
    const int nb = (A->nnz + kBlock - 1) / kBlock;
    for (int c0 = 0; c0 < k; c0 += kMaxCols) {
        const int kc = std::min(kMaxCols, k - c0);
        ColScalars s = make_scalars(kc, w + c0, nullptr, nullptr);
        if (prec == GCGE_HIP_FP64)
            k_sampled_outer<double><<<nb, kBlock, 0, ctx().stream>>>(A->nnz, rowidx, A->col,
                                                                     (const double *)X + (int64_t)c0 * ldx, ldx,
                                                                     kc, s, g_dev);
        else
            k_sampled_outer<float><<<nb, kBlock, 0, ctx().stream>>>(A->nnz, rowidx, A->col,
                                                                    (const float *)X + (int64_t)c0 * ldx, ldx,
                                                                    kc, s, g_dev);
        if (!check(hipGetLastError(), "k_sampled_outer")) return false;
    }
    return true;
}

void launch_csr_gather_sum(int nparam, const int *jrowptr, const int *jnz, const double *jval, const int *map,
                           int nnz, const double *g, double *grad, double scale, bool accumulate, double *bad)
{
    if (nparam <= 0 || failed()) return;
    k_csr_gather_sum<<<(nparam + kBlock - 1) / kBlock, kBlock, 0, ctx().stream>>>(
        nparam, jrowptr, jnz, jval, map, nnz, g, grad, scale, accumulate ? 1 : 0, bad);
    check(hipGetLastError(), "k_csr_gather_sum");
}

void launch_rows_in(int prec, int64_t n, const double *x, int64_t ldx, const int *perm, void *y, int64_t ldy, int k)
{
    if (k <= 0 || n <= 0 || failed()) return;
    if (prec == GCGE_HIP_FP64)
        k_rows_in<double><<<run_grid(n, 1, k), kBlock, 0, ctx().stream>>>(n, x, ldx, perm, (double *)y, ldy);
    else
        k_rows_in<float><<<run_grid(n, 1, k), kBlock, 0, ctx().stream>>>(n, x, ldx, perm, (float *)y, ldy);
    check(hipGetLastError(), "k_rows_in");
}

void launch_fetch(const void *host, void *dev, size_t bytes)
{
    if (bytes == 0 || failed()) return;
    const size_t units = (bytes + 15) / 16;
    k_fetch<<<(unsigned)((units + kBlock - 1) / kBlock), kBlock, 0, ctx().stream>>>((const int4 *)host, (int4 *)dev,
                                                                                    units);
    check(hipGetLastError(), "k_fetch");
}

void launch_rows_out(int prec, int64_t n, double *x, int64_t ldx, const int *perm, const void *y, int64_t ldy, int k)
{
    if (k <= 0 || n <= 0 || failed()) return;
    if (prec == GCGE_HIP_FP64)
        k_rows_out<double><<<run_grid(n, 1, k), kBlock, 0, ctx().stream>>>(n, x, ldx, perm, (const double *)y, ldy);
    else
        k_rows_out<float><<<run_grid(n, 1, k), kBlock, 0, ctx().stream>>>(n, x, ldx, perm, (const float *)y, ldy);
    check(hipGetLastError(), "k_rows_out");
}

// matrix helpers used by hip_backend.cpp
void launch_rowidx(HIP_MAT *A)
{
    k_rowidx<<<(A->n + kBlock - 1) / kBlock, kBlock, 0, ctx().stream>>>(A->n, A->rowptr, A->rowidx);
    check(hipGetLastError(), "k_rowidx");
}

void launch_to_f32(int64_t n, const double *a, float *b)
{
    k_to_f32<<<(unsigned)((n + kBlock - 1) / kBlock), kBlock, 0, ctx().stream>>>(n, a, b);
    check(hipGetLastError(), "k_to_f32");
}

}  // namespace gh

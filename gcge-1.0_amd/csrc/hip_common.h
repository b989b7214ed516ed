// hip_common.h -- internal types of the gfx950 GCGE backend.
//
// One process drives one GPU through one HIP stream (default priority).
// Multivectors are single column-major allocations whose leading dimension
// is padded to an odd multiple of 256 elements, so every column starts on a
// 2 KiB (FP64) / 1 KiB (FP32) boundary and any column range can be streamed
// with aligned, coalesced loads.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "gcge_app_hip.h"

namespace gh {

constexpr uint32_t kMagicMV = 0x4d56434fu;   // multivector
constexpr uint32_t kMagicCol = 0x4c4f4356u;  // column view / vector
constexpr uint32_t kMagicMat = 0x54414d48u;  // HIP_MAT

constexpr int kMaxCols = 128;     // per-launch column batch for per-column scalars (2.5 KB of kernel arguments)
constexpr int kMaxChunks = 512;   // split-n partial sums of reductions
constexpr size_t kHostPartials = 2048;  // most partial sums that are added on the host

struct MV;

// A vector handle (void *) is a view of one column of a multivector.
struct Col {
    uint32_t magic;
    MV *mv;
    int col;
    int owner;  // 1: this vector owns mv (created by VecCreateBy*)
};

struct MV {
    uint32_t magic;
    int prec;         // GCGE_HIP_FP64 / GCGE_HIP_FP32
    int64_t n;        // rows
    int64_t ld;       // leading dimension in elements
    int ncols;
    void *data;       // device memory, ld * ncols elements
    Col *cols;        // ncols column views
    HIP_MAT *mat;     // matrix this multivector was created from (may be NULL)
};

}  // namespace gh

// Rows with more than this many stored entries are multiplied by a whole
// wavefront each (k_spmm_long) instead of one thread (k_spmm): power-law
// graphs carry rows thousands of entries long.
constexpr int kLongRow = 64;

struct HIP_MAT_ {
    uint32_t magic;
    int n;
    int nnz;
    int *rowptr;      // device, n+1
    int *col;         // device, nnz
    int *rowidx;      // device, nnz (row of each stored entry; built on demand)
    double *val64;    // device, nnz
    float *val32;     // device, nnz (built on demand)
    int nlong;        // rows with more than kLongRow stored entries
    int *long_rows;   // device, nlong: their indices, ascending (null when none)
    double *dinv64;   // device, n: 1 / a_ii (1 where a_ii is 0 or absent; built on demand)
    float *dinv32;    // device, n: the same, rounded to FP32
    int prec;         // precision of multivectors created from this matrix
    int max_row_nnz;
    int gather_rows;  // SpMM gathers from a row-major copy of X (scattered column indices)
    double row_abs_max;  // max_i sum_j |a_ij| (Gershgorin bound of ||A||_2)
    // staged-row-block SpMM (k_spmm_halo), chosen at creation when every
    // block of up to 256 rows reads at most kHaloCap - 256 rows besides its own
    int halo;                 // 1: SpMM by k_spmm_halo
    int halo_f32;             // 1: FP32 products too (else k_spmm)
    int halo_blocks;          // row blocks
    int halo_cap;             // LDS slots per column: 256 own rows + the most extras of any block (rounded)
    int *halo_ptr;            // device, halo_blocks+1: each block's extras in halo_col
    int *halo_col;            // device: the other rows a block's entries read, ascending
    unsigned short *lcol;     // device, nnz: each entry's slot (i-th own row -> i, extra j -> 256+j)
    int *brick_rows;          // device, 256 per block: its rows, -1 for none (null: 256 consecutive rows)
    int brick_dims[3];        // box grid of brick_rows: matrices of equal dims have the same blocks
    double halo_bytes;        // device bytes of these arrays
    // row order (HIP_MatCreateFromCSROrdered): the device matrix is
    // P A P^T; multivectors created from it hold rows in the same order and
    // are permuted at host transfers.  Host arrays, null when unordered.
    int *perm_h;              // n: new position -> the caller's row
    int *iperm_h;             // n: the caller's row -> new position
    int *nzmap_h;             // nnz: the caller's entry index -> stored entry index
    int *perm_d, *nzmap_d;    // device copies of perm_h and nzmap_h (built on demand)
};

// largest LDS slot count per column of a k_spmm_halo row block
constexpr int kHaloCap = 4096;

namespace gh {

struct Ctx {
    bool init = false;
    int device = 0;
    hipStream_t stream = nullptr;
    // device scratch for partial reductions and staging (grown on demand)
    void *scratch = nullptr;
    size_t scratch_bytes = 0;
    void *rows = nullptr;  // row-major X staging of the SpMM gather path
    size_t rows_bytes = 0;
    // memory of TmpDev between calls, given back where memory is short and with
    // the last matrix
    void *tmp = nullptr;
    size_t tmp_bytes = 0;
    bool tmp_used = false;
    // pinned host buffer for results that kernels write and the host reads
    double *hbuf = nullptr;
    size_t hbuf_bytes = 0;
    // numbers that kernels write beside their results: the host takes a result
    // once its number is the launch's.  An array of its own, so that no other
    // data can look like a number; it only grows, and the numbers with it.
    unsigned long long *hseq = nullptr;
    size_t hseq_count = 0;
    unsigned long long seq = 0;  // the last launch's
    // partial sums of a small launch, in coherent host memory: the host adds them
    double *hpart = nullptr;
    double dev_bytes = 0.0;
    int num_cu = 0;
    // host->device staging ring (pinned host side, device side)
    char *stage_h = nullptr;
    char *stage_d = nullptr;
    size_t stage_cap = 0;
    size_t stage_off = 0;
};

Ctx &ctx();
bool ensure_ctx();
// device address of this GPU's no-allocation scratch array (noalloc.hip),
// looked up once per device at context set-up
bool noalloc_setup(int device);
void *scratch(size_t bytes);           // device scratch of at least bytes
void *row_stage(size_t bytes);         // device staging of row-major X copies (SpMM), at least bytes
double *host_buf(size_t count);        // pinned host doubles, writable by kernels
// The first count numbers and the next launch's (one report at a time: the
// launch, then wait_seq); null (latched) without memory.
unsigned long long *host_seq(size_t count, unsigned long long *next);
// Waits until the first count numbers are all `want`, written by kernels
// queued on the stream; false (latched) when it has drained without them.
bool wait_seq(size_t count, unsigned long long want);
// Host memory for `count` <= kHostPartials partial sums that the next launch
// writes, marked as not yet written; null (latched) without memory.
double *host_partials(size_t count);
// Waits until the launch has written all of them; false (latched) on an error.
bool wait_partials(size_t count);
// Copy small host data (coefficients) to device memory without blocking:
// the bytes go through a pinned ring whose slots are reused only after the next
// stream synchronisation, or after the results of a later launch have reached
// the host (wait_seq, wait_partials): the copies and the launches that read them
// come before it on the stream.  Returns the device address.
void *stage_to_device(const void *host, size_t bytes);
bool sync();                           // stream synchronize + error check

// ---- kernel profiler (opt-in): HIP events around each launch of a kernel
// class on the backend stream, with the algorithmic bytes and flops of the
// launch; resolved at stream synchronisation points.
enum KClass {
    K_SPMM_F64 = 0, K_SPMM_F32, K_SPMM_DOT_F64, K_SPMM_DOT_F32, K_AXPBY, K_DOTS, K_CG_UPDATE_F64, K_CG_UPDATE_F32,
    K_CG_SEARCH_F64, K_CG_SEARCH_F32,
    K_GRAM_MFMA_F64, K_GRAM_MFMA_F32, K_GRAM_THIN, K_LINCOMB_MFMA_F64, K_LINCOMB_MFMA_F32, K_LINCOMB_THIN,
    K_RESIDUAL, K_COPY, K_SWAP, K_OTHER, K_NUM
};
struct ProfScope {
    int kind;
    bool on;
    ProfScope(int kind, double bytes, double flops);
    ~ProfScope();
};
const char *kclass_name(int k);

// error latch
void latch(int code, const char *fmt, ...);
bool failed();
bool check(hipError_t e, const char *what);

inline MV *as_mv(void **h) {
    MV *m = reinterpret_cast<MV *>(h);
    return (m && m->magic == kMagicMV) ? m : nullptr;
}
inline Col *as_col(void *h) {
    Col *c = reinterpret_cast<Col *>(h);
    return (c && c->magic == kMagicCol) ? c : nullptr;
}
inline HIP_MAT *as_mat(void *h) {
    HIP_MAT *m = reinterpret_cast<HIP_MAT *>(h);
    return (m && m->magic == kMagicMat) ? m : nullptr;
}

size_t elem_size(int prec);
void *col_ptr(MV *m, int64_t c);
const float *mat_val32(HIP_MAT *A);
const int *mat_rowidx(HIP_MAT *A);
// device copies of the row order and of the entry order (built on first use;
// null without an error where there is no memory for them)
const int *mat_perm(HIP_MAT *A);
const int *mat_nzmap(HIP_MAT *A);
// 1 / diagonal of A in the given precision (built on first use)
const void *mat_dinv(HIP_MAT *A, int prec);

// ---- launchers (hip_kernels.hip) --------------------------------------
// All launchers validate nothing; callers check ranges first.
// Column j of a range is base + j * ld.

// y_j = a_j x_j + b_j y_j (branch rules of y = a x + b y), j < k <= kMaxCols
void launch_axpby(int prec, int64_t n, const void *x, int64_t ldx, void *y, int64_t ldy, int k,
                  const double *a, const double *b, const int *xidx);
// out_j = <x_j, y_j>, FP64 accumulation; result in host array out
bool dots(int prec, int64_t n, const void *x, int64_t ldx, const void *y, int64_t ldy, int k,
          double *out);
// y_j <- x_j (with precision conversion), j < k
void launch_copy(int xprec, const void *x, int64_t ldx, int yprec, void *y, int64_t ldy, int64_t n,
                 int k);
void launch_swap(int prec, void *x, int64_t ldx, void *y, int64_t ldy, int64_t n, int k);
void launch_zero_rows(int prec, void *x, int64_t ldx, int64_t n, int k, const unsigned char *mask);
// Y_j = A X_j (xidx: optional gather of X columns, k <= kMaxCols when given)
void launch_spmm(int prec, HIP_MAT *A, const void *X, int64_t ldx, void *Y, int64_t ldy, int k,
                 const int *xidx);
// Where the columns that a launch writes beside its sums are complete when the
// host has the sums: for later launches of the stream, or for other streams too
enum class Seen { in_stream, everywhere };
// Y_j = A X_j and out_j = <X_j, Y_j>
bool spmm_dot(int prec, HIP_MAT *A, const void *X, int64_t ldx, void *Y, int64_t ldy, int k,
              double *out, Seen seen);
// rnorm/xnorm/bxnorm of A x_j - lambda_j B x_j, x_j = X(:, idx[j])
bool residual_norms(int prec, HIP_MAT *A, HIP_MAT *B, const void *X, int64_t ldx, const int *idx,
                    int k, const double *lambda, double *rnorm, double *xnorm, double *bxnorm);
// x_j += alpha_j p_j ; r_j -= alpha_j w_j ; rr_j = <r_j, r_j>
bool cg_update(int prec, int64_t n, void *x, int64_t ldx, const void *p, int64_t ldp, const void *w,
               int64_t ldw, void *r, int64_t ldr, int k, const double *alpha, double *rr);
// r_j -= alpha_j w_j ; rr_j = <r_j, r_j>
bool cg_resid(int prec, int64_t n, const void *w, int64_t ldw, void *r, int64_t ldr, int k, const double *alpha,
              double *rr, Seen seen);
// r_j -= alpha_j w_j ; rz_j = <r_j, dinv .* r_j> ; rr_j = <r_j, r_j>
bool pcg_resid(int prec, int64_t n, const void *w, int64_t ldw, void *r, int64_t ldr, const void *dinv, int k,
               const double *alpha, double *rz, double *rr, Seen seen);
// dinv64[i] = 1 / a_ii (1 where a_ii is 0 or absent), dinv32 its FP32 rounding
void launch_diag_inv(HIP_MAT *A);
// x_j += alpha_j p_j (j < kx), then p_j = r_j + beta_j p_j (j < kp); with
// dinv (not null), p_j = dinv .* r_j + beta_j p_j
void launch_cg_search(int prec, int64_t n, void *x, int64_t ldx, void *p, int64_t ldp, const void *r, int64_t ldr,
                      int kx, int kp, const double *alpha, const double *beta, const void *dinv = nullptr);
// G (p x q, host, column-major ldg) = V^T W
bool gram(int prec, int64_t n, const void *V, int64_t ldv, int p, const void *W, int64_t ldw, int q,
          double *G, int ldg, bool upper_only);
// Y = beta Y + alpha X C  (C host, p x q, column-major ldc)
bool lincomb(int prec, int64_t n, const void *X, int64_t ldx, int p, void *Y, int64_t ldy, int q,
             const double *C, int ldc, double alpha, double beta);
// per-nonzero sampled outer product g_e = sum_i w_i x_i[row_e] x_i[col_e]
bool sampled_outer(int prec, HIP_MAT *A, const void *X, int64_t ldx, int k, const double *w,
                   double *g_dev);
// grad[p] = scale * sum_t jval[t] g[map[jnz[t]]] over t in [jrowptr[p],
// jrowptr[p+1]) (map null: g[jnz[t]]), added to grad[p] when accumulate; *bad
// (host memory) becomes 1 when a jnz[t] lies outside [0, nnz)
void launch_csr_gather_sum(int nparam, const int *jrowptr, const int *jnz, const double *jval, const int *map,
                           int nnz, const double *g, double *grad, double scale, bool accumulate, double *bad);
// y_j[i] = x_j[perm[i]] (perm null: x_j[i]), x in FP64 with distance ldx, and
// the reverse x_j[perm[i]] = y_j[i]; j < k
void launch_rows_in(int prec, int64_t n, const double *x, int64_t ldx, const int *perm, void *y, int64_t ldy, int k);
// bytes (rounded up to 16) from coherent host memory to device memory, both
// 16-byte aligned
void launch_fetch(const void *host, void *dev, size_t bytes);
void launch_rows_out(int prec, int64_t n, double *x, int64_t ldx, const int *perm, const void *y, int64_t ldy, int k);

}  // namespace gh

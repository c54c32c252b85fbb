// Internal definitions shared by the libommhip.so translation units.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>

#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <map>
#include <string>
#include <utility>
#include <vector>

#include "omm_hip.h"

namespace omx {

// Per-thread last error message (omx_last_error()).
void set_error(const char *fmt, ...);
void clear_error();

#define OMX_CHECK_HIP(expr)                                                                    \
    do {                                                                                       \
        hipError_t e_ = (expr);                                                                \
        if (e_ != hipSuccess) {                                                                \
            omx::set_error("%s failed: %s (%s:%d)", #expr, hipGetErrorString(e_), __FILE__,    \
                           __LINE__);                                                          \
            return OMX_ERR_HIP;                                                                \
        }                                                                                      \
    } while (0)

#define OMX_REQUIRE(cond, ...)                                                                 \
    do {                                                                                       \
        if (!(cond)) {                                                                         \
            omx::set_error(__VA_ARGS__);                                                       \
            return OMX_ERR_ARG;                                                                \
        }                                                                                      \
    } while (0)

// Event pair recorded around one launch of a timed kernel class.
struct ProfEvent {
    hipEvent_t start, stop;
    int kclass;
};

}  // namespace omx

// Launch shape of a real SpMM: blocks whose loads are issued together (1, 4, 8), waves stacked in
// rows per workgroup (1, 2, 4), block columns walked per workgroup, XCD map (0: each XCD owns
// contiguous rows; 1: each XCD walks one row chunk at a time).
struct omx_spmm_shape_s {
    int batch = 4;
    int wpg = 1;
    int jper = 1;
    int mode = 1;
};

struct omx_ctx_s {
    int device = 0;
    hipStream_t stream = nullptr;
    // Device workspace for split-K partial products and reduction partials (grown on demand).
    void *ws = nullptr;
    size_t ws_bytes = 0;
    // Small device buffer for reduction results and pinned host mirror for scalar readback.
    double *d_scalars = nullptr;
    double *h_scalars = nullptr;  // pinned; r_scalars is its address on the device
    double *r_scalars = nullptr;
    // Event timing.
    bool prof_on = false;
    std::vector<omx::ProfEvent> prof_pending;
    std::vector<hipEvent_t> prof_pool;
    double prof_ms[OMX_K_COUNT] = {0};
    int64_t prof_count[OMX_K_COUNT] = {0};
    double prof_flops[OMX_K_COUNT] = {0};  // algorithmic flops of the timed launches
    double prof_bytes[OMX_K_COUNT] = {0};  // algorithmic (minimum) HBM bytes of the timed launches
    int num_cus = 256;
    int gemm_cfg = -1;    // forced GEMM tile configuration (-1: chosen by shape)
    // Set around a product known to be symmetric: 1 = only the lower triangle is wanted, 2 = both
    // triangles.  A kernel that writes both sets 3 (no mirror pass needed).
    int gemm_sym = 0;
    bool one_part = false;  // set around products whose K is not to be split
    bool carry64 = false;   // set around FP64 products that carry their sums whatever their size
    omx_spmm_shape_s spmm_shape;  // forced SpMM launch shape (when spmm_forced)
    bool spmm_forced = false;
    bool spmm_stencil = false;  // lattice operators use the 2.5-D stencil SpMM (omx_spmm_stencil)
    // Device flag for the grouped solver: while set, GEMM, SpMM and reduction launches do nothing
    // when *launch_mask == 0, and GEMMs do not split K (no workspace, so launches can be captured).
    const int *launch_mask = nullptr;
    // autotuner: per-shape choices (configuration or SpMM launch shape, best time in ms)
    bool autotune = false;
    std::map<std::string, std::pair<int, double>> tune_gemm;
    std::map<std::string, std::pair<omx_spmm_shape_s, double>> tune_spmm;
};

struct omx_bsr_s {
    omx_ctx ctx = nullptr;
    int nb = 0;        // basis size
    int nbc = 0;       // block columns = ceil(nb/4)
    int64_t nnzb = 0;  // stored 4x4 blocks
    int is_complex = 0;
    int max_blocks_per_col = 0;
    int *d_colptr = nullptr;  // nbc+1
    int *d_rowidx = nullptr;  // nnzb
    double *d_val = nullptr;  // 16*nnzb (x2 if complex)
    int *d_walk = nullptr;    // optional order in which SpMMs visit the block columns (nbc)
    // Lx, Ly, Lz when the pattern is the periodic 7-point stencil of that lattice of 4x4 blocks
    // (recognised at upload; 0 otherwise)
    int lat[3] = {0, 0, 0};
    // LDS-staged gathers: block columns taken `group` at a time in walk order; group g gathers the
    // distinct block rows uidx[gptr[g] .. gptr[g+1]) and block l reads slot[l] of them
    int group = 0, ngroups = 0;
    int *d_gptr = nullptr, *d_uidx = nullptr;
    unsigned char *d_slot = nullptr;
};

namespace omx {

constexpr int kScalarSlots = 256;

// ---- element types -----------------------------------------------------------------------------
// Real (double, float) and complex (Cx<double>, Cx<float>: the Fortran (re, im) layout).  The
// element-wise kernels are written once over El<T>; for real types the imaginary terms are
// compiled out, so the real arithmetic (and its rounding) is exactly the real-only one.

template <typename R_>
struct Cx {
    R_ x, y;
};
template <typename T>
struct El {
    static constexpr bool cplx = false;
    __device__ static inline double re(const T &v) { return (double)v; }
    __device__ static inline double im(const T &) { return 0.0; }
    __device__ static inline T make(double r, double) { return (T)r; }
};
template <typename R_>
struct El<Cx<R_>> {
    static constexpr bool cplx = true;
    __device__ static inline double re(const Cx<R_> &v) { return (double)v.x; }
    __device__ static inline double im(const Cx<R_> &v) { return (double)v.y; }
    __device__ static inline Cx<R_> make(double r, double i) { return Cx<R_>{(R_)r, (R_)i}; }
};
template <>
struct El<double2> {
    static constexpr bool cplx = true;
    __device__ static inline double re(const double2 &v) { return v.x; }
    __device__ static inline double im(const double2 &v) { return v.y; }
    __device__ static inline double2 make(double r, double i) { return make_double2(r, i); }
};

// hipMalloc that gives back omx_malloc's idle blocks before it fails
hipError_t dev_malloc(void **p, size_t bytes);
// Gives them back; false if there are none.
bool dev_release();
// Ensure ctx->ws holds at least `bytes`.  Returns OMX_OK or an error.
int ensure_ws(omx_ctx ctx, size_t bytes);

// Look up this device's copy of the static scratch of omx_omm_pr_dots_noalloc (once per device,
// with the device current).  Returns OMX_OK or an error.
int noalloc_setup(int device);

// Begin / end a timed launch of kernel class `kclass` (no-ops unless profiling is on).
void prof_begin(omx_ctx ctx, int kclass, hipEvent_t *ev_start);
void prof_end(omx_ctx ctx, int kclass, hipEvent_t ev_start);
// Add the algorithmic work of one launch to the class totals (only while profiling is on).
inline void prof_work(omx_ctx ctx, int kclass, double flops, double bytes) {
    if (!ctx->prof_on) return;
    ctx->prof_flops[kclass] += flops;
    ctx->prof_bytes[kclass] += bytes;
}

inline bool valid_real_dt(int dt) { return dt == OMX_F64 || dt == OMX_F32; }
inline int dt_size(int dt) {
    switch (dt) {
        case OMX_F64: return 8;
        case OMX_F32: return 4;
        case OMX_BF16: return 2;
        case OMX_C128: return 16;
        case OMX_C64: return 8;
        default: return 0;
    }
}
inline bool is_trans(char op) { return op == 't' || op == 'T' || op == 'c' || op == 'C'; }
inline bool valid_op(char op) { return op == 'n' || op == 'N' || is_trans(op); }

// Waits for what a kernel writes to ctx->r_scalars, straight into ctx->h_scalars on the host: no copy command
// behind the kernel (a CG step reads back twice).
int read_scalars(omx_ctx ctx);

// Position of workgroup id w among T when each XCD (ids are dealt round-robin over 8) takes a contiguous
// band of T / 8 positions, the first T mod 8 bands one more: a bijection of 0..T-1 for every T.
__device__ inline int xcd_band(int w, int T) { return (w & 7) * (T >> 3) + min(w & 7, T & 7) + (w >> 3); }

// Tile index for workgroup id w of a tiles_m x tiles_n product: workgroup ids are dealt
// round-robin over the 8 XCDs, so each XCD is given a contiguous band of tiles; inside a band
// the tiles go in groups of 8 tile rows, column by column, so operand panels are shared in one
// XCD's L2.
__device__ inline void tile_of(int w, int tiles_m, int tiles_n, int &tm, int &tn) {
    const int t = xcd_band(w, tiles_m * tiles_n);
    constexpr int GM = 8;
    int group = t / (GM * tiles_n);
    int first_m = group * GM;
    int gm = min(tiles_m - first_m, GM);
    int in = t % (GM * tiles_n);
    tm = first_m + in % gm;
    tn = in / gm;
}

// Lower-triangle tiles (tm >= tn) of an nt x nt tile grid, nt(nt+1)/2 of them, dealt over the
// XCDs as tile_of does and enumerated by tile rows (products known to be symmetric compute only
// these and mirror them).
__device__ inline void tile_of_lower(int w, int nt, int &tm, int &tn) {
    const int t = xcd_band(w, nt * (nt + 1) / 2);
    int r = (int)((sqrtf(8.0f * (float)t + 1.0f) - 1.0f) * 0.5f);
    while (r > 0 && r * (r + 1) / 2 > t) --r;
    while ((r + 1) * (r + 2) / 2 <= t) ++r;
    tm = r;
    tn = t - r * (r + 1) / 2;
}

// Output area (elements) of the lower-triangle tiles of an n x n product with bm x bm tiles: the
// flop count of a symmetric product is 2*k times this (the MFMA work actually issued).
inline double sym_area(int n, int bm) {
    double area = 0.0;
    for (int a = 0; a * bm < n; ++a) area += (double)std::min(bm, n - a * bm) * std::min(n, (a + 1) * bm);
    return area;
}

// Launch helpers implemented in the .hip files.
int launch_gemm(omx_ctx ctx, int prec, int dt, bool trA, bool trB, int m, int n, int k, double alpha,
                const void *A, int64_t lda, const void *B, int64_t ldb, double beta, void *C, int64_t ldc);
// FP64 products of dgemm.hip (npair = 2: alpha*(A1*B1 + A2*B2), 'n','n'); OMX_ERR_UNSUPPORTED (nothing
// launched) for leading dimensions beyond 2^20.
int launch_dgemm(omx_ctx ctx, bool trA, bool trB, int npair, int m, int n, int k, double alpha, const double *A1,
                 const double *A2, int64_t lda, const double *B1, const double *B2, int64_t ldb, double beta0,
                 const double *C0, int64_t ldc0, double beta, double *C, int64_t ldc);
// nbatch products C_b := alpha*A_b*B_b ('n','n') at strides sA, sB, sC elements.
int launch_dgemm_batched(omx_ctx ctx, int m, int n, int k, double alpha, const double *A, int64_t lda, int64_t sA,
                         const double *B, int64_t ldb, int64_t sB, double *C, int64_t ldc, int64_t sC, int nbatch);
// The same for FP32 products on FP32 storage (C0 has C's leading dimension).
int launch_sgemm(omx_ctx ctx, bool trA, bool trB, int npair, int m, int n, int k, double alpha, const float *A1,
                 const float *A2, int64_t lda, const float *B1, const float *B2, int64_t ldb, double beta0, const float *C0,
                 double beta, float *C, int64_t ldc);
// C_q := A_q B^T (n x n, k columns; q = 2, 3 symmetric) in one launch, dt OMX_F64 or OMX_F32 for operands and
// products, where search_in_one finds that faster than single products.  K is not split then: the bits are
// those of single products with ctx->one_part.
bool search_in_one(omx_ctx ctx, int dt, int n, int k, int64_t lda, int64_t ldb);
int launch_search(omx_ctx ctx, int dt, int n, int k, const void *const A[4], int64_t lda, const void *B, int64_t ldb,
                  void *const C[4], int64_t ldc);
// Results of fewer than two 128 tiles per CU carry their sums over K (carry_sums), FP64 products on FP64 storage
// (carries64) and FP32 ones on FP32 storage: in 128 tiles K was split for these to fill the chip, and parts of a
// few hundred values are rounded less than one chain (FP64 Grams against 80 bits, such parts, one chain, now: 250 x 500
// 3.1e-16, 7.5e-16, 2.9e-16; 700 x 1400 3.5e-16, 1.2e-15, 3.1e-16; 2662 x 5324 1.7e-15, 1.2e-15, 5.5e-16).  Larger FP32 products are one FP32 chain over K,
// unsplit: with carried sums (1.6e-6 -> 2.5e-7 off FP64 at 8192 x 8192 x 16384) the mixed solve at n = 16384 took 670 to
// 950 low-precision steps and 22.8 to 29.9 s from six starts, against 555 to 665 steps and 18.4 to 22.3 s, and
// ended higher in energy: its stop and the FP32 recomputation of its state go by the rounding of these products.
inline bool carries(omx_ctx ctx, int m, int n) {
    return (int64_t)((m + 127) / 128) * ((n + 127) / 128) < 2 * ctx->num_cus;
}
// (a masked launch, of the grouped solver, never split K)
inline bool carries64(omx_ctx ctx, int m, int n) { return !ctx->launch_mask && (ctx->carry64 || carries(ctx, m, n)); }
// Slices of K (of nsl) between two carries, a power of two: 4 for the shortest parts that `parts` of K made, up to
// 16 for longer ones (carrying costs 1 to 3 % at 4).
inline int carry_period(int nsl, int64_t parts) {
    const int64_t len = nsl / std::max<int64_t>(1, parts);
    return len >= 32 ? 16 : len >= 16 ? 8 : 4;
}
// Parts K is split into for such a product of nsl slices of 128 bytes (es: element size); a function of the
// shape alone, so that every tile configuration and the symmetric form add in the same order.
int dgemm_k_splits(omx_ctx ctx, int m, int n, int nsl, int es);
// C := alpha*A*B^T known to be symmetric (n x n, 'n','t' operands of k columns): the lower-triangle
// tiles where the kernels allow it, then a mirror of the lower triangle onto the upper (both honour
// ctx->launch_mask).
int launch_gemm_sym(omx_ctx ctx, int prec, int dt, int n, int k, double alpha, const void *A, int64_t lda,
                    const void *B, int64_t ldb, void *C, int64_t ldc);
int launch_gemm_pair(omx_ctx ctx, int prec, int dt, int m, int n, int k, double alpha, const void *A1,
                     const void *A2, int64_t lda, const void *B1, const void *B2, int64_t ldb, double beta0,
                     const void *C0, double beta, void *C, int64_t ldc);
// Complex products (OMX_C128 on FP64 MFMA, OMX_C64 on FP32 MFMA); op 'n', 't' or 'c' (conjugate
// transpose); real alpha, beta.
int launch_zgemm(omx_ctx ctx, int dt, char opA, char opB, int m, int n, int k, double alpha, const void *A,
                 int64_t lda, const void *B, int64_t ldb, double beta, void *C, int64_t ldc);
int launch_zgemm_pair(omx_ctx ctx, int dt, int m, int n, int k, double alpha, const void *A1, const void *A2,
                      int64_t lda, const void *B1, const void *B2, int64_t ldb, double beta0, const void *C0,
                      double beta, void *C, int64_t ldc);
// Batched complex128 products (blockIdx.y = system; strides in complex elements; systems with
// active[s] == 0 skipped; no split-K).  Ops: ('n','c') and ('n','n').
int launch_zgemm_batched(omx_ctx ctx, int dt, char opA, char opB, int m, int n, int k, double alpha, const void *A,
                         int64_t lda, int64_t sA, const void *B, int64_t ldb, int64_t sB, double beta, void *C,
                         int64_t ldc, int64_t sC, int nbatch, const int *active);
// C := alpha * A * B^H for products known to be Hermitian (n x n): lower-triangle tiles, then the
// conjugated mirror.  The batched form takes the strides and mask of launch_zgemm_batched.
int launch_zgemm_herm(omx_ctx ctx, int dt, int n, int k, double alpha, const void *A, int64_t lda, const void *B,
                      int64_t ldb, void *C, int64_t ldc);
int launch_zgemm_herm_batched(omx_ctx ctx, int dt, int n, int k, double alpha, const void *A, int64_t lda,
                              int64_t sA, const void *B, int64_t ldb, int64_t sB, void *C, int64_t ldc, int64_t sC,
                              int nbatch, const int *active);
// The four line-search products of nbatch systems, X_q D^H with X_q at X + q*nbatch*sX (q = 0..3, system s at
// + s*sX) and the results likewise at C, sC apart; products 2 and 3 are Hermitian.  One launch where the
// kernel allows it.
int launch_zgemm_search_batched(omx_ctx ctx, int dt, int n, int k, const void *X, int64_t ldx, int64_t sX,
                                const void *D, int64_t ldd, int64_t sD, void *C, int64_t ldc, int64_t sC, int nbatch,
                                const int *active);
int launch_zgemm_pair_batched(omx_ctx ctx, int dt, int m, int n, int k, double alpha, const void *A1, const void *A2,
                              int64_t lda, int64_t sA, const void *B1, const void *B2, int64_t ldb, int64_t sB,
                              double beta0, const void *C0, double beta, void *C, int64_t ldc, int64_t sC, int nbatch,
                              const int *active);

// Batched pieces of the k-point solver (complex128 or complex64, systems sharing one block pattern).
int launch_spmm_z_batched(omx_ctx ctx, int dt, int no, int nb, int nbc, const int *colptr, const int *rowidx,
                          const double *val, const double *val2, int64_t sV, const void *X, int64_t ldx, int64_t sX,
                          void *Y, void *Y2, int64_t ldy, int64_t sY, int nbatch, const int *active);
// Partial sums of the line-search coefficients (13 values per workgroup, coeff_blocks(n) workgroups per
// system) and of the Polak-Ribiere dots (2 values, pr_blocks(n, m)) of nbatch systems of element type dt; a
// system s with mask && !mask[s] is skipped.  The solver's own kernels add them (omx_reduce.h).
int coeff_blocks(int n);
int pr_blocks(int n, int m);
int launch_coeff_batched(omx_ctx ctx, int dt, int n, int64_t ldm, int64_t sW, const void *HW, const void *SW,
                         const void *HWd, const void *SWd, const void *HWdd, const void *SWdd, int nbatch,
                         double *partial, const int *mask);
int launch_pr_batched(omx_ctx ctx, int dt, int n, int m, int64_t ld, int64_t sG, const void *G, const void *Gp,
                      int nbatch, double *partial, const int *mask);
// Re tr(W_s) and <W_s, W_s> to out2[2*s ...] (W_s n x n, ld = n, sW elements apart); partial holds
// 2*maxblocks values per system.
int launch_trqs_batched(omx_ctx ctx, int dt, int n, int64_t sW, const void *W, int nbatch, int maxblocks,
                        double *partial, double *out2);

}  // namespace omx

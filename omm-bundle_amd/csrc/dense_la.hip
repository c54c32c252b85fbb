// Dense factorisations for libOMM's Cholesky and preconditioned flavours (FP64, column-major):
//   omx_potrf      S = U^T U, upper (dpotrf 'u', libOMM/src/omm_ops.F90:301)
//   omx_trsm       B := alpha * op(U)^-1 * B  or  alpha * B * op(U)^-1, U upper (dtrsm)
//   omx_trmm       B := alpha * op(U) * B     or  alpha * B * op(U),     U upper (dtrmm)
//   omx_sygst      H := U^-T H U^-1, both triangles (dsygst itype 1 'u' + the mirror copy,
//                  omm_ops.F90:481-487)
//   omx_inverse_spd A := A^-1 for symmetric positive definite A (m_inverse, omm_ops.F90:1065-1075
//                  uses dsytrf/dsytri; on an SPD matrix the Cholesky route gives the same inverse)
//
// Diagonal blocks of LB = 128 are factorised and inverted by one workgroup entirely in LDS (132 KB), in
// 16x16 steps on the matrix cores; everything else is an MFMA GEMM of dgemm.hip:
//   * potrf runs the lower Cholesky of S^T (S's upper triangle, transposed into a workspace padded with
//     the identity to a multiple of 128) in panels of LB_OUT columns.  Per block of a panel: one GEMM brings
//     the block's columns up to date with the panel so far, the diagonal kernel gives L_kk and L_kk^-1,
//     and one GEMM the rest of the block column, L21 = A21 L_kk^-T.  L goes to a buffer of the panel's
//     width, from which the trailing matrix takes one lower-triangle update and the upper triangle of the
//     result is written (transposed); the strict lower triangle of the input is never read nor written (as
//     dpotrf 'u').
//   * the triangular solves work on blocks of OB = 256: one GEMM subtracts what the solved blocks
//     contribute, T = alpha B_o - op(U) X, and one applies the inverse of U's diagonal block, X_o =
//     op(U_oo)^-1 T.  The inverses come from 128x128 ones (one launch, one workgroup each) joined in
//     pairs by two batched GEMMs.  Solves whose right-hand side or result is known to be triangular
//     restrict the GEMMs to the nonzero part.
//   * sygst = a full left solve, then a right solve that forms only the block-lower part of the
//     (symmetric) result, mirrored onto the upper triangle: 5/3 n^3 flops.
//   * the SPD inverse = potrf, X = U^-1 (upper-triangular right-hand side, n^3/3 flops), then
//     A^-1 = X X^T by row chunks that skip X's zero lower part (n^3/3 flops) and a mirror.
// Multiplying by the inverse of a diagonal block instead of substituting changes rounding at the
// level of cond(block) * eps; the diagonal blocks of an SPD factor are well conditioned when S is.
#include <algorithm>

#include "omx_internal.h"
#include "omx_mfma.h"

namespace omx {

constexpr int LB = 128;       // diagonal block of one workgroup
constexpr int OB = 2 * LB;    // block of the triangular solves
constexpr int LB_OUT = 512;   // potrf's panel
constexpr int LB_S = LB + 1;  // LDS column stride
constexpr int LB_NT = 512;    // threads of the diagonal-block kernels: 8 waves
constexpr int SB = 16;        // step inside a diagonal block: the FP64 MFMA's tile
constexpr int LA_NT = 256;    // threads of the element-wise kernels
constexpr int TT = 64;        // transpose tile

// The kernels below keep an LB x LB matrix in LDS, element (i, j) at a[j * LB_S + i].  Each runs once per
// launch in one workgroup, so its time is latency, and that of fetching instructions nobody has in a cache
// counts: what runs once stays rolled (unrolled, with less waiting on LDS, the block inverse took 33 us
// instead of 28).

// v of lane `lane` (uniform), through two scalar reads; v of lane `src` (per lane), through LDS.
__device__ inline double read_lane(double v, int lane) {
    const long long b = __double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(b & 0xffffffffLL), lane);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ inline double from_lane(double v, int src) {
    const long long b = __double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_ds_bpermute(4 * src, (int)(b & 0xffffffffLL));
    const unsigned hi = (unsigned)__builtin_amdgcn_ds_bpermute(4 * src, (int)(b >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ inline double pick(const double (&x)[4], int v) { return v == 0 ? x[0] : v == 1 ? x[1] : v == 2 ? x[2] : x[3]; }

// acc += sum over k = 0 .. 15 of P(r0 + i, kp + k) Q(kq + k, c0 + j), with P(i, k) = a(i, k) and Q(k, j) = a(k, j)
// (or a(j, k) with QT), by one wave; D(i, j) in lane (i mod 4) * 16 + j, register i / 4.
template <bool QT>
__device__ inline void lds_mma(const double *a, int r0, int kp, int c0, int kq, d4v &acc) {
    const int li = threadIdx.x & 15, lk = (threadIdx.x & 63) >> 4;
#pragma unroll
    for (int k = 0; k < SB; k += 4) {
        const double x = a[(kp + k + lk) * LB_S + r0 + li];
        const double y = QT ? a[(kq + k + lk) * LB_S + c0 + li] : a[(c0 + li) * LB_S + kq + k + lk];
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(x, y, acc, 0, 0, 0);
    }
}

// s = sqrt(d) and y = 1 / s, d > 0: from the hardware's reciprocal square root (relative error e of about
// 2^-24) the series y (1 + e/2 + 3/8 e^2) of (1 - e)^-1/2 in one step, a third of the latency of the square
// root and the division one after the other.
__device__ inline void root(double d, double &s, double &y) {
    y = __builtin_amdgcn_rsq(d);
    const double e = fma(-d * y, y, 1.0);
    y = fma(y * e, fma(0.375, e, 0.5), y);
    s = d * y;
    s = fma(0.5 * y, fma(-s, s, d), s);
    const bool inf = d > 1.7976931348623157e308;
    s = inf ? d : s;
    y = inf ? 0.0 : y;
}

// Lower Cholesky of the SB x SB block at (o, o) and the inverse of its factor, by one wave: lane i < 16 holds
// row i of the block, lane 16 + c column c of the identity.  Both take the same step: with m = r[k] /
// L(k, k), element L(i, k) or X(k, c), r[j] -= m L(j, k) for j > k, L(j, k) broadcast through scalar reads.  L
// goes to Lout (ld ldl), X = L^-1 (zeros above the diagonal) in its place in a.  A non-positive pivot is
// replaced by 1, the first one (gk + k < n) noted in *bad.  Unrolled all the same: the code is reused for
// the 8 steps of a block, and rolled, with rows and columns through LDS shuffles, a pivot took 367 ns.
__device__ inline void chol_step(double *a, int o, int gk, int n, double *__restrict__ Lout, int64_t ldl, int *bad) {
    const int lane = threadIdx.x & 63, i = lane & 15;
    const bool rows = lane < SB;
    double r[SB];
#pragma unroll
    for (int j = 0; j < SB; ++j) {
        const double v = a[(o + min(i, j)) * LB_S + o + max(i, j)];
        r[j] = rows ? v : (i == j ? 1.0 : 0.0);
    }
    int first = SB;
#pragma unroll
    for (int k = 0; k < SB; ++k) {
        double d = read_lane(r[k], k), dk, rdk;
        first = !(d > 0.0) && first == SB ? k : first;
        d = d > 0.0 ? d : 1.0;
        root(d, dk, rdk);
        const double m = r[k] * rdk;
        r[k] = rows && i == k ? dk : m;
#pragma unroll
        for (int j = k + 1; j < SB; ++j) r[j] = fma(-m, read_lane(m, j), r[j]);
    }
    if (lane == 0 && first < SB && gk + first < n && *bad == 0) *bad = gk + first + 1;
    if (rows) {
#pragma unroll
        for (int j = 0; j < SB; ++j)
            if (i >= j) Lout[i + (int64_t)j * ldl] = r[j];
    } else if (lane < 2 * SB) {
#pragma unroll
        for (int j = 0; j < SB; ++j) a[(o + i) * LB_S + o + j] = j >= i ? r[j] : 0.0;  // X(j, i)
    }
}

// Joins the inverses of the SB x SB diagonal blocks of a lower-triangular matrix in a (diagonal blocks already
// inverted, zeros above their diagonals; the blocks above are scratch) to the whole inverse, 8 waves: for
// pairs of inverted blocks of 16, 32 and 64, X21 = -X22 (L21 X11), the inner product parked in the block's
// mirror image above the diagonal.
__device__ inline void join_inverses(double *a) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, lq = lane >> 4;
#pragma unroll 1
    for (int lg = 0; lg < 3; ++lg) {
        const int b = SB << lg, work = 4 << lg;  // 16x16 tiles of all pairs' blocks
#pragma unroll 1
        for (int phase = 0; phase < 2; ++phase) {
            d4v acc[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                acc[h] = d4v{0, 0, 0, 0};
                const int w = wave + 8 * h, q = w & ((1 << 2 * lg) - 1);
                if (w >= work) continue;
                const int o1 = (w >> 2 * lg) * 2 * b, o2 = o1 + b, ti = (q & ((1 << lg) - 1)) * SB, tj = (q >> lg) * SB;
                // T = L21 X11 (X11 lower: from tj), then X21 = -X22 T (X22 lower: up to ti; T(k, j) at (o1 + k, o2 + j))
                const int kb = phase ? 0 : tj, ke = phase ? ti + SB : b, kp = phase ? o2 : o1, c0 = phase ? o2 : o1;
#pragma unroll 1
                for (int k = kb; k < ke; k += SB) lds_mma<false>(a, o2 + ti, kp + k, c0 + tj, o1 + k, acc[h]);
            }
            __syncthreads();
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int w = wave + 8 * h, q = w & ((1 << 2 * lg) - 1);
                if (w >= work) continue;
                const int o1 = (w >> 2 * lg) * 2 * b, o2 = o1 + b, ti = (q & ((1 << lg) - 1)) * SB, tj = (q >> lg) * SB;
                double *to = a + ((phase ? o1 : o2) + tj + li) * LB_S + (phase ? o2 : o1) + ti + lq;
#pragma unroll
                for (int v = 0; v < 4; ++v) to[4 * v] = phase ? -acc[h][v] : acc[h][v];
            }
            __syncthreads();
        }
    }
}

// The LB x LB diagonal block of W at (k0, k0) by one workgroup: L into Lout (ld ldl), L^-1 (zeros above the
// diagonal) into LI (LB x LB); *info := global index + 1 of the first non-positive pivot below n (replaced
// by 1, so the remaining blocks stay finite).  W is padded with the identity beyond n, so the block is
// always whole.  Right-looking in steps of SB: wave 0 factorises and inverts the diagonal block of the step
// while the other waves finish the previous step's update; the blocks below become A L_ss^-T, one wave
// each; the next diagonal block is updated first, by wave 0.
// What bounds it: the chain of 128 pivots.  The one-wave 64x64 form before it, unrolled, took 59 us per 64
// columns (64 launches, 3.7 ms of an order-4000 factorisation).
__global__ __launch_bounds__(LB_NT) void k_chol_block(const double *__restrict__ W, int64_t ldw, int k0, int n,
                                                      double *__restrict__ Lout, int64_t ldl, double *__restrict__ LI,
                                                      int *__restrict__ info) {
    __shared__ double a[LB * LB_S];
    __shared__ int bad;
    constexpr int NB = LB / SB;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, li = lane & 15, lq = lane >> 4;
    const double *Wkk = W + k0 + (int64_t)k0 * ldw;
    const int r = t % LB, c0 = t / LB;  // four columns at a time
#pragma unroll 1
    for (int c = c0; c < LB; c += 32) {  // whole columns (the part above the diagonal is scratch), 8 in flight
        double v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = Wkk[r + (int64_t)(c + 4 * q) * ldw];
#pragma unroll
        for (int q = 0; q < 8; ++q) a[(c + 4 * q) * LB_S + r] = v[q];
    }
    if (t == 0) bad = 0;
    __syncthreads();
    auto update = [&](int o, int I, int J) {  // a(I, J) -= L(I, o) L(J, o)^T, SB x SB blocks
        d4v acc{0, 0, 0, 0};
        lds_mma<true>(a, I * SB, o, J * SB, o, acc);
#pragma unroll
        for (int v = 0; v < 4; ++v) a[(J * SB + li) * LB_S + I * SB + lq + 4 * v] -= acc[v];
    };
#pragma unroll 1
    for (int s = 0; s < NB; ++s) {
        const int o = s * SB, po = o - SB;
        if (wave == 0) {
            if (s) update(po, s, s);
            chol_step(a, o, k0 + o, n, Lout + o + (int64_t)o * ldl, ldl, &bad);
        } else if (s) {  // the rest of the previous step's update: block columns s.., tiles after the first
            for (int J = s, w = wave; J < NB; ++J) {
                for (; w < NB - J; w += LB_NT / 64 - 1) update(po, J + w, J);
                w -= NB - J;
            }
        }
        __syncthreads();
        if (s + 1 + wave < NB) {  // block row s + 1 + wave: A L_ss^-T
            const int I = s + 1 + wave;
            d4v acc{0, 0, 0, 0};
            lds_mma<true>(a, I * SB, o, o, o, acc);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int i = I * SB + lq + 4 * v, j = o + li;
                a[j * LB_S + i] = acc[v];
                Lout[i + (int64_t)j * ldl] = acc[v];
            }
        }
        __syncthreads();
    }
    join_inverses(a);
#pragma unroll 1
    for (int c = c0; c < LB; c += 32)
#pragma unroll
        for (int q = 0; q < 8; ++q) LI[r + (c + 4 * q) * LB] = (r >= c + 4 * q) ? a[(c + 4 * q) * LB_S + r] : 0.0;
    if (t == 0 && bad && *info == 0) *info = bad;
}

// Inverses of the LB diagonal blocks of the upper-triangular U (order nu), one workgroup per block:
// block b lands at rows and columns (b & 1) * LB of the OB x OB matrix UI + (b / 2) * OB^2 (upper, zeros
// below the diagonal, and in the whole block below it); a partial last block is padded with the identity.
// U_bb^T is inverted as a lower matrix in LDS.
__global__ __launch_bounds__(LB_NT) void k_trinv_upper_blocks(int nu, const double *__restrict__ U, int64_t ldu,
                                                              double *__restrict__ UI) {
    __shared__ double a[LB * LB_S];
    const int t = threadIdx.x, b = blockIdx.x, k0 = b * LB, nb = min(LB, nu - k0);
    const double *Ubb = U + k0 + (int64_t)k0 * ldu;
    const int r = t % LB, c0 = t / LB;  // a(c, r) = U(r, c) for r <= c; loads stay inside the block
#pragma unroll 1
    for (int c = c0; c < LB; c += 32) {
        double v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = Ubb[min(r, nb - 1) + (int64_t)min(c + 4 * q, nb - 1) * ldu];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int i = c + 4 * q;
            a[r * LB_S + i] = (i < r) ? 0.0 : (i < nb) ? v[q] : (i == r ? 1.0 : 0.0);
        }
    }
    __syncthreads();
    {  // the wave's diagonal block: row operations on the identity, 4 elements per lane
        const int o = (t >> 6) * SB, lane = t & 63, j = lane & 15, iq = lane >> 4;
        double y[4];
        const double rdiag = 1.0 / a[(o + j) * LB_S + o + j];
#pragma unroll
        for (int v = 0; v < 4; ++v) y[v] = iq + 4 * v == j ? 1.0 : 0.0;
#pragma unroll 1
        for (int k = 0; k < SB; ++k) {
            const double *L = a + (o + k) * LB_S + o;
            const double yk = from_lane(pick(y, k >> 2), (k & 3) * 16 + j) * read_lane(rdiag, k);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int i = iq + 4 * v;
                y[v] = i > k ? fma(-L[i], yk, y[v]) : (i == k ? yk : y[v]);
            }
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int v = 0; v < 4; ++v) a[(o + j) * LB_S + o + iq + 4 * v] = iq + 4 * v >= j ? y[v] : 0.0;
    }
    __syncthreads();
    join_inverses(a);
    double *out = UI + (int64_t)(b / 2) * OB * OB + (b & 1) * (LB + (int64_t)LB * OB);
#pragma unroll 1
    for (int c = c0; c < LB; c += 4) {  // U_bb^-1 (r, c) = X(c, r)
        out[r + (int64_t)c * OB] = (r <= c) ? a[r * LB_S + c] : 0.0;
        if (b & 1) out[r + (int64_t)(c - LB) * OB] = 0.0;
    }
}

// Transposed copies of triangles through 64 x 64 LDS tiles (coalesced on both sides).
//   UP_TO_LOWER: dst = W (N x N, N >= n, ld ldd) from the upper triangle of src (n x n):
//     W(i, j) = src(j, i) for j <= i < n; the identity where i or j >= n; 0 above the diagonal.
//   else: rows r0 .. r0 + N of the upper triangle of dst (n x n) from a panel of the lower triangle: dst(i, j)
//     = src(j, i - r0) for r0 <= i < r0 + N, i <= j < n; nothing else is written.
template <bool UP_TO_LOWER>
__global__ __launch_bounds__(LA_NT) void k_tri_transpose(int n, int N, const double *__restrict__ src, int64_t lds,
                                                         double *__restrict__ dst, int64_t ldd, int r0) {
    __shared__ double tile[TT][TT + 1];
    const int i0 = (UP_TO_LOWER ? 0 : r0) + blockIdx.x * TT, j0 = blockIdx.y * TT;  // dst tile rows i0.., columns j0..
    const int tx = threadIdx.x % TT, ty = threadIdx.x / TT;  // 64 x 4
    const bool need = UP_TO_LOWER ? (i0 + TT - 1 >= j0) : (i0 <= j0 + TT - 1);
    if (!need) {
        if (UP_TO_LOWER)
            for (int c = ty; c < TT; c += 4)
                if (i0 + tx < N && j0 + c < N) dst[(i0 + tx) + (int64_t)(j0 + c) * ldd] = 0.0;
        return;
    }
    // src(j, i) for j in the dst column range, i in the dst row range: coalesced over j
    for (int c = ty; c < TT; c += 4) {
        const int i = i0 + c, j = j0 + tx;
        double v = 0.0;
        if (UP_TO_LOWER ? (j <= i && i < n) : (i <= j && j < n && i < r0 + N))
            v = src[j + (int64_t)(UP_TO_LOWER ? i : i - r0) * lds];
        tile[c][tx] = v;  // tile[i - i0][j - j0]
    }
    __syncthreads();
    for (int c = ty; c < TT; c += 4) {
        const int i = i0 + tx, j = j0 + c;
        const double v = tile[tx][c];
        if (UP_TO_LOWER) {
            double w = 0.0;
            if (i >= j) w = (i < n && j < n) ? v : (i == j ? 1.0 : 0.0);
            if (i < N && j < N) dst[i + (int64_t)j * ldd] = w;
        } else if (i <= j && j < n && i < r0 + N) {
            dst[i + (int64_t)j * ldd] = v;
        }
    }
}

// Lower triangle -> upper triangle (symmetrise), 64 x 64 tiles through LDS.
__global__ __launch_bounds__(LA_NT) void k_mirror_lower(int n, double *__restrict__ A, int64_t lda) {
    __shared__ double tile[TT][TT + 1];
    const int i0 = blockIdx.x * TT, j0 = blockIdx.y * TT;  // upper tile (i0 <= j0)
    if (i0 > j0) return;
    const int tx = threadIdx.x % TT, ty = threadIdx.x / TT;
    for (int c = ty; c < TT; c += 4) {  // read A(j, i) from the lower tile: rows j0.., columns i0..
        const int j = j0 + tx, i = i0 + c;
        tile[c][tx] = (j < n && i < n) ? A[j + (int64_t)i * lda] : 0.0;
    }
    __syncthreads();
    for (int c = ty; c < TT; c += 4) {
        const int i = i0 + tx, j = j0 + c;
        if (i < j && j < n) A[i + (int64_t)j * lda] = tile[tx][c];
    }
}

// W := upper triangle of U (zeros below), n x n, ld n.
__global__ __launch_bounds__(LA_NT) void k_triu_copy(int n, const double *__restrict__ U, int64_t ldu,
                                                     double *__restrict__ W) {
    const int64_t total = (int64_t)n * n;
    for (int64_t q = (int64_t)blockIdx.x * LA_NT + threadIdx.x; q < total; q += (int64_t)gridDim.x * LA_NT) {
        const int64_t i = q % n, j = q / n;
        W[q] = (i <= j) ? U[i + j * ldu] : 0.0;
    }
}

__global__ void k_set_identity(int n, double *__restrict__ A, int64_t lda) {
    const int64_t total = (int64_t)n * n;
    for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < total; q += (int64_t)gridDim.x * blockDim.x) {
        const int64_t i = q % n, j = q / n;
        A[i + j * lda] = (i == j) ? 1.0 : 0.0;
    }
}

static inline int la_grid(int64_t total) {
    return (int)std::max<int64_t>(1, std::min<int64_t>((total + LA_NT - 1) / LA_NT, 65536));
}

static int gemm64(omx_ctx ctx, bool trA, bool trB, int m, int n, int k, double alpha, const double *A, int64_t lda,
                  const double *B, int64_t ldb, double beta, double *C, int64_t ldc) {
    if (m <= 0 || n <= 0 || k <= 0) return OMX_OK;
    return launch_gemm(ctx, OMX_PREC_F64, OMX_F64, trA, trB, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
}

// C := alpha op(A) op(B) + beta0 C0 (none: C0 null), with a leading dimension of its own for C0.  The products of
// the solves carry their sums, every 64 values of K: a solve subtracts the solved blocks from the right-hand side in
// one product, and in one chain over its whole K every step is rounded at the size of the full sum.  Against 64 bits,
// order 600, with and without: solves with a factor of condition number 3 3.3e-16 and 5.7e-16 (updates of 128 columns
// at a time, as before, 3.4e-16), potrf at condition number 1e4 4.8e-15 and 8.2e-15 (64 columns: 3.9e-15); the
// reduction at order 4000 takes 5.39 ms with and 5.31 without.
static int gemm64_from(omx_ctx ctx, bool trA, bool trB, int m, int n, int k, double alpha, const double *A, int64_t lda,
                       const double *B, int64_t ldb, double beta0, const double *C0, int64_t ldc0, double *C,
                       int64_t ldc) {
    if (m <= 0 || n <= 0) return OMX_OK;
    if (k > 0) {
        ctx->carry64 = true;
        const int rc = launch_dgemm(ctx, trA, trB, 1, m, n, k, alpha, A, A, lda, B, B, ldb, beta0, C0, ldc0, 0.0, C, ldc);
        ctx->carry64 = false;
        if (rc != OMX_ERR_UNSUPPORTED) return rc;
    }
    const int rc = C0 ? omx_add(ctx, OMX_F64, 'n', m, n, beta0, C0, ldc0, 0.0, C, ldc) : OMX_OK;
    return rc ? rc : gemm64(ctx, trA, trB, m, n, k, alpha, A, lda, B, ldb, C0 ? 1.0 : 0.0, C, ldc);
}

// C (n x n) := alpha A B^T + beta C on the lower-triangle tiles where the kernel can restrict itself
// to them (the caller reads only the lower triangle), A, B n x k.
static int gemm64_lower(omx_ctx ctx, int n, int k, double alpha, const double *A, int64_t lda, const double *B,
                        int64_t ldb, double beta, double *C, int64_t ldc) {
    if (n <= 0 || k <= 0) return OMX_OK;
    ctx->gemm_sym = 1;
    const int rc = launch_gemm(ctx, OMX_PREC_F64, OMX_F64, false, true, n, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
    ctx->gemm_sym = 0;
    return rc;
}

// Stream-ordered device buffers released when the scope ends.
struct DevBuf {
    omx_ctx ctx;
    double *p = nullptr;
    DevBuf(omx_ctx c) : ctx(c) {}
    int alloc(size_t count) {
        const size_t bytes = sizeof(double) * std::max<size_t>(count, 1);
        hipError_t e = hipMallocAsync((void **)&p, bytes, ctx->stream);
        if (e != hipSuccess && dev_release()) e = hipMallocAsync((void **)&p, bytes, ctx->stream);
        if (e != hipSuccess) {
            p = nullptr;
            set_error("dense factorisation: device allocation of %zu doubles failed", count);
            return OMX_ERR_NOMEM;
        }
        return OMX_OK;
    }
    ~DevBuf() {
        if (p) (void)hipFreeAsync(p, ctx->stream);
    }
};

// Shape of the solution known in advance, so the GEMMs can skip what stays zero or is not needed:
//   TRI_NONE:   full solve;
//   TRI_COLS_GE (left 'n'):  B is upper triangular with the block structure of U (B = I at the
//               start): block row b of X lives in columns >= b*LB;
//   TRI_ROWS_GE (right 'n'): only the block-lower part of X is wanted: block column b for rows >= b*LB.
enum TriShape { TRI_NONE = 0, TRI_COLS_GE = 1, TRI_ROWS_GE = 2 };

// UI := the inverses of U's OB diagonal blocks (order nu), OB x OB each, padded with the identity.
static int block_inverses(omx_ctx ctx, int nu, const double *U, int64_t ldu, double *UI, double *T) {
    const int nblk = (nu + LB - 1) / LB, whole = nu / OB, rest = nu - whole * OB;
    hipLaunchKernelGGL(k_trinv_upper_blocks, dim3(nblk), dim3(LB_NT), 0, ctx->stream, nu, U, ldu, UI);
    // X12 = -X11 (U12 X22) of every pair; the last one's second block may be partial
    const int64_t o12 = (int64_t)LB * OB, o22 = LB + o12, so = (int64_t)OB * OB, su = OB * (ldu + 1);
    int rc = OMX_OK;
    auto join = [&](int b, int n2) {  // one pair, second block of order n2
        double *X = UI + b * so;
        rc = gemm64(ctx, false, false, LB, n2, n2, 1.0, U + b * su + LB * ldu, ldu, X + o22, OB, 0.0, T, LB);
        if (!rc) rc = gemm64(ctx, false, false, LB, n2, LB, -1.0, X, OB, T, LB, 0.0, X + o12, OB);
        return rc;
    };
    if (whole) {
        rc = launch_dgemm_batched(ctx, LB, LB, LB, 1.0, U + LB * ldu, ldu, su, UI + o22, OB, so, T, LB, (int64_t)LB * LB,
                                  whole);
        if (!rc)
            rc = launch_dgemm_batched(ctx, LB, LB, LB, -1.0, UI, OB, so, T, LB, (int64_t)LB * LB, UI + o12, OB, so, whole);
        if (rc == OMX_ERR_UNSUPPORTED) {
            rc = OMX_OK;
            for (int b = 0; b < whole && !rc; ++b) join(b, LB);
        }
        if (rc) return rc;
    }
    if (rest > LB) join(whole, rest - LB);
    return rc;
}

static int trsm_impl(omx_ctx ctx, char side, char trans, int m, int n, double alpha, const double *U, int64_t ldu,
                     double *B, int64_t ldb, TriShape shape = TRI_NONE) {
    const bool left = (side == 'l' || side == 'L');
    const bool tr = is_trans(trans);
    const int nu = left ? m : n;  // order of U
    const int nout = (nu + OB - 1) / OB;
    DevBuf UI(ctx), T(ctx);
    int rc = UI.alloc((size_t)nout * OB * OB);
    if (!rc) rc = T.alloc(std::max((size_t)OB * (left ? n : m), (size_t)nout * LB * LB));
    if (!rc) rc = block_inverses(ctx, nu, U, ldu, UI.p, T.p);
    if (rc) return rc;
    const bool fwd = left ? tr : !tr;  // forward solves take the blocks in order, backward in reverse
    for (int so = 0; so < nout; ++so) {
        const int o = fwd ? so : nout - 1 - so;
        const int o0 = o * OB, ob = std::min(OB, nu - o0), end = o0 + ob;
        const double *Ui = UI.p + (int64_t)o * OB * OB;
        const int d0 = fwd ? 0 : end, nd = fwd ? o0 : nu - end;  // the blocks solved before this one
        if (left) {
            // T = alpha B_o - op(U)(o, solved) X(solved), X_o = op(U_oo)^-1 T
            const int c0 = shape == TRI_COLS_GE ? o0 : 0, nc = n - c0;
            double *Bo = B + o0 + (int64_t)c0 * ldb;
            const double *Uo = tr ? U + d0 + (int64_t)o0 * ldu : U + o0 + (int64_t)d0 * ldu;
            rc = gemm64_from(ctx, tr, false, ob, nc, nd, -1.0, Uo, ldu, B + d0 + (int64_t)c0 * ldb, ldb, alpha, Bo, ldb, T.p,
                             ob);
            if (!rc) rc = gemm64_from(ctx, tr, false, ob, nc, ob, 1.0, Ui, OB, T.p, ob, 0.0, nullptr, 0, Bo, ldb);
        } else {
            // T = alpha B_o - X(solved) op(U)(solved, o), X_o = T op(U_oo)^-1
            const int r0 = shape == TRI_ROWS_GE ? o0 : 0, nr = m - r0;
            double *Bo = B + r0 + (int64_t)o0 * ldb;
            const double *Uo = tr ? U + o0 + (int64_t)d0 * ldu : U + d0 + (int64_t)o0 * ldu;
            rc = gemm64_from(ctx, false, tr, nr, ob, nd, -1.0, B + r0 + (int64_t)d0 * ldb, ldb, Uo, ldu, alpha, Bo, ldb, T.p,
                             nr);
            if (!rc) rc = gemm64_from(ctx, false, tr, nr, ob, ob, 1.0, T.p, nr, Ui, OB, 0.0, nullptr, 0, Bo, ldb);
        }
        if (rc) return rc;
    }
    OMX_CHECK_HIP(hipGetLastError());
    return OMX_OK;
}

// Upper Cholesky of A (order n) through the lower Cholesky of its transposed upper triangle, in panels of
// LB_OUT columns (see the head of this file).
static int potrf_impl(omx_ctx ctx, int n, double *A, int64_t lda, int *info) {
    const int N = (n + LB - 1) / LB * LB;
    int *d_info = (int *)(ctx->d_scalars + (kScalarSlots - 1));  // the GEMMs use the workspace
    OMX_CHECK_HIP(hipMemsetAsync(d_info, 0, sizeof(int), ctx->stream));
    DevBuf W(ctx), V(ctx), LI(ctx);
    int rc = W.alloc((size_t)N * N);
    if (!rc) rc = V.alloc((size_t)N * std::min(N, LB_OUT));
    if (!rc) rc = LI.alloc((size_t)LB * LB);
    if (rc) return rc;
    hipLaunchKernelGGL(k_tri_transpose<true>, dim3(N / TT, N / TT), dim3(LA_NT), 0, ctx->stream, n, N,
                       (const double *)A, lda, W.p, (int64_t)N, 0);
    for (int o0 = 0; o0 < N; o0 += LB_OUT) {
        const int end = std::min(N, o0 + LB_OUT);
        // V(:, k - o0) holds column k of L for the panel's columns k (rows counted from 0)
        for (int k0 = o0; k0 < end; k0 += LB) {
            double *Wk = W.p + k0 + (int64_t)k0 * N, *Vk = V.p + (int64_t)(k0 - o0) * N;
            if (k0 > o0 && (rc = gemm64_from(ctx, false, true, N - k0, LB, k0 - o0, -1.0, V.p + k0, N, V.p + k0, N, 1.0, Wk, N,
                                             Wk, N)))
                return rc;
            hipLaunchKernelGGL(k_chol_block, dim3(1), dim3(LB_NT), 0, ctx->stream, (const double *)W.p, (int64_t)N, k0, n,
                               Vk + k0, (int64_t)N, LI.p, d_info);
            const int rest = N - k0 - LB;
            if (rest > 0 &&
                (rc = gemm64_from(ctx, false, true, rest, LB, LB, 1.0, Wk + LB, N, LI.p, LB, 0.0, nullptr, 0, Vk + k0 + LB, N)))
                return rc;
        }
        const int rest = N - end;
        if (rest > 0 && (rc = gemm64_lower(ctx, rest, end - o0, -1.0, V.p + end, N, V.p + end, N, 1.0,
                                           W.p + end + (int64_t)end * N, N)))
            return rc;
        const int rows = std::min(end, n) - o0;  // this panel's rows of the result
        if (rows > 0)
            hipLaunchKernelGGL(k_tri_transpose<false>, dim3((rows + TT - 1) / TT, (n + TT - 1) / TT), dim3(LA_NT), 0,
                               ctx->stream, n, rows, (const double *)V.p, (int64_t)N, A, lda, o0);
    }
    OMX_CHECK_HIP(hipGetLastError());
    int h_info = 0;
    OMX_CHECK_HIP(hipMemcpyAsync(&h_info, d_info, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
    OMX_CHECK_HIP(hipStreamSynchronize(ctx->stream));
    *info = h_info;
    return OMX_OK;
}

}  // namespace omx

using namespace omx;

extern "C" {

int omx_potrf(omx_ctx ctx, int dt, int n, void *A, int64_t lda, int *info) {
    OMX_REQUIRE(ctx && info && n >= 0 && lda >= std::max(1, n), "omx_potrf: bad arguments");
    OMX_REQUIRE(dt == OMX_F64, "omx_potrf: FP64 only");
    *info = 0;
    if (n == 0) return OMX_OK;
    OMX_REQUIRE(A, "omx_potrf: null operand");
    return potrf_impl(ctx, n, (double *)A, lda, info);
}

int omx_trsm(omx_ctx ctx, int dt, char side, char trans, int m, int n, double alpha, const void *U, int64_t ldu,
             void *B, int64_t ldb) {
    OMX_REQUIRE(ctx && m >= 0 && n >= 0 && valid_op(trans), "omx_trsm: bad arguments");
    OMX_REQUIRE(side == 'l' || side == 'L' || side == 'r' || side == 'R', "omx_trsm: side must be l or r");
    OMX_REQUIRE(dt == OMX_F64, "omx_trsm: FP64 only");
    const bool left = (side == 'l' || side == 'L');
    OMX_REQUIRE(ldu >= std::max(1, left ? m : n) && ldb >= std::max(1, m), "omx_trsm: bad leading dimension");
    if (!m || !n) return OMX_OK;
    OMX_REQUIRE(U && B, "omx_trsm: null operand");
    return trsm_impl(ctx, side, trans, m, n, alpha, (const double *)U, ldu, (double *)B, ldb);
}

int omx_trmm(omx_ctx ctx, int dt, char side, char trans, int m, int n, double alpha, const void *U, int64_t ldu,
             void *B, int64_t ldb) {
    OMX_REQUIRE(ctx && m >= 0 && n >= 0 && valid_op(trans), "omx_trmm: bad arguments");
    OMX_REQUIRE(side == 'l' || side == 'L' || side == 'r' || side == 'R', "omx_trmm: side must be l or r");
    OMX_REQUIRE(dt == OMX_F64, "omx_trmm: FP64 only");
    const bool left = (side == 'l' || side == 'L');
    const int nu = left ? m : n;
    OMX_REQUIRE(ldu >= std::max(1, nu) && ldb >= std::max(1, m), "omx_trmm: bad leading dimension");
    if (!m || !n) return OMX_OK;
    OMX_REQUIRE(U && B, "omx_trmm: null operand");
    // W = triu(U) (n_u^2) and T = copy of B (m*n) in stream-ordered buffers of their own (the GEMM
    // uses the context workspace), then B = alpha * op(W) * T or T * op(W)
    DevBuf W(ctx), T(ctx);
    int rc = W.alloc((size_t)nu * nu);
    if (!rc) rc = T.alloc((size_t)m * n);
    if (rc) return rc;
    hipLaunchKernelGGL(k_triu_copy, dim3(la_grid((int64_t)nu * nu)), dim3(LA_NT), 0, ctx->stream, nu,
                       (const double *)U, ldu, W.p);
    OMX_CHECK_HIP(hipMemcpy2DAsync(T.p, sizeof(double) * m, B, sizeof(double) * ldb, sizeof(double) * m, n,
                                   hipMemcpyDeviceToDevice, ctx->stream));
    const bool tr = is_trans(trans);
    if (left)
        rc = gemm64(ctx, tr, false, m, n, m, alpha, W.p, nu, T.p, m, 0.0, (double *)B, ldb);
    else
        rc = gemm64(ctx, false, tr, m, n, n, alpha, T.p, m, W.p, nu, 0.0, (double *)B, ldb);
    if (rc) return rc;
    OMX_CHECK_HIP(hipGetLastError());
    return OMX_OK;
}

int omx_sygst(omx_ctx ctx, int dt, int n, void *H, int64_t ldh, const void *U, int64_t ldu) {
    OMX_REQUIRE(ctx && n >= 0 && ldh >= std::max(1, n) && ldu >= std::max(1, n), "omx_sygst: bad arguments");
    OMX_REQUIRE(dt == OMX_F64, "omx_sygst: FP64 only");
    if (!n) return OMX_OK;
    OMX_REQUIRE(H && U, "omx_sygst: null operand");
    // Y := U^-T H (full), then the block-lower part of Y U^-1, mirrored: the result is symmetric, as
    // the reference's after dsygst and its mirror copy.
    int rc = trsm_impl(ctx, 'l', 't', n, n, 1.0, (const double *)U, ldu, (double *)H, ldh);
    if (rc) return rc;
    rc = trsm_impl(ctx, 'r', 'n', n, n, 1.0, (const double *)U, ldu, (double *)H, ldh, TRI_ROWS_GE);
    if (rc) return rc;
    const int nt = (n + TT - 1) / TT;
    hipLaunchKernelGGL(k_mirror_lower, dim3(nt, nt), dim3(LA_NT), 0, ctx->stream, n, (double *)H, ldh);
    OMX_CHECK_HIP(hipGetLastError());
    return OMX_OK;
}

int omx_inverse_spd(omx_ctx ctx, int dt, int n, void *A, int64_t lda, int *info) {
    OMX_REQUIRE(ctx && info && n >= 0 && lda >= std::max(1, n), "omx_inverse_spd: bad arguments");
    OMX_REQUIRE(dt == OMX_F64, "omx_inverse_spd: FP64 only");
    *info = 0;
    if (!n) return OMX_OK;
    OMX_REQUIRE(A, "omx_inverse_spd: null operand");
    // U = chol(A) in a workspace copy; X = U^-1 (upper triangular: the solve skips the zero block
    // columns); A^-1 = X X^T by row chunks of LB_OUT: rows [r0, r0 + w) against columns [0, r0 + w)
    // need only p >= r0 (X(i, p) = 0 for p < i), so each chunk is one product with K = n - r0
    // (n^3/3 flops in all), then the lower triangle is mirrored
    DevBuf U(ctx), X(ctx);
    int rc = U.alloc((size_t)n * n);
    if (!rc) rc = X.alloc((size_t)n * n);
    if (rc) return rc;
    OMX_CHECK_HIP(hipMemcpy2DAsync(U.p, sizeof(double) * n, A, sizeof(double) * lda, sizeof(double) * n, n,
                                   hipMemcpyDeviceToDevice, ctx->stream));
    rc = potrf_impl(ctx, n, U.p, n, info);
    if (rc || *info) return rc;
    hipLaunchKernelGGL(k_set_identity, dim3(la_grid((int64_t)n * n)), dim3(LA_NT), 0, ctx->stream, n, X.p,
                       (int64_t)n);
    if ((rc = trsm_impl(ctx, 'l', 'n', n, n, 1.0, U.p, n, X.p, n, TRI_COLS_GE))) return rc;
    double *Ad = (double *)A;
    for (int r0 = 0; r0 < n; r0 += LB_OUT) {
        const int w = std::min(LB_OUT, n - r0);
        if ((rc = gemm64(ctx, false, true, w, r0 + w, n - r0, 1.0, X.p + r0 + (int64_t)r0 * n, n, X.p + (int64_t)r0 * n,
                         n, 0.0, Ad + r0, lda)))
            return rc;
    }
    const int nt = (n + TT - 1) / TT;
    hipLaunchKernelGGL(k_mirror_lower, dim3(nt, nt), dim3(LA_NT), 0, ctx->stream, n, Ad, lda);
    OMX_CHECK_HIP(hipGetLastError());
    OMX_CHECK_HIP(hipStreamSynchronize(ctx->stream));
    return OMX_OK;
}

}  // extern "C"

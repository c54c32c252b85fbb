// Complex dense products on the CDNA4 matrix cores: C := alpha*op(A)*op(B) + beta*C for
// complex128 (FP64 MFMA) and complex64 (FP32 MFMA), op = 'n', 't' or 'c' (conjugate transpose),
// real alpha and beta (the only scalars the OMM loop uses).  These are MatrixSwitch's
// mm_zmultiply products (MatrixSwitch/src/MatrixSwitch.F90:1395-1726, 'ref' semantics of
// MatrixSwitch_mm_multiply.F90:85-185) for the k-point solves.
//
// Storage is the Fortran complex layout: (re, im) interleaved, column-major.  Each 16x16 output block
// keeps a real and an imaginary accumulator, four real MFMAs per block and k step:
//     acc_re += a_re*b_re - a_im*b_im,    acc_im += a_re*b_im + a_im*b_re.
// k_zgemm_dl (operands straight into LDS) takes every product with leading dimensions up to 2^20; past
// that k_zgemm stages
// through registers into real and imaginary k-major LDS planes (conjugation negates the imaginary plane).
// K slices are double-buffered in both; split-K with an in-order reduction covers shapes with too few
// tiles; the pair mode (two contractions back to back over one K range) gives calc_G in one launch.
#include <algorithm>

#include "omx_internal.h"
#include "omx_mfma.h"

namespace omx {

typedef double zd4v __attribute__((ext_vector_type(4)));
typedef float zf4v __attribute__((ext_vector_type(4)));

template <typename R>
struct ZPrec;
template <>
struct ZPrec<double> {
    typedef zd4v accv;
    typedef double2 cplx;
    __device__ static inline accv mfma(double a, double b, accv c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    // result lane l, register v -> row (l/16) + 4v
    __device__ static inline int out_row(int lq, int v) { return lq + 4 * v; }
};
template <>
struct ZPrec<float> {
    typedef zf4v accv;
    typedef float2 cplx;
    __device__ static inline accv mfma(float a, float b, accv c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    // result lane l, register v -> row 4(l/16) + v
    __device__ static inline int out_row(int lq, int v) { return 4 * lq + v; }
};

constexpr int ZBM = 64, ZBN = 128, ZBK = 8, ZNT = 256, ZPAD = 4;

// Batched products: blockIdx.y selects the system; operand and result offsets are the system index
// times these strides (complex elements); systems with active[s] == 0 are skipped.
struct ZBatch {
    int64_t sA = 0, sB = 0, sC = 0;
    const int *active = nullptr;
    // several products per system (direct-to-LDS kernel only): entry y of the batch is product y / nsys of
    // system y % nsys, B is the system's, and with sym the products from entry `herm` on are Hermitian
    int nsys = 0, herm = 0;
};
constexpr int ZWM = ZBM / 2, ZWN = ZBN / 2, ZFBM = ZWM / 16, ZFBN = ZWN / 16;
static_assert(ZBN == 2 * ZBM, "the lower-triangle tile count assumes tiles twice as wide as tall");

// Tiles of an n x n product that hold lower-triangle elements (row >= column): tile row tm (ZBM
// rows) reaches column ZBM*tm + ZBM-1, so it holds tm/2 + 1 tiles of ZBN columns, and tile rows
// 2a and 2a+1 hold a+1 each.  Ids are dealt over the XCDs as tile_of does; within a band the
// tiles go by rows.
static inline int lower_tiles_z(int tiles_m) {
    int t = 0;
    for (int r = 0; r < tiles_m; ++r) t += r / 2 + 1;
    return t;
}
__device__ inline void tile_of_lower_z(int w, int T, int &tm, int &tn) {
    int t = w;
    if ((T & 7) == 0) t = (w & 7) * (T >> 3) + (w >> 3);
    int a = (int)((sqrtf(4.0f * (float)t + 1.0f) - 1.0f) * 0.5f);
    while (a > 0 && a * (a + 1) > t) --a;
    while ((a + 1) * (a + 2) <= t) ++a;
    const int r = t - a * (a + 1);
    tm = 2 * a + r / (a + 1);
    tn = r % (a + 1);
}

// One BK slice of op(A) (BM x BK, "rows" r = i) or op(B)^T (BN x BK, r = j) into registers.
// CONTIG_R: r is the contiguous index in memory (A 'n', B 't'/'c'); otherwise k is.
template <typename R, bool CONTIG_R, bool CONJ, int ROWS>
struct ZStage {
    typedef typename ZPrec<R>::cplx C2;
    static constexpr int NE = ROWS * ZBK / ZNT;
    R re[NE], im[NE];
    __device__ static inline void coord(int t, int q, int &r, int &k) {
        const int idx = t + ZNT * q;
        if constexpr (CONTIG_R) {
            r = idx % ROWS;
            k = idx / ROWS;
        } else {
            k = idx % ZBK;
            r = idx / ZBK;
        }
    }
    __device__ inline void load(const C2 *__restrict__ P, int64_t ld, int r0, int k0, int rlim, int klim, int t) {
#pragma unroll
        for (int q = 0; q < NE; ++q) {
            int r, k;
            coord(t, q, r, k);
            const int gr = r0 + r, gk = k0 + k;
            C2 v;
            if (gr < rlim && gk < klim) {
                v = CONTIG_R ? P[(int64_t)gr + (int64_t)gk * ld] : P[(int64_t)gk + (int64_t)gr * ld];
            } else {
                v.x = (R)0;
                v.y = (R)0;
            }
            re[q] = v.x;
            im[q] = CONJ ? -v.y : v.y;
        }
    }
    __device__ inline void store(R *lre, R *lim, int t) const {
#pragma unroll
        for (int q = 0; q < NE; ++q) {
            int r, k;
            coord(t, q, r, k);
            lre[k * (ROWS + ZPAD) + r] = re[q];
            lim[k * (ROWS + ZPAD) + r] = im[q];
        }
    }
};

template <typename R, bool TRA, bool CJA, bool TRB, bool CJB, int NPAIR>
__global__ __launch_bounds__(ZNT, 2) void k_zgemm(int m, int n, int k, double alpha,
                                               const typename ZPrec<R>::cplx *__restrict__ A1,
                                               const typename ZPrec<R>::cplx *__restrict__ A2, int64_t lda,
                                               const typename ZPrec<R>::cplx *__restrict__ B1,
                                               const typename ZPrec<R>::cplx *__restrict__ B2, int64_t ldb,
                                               double beta0, const typename ZPrec<R>::cplx *__restrict__ C0,
                                               double beta, typename ZPrec<R>::cplx *__restrict__ C, int64_t ldc,
                                               int k_per_split, R *__restrict__ partial, int sym_tiles,
                                               ZBatch bat) {
    typedef typename ZPrec<R>::accv AV;
    typedef typename ZPrec<R>::cplx C2;
    constexpr int LA = ZBK * (ZBM + ZPAD), LB = ZBK * (ZBN + ZPAD);
    constexpr int STAGE = 2 * (LA + LB);  // re and im planes of A and B
    __shared__ R smem[2 * STAGE];

    const int bsys = blockIdx.y;
    if (bat.active && !bat.active[bsys]) return;  // whole workgroup, before any barrier
    A1 += bsys * bat.sA;
    A2 += bsys * bat.sA;
    B1 += bsys * bat.sB;
    B2 += bsys * bat.sB;
    C += bsys * bat.sC;
    if (C0) C0 += bsys * bat.sC;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int tiles_m = (m + ZBM - 1) / ZBM, tiles_n = (n + ZBN - 1) / ZBN;
    int tm, tn;
    if (sym_tiles)
        tile_of_lower_z(blockIdx.x, sym_tiles, tm, tn);
    else
        tile_of(blockIdx.x, tiles_m, tiles_n, tm, tn);
    const int i0 = tm * ZBM, j0 = tn * ZBN;
    const int ktot = NPAIR * k;
    const int kb = blockIdx.z * k_per_split;
    const int ke = min(ktot, kb + k_per_split);

    AV are[ZFBM][ZFBN], aim[ZFBM][ZFBN];
#pragma unroll
    for (int a = 0; a < ZFBM; ++a)
#pragma unroll
        for (int b = 0; b < ZFBN; ++b) {
            are[a][b] = AV{0, 0, 0, 0};
            aim[a][b] = AV{0, 0, 0, 0};
        }

    ZStage<R, !TRA, CJA, ZBM> sa;
    ZStage<R, TRB, CJB, ZBN> sb;
    auto fetch = [&](int kk) {
        const C2 *Ap = A1, *Bp = B1;
        int kl = kk;
        if (NPAIR == 2 && kk >= k) {
            Ap = A2;
            Bp = B2;
            kl = kk - k;
        }
        const int klim = min(k, kl + (ke - kk));
        sa.load(Ap, lda, i0, kl, m, klim, t);
        sb.load(Bp, ldb, j0, kl, n, klim, t);
    };
    auto planes = [&](int buf, R *&Are, R *&Aim, R *&Bre, R *&Bim) {
        R *base = smem + buf * STAGE;
        Are = base;
        Aim = base + LA;
        Bre = base + 2 * LA;
        Bim = base + 2 * LA + LB;
    };

    const int li = lane & 15, lk = lane >> 4;
    const int nslices = (ke - kb + ZBK - 1) / ZBK;
    if (nslices > 0) {
        R *Are, *Aim, *Bre, *Bim;
        fetch(kb);
        planes(0, Are, Aim, Bre, Bim);
        sa.store(Are, Aim, t);
        sb.store(Bre, Bim, t);
        __syncthreads();
        for (int s = 0; s < nslices; ++s) {
            const bool more = (s + 1 < nslices);
            if (more) fetch(kb + (s + 1) * ZBK);
            planes(s & 1, Are, Aim, Bre, Bim);
#pragma unroll
            for (int ks = 0; ks < ZBK; ks += 4) {
                R xr[ZFBM], xi[ZFBM], nxi[ZFBM], yr[ZFBN], yi[ZFBN];
#pragma unroll
                for (int f = 0; f < ZFBM; ++f) {
                    const int o = (ks + lk) * (ZBM + ZPAD) + wm * ZWM + f * 16 + li;
                    xr[f] = Are[o];
                    xi[f] = Aim[o];
                    nxi[f] = -xi[f];
                }
#pragma unroll
                for (int f = 0; f < ZFBN; ++f) {
                    const int o = (ks + lk) * (ZBN + ZPAD) + wn * ZWN + f * 16 + li;
                    yr[f] = Bre[o];
                    yi[f] = Bim[o];
                }
#pragma unroll
                for (int fm = 0; fm < ZFBM; ++fm)
#pragma unroll
                    for (int fn = 0; fn < ZFBN; ++fn) {
                        are[fm][fn] = ZPrec<R>::mfma(xr[fm], yr[fn], are[fm][fn]);
                        are[fm][fn] = ZPrec<R>::mfma(nxi[fm], yi[fn], are[fm][fn]);
                        aim[fm][fn] = ZPrec<R>::mfma(xr[fm], yi[fn], aim[fm][fn]);
                        aim[fm][fn] = ZPrec<R>::mfma(xi[fm], yr[fn], aim[fm][fn]);
                    }
            }
            if (more) {
                planes((s + 1) & 1, Are, Aim, Bre, Bim);
                sa.store(Are, Aim, t);
                sb.store(Bre, Bim, t);
            }
            __syncthreads();
        }
    }

    const int lq = lane >> 4;
#pragma unroll
    for (int fm = 0; fm < ZFBM; ++fm)
#pragma unroll
        for (int fn = 0; fn < ZFBN; ++fn) {
            const int j = j0 + wn * ZWN + fn * 16 + li;
            if (j >= n) continue;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int i = i0 + wm * ZWM + fm * 16 + ZPrec<R>::out_row(lq, v);
                if (i >= m) continue;
                const R vr = are[fm][fn][v], vi = aim[fm][fn][v];
                if (partial) {
                    const int64_t off = 2 * ((int64_t)blockIdx.z * m * n + (int64_t)i + (int64_t)j * m);
                    partial[off] = vr;
                    partial[off + 1] = vi;
                } else {
                    const int64_t off = (int64_t)i + (int64_t)j * ldc;
                    double rr = alpha * (double)vr, ri = alpha * (double)vi;
                    if (C0) {
                        rr += beta0 * (double)C0[off].x;
                        ri += beta0 * (double)C0[off].y;
                    }
                    if (beta != 0.0) {
                        rr += beta * (double)C[off].x;
                        ri += beta * (double)C[off].y;
                    }
                    C2 o;
                    o.x = (R)rr;
                    o.y = (R)ri;
                    C[off] = o;
                }
            }
        }
}

template <typename R>
__global__ void k_zsplitk_reduce(int m, int n, int splits, const R *__restrict__ partial, double alpha, double beta0,
                                 const typename ZPrec<R>::cplx *__restrict__ C0, double beta,
                                 typename ZPrec<R>::cplx *__restrict__ C, int64_t ldc) {
    const int64_t total = (int64_t)m * n;
    for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < total; q += (int64_t)gridDim.x * blockDim.x) {
        const int64_t i = q % m, j = q / m;
        R sr = partial[2 * q], si = partial[2 * q + 1];
        for (int z = 1; z < splits; ++z) {
            sr += partial[2 * ((int64_t)z * total + q)];
            si += partial[2 * ((int64_t)z * total + q) + 1];
        }
        const int64_t off = i + j * ldc;
        double rr = alpha * (double)sr, ri = alpha * (double)si;
        if (C0) {
            rr += beta0 * (double)C0[off].x;
            ri += beta0 * (double)C0[off].y;
        }
        if (beta != 0.0) {
            rr += beta * (double)C[off].x;
            ri += beta * (double)C[off].y;
        }
        typename ZPrec<R>::cplx o;
        o.x = (R)rr;
        o.y = (R)ri;
        C[off] = o;
    }
}

// ---------------------------------------------------------------------------------------------
// Direct-to-LDS products, for every m, n, k and leading dimensions up to 2^20.
//
// The operands stay interleaved (re, im) in LDS: an element is read whole (16 or 8 bytes), and the signs
// that conjugation and the real part need are put on A's values in registers.  K is taken in slices of
// 128 bytes of elements (8 complex128, 16 complex64), loaded with buffer_load_dwordx4 ... lds through
// descriptors that end where the operand ends (dwords past it arrive as zero); a row-contiguous operand
// lands k-major, a k-contiguous one in 128-byte rows whose 16-byte chunks are swizzled by row, and the
// last slice of such a row is cleared past k.  Tiles: 64x64 (4 waves of 32x32, two stages: a third stage
// leaves room for one workgroup fewer per CU and costs 2-4 %) and 32x32 (4 waves of 16x16, two stages of
// four slices); the K chain per element does not depend on the tile.
// What bounds it: the matrix cores (a 64x64 complex tile moves as few bytes per operation as a real
// 128x128 one), or, where the tiles do not fill the chip, the serial chain of slices of one tile.  The
// register-staged kernel below ran 64x128 tiles only: the 2000 x 2000 x 4000 complex128 Hermitian Gram
// took 1.60 ms (now 1.14), the full Gram 2.24 (1.85, 69 TF/s), 16 Grams of 128 x 128 x 256 on 32 workgroups
// 92 us (now 19).
// ---------------------------------------------------------------------------------------------
template <typename R>
struct ZGeo {
    static constexpr int ES = 2 * sizeof(R), EPC = 16 / ES, DK = 128 / ES;
    // the chunk swizzle of k-contiguous rows: complex128 reads one 16-byte chunk of 16 rows (16 distinct
    // bank groups), complex64 half a chunk
    __device__ static inline int swz(int r) { return ES == 16 ? (r & 7) ^ ((r >> 3) & 1) : dl_swz(r); }
};
// Byte offset of lane `lane` of wave load `ins` of an operand tile (ROWS rows) from the slice's base.
template <typename R, int ROWS, bool KC>
__device__ inline int zl_voff(int ins, int lane, int ld) {
    typedef ZGeo<R> G;
    if constexpr (KC) {
        const int r = ins * 8 + (lane >> 3);
        return r * ld * G::ES + 16 * ((lane & 7) ^ G::swz(r));
    } else {
        constexpr int LPR = ROWS * G::ES / 16;  // lanes per k-row
        return (ins * (64 / LPR) + lane / LPR) * ld * G::ES + 16 * (lane % LPR);
    }
}
// Place (in elements) of row r, k kk in a staged tile.
template <typename R, int ROWS, bool KC>
__device__ inline int zl_at(int r, int kk) {
    typedef ZGeo<R> G;
    return KC ? r * G::DK + ((kk / G::EPC) ^ G::swz(r)) * G::EPC + kk % G::EPC : kk * ROWS + r;
}

template <int B_, int NST_, int U_>
struct ZlCfg {
    static constexpr int B = B_, NST = NST_, U = U_, W = B_ / 2, FB = W / 16;
};
typedef ZlCfg<64, 2, 1> Zl64;
typedef ZlCfg<32, 2, 4> Zl32;

// CARRY (single products: complex64, every 32 values of K, and the complex128 ones of zl_carry): sums of `carry` slices are
// added up apart (see carry_sums), which keeps the error at or below that of the many parts K used to be split into (complex64 Gram
// 54 x 108: 1.6e-7 -> 1.4e-7, 2000 x 4000: 1.6e-6 -> 2.5e-7; with one chain 900 x 2916 1.3e-6) for 3 %.  Batched
// products keep one chain: their roundings are part of a k-point solve's trajectory.
template <typename R, class CF, bool TRA, bool CJA, bool TRB, bool CJB, int NPAIR, bool CARRY>
__global__ __launch_bounds__(256, 2) void k_zgemm_dl(int m, int n, int k, double alpha,
                                                    const typename ZPrec<R>::cplx *__restrict__ A1,
                                                    const typename ZPrec<R>::cplx *__restrict__ A2, int64_t lda,
                                                    const typename ZPrec<R>::cplx *__restrict__ B1,
                                                    const typename ZPrec<R>::cplx *__restrict__ B2, int64_t ldb,
                                                    double beta0, const typename ZPrec<R>::cplx *__restrict__ C0,
                                                    double beta, typename ZPrec<R>::cplx *__restrict__ C, int64_t ldc,
                                                    int sym, int sps, typename ZPrec<R>::cplx *__restrict__ partial,
                                                    int carry, ZBatch bat) {
    typedef ZGeo<R> G;
    typedef typename ZPrec<R>::cplx C2;
    typedef typename ZPrec<R>::accv AV;
    constexpr int B = CF::B, NST = CF::NST, U = CF::U, W = CF::W, FB = CF::FB, DK = G::DK;
    constexpr int LPW = 2 * B * 128 / 1024 / 4;          // wave loads per slice and wave
    constexpr int SLICE = 2 * B * DK, STAGE = U * SLICE;  // elements: A, then B
    constexpr bool KCA = TRA, KCB = !TRB;
    __shared__ __align__(16) C2 smem[NST * STAGE];
    const int bsys = blockIdx.y, sys = bat.nsys ? bsys % bat.nsys : bsys;
    if (bat.active && !bat.active[sys]) return;  // whole workgroup, before any barrier
    if (bat.nsys) {
        const int T = (m + B - 1) / B;
        if (bsys < bat.herm)
            sym = 0;
        else if (sym && (int)blockIdx.x >= T * (T + 1) / 2)
            return;  // the tiles above the diagonal
    }
    A1 += bsys * bat.sA;
    A2 += bsys * bat.sA;
    B1 += sys * bat.sB;
    B2 += sys * bat.sB;
    C += bsys * bat.sC;
    if (C0) C0 += bsys * bat.sC;
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    int tm, tn;
    if (sym)
        tile_of_lower(blockIdx.x, (m + B - 1) / B, tm, tn);
    else
        tile_of(blockIdx.x, (m + B - 1) / B, (n + B - 1) / B, tm, tn);
    const int i0 = tm * B, j0 = tn * B, wi = i0 + wm * W, wj = j0 + wn * W;
    const bool live = wi < m && wj < n && !(sym && wj > wi + W - 1);
    const int nsl = (k + DK - 1) / DK, sb = blockIdx.z * sps, ns = min(NPAIR * nsl, sb + sps) - sb;

    AV are[FB][FB], aim[FB][FB];
#pragma unroll
    for (int a = 0; a < FB; ++a)
#pragma unroll
        for (int b = 0; b < FB; ++b) {
            are[a][b] = AV{0, 0, 0, 0};
            aim[a][b] = AV{0, 0, 0, 0};
        }
    AV tre[CARRY ? FB : 1][CARRY ? FB : 1], tim[CARRY ? FB : 1][CARRY ? FB : 1];
    if constexpr (CARRY) {
#pragma unroll
        for (int a = 0; a < FB; ++a)
#pragma unroll
            for (int b = 0; b < FB; ++b) {
                tre[a][b] = AV{0, 0, 0, 0};
                tim[a][b] = AV{0, 0, 0, 0};
            }
    }
    // waves 0 and 1 load A, 2 and 3 B; the wave's descriptor advances by one slice each time and starts
    // over at the second product of a pair
    const bool on_b = wave >= 2;
    int voff[LPW];
#pragma unroll
    for (int q = 0; q < LPW; ++q) {
        const int ins = (wave & 1) * LPW + q;
        voff[q] = on_b ? zl_voff<R, B, KCB>(ins, lane, (int)ldb) : zl_voff<R, B, KCA>(ins, lane, (int)lda);
    }
    const bool kc = on_b ? KCB : KCA;
    const int64_t ld = on_b ? ldb : lda;
    const int x0 = on_b ? j0 : i0, ext = on_b ? n : m;
    const int64_t step = G::ES * (kc ? DK : DK * ld), at = G::ES * (kc ? x0 * ld : (int64_t)x0);
    const int64_t all = G::ES * (kc ? (int64_t)(ext - 1 - x0) * ld + k : (int64_t)(k - 1) * ld + (ext - x0));
    const char *const first = (const char *)(on_b ? B1 : A1) + at, *const second = (const char *)(on_b ? B2 : A2) + at;
    const int sb_in = NPAIR == 2 && sb >= nsl ? sb - nsl : sb;
    const char *pos = (NPAIR == 2 && sb >= nsl ? second : first) + sb_in * step;
    int64_t left = all - sb_in * step;
    // slice (of this part) where the second product starts; the last slice of each product if partial
    const int sw = nsl - sb, t1 = k % DK ? sw - 1 : -1, t2 = NPAIR == 2 && k % DK ? sw + nsl - 1 : -1;
    auto issue = [&](int s) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int sl = s * U + u;
            if (U > 1 && sl >= ns) break;
            C2 *st = smem + (s % NST) * STAGE + u * SLICE + wave * LPW * (1024 / G::ES);
            if (NPAIR == 2 && sl == sw) {
                pos = second;
                left = all;
            }
            const __amdgpu_buffer_rsrc_t r = raw_rsrc(pos, (uint32_t)((uint64_t)left >> 31) ? 0x7ffffff8 : (int)left);
            pos += step;
            left -= step;
#pragma unroll
            for (int q = 0; q < LPW; ++q) {
                const int vo = voff[q];
                __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void *)(st + q * (1024 / G::ES)), 16, vo, 0, 0, 0);
            }
        }
    };
    const int li = lane & 15, lk = lane >> 4;
    // a = x, b = y of op(A), op(B) before conjugation:
    //   re += xr yr + s xi yi, im += (sB) xr yi + (sA) xi yr, with sA, sB = -1 where conjugated and s = -sA sB
    constexpr bool NEG_S = (CJA == CJB), NEG_B = CJB, NEG_A = CJA;
    auto slice = [&](const C2 *As, const C2 *Bs) {
        C2 a[2][FB], b[2][FB];
        auto frag = [&](int ks, C2 (&fa)[FB], C2 (&fb)[FB]) {
#pragma unroll
            for (int f = 0; f < FB; ++f) fa[f] = As[zl_at<R, B, KCA>(wm * W + f * 16 + li, ks + lk)];
#pragma unroll
            for (int f = 0; f < FB; ++f) fb[f] = Bs[zl_at<R, B, KCB>(wn * W + f * 16 + li, ks + lk)];
        };
        frag(0, a[0], b[0]);
#pragma unroll
        for (int ks = 0; ks < DK; ks += 4) {
            const int cur = (ks / 4) & 1;
            if (ks + 4 < DK) frag(ks + 4, a[cur ^ 1], b[cur ^ 1]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int fm = 0; fm < FB; ++fm) {
                const C2 x = a[cur][fm];
                const R xs = NEG_S ? -x.y : x.y, xb = NEG_B ? -x.x : x.x, xa = NEG_A ? -x.y : x.y;
#pragma unroll
                for (int fn = 0; fn < FB; ++fn) {  // (y, x): the result's columns run along i
                    const C2 y = b[cur][fn];
                    are[fm][fn] = ZPrec<R>::mfma(y.x, x.x, are[fm][fn]);
                    aim[fm][fn] = ZPrec<R>::mfma(y.y, xb, aim[fm][fn]);
                    are[fm][fn] = ZPrec<R>::mfma(y.y, xs, are[fm][fn]);
                    aim[fm][fn] = ZPrec<R>::mfma(y.x, xa, aim[fm][fn]);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    const int nst = (ns + U - 1) / U, nfull = ns / U;
#pragma unroll
    for (int s = 0; s < NST - 1; ++s)
        if (s < nst) issue(s);
    auto march = [&](auto work) {  // waves outside the result only load, clear and wait
        for (int s = 0; s < nst; ++s) {
            if (NST > 2 && s + NST - 2 < nfull)
                __builtin_amdgcn_s_waitcnt(waitcnt_vmcnt(LPW * U * (NST - 2)));
            else
                __builtin_amdgcn_s_waitcnt(waitcnt_vmcnt(0));
            wg_barrier();  // stage s has landed for every wave; stage s-1 is no longer read
            if (s + NST - 1 < nst) issue(s + NST - 1);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int sl = s * U + u;
                if (U > 1 && sl >= ns) break;
                C2 *As = smem + (s % NST) * STAGE + u * SLICE, *Bs = As + B * DK;
                if ((KCA || KCB) && (sl == t1 || (NPAIR == 2 && sl == t2))) {  // k-contiguous rows end at k
                    for (int e = t; e < B * DK; e += 256)
                        if (e % DK >= k % DK) {
                            if (KCA) As[zl_at<R, B, true>(e / DK, e % DK)] = C2{0, 0};
                            if (KCB) Bs[zl_at<R, B, true>(e / DK, e % DK)] = C2{0, 0};
                        }
                    wg_barrier();
                }
                if (decltype(work)::value) {
                    slice(As, Bs);
                    if constexpr (CARRY) {
                        const bool end = sizeof(R) == 4 ? sl % 2 == 1 : u == U - 1 && (sl & (carry - 1)) == carry - 1;
                        if (end || (NPAIR == 2 && sl + 1 == sw)) {
                            carry_sums(are, tre);
                            carry_sums(aim, tim);
                        }
                    }
                }
            }
        }
    };
    if (!live) {
        march(std::false_type{});
        return;
    }
    march(std::true_type{});
    if constexpr (CARRY) {
#pragma unroll
        for (int a = 0; a < FB; ++a)
#pragma unroll
            for (int b = 0; b < FB; ++b) {
                are[a][b] = tre[a][b] + are[a][b];
                aim[a][b] = tim[a][b] + aim[a][b];
            }
    }
    const int lq = lane >> 4;
#pragma unroll
    for (int fm = 0; fm < FB; ++fm)
#pragma unroll
        for (int fn = 0; fn < FB; ++fn) {
            const int i = wi + fm * 16 + li;
            if (i >= m) continue;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int j = wj + fn * 16 + ZPrec<R>::out_row(lq, v);
                if (j >= n || (sym && j > i)) continue;
                const R vr = are[fm][fn][v], vi = aim[fm][fn][v];
                if (partial) {  // a part of K: the raw sums, reduced in part order later
                    partial[(int64_t)blockIdx.z * m * n + (int64_t)i + (int64_t)j * m] = C2{vr, vi};
                    continue;
                }
                const int64_t off = (int64_t)i + (int64_t)j * ldc;
                double rr = alpha * (double)vr, ri = alpha * (double)vi;
                if (C0) {
                    rr += beta0 * (double)C0[off].x;
                    ri += beta0 * (double)C0[off].y;
                }
                if (beta != 0.0) {
                    rr += beta * (double)C[off].x;
                    ri += beta * (double)C[off].y;
                }
                C[off] = C2{(R)rr, (R)ri};
                if (sym == 2 && j < i) C[(int64_t)j + (int64_t)i * ldc] = C2{(R)rr, (R)-ri};
            }
        }
}

// C := alpha * (sum of the K parts, in part order) + beta0*C0 + beta*C; sym: the lower triangle, and with
// sym == 2 its conjugate mirror.
template <typename R>
__global__ __launch_bounds__(256) void k_zl_reduce(int m, int n, int sym, int splits,
                                                   const typename ZPrec<R>::cplx *__restrict__ partial, double alpha,
                                                   double beta0, const typename ZPrec<R>::cplx *__restrict__ C0,
                                                   double beta, typename ZPrec<R>::cplx *__restrict__ C, int64_t ldc) {
    typedef typename ZPrec<R>::cplx C2;
    const int64_t total = (int64_t)m * n;
    for (int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x; q < total; q += (int64_t)gridDim.x * 256) {
        const int64_t i = q % m, j = q / m;
        if (sym && j > i) continue;
        C2 s = partial[q];
        for (int z = 1; z < splits; ++z) {
            const C2 p = partial[(int64_t)z * total + q];
            s.x += p.x;
            s.y += p.y;
        }
        const int64_t off = i + j * ldc;
        double rr = alpha * (double)s.x, ri = alpha * (double)s.y;
        if (C0) {
            rr += beta0 * (double)C0[off].x;
            ri += beta0 * (double)C0[off].y;
        }
        if (beta != 0.0) {
            rr += beta * (double)C[off].x;
            ri += beta * (double)C[off].y;
        }
        C[off] = C2{(R)rr, (R)ri};
        if (sym == 2 && j < i) C[j + i * ldc] = C2{(R)rr, (R)-ri};
    }
}

static int64_t zl_tiles(int m, int n, int b, bool sym) {
    const int64_t tm = (m + b - 1) / b, tn = (n + b - 1) / b;
    return sym ? tm * (tm + 1) / 2 : tm * tn;
}
// Tile and parts of K with the least time: rounds of workgroups over the CUs times the slices of a part,
// plus the reduction of the parts.  round[r] is a CU's time (us) for one slice of r workgroups resident
// together (up to four of the 64 tile, two of the 32 one), measured with 250 to 2000 states: a lone
// workgroup leaves the matrix cores idle while it waits, 1.37 us per slice against 0.92 in a full CU.
static void zl_shape(omx_ctx ctx, int m, int n, int nsl, bool sym, int nbatch, bool split, bool seam, int &tile,
                     int &splits) {
    const int edge[2] = {64, 32}, full[2] = {4, 2};
    const double round[2][5] = {{0.0, 1.37, 1.96, 2.87, 3.69}, {0.0, 0.29, 0.55, 0.0, 0.0}};
    double cost = 0.0;
    tile = 0;
    for (int q = 0; q < 2; ++q)
        for (int s : {1, 2, 3, 4, 5, 6, 8, 12}) {
            if (s > 1 && (!split || nsl < 4 * s)) break;
            if (s == 1 && seam && split && nsl >= 8) continue;  // two parts at the least
            const int64_t units = zl_tiles(m, n, edge[q], sym) * nbatch * s;
            const int64_t rounds = (units + ctx->num_cus - 1) / ctx->num_cus;
            const double per = (double)(rounds / full[q]) * round[q][full[q]] + round[q][rounds % full[q]];
            const double c = 0.55 * rounds + per * ((nsl + s - 1) / s) +
                             (s > 1 ? 5.3 + 16e-6 * (s + 1) * m * n / 4.9 : 0.0);
            if (!tile || c < cost) {
                tile = edge[q];
                splits = s;
                cost = c;
            }
        }
}

// Slices of K (of nsl) between the carries of a complex128 product, 0 for none: carried where its parts of K (sps
// slices) are a quarter longer than those that 64x128 tiles were split into to fill the chip (up to four for the
// lower triangle of a Hermitian product).  Against 80 bits, with those parts, without and with carried sums: Gram
// 250 x 500 2.8e-16, 4.6e-16, 2.4e-16, 700 x 1400 5.3e-16, 1.7e-15, 3.5e-16; Hermitian 2000 x 4000 1.15e-15, 2.8e-15,
// 3.7e-16 (1.09 -> 1.14 ms).
static int zl_carry(omx_ctx ctx, int m, int n, bool lower, int nsl, int sps) {
    const int64_t tm = (m + ZBM - 1) / ZBM, tn = (n + ZBN - 1) / ZBN, tiles = lower ? (tm * tn + tm) / 2 : tm * tn;
    const int64_t fill = tiles < 2 * ctx->num_cus ? (2 * ctx->num_cus + tiles - 1) / tiles : 1;
    const int64_t parts = std::min<int64_t>(std::min<int64_t>(fill, lower ? 4 : 64), std::max(1, nsl / 4));
    return 4 * sps * parts > 5 * (int64_t)nsl ? carry_period(nsl, parts) : 0;
}

// Launches the direct-to-LDS product; OMX_ERR_UNSUPPORTED for leading dimensions beyond 2^20.
template <typename R, bool TRA, bool CJA, bool TRB, bool CJB, int NPAIR>
static int run_zgemm_dl(omx_ctx ctx, int m, int n, int k, double alpha, const void *A1, const void *A2, int64_t lda,
                        const void *B1, const void *B2, int64_t ldb, double beta0, const void *C0, double beta, void *C,
                        int64_t ldc, int nbatch, const ZBatch &bat, bool allow_split) {
    typedef typename ZPrec<R>::cplx C2;
    if (m <= 0 || n <= 0 || k <= 0 || lda > (1 << 20) || ldb > (1 << 20)) return OMX_ERR_UNSUPPORTED;
    // A complex64 gradient of an order that is no multiple of 8 stays in three passes: their roundings of
    // the intermediate results to FP32 are part of a solve's trajectory (one product instead moves an
    // energy by 3e-6 within 20 CG steps).
    if (NPAIR == 2 && sizeof(R) == 4 && k % ZBK != 0) return OMX_ERR_UNSUPPORTED;
    const int sym = (NPAIR == 1 && m == n && !TRA && TRB && CJB) ? ctx->gemm_sym : 0;
    const int nsl = NPAIR * ((k + ZGeo<R>::DK - 1) / ZGeo<R>::DK);
    // The two products of a complex128 pair whose K is no multiple of 8 used to be made in separate passes: the chains
    // are no longer than theirs (pairs against 80 bits, separate passes, one chain over both, now: 701 states 5.8e-16,
    // 9.2e-16, 3.9e-16, 0.22 -> 0.23 ms; 2001 2.05e-15, 2.99e-15, 2.05e-15, 4.06 -> 4.09 ms).
    const bool seam = NPAIR == 2 && k % ZBK != 0;
    int tile, splits;
    // batched launches never split K: no workspace, so the launch can be graph-captured
    const bool lower = sym && !bat.nsys;  // a grid of lower-triangle tiles
    zl_shape(ctx, m, n, nsl, lower, bat.nsys ? (nbatch + bat.herm) / 2 : nbatch, allow_split && nbatch == 1, seam, tile,
             splits);
    int sps = (nsl + splits - 1) / splits;
    splits = (nsl + sps - 1) / sps;
    C2 *partial = nullptr;
    if (splits > 1) {
        const int rc = ensure_ws(ctx, sizeof(C2) * (size_t)splits * m * n);
        if (rc == OMX_ERR_NOMEM) {  // no room for the parts: K whole, which needs none
            clear_error();
            splits = 1;
            sps = nsl;
        } else if (rc) {
            return rc;
        } else {
            partial = (C2 *)ctx->ws;
        }
    }
    const int64_t tiles = zl_tiles(m, n, tile, lower);
    OMX_REQUIRE(tiles < (1LL << 31), "complex product: grid too large");
    const int cls = NPAIR == 2 ? OMX_K_GEMM_PAIR : OMX_K_GEMM, nherm = sym ? nbatch - bat.herm : 0;
    hipEvent_t ev;
    prof_begin(ctx, cls, &ev);
    prof_work(ctx, cls, 8.0 * (nherm * (nherm ? sym_area(m, tile) : 0.0) + (nbatch - nherm) * (double)m * n) * NPAIR * k,
              nbatch * 2.0 * sizeof(R) * ((double)NPAIR * ((double)m * k + (double)k * n) +
                                          (double)m * n * (1 + (C0 ? 1 : 0) + (beta != 0.0 ? 1 : 0))));
    const dim3 grid((unsigned)tiles, nbatch, splits);
#define OMX_ZL_RUN(CF, CY)                                                                                          \
    hipLaunchKernelGGL((k_zgemm_dl<R, CF, TRA, CJA, TRB, CJB, NPAIR, CY>), grid, dim3(256), 0, ctx->stream, m, n, k, alpha, \
                       (const C2 *)A1, (const C2 *)A2, lda, (const C2 *)B1, (const C2 *)B2, ldb, beta0,             \
                       (const C2 *)C0, beta, (C2 *)C, ldc, sym, sps, partial, carry, bat)
    const int carry = !allow_split ? 0 : sizeof(R) == 4 ? 2 : zl_carry(ctx, m, n, lower, seam ? nsl / 2 : nsl, sps);
    if (tile == 64 && carry)
        OMX_ZL_RUN(Zl64, true);
    else if (tile == 64)
        OMX_ZL_RUN(Zl64, false);
    else if (carry)
        OMX_ZL_RUN(Zl32, true);
    else
        OMX_ZL_RUN(Zl32, false);
#undef OMX_ZL_RUN
    if (partial)
        hipLaunchKernelGGL((k_zl_reduce<R>), dim3((unsigned)std::min<int64_t>(((int64_t)m * n + 255) / 256, 8192)),
                           dim3(256), 0, ctx->stream, m, n, sym, splits, partial, alpha, beta0, (const C2 *)C0, beta,
                           (C2 *)C, ldc);
    prof_end(ctx, cls, ev);
    OMX_CHECK_HIP(hipGetLastError());
    if (sym == 2) ctx->gemm_sym = 3;  // the upper triangle is written too
    return OMX_OK;
}

template <typename R, bool TRA, bool CJA, bool TRB, bool CJB, int NPAIR>
static int run_zgemm(omx_ctx ctx, int m, int n, int k, double alpha, const void *A1, const void *A2, int64_t lda,
                     const void *B1, const void *B2, int64_t ldb, double beta0, const void *C0, double beta, void *C,
                     int64_t ldc, int nbatch = 1, ZBatch bat = ZBatch(), bool allow_split = true) {
    typedef typename ZPrec<R>::cplx C2;
    {
        const int rc = run_zgemm_dl<R, TRA, CJA, TRB, CJB, NPAIR>(ctx, m, n, k, alpha, A1, A2, lda, B1, B2, ldb, beta0, C0,
                                                                  beta, C, ldc, nbatch, bat, allow_split);
        if (rc != OMX_ERR_UNSUPPORTED) return rc;
        if (NPAIR == 2 && k % ZBK != 0) return rc;  // the staged pair's boundary must fall on a slice boundary
    }
    const int full_tiles = ((m + ZBM - 1) / ZBM) * ((n + ZBN - 1) / ZBN);
    const int ktot = NPAIR * k;
    int splits = 1;
    const int target = 2 * ctx->num_cus;
    // products known to be Hermitian (A B^H, ctx->gemm_sym): lower-triangle tiles only.  Split along
    // K when the tiles fill less than two workgroups per CU; the reduction also writes the upper
    // elements no tile computed, which the caller's mirror then overwrites.
    const int sym_tiles =
        (ctx->gemm_sym && NPAIR == 1 && m == n && !TRA && TRB && CJB) ? lower_tiles_z((m + ZBM - 1) / ZBM) : 0;
    const int tiles = sym_tiles ? sym_tiles : full_tiles;
    // batched launches never split K: no workspace, so the launch can be graph-captured
    if (allow_split && nbatch == 1 && tiles < target) {
        const int max_splits = std::max(1, ktot / (4 * ZBK));
        splits = std::max(1, std::min(std::min(max_splits, (target + tiles - 1) / tiles), 64));
        if (sym_tiles) {
            // the fewest rounds of workgroups per unit of K, up to 4 splits (272 tiles: 3 splits,
            // two rounds of thirds, not 2 splits and a second round of 32 workgroups)
            auto cost = [&](int q) { return (double)((tiles * q + target - 1) / target) / q; };
            splits = 1;
            for (int q = 2; q <= std::min(max_splits, 4); ++q)
                if (cost(q) < cost(splits)) splits = q;
        }
    }
    int kps = (ktot + splits - 1) / splits;
    kps = (kps + ZBK - 1) / ZBK * ZBK;
    splits = (ktot + kps - 1) / kps;
    R *partial = nullptr;
    if (splits > 1) {
        int rc = ensure_ws(ctx, sizeof(R) * 2 * (size_t)splits * m * n);
        if (rc) return rc;
        partial = (R *)ctx->ws;
    }
    hipEvent_t ev;
    prof_begin(ctx, NPAIR == 2 ? OMX_K_GEMM_PAIR : OMX_K_GEMM, &ev);
    prof_work(ctx, NPAIR == 2 ? OMX_K_GEMM_PAIR : OMX_K_GEMM,
              nbatch * 8.0 * m * n * (double)ktot * ((double)tiles / full_tiles),
              nbatch * 2.0 * sizeof(R) * ((double)NPAIR * ((double)m * k + (double)k * n) +
                                          (double)m * n * (1 + (C0 ? 1 : 0) + (beta != 0.0 ? 1 : 0))));
    hipLaunchKernelGGL((k_zgemm<R, TRA, CJA, TRB, CJB, NPAIR>), dim3(tiles, nbatch, splits), dim3(ZNT), 0, ctx->stream,
                       m, n, k, alpha, (const C2 *)A1, (const C2 *)A2, lda, (const C2 *)B1, (const C2 *)B2, ldb, beta0,
                       (const C2 *)C0, beta, (C2 *)C, ldc, kps, partial, sym_tiles, bat);
    if (splits > 1) {
        const int64_t total = (int64_t)m * n;
        const int grid = (int)std::min<int64_t>((total + 255) / 256, 8192);
        hipLaunchKernelGGL((k_zsplitk_reduce<R>), dim3(grid), dim3(256), 0, ctx->stream, m, n, splits, partial, alpha,
                           beta0, (const C2 *)C0, beta, (C2 *)C, ldc);
    }
    prof_end(ctx, NPAIR == 2 ? OMX_K_GEMM_PAIR : OMX_K_GEMM, ev);
    OMX_CHECK_HIP(hipGetLastError());
    return OMX_OK;
}

// op -> (transposed, conjugated) template arguments.
template <typename R, bool TRB, bool CJB>
static int zdispatch_a(omx_ctx ctx, char opA, int m, int n, int k, double alpha, const void *A, int64_t lda,
                       const void *B, int64_t ldb, double beta, void *C, int64_t ldc) {
    if (opA == 'n' || opA == 'N')
        return run_zgemm<R, false, false, TRB, CJB, 1>(ctx, m, n, k, alpha, A, A, lda, B, B, ldb, 0.0, nullptr, beta,
                                                       C, ldc);
    if (opA == 't' || opA == 'T')
        return run_zgemm<R, true, false, TRB, CJB, 1>(ctx, m, n, k, alpha, A, A, lda, B, B, ldb, 0.0, nullptr, beta, C,
                                                      ldc);
    return run_zgemm<R, true, true, TRB, CJB, 1>(ctx, m, n, k, alpha, A, A, lda, B, B, ldb, 0.0, nullptr, beta, C,
                                                 ldc);
}

template <typename R>
static int zdispatch(omx_ctx ctx, char opA, char opB, int m, int n, int k, double alpha, const void *A, int64_t lda,
                     const void *B, int64_t ldb, double beta, void *C, int64_t ldc) {
    if (opB == 'n' || opB == 'N')
        return zdispatch_a<R, false, false>(ctx, opA, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
    if (opB == 't' || opB == 'T')
        return zdispatch_a<R, true, false>(ctx, opA, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
    return zdispatch_a<R, true, true>(ctx, opA, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
}

int launch_zgemm(omx_ctx ctx, int dt, char opA, char opB, int m, int n, int k, double alpha, const void *A,
                 int64_t lda, const void *B, int64_t ldb, double beta, void *C, int64_t ldc) {
    if (dt == OMX_C128) return zdispatch<double>(ctx, opA, opB, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
    if (dt == OMX_C64) return zdispatch<float>(ctx, opA, opB, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
    set_error("complex product: unsupported element type %d", dt);
    return OMX_ERR_UNSUPPORTED;
}

// Batched complex products (complex128 or complex64) over nbatch systems with element strides sA, sB,
// sC (result and C0).
template <typename R>
static int zgemm_batched_r(omx_ctx ctx, char opA, char opB, int m, int n, int k, double alpha, const void *A,
                           int64_t lda, const void *B, int64_t ldb, double beta, void *C, int64_t ldc, int nbatch,
                           const ZBatch &bat) {
    const bool ta = (opA != 'n' && opA != 'N');
    const bool tb = (opB != 'n' && opB != 'N'), cb = (opB == 'c' || opB == 'C');
    if (!ta && tb && cb)  // the Gram products X Y^H
        return run_zgemm<R, false, false, true, true, 1>(ctx, m, n, k, alpha, A, A, lda, B, B, ldb, 0.0, nullptr,
                                                         beta, C, ldc, nbatch, bat, false);
    if (!ta && !tb)
        return run_zgemm<R, false, false, false, false, 1>(ctx, m, n, k, alpha, A, A, lda, B, B, ldb, 0.0, nullptr,
                                                           beta, C, ldc, nbatch, bat, false);
    set_error("batched complex product: op (%c,%c) not available", opA, opB);
    return OMX_ERR_UNSUPPORTED;
}

int launch_zgemm_batched(omx_ctx ctx, int dt, char opA, char opB, int m, int n, int k, double alpha, const void *A,
                         int64_t lda, int64_t sA, const void *B, int64_t ldb, int64_t sB, double beta, void *C,
                         int64_t ldc, int64_t sC, int nbatch, const int *active) {
    ZBatch bat;
    bat.sA = sA;
    bat.sB = sB;
    bat.sC = sC;
    bat.active = active;
    if (dt == OMX_C128)
        return zgemm_batched_r<double>(ctx, opA, opB, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, nbatch, bat);
    if (dt == OMX_C64)
        return zgemm_batched_r<float>(ctx, opA, opB, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, nbatch, bat);
    set_error("batched complex product: unsupported element type %d", dt);
    return OMX_ERR_UNSUPPORTED;
}

// C(i, j) := conj(C(j, i)) for i < j in each system's n x n block: copies the lower triangle of a
// Hermitian product onto the upper one.  One 32 x 32 tile pair per workgroup (the diagonal tiles
// on themselves), through an LDS transpose so that reads and writes run along columns.
template <typename R>
__global__ __launch_bounds__(256) void k_herm_mirror(int n, typename ZPrec<R>::cplx *__restrict__ C, int64_t ldc,
                                                     ZBatch bat) {
    typedef typename ZPrec<R>::cplx C2;
    constexpr int T = 32;
    __shared__ C2 tile[T][T + 1];
    const int bsys = blockIdx.y;
    if (bat.active && !bat.active[bsys]) return;
    C += bsys * bat.sC;
    int a, b;  // lower tile (a, b), a >= b; it fills the upper tile (b, a)
    tile_of_lower(blockIdx.x, (n + T - 1) / T, a, b);
    const int r0 = a * T, c0 = b * T;
    for (int q = threadIdx.x; q < T * T; q += 256) {
        const int r = q % T, c = q / T;
        if (r0 + r < n && c0 + c < n) tile[c][r] = C[(int64_t)(r0 + r) + (int64_t)(c0 + c) * ldc];
    }
    __syncthreads();
    for (int q = threadIdx.x; q < T * T; q += 256) {
        const int i = q % T, j = q / T;  // upper element (c0 + i, r0 + j)
        const int gi = c0 + i, gj = r0 + j;
        if (gi < gj && gj < n) {
            C2 v = tile[i][j];
            v.y = -v.y;
            C[(int64_t)gi + (int64_t)gj * ldc] = v;
        }
    }
}

// C := alpha * A * B^H for a product known to be Hermitian (n x n; A, B n x k), as AW = (C*H)*C^H in
// omm()'s calc_AW (omm_ops.F90:44-64) on complex storage.  The kernel computes the lower-triangle
// tiles where it can, and the lower triangle is then mirrored, so C is exactly Hermitian.
template <typename R>
static int zgemm_herm_r(omx_ctx ctx, int n, int k, double alpha, const void *A, int64_t lda, const void *B,
                        int64_t ldb, void *C, int64_t ldc, int nbatch, const ZBatch &bat, bool allow_split) {
    ctx->gemm_sym = 2;
    int rc = run_zgemm<R, false, false, true, true, 1>(ctx, n, n, k, alpha, A, A, lda, B, B, ldb, 0.0, nullptr, 0.0,
                                                       C, ldc, nbatch, bat, allow_split);
    const bool whole = ctx->gemm_sym == 3;  // the product wrote the upper triangle too
    ctx->gemm_sym = 0;
    if (rc || whole) return rc;
    const int nt = (n + 31) / 32;
    hipLaunchKernelGGL(k_herm_mirror<R>, dim3(nt * (nt + 1) / 2, nbatch), dim3(256), 0, ctx->stream, n,
                       (typename ZPrec<R>::cplx *)C, ldc, bat);
    OMX_CHECK_HIP(hipGetLastError());
    return OMX_OK;
}

int launch_zgemm_herm(omx_ctx ctx, int dt, int n, int k, double alpha, const void *A, int64_t lda, const void *B,
                      int64_t ldb, void *C, int64_t ldc) {
    if (dt == OMX_C128) return zgemm_herm_r<double>(ctx, n, k, alpha, A, lda, B, ldb, C, ldc, 1, ZBatch(), true);
    if (dt == OMX_C64) return zgemm_herm_r<float>(ctx, n, k, alpha, A, lda, B, ldb, C, ldc, 1, ZBatch(), true);
    set_error("Hermitian product: unsupported element type %d", dt);
    return OMX_ERR_UNSUPPORTED;
}

int launch_zgemm_search_batched(omx_ctx ctx, int dt, int n, int k, const void *X, int64_t ldx, int64_t sX,
                                const void *D, int64_t ldd, int64_t sD, void *C, int64_t ldc, int64_t sC, int nbatch,
                                const int *active) {
    OMX_REQUIRE(dt == OMX_C128 || dt == OMX_C64, "batched complex products: unsupported element type %d", dt);
    int rc = OMX_ERR_UNSUPPORTED;
    if (4LL * nbatch < 65536) {
        ZBatch bat;
        bat.sA = sX;
        bat.sB = sD;
        bat.sC = sC;
        bat.active = active;
        bat.nsys = nbatch;
        bat.herm = 2 * nbatch;
        ctx->gemm_sym = 2;
        rc = dt == OMX_C128 ? run_zgemm_dl<double, false, false, true, true, 1>(ctx, n, n, k, 1.0, X, X, ldx, D, D, ldd, 0.0,
                                                                                nullptr, 0.0, C, ldc, 4 * nbatch, bat, false)
                            : run_zgemm_dl<float, false, false, true, true, 1>(ctx, n, n, k, 1.0, X, X, ldx, D, D, ldd, 0.0,
                                                                               nullptr, 0.0, C, ldc, 4 * nbatch, bat, false);
        ctx->gemm_sym = 0;
    }
    if (rc != OMX_ERR_UNSUPPORTED) return rc;
    const size_t es = dt == OMX_C128 ? 16 : 8;
    for (int q = 0; q < 4; ++q) {
        const void *x = (const char *)X + es * q * nbatch * sX;
        void *c = (char *)C + es * q * nbatch * sC;
        rc = q < 2 ? launch_zgemm_batched(ctx, dt, 'n', 'c', n, n, k, 1.0, x, ldx, sX, D, ldd, sD, 0.0, c, ldc, sC, nbatch,
                                          active)
                   : launch_zgemm_herm_batched(ctx, dt, n, k, 1.0, x, ldx, sX, D, ldd, sD, c, ldc, sC, nbatch, active);
        if (rc) return rc;
    }
    return OMX_OK;
}
int launch_zgemm_herm_batched(omx_ctx ctx, int dt, int n, int k, double alpha, const void *A, int64_t lda,
                              int64_t sA, const void *B, int64_t ldb, int64_t sB, void *C, int64_t ldc, int64_t sC,
                              int nbatch, const int *active) {
    ZBatch bat;
    bat.sA = sA;
    bat.sB = sB;
    bat.sC = sC;
    bat.active = active;
    if (dt == OMX_C128) return zgemm_herm_r<double>(ctx, n, k, alpha, A, lda, B, ldb, C, ldc, nbatch, bat, false);
    if (dt == OMX_C64) return zgemm_herm_r<float>(ctx, n, k, alpha, A, lda, B, ldb, C, ldc, nbatch, bat, false);
    set_error("batched Hermitian product: unsupported element type %d", dt);
    return OMX_ERR_UNSUPPORTED;
}

int launch_zgemm_pair_batched(omx_ctx ctx, int dt, int m, int n, int k, double alpha, const void *A1, const void *A2,
                              int64_t lda, int64_t sA, const void *B1, const void *B2, int64_t ldb, int64_t sB,
                              double beta0, const void *C0, double beta, void *C, int64_t ldc, int64_t sC, int nbatch,
                              const int *active) {
    ZBatch bat;
    bat.sA = sA;
    bat.sB = sB;
    bat.sC = sC;
    bat.active = active;
    if (dt == OMX_C64)
        return run_zgemm<float, false, false, false, false, 2>(ctx, m, n, k, alpha, A1, A2, lda, B1, B2, ldb, beta0,
                                                               C0, beta, C, ldc, nbatch, bat, false);
    return run_zgemm<double, false, false, false, false, 2>(ctx, m, n, k, alpha, A1, A2, lda, B1, B2, ldb, beta0, C0,
                                                            beta, C, ldc, nbatch, bat, false);
}

int launch_zgemm_pair(omx_ctx ctx, int dt, int m, int n, int k, double alpha, const void *A1, const void *A2,
                      int64_t lda, const void *B1, const void *B2, int64_t ldb, double beta0, const void *C0,
                      double beta, void *C, int64_t ldc) {
    if (dt == OMX_C128)
        return run_zgemm<double, false, false, false, false, 2>(ctx, m, n, k, alpha, A1, A2, lda, B1, B2, ldb, beta0,
                                                                C0, beta, C, ldc);
    if (dt == OMX_C64)
        return run_zgemm<float, false, false, false, false, 2>(ctx, m, n, k, alpha, A1, A2, lda, B1, B2, ldb, beta0,
                                                               C0, beta, C, ldc);
    set_error("complex calc_G: unsupported element type %d", dt);
    return OMX_ERR_UNSUPPORTED;
}

}  // namespace omx

// Dense products on the CDNA4 matrix cores: C := alpha*op(A)*op(B) + beta*C.
//
// One kernel template covers the OMM products
//   Gram      (No x Nb)(Nb x No)  -> op = ('n','t'): HWd = HC*D^T, SWd = SC*D^T, HWdd = HG*D^T, ...
//   gradient  (No x No)(No x Nb)  -> op = ('n','n'): SW*HC, HW*SC (fused pair: calc_G)
//   density   (Nb x No)(No x Nb)  -> op = ('t','n'): D_min = C^T*(QW*C)
// and the three precisions:
//   FP64: v_mfma_f64_16x16x4f64, FP64 accumulate (the oracle-grade path);
//   FP32: operands rounded to FP32, v_mfma_f32_16x16x4f32, FP32 accumulate;
//   BF16: operands rounded to BF16 (one rounding from the stored value),
//         v_mfma_f32_16x16x32_bf16, FP32 accumulate.
//
// Work decomposition: a workgroup of WGM x WGN wave64s owns a BM x BN tile of C; each wave owns
// a (BM/WGM) x (BN/WGN) sub-tile held as 16x16 MFMA accumulator blocks.  K is consumed in BK
// slices staged through LDS and double-buffered: the next slice is fetched from HBM/L2 into
// registers (16-byte vector loads along the contiguous index) while the current slice feeds the
// MFMAs.  When the tile count cannot fill the chip, K is split over grid.z into partial tiles
// that a second kernel adds in split order (deterministic).  The linear workgroup id is remapped
// so that each XCD (ids are dealt round-robin over the 8 XCDs) walks a contiguous band of tiles,
// grouped GM tile-rows at a time, so operand panels are shared inside one XCD's L2.
#include <algorithm>
#include <type_traits>

#include "omx_internal.h"
#include "omx_mfma.h"

namespace omx {

// ---------------------------------------------------------------------------------------------
// Precision traits: K slice, LDS element type, accumulator type and result lane layout.
// ---------------------------------------------------------------------------------------------
template <int PREC>
struct Prec;

template <>
struct Prec<OMX_PREC_F64> {
    static constexpr int BK = 16;
    typedef double lds_t;
    typedef double acc_t;
    typedef d4v accv;
    // v_mfma_f64_16x16x4f64 result: lane l, register pair v -> row (l/16) + 4v, column l%16
    __device__ static inline int out_row(int lq, int v) { return lq + 4 * v; }
};
template <>
struct Prec<OMX_PREC_F32> {
    static constexpr int BK = 32;
    typedef float lds_t;
    typedef float acc_t;
    typedef f4v accv;
    // v_mfma_f32_16x16x4f32 result: lane l, register v -> row 4(l/16) + v, column l%16
    __device__ static inline int out_row(int lq, int v) { return 4 * lq + v; }
};
template <>
struct Prec<OMX_PREC_BF16> {
    static constexpr int BK = 64;
    typedef __bf16 lds_t;
    typedef float acc_t;
    typedef f4v accv;
    // v_mfma_f32_16x16x32_bf16 result: lane l, register v -> row 4(l/16) + v, column l%16
    __device__ static inline int out_row(int lq, int v) { return 4 * lq + v; }
};

template <typename TS, int PREC>
__device__ inline typename Prec<PREC>::lds_t to_lds(TS v) {
    return (typename Prec<PREC>::lds_t)v;
}

// ---------------------------------------------------------------------------------------------
// Tile configurations.
// ---------------------------------------------------------------------------------------------
template <int BM_, int BN_, int WGM_, int WGN_, int MINW_>
struct Cfg {
    static constexpr int BM = BM_, BN = BN_, WGM = WGM_, WGN = WGN_;
    static constexpr int NT = 64 * WGM * WGN;
    static constexpr int WM = BM / WGM, WN = BN / WGN;
    static constexpr int FBM = WM / 16, FBN = WN / 16;
    static constexpr int MINW = MINW_;  // waves per SIMD the register budget must allow
};
// Ids used by the selector and by omx_gemm_set_tile().
typedef Cfg<128, 128, 2, 2, 2> Cfg0;  // 4 waves, 64x64 per wave, two workgroups per CU
typedef Cfg<128, 128, 2, 2, 1> Cfg1;  // 4 waves, 64x64 per wave, one workgroup per CU
typedef Cfg<256, 128, 2, 2, 1> Cfg2;  // 4 waves, 128x64 per wave
typedef Cfg<128, 256, 2, 2, 1> Cfg3;  // 4 waves, 64x128 per wave
typedef Cfg<256, 256, 2, 4, 1> Cfg4;  // 8 waves, 128x64 per wave (BF16 products)
typedef Cfg<128, 128, 4, 2, 2> Cfg5;  // 8 waves, 32x64 per wave, two workgroups per CU (FP64)
typedef Cfg<128, 128, 2, 4, 2> Cfg6;  // 8 waves, 64x32 per wave, two workgroups per CU (FP64)
constexpr int kNumCfg = 8;  // 7: direct-to-LDS staging (FP64 and FP32 products)

// LDS layouts.  FP64/FP32: k-major ([k][i], i contiguous): one element per lane per MFMA step,
// lanes 0..15 read 16 consecutive i.  BF16: i-major ([i][k], k contiguous): each lane feeds 8
// consecutive k values per MFMA step as one 16-byte read.
template <int PREC, int ROWS>
struct LdsT {
    static constexpr int BK = Prec<PREC>::BK;
    static constexpr bool KMAJOR = (PREC != OMX_PREC_BF16);
    static constexpr int PAD = KMAJOR ? 4 : 8;
    static constexpr int ELEMS = KMAJOR ? BK * (ROWS + PAD) : ROWS * (BK + PAD);
    __device__ static inline int off(int r, int k) { return KMAJOR ? k * (ROWS + PAD) + r : r * (BK + PAD) + k; }
};

// ---------------------------------------------------------------------------------------------
// Global -> register staging of one BK slice of op(A) (BM x BK) or op(B)^T (BN x BK).
// "Row" index r (i for A, j for B) and k.  CONTIG_R: r is contiguous in memory (A 'n', B 't');
// otherwise k is (A 't', B 'n').  Loads are VEC-wide vectors along the contiguous index when
// the vector lies inside the matrix and the leading dimension keeps it 16-byte aligned.
// ---------------------------------------------------------------------------------------------
template <typename TS, int PREC, bool CONTIG_R, int ROWS, int NT>
struct Stage {
    static constexpr int BK = Prec<PREC>::BK;
    static constexpr int VEC = 16 / sizeof(TS);
    // BF16 with contiguous rows: a thread owns a micro-tile of TR rows x TK consecutive k, loaded
    // as TK vectors along the rows and written to the i-major LDS tile as TR runs of TK k values
    // (a register transpose).  Every other case: vectors along the contiguous index.
    static constexpr bool MICRO = (PREC == OMX_PREC_BF16 && CONTIG_R);
    static constexpr int TR = 4, TK = 8;
    static constexpr int NE = ROWS * BK / NT;  // elements per thread
    static constexpr int NV = NE / VEC;
    static_assert(NE % VEC == 0, "slice not divisible into vectors");
    static_assert(!MICRO || (NE == TR * TK && TR % VEC == 0), "micro-tile shape");
    typename Prec<PREC>::lds_t v[NE];

    // Vector q of this thread -> (r, k) of its first element (non-MICRO modes).
    __device__ static inline void coord(int t, int q, int &r, int &k) {
        if constexpr (CONTIG_R) {
            int idx = t + NT * q;
            r = (idx % (ROWS / VEC)) * VEC;
            k = idx / (ROWS / VEC);
        } else {
            int idx = t + NT * q;
            k = (idx % (BK / VEC)) * VEC;
            r = idx / (BK / VEC);
        }
    }
    // MICRO mode: micro-tile origin of thread t.
    __device__ static inline void micro_origin(int t, int &r, int &k) {
        r = (t % (ROWS / TR)) * TR;
        k = (t / (ROWS / TR)) * TK;
    }

    __device__ inline void load(const TS *__restrict__ P, int64_t ld, int r0, int k0, int rlim, int klim, bool vec_ok,
                                int t) {
        if constexpr (MICRO) {
            int r, k;
            micro_origin(t, r, k);
            const int gr = r0 + r;
#pragma unroll
            for (int kk = 0; kk < TK; ++kk) {
                const int gk = k0 + k + kk;
                const TS *src = P + (int64_t)gr + (int64_t)gk * ld;
                TS x[TR];
                if (vec_ok && gr + TR <= rlim && gk < klim && TR % VEC == 0) {
                    typedef TS V __attribute__((ext_vector_type(VEC)));
#pragma unroll
                    for (int h = 0; h < TR / VEC; ++h) {
                        V w = *reinterpret_cast<const V *>(src + h * VEC);
#pragma unroll
                        for (int e = 0; e < VEC; ++e) x[h * VEC + e] = w[e];
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < TR; ++e) x[e] = (gr + e < rlim && gk < klim) ? src[e] : (TS)0;
                }
#pragma unroll
                for (int e = 0; e < TR; ++e) v[e * TK + kk] = to_lds<TS, PREC>(x[e]);
            }
        } else {
#pragma unroll
            for (int q = 0; q < NV; ++q) {
                int r, k;
                coord(t, q, r, k);
                const int gr = r0 + r, gk = k0 + k;
                const bool full = CONTIG_R ? (gr + VEC <= rlim && gk < klim) : (gr < rlim && gk + VEC <= klim);
                const TS *src = CONTIG_R ? P + (int64_t)gr + (int64_t)gk * ld : P + (int64_t)gk + (int64_t)gr * ld;
                TS x[VEC];
                if (vec_ok && full) {
                    typedef TS V __attribute__((ext_vector_type(VEC)));
                    V w = *reinterpret_cast<const V *>(src);
#pragma unroll
                    for (int e = 0; e < VEC; ++e) x[e] = w[e];
                } else {
#pragma unroll
                    for (int e = 0; e < VEC; ++e) {
                        const bool in = CONTIG_R ? (gr + e < rlim && gk < klim) : (gr < rlim && gk + e < klim);
                        x[e] = in ? src[e] : (TS)0;
                    }
                }
#pragma unroll
                for (int e = 0; e < VEC; ++e) v[q * VEC + e] = to_lds<TS, PREC>(x[e]);
            }
        }
    }

    __device__ inline void store(typename Prec<PREC>::lds_t *lds, int t) const {
        if constexpr (MICRO) {
            // one 16-byte write of TK = 8 consecutive k per row of the micro-tile
            int r, k;
            micro_origin(t, r, k);
#pragma unroll
            for (int e = 0; e < TR; ++e) {
                bf8v w;
#pragma unroll
                for (int kk = 0; kk < TK; ++kk) w[kk] = v[e * TK + kk];
                *reinterpret_cast<bf8v *>(&lds[LdsT<PREC, ROWS>::off(r + e, k)]) = w;
            }
        } else {
#pragma unroll
            for (int q = 0; q < NV; ++q) {
                int r, k;
                coord(t, q, r, k);
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    if (CONTIG_R)
                        lds[LdsT<PREC, ROWS>::off(r + e, k)] = v[q * VEC + e];
                    else
                        lds[LdsT<PREC, ROWS>::off(r, k + e)] = v[q * VEC + e];
                }
            }
        }
    }
};

// ---------------------------------------------------------------------------------------------
// MFMA step over one BK slice held in LDS.
// ---------------------------------------------------------------------------------------------
template <int PREC, class CF>
__device__ inline void mma_slice(const typename Prec<PREC>::lds_t *As, const typename Prec<PREC>::lds_t *Bs,
                                 typename Prec<PREC>::accv (&acc)[CF::FBM][CF::FBN], int wm, int wn, int lane) {
    constexpr int BK = Prec<PREC>::BK;
    typedef LdsT<PREC, CF::BM> LA;
    typedef LdsT<PREC, CF::BN> LB;
    const int li = lane & 15, lk = lane >> 4;
    if constexpr (PREC == OMX_PREC_F64 || PREC == OMX_PREC_F32) {
        typedef typename Prec<PREC>::lds_t T;
#pragma unroll
        for (int ks = 0; ks < BK; ks += 4) {
            T a[CF::FBM], b[CF::FBN];
#pragma unroll
            for (int f = 0; f < CF::FBM; ++f) a[f] = As[LA::off(wm * CF::WM + f * 16 + li, ks + lk)];
#pragma unroll
            for (int f = 0; f < CF::FBN; ++f) b[f] = Bs[LB::off(wn * CF::WN + f * 16 + li, ks + lk)];
#pragma unroll
            for (int fm = 0; fm < CF::FBM; ++fm)
#pragma unroll
                for (int fn = 0; fn < CF::FBN; ++fn) {
                    if constexpr (PREC == OMX_PREC_F64)
                        acc[fm][fn] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[fm], b[fn], acc[fm][fn], 0, 0, 0);
                    else
                        acc[fm][fn] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[fm], b[fn], acc[fm][fn], 0, 0, 0);
                }
        }
    } else {
#pragma unroll
        for (int ks = 0; ks < BK; ks += 32) {
            bf8v a[CF::FBM], b[CF::FBN];
#pragma unroll
            for (int f = 0; f < CF::FBM; ++f)
                a[f] = *reinterpret_cast<const bf8v *>(&As[LA::off(wm * CF::WM + f * 16 + li, ks + 8 * lk)]);
#pragma unroll
            for (int f = 0; f < CF::FBN; ++f)
                b[f] = *reinterpret_cast<const bf8v *>(&Bs[LB::off(wn * CF::WN + f * 16 + li, ks + 8 * lk)]);
#pragma unroll
            for (int fm = 0; fm < CF::FBM; ++fm)
#pragma unroll
                for (int fn = 0; fn < CF::FBN; ++fn)
                    acc[fm][fn] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[fm], b[fn], acc[fm][fn], 0, 0, 0);
        }
    }
}

// Pair mode (NPAIR = 2): C := alpha*(A1*B1 + A2*B2) + beta0*C0 + beta*C over a K range made of
// the two contractions back to back (calc_G).  NPAIR = 1: the plain product.
template <typename TS, int PREC, bool TRA, bool TRB, int NPAIR, class CF>
__global__ __launch_bounds__(CF::NT, CF::MINW) void k_gemm(int m, int n, int k, double alpha, const TS *__restrict__ A1,
                                                 const TS *__restrict__ A2, int64_t lda, const TS *__restrict__ B1,
                                                 const TS *__restrict__ B2, int64_t ldb, double beta0,
                                                 const TS *__restrict__ C0, double beta, TS *__restrict__ C,
                                                 int64_t ldc, int k_per_split, int vec_a, int vec_b, int sym,
                                                 typename Prec<PREC>::acc_t *__restrict__ partial,
                                                 const int *__restrict__ mask, int carry) {
    typedef typename Prec<PREC>::lds_t LT;
    typedef typename Prec<PREC>::acc_t AT;
    typedef typename Prec<PREC>::accv AV;
    typedef LdsT<PREC, CF::BM> LA;
    typedef LdsT<PREC, CF::BN> LB;
    constexpr int BK = Prec<PREC>::BK;
    __shared__ LT smem[2 * (LA::ELEMS + LB::ELEMS)];
    if (mask && !*mask) return;  // whole workgroup, before any barrier

    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int wm = wave / CF::WGN, wn = wave % CF::WGN;
    const int tiles_m = (m + CF::BM - 1) / CF::BM, tiles_n = (n + CF::BN - 1) / CF::BN;
    int tm, tn;
    if (sym)
        tile_of_lower(blockIdx.x, tiles_m, tm, tn);
    else
        tile_of(blockIdx.x, tiles_m, tiles_n, tm, tn);
    const int i0 = tm * CF::BM, j0 = tn * CF::BN;

    // K range of this split over the virtual contraction [0, NPAIR*k).
    const int ktot = NPAIR * k;
    const int kb = blockIdx.z * k_per_split;
    const int ke = min(ktot, kb + k_per_split);

    AV acc[CF::FBM][CF::FBN];
#pragma unroll
    for (int a = 0; a < CF::FBM; ++a)
#pragma unroll
        for (int b = 0; b < CF::FBN; ++b) acc[a][b] = AV{0, 0, 0, 0};

    constexpr bool CARRY = PREC == OMX_PREC_F32 && sizeof(TS) == 4;
    AV tot[CARRY ? CF::FBM : 1][CARRY ? CF::FBN : 1];  // (see carry_sums)
    if constexpr (CARRY) {
#pragma unroll
        for (int a = 0; a < CF::FBM; ++a)
#pragma unroll
            for (int b = 0; b < CF::FBN; ++b) tot[a][b] = AV{0, 0, 0, 0};
    }

    Stage<TS, PREC, !TRA, CF::BM, CF::NT> sa;
    Stage<TS, PREC, TRB, CF::BN, CF::NT> sb;

    auto fetch = [&](int kk) {
        // kk is a virtual K index; pick the operand pair it falls in.
        const TS *Ap = A1, *Bp = B1;
        int kl = kk;
        if (NPAIR == 2 && kk >= k) {
            Ap = A2;
            Bp = B2;
            kl = kk - k;
        }
        int klim = min(k, kl + (ke - kk));  // stop at the split end and at the pair end
        sa.load(Ap, lda, i0, kl, m, klim, vec_a != 0, t);
        sb.load(Bp, ldb, j0, kl, n, klim, vec_b != 0, t);
    };

    LT *As0 = smem, *Bs0 = smem + LA::ELEMS;
    LT *As1 = smem + LA::ELEMS + LB::ELEMS, *Bs1 = As1 + LA::ELEMS;

    // In pair mode the host guarantees k % BK == 0, so no slice straddles the pair boundary.
    const int nslices = (ke - kb + BK - 1) / BK;
    if (nslices > 0) {
        fetch(kb);
        sa.store(As0, t);
        sb.store(Bs0, t);
        __syncthreads();
        for (int s = 0; s < nslices; ++s) {
            LT *Ac = (s & 1) ? As1 : As0, *Bc = (s & 1) ? Bs1 : Bs0;
            LT *An = (s & 1) ? As0 : As1, *Bn = (s & 1) ? Bs0 : Bs1;
            const bool more = (s + 1 < nslices);
            if (more) fetch(kb + (s + 1) * BK);
            mma_slice<PREC, CF>(Ac, Bc, acc, wm, wn, lane);
            if constexpr (CARRY) {
                if (carry && (s % 4 == 3 || (NPAIR == 2 && kb + (s + 1) * BK == k))) carry_sums(acc, tot);
            }
            if (more) {
                sa.store(An, t);
                sb.store(Bn, t);
            }
            __syncthreads();
        }
    }

    if constexpr (CARRY) {
#pragma unroll
        for (int a = 0; a < CF::FBM; ++a)
#pragma unroll
            for (int b = 0; b < CF::FBN; ++b) acc[a][b] = tot[a][b] + acc[a][b];
    }
    // Epilogue.  Accumulator v of block (fm, fn) holds column lane%16 and row out_row(lane/16, v).
    const int li = lane & 15, lq = lane >> 4;
#pragma unroll
    for (int fm = 0; fm < CF::FBM; ++fm)
#pragma unroll
        for (int fn = 0; fn < CF::FBN; ++fn) {
            const int j = j0 + wn * CF::WN + fn * 16 + li;
            if (j >= n) continue;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int i = i0 + wm * CF::WM + fm * 16 + Prec<PREC>::out_row(lq, v);
                if (i >= m) continue;
                const AT val = acc[fm][fn][v];
                if (partial) {
                    partial[(int64_t)blockIdx.z * m * n + (int64_t)i + (int64_t)j * m] = val;
                } else {
                    double r = alpha * (double)val;
                    if (C0) r += beta0 * (double)C0[(int64_t)i + (int64_t)j * ldc];
                    if (beta != 0.0) r += beta * (double)C[(int64_t)i + (int64_t)j * ldc];
                    C[(int64_t)i + (int64_t)j * ldc] = (TS)r;
                }
            }
        }
}

// Reduction of split-K partials in split order, then the alpha/beta epilogue.
template <typename TS, typename AT>
__global__ void k_splitk_reduce(int m, int n, int splits, const AT *__restrict__ partial, double alpha, double beta0,
                                const TS *__restrict__ C0, double beta, TS *__restrict__ C, int64_t ldc) {
    int64_t total = (int64_t)m * n;
    for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < total; q += (int64_t)gridDim.x * blockDim.x) {
        int64_t i = q % m, j = q / m;
        AT s = partial[q];
        for (int z = 1; z < splits; ++z) s += partial[(int64_t)z * total + q];
        double r = alpha * (double)s;
        if (C0) r += beta0 * (double)C0[i + j * ldc];
        if (beta != 0.0) r += beta * (double)C[i + j * ldc];
        C[i + j * ldc] = (TS)r;
    }
}

static bool aligned16(const void *p) { return ((uintptr_t)p & 15) == 0; }

template <typename TS, int PREC, bool TRA, bool TRB, int NPAIR, class CF>
static int run_cfg(omx_ctx ctx, int m, int n, int k, double alpha, const TS *A1, const TS *A2, int64_t lda,
                   const TS *B1, const TS *B2, int64_t ldb, double beta0, const TS *C0, double beta, TS *C,
                   int64_t ldc) {
    typedef typename Prec<PREC>::acc_t AT;
    constexpr int BK = Prec<PREC>::BK;
    constexpr int VEC = 16 / sizeof(TS);
    const int tiles = ((m + CF::BM - 1) / CF::BM) * ((n + CF::BN - 1) / CF::BN);
    const int ktot = NPAIR * k;
    // Split K when the tile count cannot fill the chip (aim for >= 2 workgroups per CU), or as the direct-to-LDS
    // kernel splits where that adds in the same way (FP64 small results reach this kernel only by leading dimensions
    // beyond 2^20).
    int splits = 1;
    const int target = 2 * ctx->num_cus;
    constexpr bool f64 = PREC == OMX_PREC_F64 && sizeof(TS) == 8, f32 = PREC == OMX_PREC_F32 && sizeof(TS) == 4;
    if ((f64 && !carries64(ctx, m, n)) || f32) {
        splits = dgemm_k_splits(ctx, m, n, (ktot + BK - 1) / BK, PREC == OMX_PREC_F64 ? 8 : 4);
    } else if (tiles < target && !ctx->launch_mask) {
        int max_splits = std::max(1, ktot / (4 * BK));
        splits = std::min(max_splits, (target + tiles - 1) / tiles);
        splits = std::max(1, std::min(splits, 64));
    }
    int kps = (ktot + splits - 1) / splits;
    kps = (kps + BK - 1) / BK * BK;  // slices never straddle a split
    splits = (ktot + kps - 1) / kps;
    AT *partial = nullptr;
    if (splits > 1) {
        size_t bytes = sizeof(AT) * (size_t)splits * m * n;
        int rc = ensure_ws(ctx, bytes);
        if (rc) return rc;
        partial = (AT *)ctx->ws;
    }
    const int vec_a = (lda % VEC == 0) && aligned16(A1) && aligned16(A2);
    const int vec_b = (ldb % VEC == 0) && aligned16(B1) && aligned16(B2);
    // products known to be symmetric (omx_gemm_sym): lower-triangle tiles only, when one split
    // covers K and the tiles are square
    const int tiles_m = (m + CF::BM - 1) / CF::BM;
    const bool sym = ctx->gemm_sym && m == n && CF::BM == CF::BN && splits == 1;
    const int grid = sym ? tiles_m * (tiles_m + 1) / 2 : tiles;
    hipEvent_t ev;
    prof_begin(ctx, NPAIR == 2 ? OMX_K_GEMM_PAIR : OMX_K_GEMM, &ev);
    prof_work(ctx, NPAIR == 2 ? OMX_K_GEMM_PAIR : OMX_K_GEMM, 2.0 * (sym ? sym_area(m, CF::BM) : (double)m * n) * (double)ktot,
              sizeof(TS) * ((double)NPAIR * ((double)m * k + (double)k * n) +
                            (double)m * n * (1 + (C0 ? 1 : 0) + (beta != 0.0 ? 1 : 0))));
    hipLaunchKernelGGL((k_gemm<TS, PREC, TRA, TRB, NPAIR, CF>), dim3(grid, 1, splits), dim3(CF::NT), 0, ctx->stream,
                       m, n, k, alpha, A1, A2, lda, B1, B2, ldb, beta0, C0, beta, C, ldc, kps, vec_a, vec_b, (int)sym,
                       partial, ctx->launch_mask, (int)carries(ctx, m, n));
    if (splits > 1) {
        int64_t total = (int64_t)m * n;
        int grid = (int)std::min<int64_t>((total + 255) / 256, 8192);
        hipLaunchKernelGGL((k_splitk_reduce<TS, AT>), dim3(grid), dim3(256), 0, ctx->stream, m, n, splits, partial,
                           alpha, beta0, C0, beta, C, ldc);
    }
    prof_end(ctx, NPAIR == 2 ? OMX_K_GEMM_PAIR : OMX_K_GEMM, ev);
    OMX_CHECK_HIP(hipGetLastError());
    return OMX_OK;
}

// Tile configurations that apply to a product: FP64 products with A not transposed ('n','t' Grams,
// 'n','n' products and the calc_G pair) carry 0-3 and 5-7 (7 on FP64 storage); the BF16 Grams and pairs on
// FP32 storage 0 and 4, FP32 products on FP32 storage 0 and 7; every other product uses 0.
template <typename TS, int PREC, bool TRA, bool TRB, int NPAIR>
struct CfgSet {
    static constexpr bool f64 = (PREC == OMX_PREC_F64) && !TRA;
    static constexpr bool dl = (PREC == OMX_PREC_F64) && std::is_same<TS, double>::value;
    static constexpr bool lowp = (PREC == OMX_PREC_BF16) && std::is_same<TS, float>::value && !TRA && (TRB || NPAIR == 2);
    static constexpr bool sdl = (PREC == OMX_PREC_F32) && std::is_same<TS, float>::value;
    static std::vector<int> ids() {
        if (dl && f64) return {7, 0, 1, 2, 3, 5, 6};
        if (dl) return {7, 0};
        if (sdl) return {7, 0};
        if (lowp) return {0, 4};
        return {0};
    }
};

template <typename TS, int PREC, bool TRA, bool TRB, int NPAIR>
static int run_cfg_id(int id, omx_ctx ctx, int m, int n, int k, double alpha, const TS *A1, const TS *A2,
                      int64_t lda, const TS *B1, const TS *B2, int64_t ldb, double beta0, const TS *C0, double beta,
                      TS *C, int64_t ldc) {
    typedef CfgSet<TS, PREC, TRA, TRB, NPAIR> CS;
    if constexpr (CS::dl) {
        if (id == 7) {
            int rc = launch_dgemm(ctx, TRA, TRB, NPAIR, m, n, k, alpha, A1, A2, lda, B1, B2, ldb, beta0, C0, ldc, beta,
                                  C, ldc);
            if (rc != OMX_ERR_UNSUPPORTED) return rc;
            id = 5;  // the staged kernel (5 tiles; 0 with A transposed) for leading dimensions beyond 2^20
        }
    }
    if constexpr (CS::f64) {
        switch (id) {
            case 1:
                return run_cfg<TS, PREC, TRA, TRB, NPAIR, Cfg1>(ctx, m, n, k, alpha, A1, A2, lda, B1, B2, ldb, beta0,
                                                                C0, beta, C, ldc);
            case 2:
                return run_cfg<TS, PREC, TRA, TRB, NPAIR, Cfg2>(ctx, m, n, k, alpha, A1, A2, lda, B1, B2, ldb, beta0,
                                                                C0, beta, C, ldc);
            case 3:
                return run_cfg<TS, PREC, TRA, TRB, NPAIR, Cfg3>(ctx, m, n, k, alpha, A1, A2, lda, B1, B2, ldb, beta0,
                                                                C0, beta, C, ldc);
            case 5:
                return run_cfg<TS, PREC, TRA, TRB, NPAIR, Cfg5>(ctx, m, n, k, alpha, A1, A2, lda, B1, B2, ldb, beta0,
                                                                C0, beta, C, ldc);
            case 6:
                return run_cfg<TS, PREC, TRA, TRB, NPAIR, Cfg6>(ctx, m, n, k, alpha, A1, A2, lda, B1, B2, ldb, beta0,
                                                                C0, beta, C, ldc);
            default:
                break;
        }
    }
    if constexpr (CS::sdl) {
        if (id == 7) {
            int rc = launch_sgemm(ctx, TRA, TRB, NPAIR, m, n, k, alpha, A1, A2, lda, B1, B2, ldb, beta0, C0, beta, C, ldc);
            if (rc != OMX_ERR_UNSUPPORTED) return rc;
            id = 0;  // the staged kernel for leading dimensions beyond 2^20
        }
    }
    if constexpr (CS::lowp) {
        if (id == 4)
            return run_cfg<TS, PREC, TRA, TRB, NPAIR, Cfg4>(ctx, m, n, k, alpha, A1, A2, lda, B1, B2, ldb, beta0, C0,
                                                            beta, C, ldc);
    }
    return run_cfg<TS, PREC, TRA, TRB, NPAIR, Cfg0>(ctx, m, n, k, alpha, A1, A2, lda, B1, B2, ldb, beta0, C0, beta,
                                                    C, ldc);
}

// Autotuner: the first time a product shape is seen with tuning on, every applicable tile
// configuration is timed (one warm-up and one timed launch each, with HIP events on the library
// stream, into a scratch result so the caller's C is untouched) and the fastest is remembered for
// that shape on this context.  Tuning synchronises and allocates, so it must not run under graph
// capture.
template <typename TS, int PREC, bool TRA, bool TRB, int NPAIR>
static int tuned_cfg(omx_ctx ctx, int m, int n, int k, const TS *A1, const TS *A2, int64_t lda, const TS *B1,
                     const TS *B2, int64_t ldb, int &out) {
    typedef CfgSet<TS, PREC, TRA, TRB, NPAIR> CS;
    char key[128];
    snprintf(key, sizeof key, "gemm prec=%d es=%d op=%c%c pair=%d m=%d n=%d k=%d", PREC, (int)sizeof(TS),
             TRA ? 't' : 'n', TRB ? 't' : 'n', NPAIR, m, n, k);
    auto it = ctx->tune_gemm.find(key);
    if (it != ctx->tune_gemm.end()) {
        out = it->second.first;
        return OMX_OK;
    }
    std::vector<int> ids = CS::ids();
    if (CS::dl && carries64(ctx, m, n)) ids = {7};
    if (ids.size() == 1) {
        ctx->tune_gemm[key] = {ids[0], 0.0};
        out = ids[0];
        return OMX_OK;
    }
    TS *tmp = nullptr;
    OMX_CHECK_HIP(dev_malloc((void **)&tmp, sizeof(TS) * (size_t)std::max(m, 1) * std::max(n, 1)));
    hipEvent_t e0, e1;
    OMX_CHECK_HIP(hipEventCreate(&e0));
    OMX_CHECK_HIP(hipEventCreate(&e1));
    const bool prof = ctx->prof_on;
    const int sym = ctx->gemm_sym;
    ctx->prof_on = false;
    int best = ids[0], rc = OMX_OK;
    float best_ms = 0.0f;
    for (int id : ids) {
        float ms = 0.0f;
        for (int rep = 0; rep < 2 && rc == OMX_OK; ++rep) {
            (void)hipEventRecord(e0, ctx->stream);
            rc = run_cfg_id<TS, PREC, TRA, TRB, NPAIR>(id, ctx, m, n, k, 1.0, A1, A2, lda, B1, B2, ldb, 0.0, nullptr,
                                                       0.0, tmp, std::max(m, 1));
            ctx->gemm_sym = sym;
            (void)hipEventRecord(e1, ctx->stream);
            (void)hipEventSynchronize(e1);
            (void)hipEventElapsedTime(&ms, e0, e1);
        }
        if (rc) break;
        if (id == ids[0] || ms < best_ms) {
            best = id;
            best_ms = ms;
        }
    }
    ctx->prof_on = prof;
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    (void)hipFree(tmp);
    if (rc) return rc;
    ctx->tune_gemm[key] = {best, (double)best_ms};
    out = best;
    return OMX_OK;
}

template <typename TS, int PREC, bool TRA, bool TRB, int NPAIR>
static int run_gemm(omx_ctx ctx, int m, int n, int k, double alpha, const TS *A1, const TS *A2, int64_t lda,
                    const TS *B1, const TS *B2, int64_t ldb, double beta0, const TS *C0, double beta, TS *C,
                    int64_t ldc) {
    // default: the direct-to-LDS kernel for FP64 products on FP64 storage and FP32 ones on FP32 storage (past leading
    // dimensions of 2^20 it hands over to the staged 8-wave tile 5, or 0), 0 otherwise
    typedef CfgSet<TS, PREC, TRA, TRB, NPAIR> CS;
    int id = (CS::dl || CS::sdl) ? 7 : 0;
    if (ctx->gemm_cfg >= 0) {
        id = ctx->gemm_cfg;  // forced (omx_gemm_set_tile); a configuration that does not apply falls back to 0
    } else if (ctx->autotune) {
        int rc = tuned_cfg<TS, PREC, TRA, TRB, NPAIR>(ctx, m, n, k, A1, A2, lda, B1, B2, ldb, id);
        if (rc) return rc;
    }
    // 7 alone carries its sums in FP64 (a masked launch may have left another choice for the shape)
    if (CS::dl && carries64(ctx, m, n)) id = 7;
    return run_cfg_id<TS, PREC, TRA, TRB, NPAIR>(id, ctx, m, n, k, alpha, A1, A2, lda, B1, B2, ldb, beta0, C0, beta,
                                                 C, ldc);
}

// ---------------------------------------------------------------------------------------------
// BF16 products of FP32 matrices through k-contiguous BF16 copies, for every m, n, k (k is padded with
// zeros to whole slices: 5488 x 5488 x 10976 2.03 -> 0.72 ms, 250 x 250 x 500 44 -> 16 us, against the
// staged kernel, which reads and rounds the FP32 operands again for every tile).
//
// The operands are first rounded to BF16 (round to nearest even, the same rounding as the
// staging conversion of k_gemm) into k-contiguous panels: op(A) as At[kk + i*K] and op(B) as
// Bt[kk + j*K].  The GEMM then moves half the bytes of FP32 operands, loads 16-byte vectors of 8
// consecutive k straight into the i-major LDS tiles, and skips the per-tile conversion.  With
// split = true each operand is also written as a second BF16 term, lo = bf16(a - hi), and the
// product runs over a K three times longer, [Ah Ah Al] x [Bh; Bl; Bh]: hi*hi + hi*lo + lo*hi,
// which keeps about 16 significant bits of each operand (the BF16x3 product).
// ---------------------------------------------------------------------------------------------

constexpr int BG_T = 64;  // conversion tile (rows x cols)

// The terms each k block of a panel holds, A's and B's (1 = hi = bf16(a), 2 = mid = bf16(a - hi), 3 = lo =
// bf16(a - hi - mid), each difference taken exactly in the source precision).  For FP32 sources hi +
// mid + lo is the value exactly; hi + mid keeps about 16 significant bits.  NS = 1: BF16; 2: BF16x3;
// 3: BF16x6 (the term products in order, smallest first).
template <int NS>
struct BgTerms;
template <>
struct BgTerms<1> {
    static constexpr int n = 1;
    static constexpr int of[2][1] = {{1}, {1}};
};
template <>
struct BgTerms<2> {
    static constexpr int n = 3;
    static constexpr int of[2][3] = {{1, 1, 2}, {1, 2, 1}};
};
template <>
struct BgTerms<3> {
    static constexpr int n = 6;
    static constexpr int of[2][6] = {{1, 3, 2, 1, 2, 1}, {3, 1, 2, 2, 1, 1}};
};

// One operand's conversion: src (rows x cols, ld lds) into the panel at dst, whose rows (ld ldd) hold
// the k blocks of length kp one after another.  trans: element (r, c) goes to dst[c + r*ldd] (k runs
// along the columns), else to dst[r + c*ldd] (k runs along the rows).
struct BgJob {
    const void *src;
    int64_t lds;
    __bf16 *dst;
    int rows, cols, trans, side;  // side: 0 = A, 1 = B
    int first, nbx;               // first workgroup and workgroups along the rows
};
struct BgJobs {
    BgJob j[4];
    int n, kp;
    int64_t ldd;
};

// All conversions of a product in one launch (a launch each costs 2-3 us, as much as a small product),
// each value rounded once from the stored one.  One 64 x 64 tile per workgroup: 16-byte loads along
// the rows, and 16-byte stores of 8 BF16 along k (through an LDS transpose for trans); k is padded with
// zeros up to kp (a multiple of 64, so every store is whole and aligned).  Edges and unaligned operands
// load element by element.
template <typename TS, int NS>
__global__ __launch_bounds__(256) void k_to_bf16(BgJobs jobs) {
    typedef BgTerms<NS> TT;
    constexpr int VEC = 16 / sizeof(TS);  // elements per 16-byte load
    __shared__ TS tile[BG_T][BG_T + 1];   // [c][r]
    int q = 0;
    while (q + 1 < jobs.n && (int)blockIdx.x >= jobs.j[q + 1].first) ++q;
    const BgJob job = jobs.j[q];
    const int t = threadIdx.x, w = blockIdx.x - job.first, kp = jobs.kp, rows = job.rows, cols = job.cols;
    const int64_t ldd = jobs.ldd;
    const TS *src = (const TS *)job.src;
    const int r0 = (w % job.nbx) * BG_T, c0 = (w / job.nbx) * BG_T;
    const bool vld = (job.lds % VEC) == 0 && ((uintptr_t)src & 15) == 0;
    auto load = [&](int gr, int gc, int count, TS *x) {  // x[0..count) = src(gr.., gc), zero outside
        const TS *p = src + (int64_t)gr + (int64_t)gc * job.lds;
        if (vld && gc < cols && gr + count <= rows) {
#pragma unroll
            for (int e = 0; e < count; e += VEC) {
                typedef TS vec_t __attribute__((ext_vector_type(VEC)));
                const vec_t v = *reinterpret_cast<const vec_t *>(p + e);
#pragma unroll
                for (int h = 0; h < VEC; ++h) x[e + h] = v[h];
            }
        } else {
#pragma unroll
            for (int e = 0; e < count; ++e) x[e] = (gc < cols && gr + e < rows) ? p[e] : (TS)0;
        }
    };
    auto store8 = [&](const TS *x, int64_t off) {  // the terms of 8 values to every k block
        bf8v t1, t2, t3;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const __bf16 h = (__bf16)x[e];
            const TS r1 = x[e] - (TS)h;
            const __bf16 md = (__bf16)r1;
            t1[e] = h;
            t2[e] = md;
            t3[e] = (__bf16)(r1 - (TS)md);
        }
#pragma unroll
        for (int b = 0; b < TT::n; ++b) {
            const int tb = job.side ? TT::of[1][b] : TT::of[0][b];
            *reinterpret_cast<bf8v *>(job.dst + off + (int64_t)b * kp) = tb == 1 ? t1 : (tb == 2 ? t2 : t3);
        }
    };
    if (job.trans) {
        constexpr int VPC = BG_T / VEC;  // load vectors per tile column
        for (int v = t; v < BG_T * VPC; v += 256) {
            const int c = v / VPC, rv = (v % VPC) * VEC;
            TS x[VEC];
            load(r0 + rv, c0 + c, VEC, x);
#pragma unroll
            for (int e = 0; e < VEC; ++e) tile[c][rv + e] = x[e];
        }
        __syncthreads();
        for (int u = t; u < BG_T * (BG_T / 8); u += 256) {
            const int r = u / (BG_T / 8), c8 = (u % (BG_T / 8)) * 8;
            if (r0 + r >= rows || c0 + c8 >= kp) continue;
            TS x[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = tile[c8 + e][r];
            store8(x, (int64_t)(c0 + c8) + (int64_t)(r0 + r) * ldd);
        }
    } else {
        for (int u = t; u < BG_T * (BG_T / 8); u += 256) {
            const int c = u / (BG_T / 8), r8 = (u % (BG_T / 8)) * 8;
            if (r0 + r8 >= kp || c0 + c >= cols) continue;
            TS x[8];
            load(r0 + r8, c0 + c, 8, x);
            store8(x, (int64_t)(r0 + r8) + (int64_t)(c0 + c) * ldd);
        }
    }
}

// LDS tile of the BF16 panel product: i-major rows of BK = 64 BF16 (128 bytes, 8 chunks of 16 B),
// no padding.  Logical chunk c of row r is stored at physical chunk c ^ bg_swz(r).  A fragment
// read takes one chunk of 16 consecutive rows; with this swizzle those 16 reads cover 16
// distinct 16-byte bank groups, so the read is free of bank conflicts.
__device__ inline int bg_swz(int r) { return (r & 7) ^ ((r >> 3) & 1); }


// One BK = 64 slice of the BF16 panel product, software-pipelined: the wave's MFMAs run in groups
// (one A fragment x the FBN B fragments of a 32-wide k step), and the LDS reads for group g + LEAD
// are issued before the MFMAs of group g, so that LEAD groups of reads are in flight behind the
// matrix core (the waits become lgkmcnt(n > 0) instead of a full drain after every read).  The
// scheduling fences keep the compiler from regrouping the reads.
template <class CF, int LEAD>
__device__ inline void mma_slice_bf16_pipe(const __bf16 *As, const __bf16 *Bs, f4v (&acc)[CF::FBM][CF::FBN], int wm,
                                           int wn, int lane) {
    constexpr int BK = Prec<OMX_PREC_BF16>::BK, NKS = BK / 32, NG = NKS * CF::FBM;
    const int li = lane & 15, lk = lane >> 4;
    bf8v fa[NKS][CF::FBM], fb[NKS][CF::FBN];
#pragma unroll
    for (int g = -LEAD; g < NG; ++g) {
        const int lg = g + LEAD;
        if (lg >= 0 && lg < NG) {
            const int ks = lg / CF::FBM, fm = lg % CF::FBM;
            const int c = ks * 4 + lk;  // logical 16-byte chunk: k = 8c .. 8c+7
            if (fm == 0) {
#pragma unroll
                for (int f = 0; f < CF::FBN; ++f) {
                    const int r = wn * CF::WN + f * 16 + li;
                    fb[ks][f] = *reinterpret_cast<const bf8v *>(&Bs[r * BK + (c ^ bg_swz(r)) * 8]);
                }
            }
            const int r = wm * CF::WM + fm * 16 + li;
            fa[ks][fm] = *reinterpret_cast<const bf8v *>(&As[r * BK + (c ^ bg_swz(r)) * 8]);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (g >= 0) {
            const int ks = g / CF::FBM, fm = g % CF::FBM;
#pragma unroll
            for (int fn = 0; fn < CF::FBN; ++fn)
                acc[fm][fn] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[ks][fm], fb[ks][fn], acc[fm][fn], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// C := alpha * sum_kk At[kk + i*lda] * Bt[kk + j*ldb] + beta0*C0 + beta*C over kk < K (K % 64 == 0,
// lda, ldb multiples of 8, 16-byte aligned panels), FP32 accumulation; C, C0 of type TO (the
// storage type, FP32 or FP64).
//
// Operand rows go straight from the panels into LDS: one buffer_load_dwordx4 ... lds per wave moves
// 8 rows of a slice (1 KB, lane l landing at byte 16*l), each lane fetching the logical chunk that
// belongs at its physical position under bg_swz.  No staging registers and no LDS write
// instructions; two LDS stages, the loads of slice s+1 in flight while slice s feeds the MFMAs.
// The buffer form rather than global_load_lds: while a FLAT-encoded load into LDS is in flight the
// compiler's wait insertion cannot count LDS reads in order and drains every one of them
// (lgkmcnt(0)) before each use, which serialises the fragment reads the slice pipeline issues ahead;
// with the buffer form the waits count only the reads a group needs.  Requires BM * K * 2 bytes
// below 2^31 (byte offsets inside the tile's rows are 32-bit).
// Rows past m or n are fetched from the last valid row and their results are not stored.
template <class CF, typename TO>
__global__ __launch_bounds__(CF::NT, CF::MINW) void k_bgemm_tn(int m, int n, int K, double alpha,
                                                     const __bf16 *__restrict__ At, int64_t lda,
                                                     const __bf16 *__restrict__ Bt, int64_t ldb, double beta0,
                                                     const TO *__restrict__ C0, double beta, TO *__restrict__ C,
                                                     int64_t ldc, int sym, int kps,
                                                     float *__restrict__ partial) {
    constexpr int BK = Prec<OMX_PREC_BF16>::BK;
    constexpr int NW = CF::WGM * CF::WGN;
    constexpr int INS = (CF::BM + CF::BN) / 8;  // wave loads per slice, 8 rows each
    constexpr int LPW = INS / NW;
    constexpr int STAGE = (CF::BM + CF::BN) * BK;  // BF16 per LDS stage
    static_assert(LPW * NW == INS && CF::BM % 8 == 0, "rows per wave");
    __shared__ __bf16 smem[2 * STAGE];

    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int wm = wave / CF::WGN, wn = wave % CF::WGN;
    const int tiles_m = (m + CF::BM - 1) / CF::BM, tiles_n = (n + CF::BN - 1) / CF::BN;
    int tm, tn;
    if (sym)
        tile_of_lower(blockIdx.x, tiles_m, tm, tn);
    else
        tile_of(blockIdx.x, tiles_m, tiles_n, tm, tn);
    const int i0 = tm * CF::BM, j0 = tn * CF::BN;

    f4v acc[CF::FBM][CF::FBN];
#pragma unroll
    for (int a = 0; a < CF::FBM; ++a)
#pragma unroll
        for (int b = 0; b < CF::FBN; ++b) acc[a][b] = f4v{0, 0, 0, 0};

    // Buffer descriptors over the tile's A rows and B rows; each lane's byte offset of its chunk
    // in slice 0 is fixed for the whole K loop (slice s adds 2*s*BK).
    const __amdgpu_buffer_rsrc_t ra = raw_rsrc(At + (int64_t)i0 * lda, (int)(2 * ((int64_t)min(CF::BM, m - i0) * lda)));
    const __amdgpu_buffer_rsrc_t rb = raw_rsrc(Bt + (int64_t)j0 * ldb, (int)(2 * ((int64_t)min(CF::BN, n - j0) * ldb)));
    const int uwave = __builtin_amdgcn_readfirstlane(wave);
    int voff[LPW];
#pragma unroll
    for (int q = 0; q < LPW; ++q) {
        const int ins = uwave * LPW + q;       // A rows first, then B rows
        const int rr = ins * 8 + (lane >> 3);  // tile row this lane fills
        const int p = lane & 7;                // physical chunk it fills
        if (ins * 8 < CF::BM)
            voff[q] = 2 * (int)(min(rr, m - 1 - i0) * lda + (p ^ bg_swz(rr)) * 8);
        else
            voff[q] = 2 * (int)(min(rr - CF::BM, n - 1 - j0) * ldb + (p ^ bg_swz(rr - CF::BM)) * 8);
    }
    const int s0 = blockIdx.z * kps, nslices = min(K / BK - s0, kps);  // this part of K, in slices
    auto issue = [&](int s) {
        __bf16 *st = smem + (s & 1) * STAGE;
        const int kb = 2 * (s0 + s) * BK;
#pragma unroll
        for (int q = 0; q < LPW; ++q) {
            const int ins = uwave * LPW + q;
            const int vo = voff[q] + kb;
            // An if over two calls, and the offset in a local: with a conditional expression over the
            // two descriptors, or an array element in the argument, the host compilation pass drops
            // the kernel's launch stub without a diagnostic (build.sh checks for that).
            if (ins * 8 < CF::BM)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_void *)(st + ins * 8 * BK), 16, vo, 0, 0, 0);
            else
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_void *)(st + ins * 8 * BK), 16, vo, 0, 0, 0);
        }
    };

    if (nslices > 0) issue(0);
    for (int s = 0; s < nslices; ++s) {
        __builtin_amdgcn_s_waitcnt(waitcnt_vmcnt(0));  // this wave's rows of slice s have landed
        __syncthreads();                               // everyone's have; slice s-1 is no longer read
        if (s + 1 < nslices) issue(s + 1);
        const __bf16 *As = smem + (s & 1) * STAGE, *Bs = As + CF::BM * BK;
        mma_slice_bf16_pipe<CF, 2>(As, Bs, acc, wm, wn, lane);
    }

    const int li = lane & 15, lq = lane >> 4;
#pragma unroll
    for (int fm = 0; fm < CF::FBM; ++fm)
#pragma unroll
        for (int fn = 0; fn < CF::FBN; ++fn) {
            const int j = j0 + wn * CF::WN + fn * 16 + li;
            if (j >= n) continue;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int i = i0 + wm * CF::WM + fm * 16 + Prec<OMX_PREC_BF16>::out_row(lq, v);
                if (i >= m) continue;
                if (partial) {  // a part of K: reduced in part order later
                    partial[(int64_t)blockIdx.z * m * n + (int64_t)i + (int64_t)j * m] = acc[fm][fn][v];
                    continue;
                }
                double r = alpha * (double)acc[fm][fn][v];
                if (C0) r += beta0 * (double)C0[(int64_t)i + (int64_t)j * ldc];
                if (beta != 0.0) r += beta * (double)C[(int64_t)i + (int64_t)j * ldc];
                C[(int64_t)i + (int64_t)j * ldc] = (TO)r;
            }
        }
}

// One operand term of a BF16 panel product: op(X) with X rows x cols (ld ldx); as a k-contiguous
// panel it is `extent` x K (extent = m for A, n for B).
struct BgTerm {
    const void *X;  // FP32 or FP64 (the product's storage type)
    int64_t ldx;
    bool trans;  // true: X is stored K x extent (already k-contiguous)
};

// The job of one operand (extent x k as a panel): the columns of X hold k where X is transposed.
static void bg_job(BgJobs &jobs, int &grid, const BgTerm &tm, int extent, int k, int side, __bf16 *dst) {
    BgJob &j = jobs.j[jobs.n++];
    j = BgJob{tm.X, tm.ldx, dst, tm.trans ? k : extent, tm.trans ? extent : k, !tm.trans, side, grid, 0};
    const int along_r = tm.trans ? jobs.kp : extent, along_c = tm.trans ? extent : jobs.kp;
    j.nbx = (along_r + BG_T - 1) / BG_T;
    grid += j.nbx * ((along_c + BG_T - 1) / BG_T);
}

// Tile (256: 8 waves of 128x64, 128: 4 waves of 64x64, two workgroups per CU) and the parts K is split
// into: the least of rounds of workgroups over the CUs times the 64-wide slices of a part, plus the
// reduction of the parts.  Slice times (us) measured on Grams and gradients of 2662 to 5488 states, alone
// with one workgroup on a CU; over 34 products of 54 to 5488 states the choice is within 3 % of the
// fastest of both tiles and 1 to 8 parts on average.  A 256 tile moves half the bytes per operation, a 128
// tile leaves less of the chip idle in the last round: 4394 states 0.46 ms against 0.53, 5488 0.89
// against 0.72.  The choice depends on the full product's shape alone, so a symmetric product adds as the
// full one does.
static void bg_shape(omx_ctx ctx, int m, int n, int slices, int &tile, int &splits) {
    const int edge[2] = {256, 128};
    const double slice[2] = {1.75, 0.565}, alone[2] = {1.75, 0.77};
    double cost = 0.0;
    tile = 0;
    for (int q = 0; q < 2; ++q)
        for (int s : {1, 2, 3, 4, 6, 8}) {
            if (s > 1 && slices < 2 * s) break;
            const int64_t tiles = (int64_t)((m + edge[q] - 1) / edge[q]) * ((n + edge[q] - 1) / edge[q]) * s;
            const int64_t rounds = (tiles + ctx->num_cus - 1) / ctx->num_cus;
            const double c = std::max(slice[q] * rounds, alone[q]) * ((slices + s - 1) / s) +
                             (s > 1 ? 3.5 + 4e-6 * (s + 1) * m * n / 4.5 : 0.0);
            if (!tile || c < cost) {
                tile = edge[q];
                splits = s;
                cost = c;
            }
        }
}

// C := alpha * sum_t op(A_t) op(B_t) + beta0*C0 + beta*C for nterm products of inner size k on
// TS storage (FP32 or FP64) through k-contiguous BF16 panels in the workspace.  nsplit = 1: BF16
// operands.  nsplit = 2 (BF16x3): hi*hi + hi*mid + mid*hi, about 16 significant bits per operand.
// nsplit = 3 (BF16x6): the six term products of order >= 2^-16 of the operands' three-term splits,
// smallest first (hi*lo + lo*hi + mid*mid + hi*mid + mid*hi + hi*hi), FP32-grade products.
// Returns OMX_ERR_UNSUPPORTED (nothing launched) when the shape does not suit the panels.
template <typename TS>
static int bgemm_panels(omx_ctx ctx, int m, int n, int k, int nterm, const BgTerm *A, const BgTerm *B, int nsplit,
                        double alpha, double beta0, const TS *C0, double beta, TS *C, int64_t ldc) {
    constexpr int BK = Prec<OMX_PREC_BF16>::BK;
    if (ctx->launch_mask) return OMX_ERR_UNSUPPORTED;
    // the split products run in FP32 outside these shapes; BF16 takes any
    if (nsplit > 1 && (k % BK != 0 || m < 256 || n < 256 || k < 4 * BK)) return OMX_ERR_UNSUPPORTED;
    const int kp = (k + BK - 1) / BK * BK;  // each k block of a panel ends in zeros up to a whole slice
    static const int nblk[3] = {1, 3, 6};  // k blocks per product term
    OMX_REQUIRE(nsplit >= 1 && nsplit <= 3, "bf16 panels: split %d", nsplit);
    const int reps = nblk[nsplit - 1];
    const int64_t K = (int64_t)kp * nterm * reps;
    if ((int64_t)Cfg4::BM * K * (int64_t)sizeof(__bf16) >= (1LL << 31)) return OMX_ERR_UNSUPPORTED;  // 32-bit offsets
    const size_t bytes_a = sizeof(__bf16) * (size_t)K * m, bytes_b = sizeof(__bf16) * (size_t)K * n;
    int tile, splits;
    bg_shape(ctx, m, n, (int)(K / BK), tile, splits);
    const int kps = ((int)(K / BK) + splits - 1) / splits;
    splits = ((int)(K / BK) + kps - 1) / kps;
    const size_t panels = (bytes_a + 255) / 256 * 256 + (bytes_b + 255) / 256 * 256;
    int rc = ensure_ws(ctx, panels + (splits > 1 ? sizeof(float) * (size_t)splits * m * n : 0));
    if (rc == OMX_ERR_NOMEM && nsplit == 1) {  // no room for the panels: the staged kernel
        clear_error();
        return OMX_ERR_UNSUPPORTED;
    }
    if (rc) return rc;
    float *partial = splits > 1 ? (float *)((char *)ctx->ws + panels) : nullptr;
    __bf16 *At = (__bf16 *)ctx->ws;
    __bf16 *Bt = (__bf16 *)((char *)ctx->ws + ((bytes_a + 255) / 256) * 256);
    const bool sym = ctx->gemm_sym && m == n && nterm == 1;  // lower-triangle tiles of a symmetric product
    hipEvent_t ev;
    prof_begin(ctx, nterm == 2 ? OMX_K_GEMM_PAIR : OMX_K_GEMM, &ev);
    prof_work(ctx, nterm == 2 ? OMX_K_GEMM_PAIR : OMX_K_GEMM,
              2.0 * (sym ? sym_area(m, tile) : (double)m * n) * (double)k * nterm,
              sizeof(TS) * (nterm * ((double)m * k + (double)k * n) + (double)m * n * (1 + (C0 ? 1 : 0) + (beta != 0.0))));
    // Rows of At are m panels of length K (ld K), rows of Bt n of length K; product term tt takes
    // the K range [tt*reps*k, (tt+1)*reps*k), block b of it holding the A and B terms of pair b.
    BgJobs jobs{};
    jobs.kp = kp;
    jobs.ldd = K;
    int cgrid = 0;
    for (int tt = 0; tt < nterm; ++tt) {
        bg_job(jobs, cgrid, A[tt], m, k, 0, At + (int64_t)tt * reps * kp);
        bg_job(jobs, cgrid, B[tt], n, k, 1, Bt + (int64_t)tt * reps * kp);
    }
    if (nsplit == 1)
        hipLaunchKernelGGL((k_to_bf16<TS, 1>), dim3(cgrid), dim3(256), 0, ctx->stream, jobs);
    else if (nsplit == 2)
        hipLaunchKernelGGL((k_to_bf16<TS, 2>), dim3(cgrid), dim3(256), 0, ctx->stream, jobs);
    else
        hipLaunchKernelGGL((k_to_bf16<TS, 3>), dim3(cgrid), dim3(256), 0, ctx->stream, jobs);
    {
        const int tm = (m + tile - 1) / tile, tn = (n + tile - 1) / tile;
        const dim3 grid(sym ? tm * (tm + 1) / 2 : tm * tn, 1, splits);
        if (tile == 256)
            hipLaunchKernelGGL((k_bgemm_tn<Cfg4, TS>), grid, dim3(Cfg4::NT), 0, ctx->stream, m, n, (int)K, alpha, At, K,
                               Bt, K, beta0, C0, beta, C, ldc, (int)sym, kps, partial);
        else
            hipLaunchKernelGGL((k_bgemm_tn<Cfg0, TS>), grid, dim3(Cfg0::NT), 0, ctx->stream, m, n, (int)K, alpha, At, K,
                               Bt, K, beta0, C0, beta, C, ldc, (int)sym, kps, partial);
        // (a symmetric product's elements above its tiles are not written: the mirror overwrites them)
        if (partial)
            hipLaunchKernelGGL((k_splitk_reduce<TS, float>), dim3((int)std::min<int64_t>(((int64_t)m * n + 255) / 256, 8192)),
                               dim3(256), 0, ctx->stream, m, n, splits, partial, alpha, beta0, C0, beta, C, ldc);
        rc = hipGetLastError() == hipSuccess ? OMX_OK : OMX_ERR_HIP;
        if (rc) set_error("bf16 panel GEMM launch failed");
    }
    prof_end(ctx, nterm == 2 ? OMX_K_GEMM_PAIR : OMX_K_GEMM, ev);
    return rc;
}

// BF16 panel split of a product precision: 1 term (BF16), 2 (BF16x3) or 3 (BF16x6).
static int split_of(int prec) { return prec == OMX_PREC_BF16X6 ? 3 : prec == OMX_PREC_BF16X3 ? 2 : 1; }

template <typename TS, int PREC>
static int dispatch_ops(omx_ctx ctx, bool trA, bool trB, int m, int n, int k, double alpha, const void *A,
                        int64_t lda, const void *B, int64_t ldb, double beta, void *C, int64_t ldc) {
    const TS *a = (const TS *)A, *b = (const TS *)B;
    TS *c = (TS *)C;
    if (!trA && !trB)
        return run_gemm<TS, PREC, false, false, 1>(ctx, m, n, k, alpha, a, a, lda, b, b, ldb, 0.0, nullptr, beta, c, ldc);
    if (!trA && trB)
        return run_gemm<TS, PREC, false, true, 1>(ctx, m, n, k, alpha, a, a, lda, b, b, ldb, 0.0, nullptr, beta, c, ldc);
    if (trA && !trB)
        return run_gemm<TS, PREC, true, false, 1>(ctx, m, n, k, alpha, a, a, lda, b, b, ldb, 0.0, nullptr, beta, c, ldc);
    return run_gemm<TS, PREC, true, true, 1>(ctx, m, n, k, alpha, a, a, lda, b, b, ldb, 0.0, nullptr, beta, c, ldc);
}

int launch_gemm(omx_ctx ctx, int prec, int dt, bool trA, bool trB, int m, int n, int k, double alpha, const void *A,
                int64_t lda, const void *B, int64_t ldb, double beta, void *C, int64_t ldc) {
    if (dt == OMX_F64) {
        if (prec == OMX_PREC_BF16 || prec == OMX_PREC_BF16X3 || prec == OMX_PREC_BF16X6) {
            const BgTerm a{A, lda, trA}, b{B, ldb, !trB};
            int rc = bgemm_panels<double>(ctx, m, n, k, 1, &a, &b, split_of(prec), alpha, 0.0, nullptr, beta,
                                          (double *)C, ldc);
            if (rc != OMX_ERR_UNSUPPORTED) return rc;
            if (prec != OMX_PREC_BF16) prec = OMX_PREC_F32;  // the panels do not cover this shape
        }
        if (prec == OMX_PREC_F64)
            return dispatch_ops<double, OMX_PREC_F64>(ctx, trA, trB, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
        if (prec == OMX_PREC_F32)
            return dispatch_ops<double, OMX_PREC_F32>(ctx, trA, trB, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
        if (prec == OMX_PREC_BF16)
            return dispatch_ops<double, OMX_PREC_BF16>(ctx, trA, trB, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
    } else if (dt == OMX_F32) {
        if (prec == OMX_PREC_BF16 || prec == OMX_PREC_BF16X3 || prec == OMX_PREC_BF16X6) {
            // k-contiguous BF16 panels (A 't' and B 'n' are already k-contiguous)
            const BgTerm a{A, lda, trA}, b{B, ldb, !trB};
            int rc = bgemm_panels<float>(ctx, m, n, k, 1, &a, &b, split_of(prec), alpha, 0.0, nullptr, beta,
                                         (float *)C, ldc);
            if (rc != OMX_ERR_UNSUPPORTED) return rc;
            if (prec != OMX_PREC_BF16) prec = OMX_PREC_F32;  // the panels do not cover this shape
        }
        if (prec == OMX_PREC_F32)
            return dispatch_ops<float, OMX_PREC_F32>(ctx, trA, trB, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
        if (prec == OMX_PREC_BF16)
            return dispatch_ops<float, OMX_PREC_BF16>(ctx, trA, trB, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
    }
    set_error("omx_gemm: unsupported (dt=%d, prec=%d)", dt, prec);
    return OMX_ERR_UNSUPPORTED;
}

// C := alpha*(A1*B1 + A2*B2) + beta0*C0 + beta*C with A* m x k ('n'), B* k x n ('n').
int launch_gemm_pair(omx_ctx ctx, int prec, int dt, int m, int n, int k, double alpha, const void *A1,
                     const void *A2, int64_t lda, const void *B1, const void *B2, int64_t ldb, double beta0,
                     const void *C0, double beta, void *C, int64_t ldc) {
    if ((dt == OMX_F32 || dt == OMX_F64) &&
        (prec == OMX_PREC_BF16 || prec == OMX_PREC_BF16X3 || prec == OMX_PREC_BF16X6)) {
        const BgTerm a[2] = {{A1, lda, false}, {A2, lda, false}};
        const BgTerm b[2] = {{B1, ldb, true}, {B2, ldb, true}};
        const int split = split_of(prec);
        int rc = dt == OMX_F32 ? bgemm_panels<float>(ctx, m, n, k, 2, a, b, split, alpha, beta0, (const float *)C0,
                                                     beta, (float *)C, ldc)
                               : bgemm_panels<double>(ctx, m, n, k, 2, a, b, split, alpha, beta0, (const double *)C0,
                                                      beta, (double *)C, ldc);
        if (rc != OMX_ERR_UNSUPPORTED) return rc;
        if (prec != OMX_PREC_BF16) prec = OMX_PREC_F32;
    }
    const int bk = (prec == OMX_PREC_F64)   ? Prec<OMX_PREC_F64>::BK
                   : (prec == OMX_PREC_F32) ? Prec<OMX_PREC_F32>::BK
                                            : Prec<OMX_PREC_BF16>::BK;
    // The pair boundary must fall on a K-slice boundary of the staged kernels (the direct-to-LDS FP64 and
    // FP32 kernels pad each product's last slice); otherwise the caller runs separate passes.
    if (k % bk != 0) {
        if (dt == OMX_F64 && prec == OMX_PREC_F64 && (ctx->gemm_cfg < 0 || ctx->gemm_cfg == 7 || carries64(ctx, m, n)))
            return launch_dgemm(ctx, false, false, 2, m, n, k, alpha, (const double *)A1, (const double *)A2, lda,
                                (const double *)B1, (const double *)B2, ldb, beta0, (const double *)C0, ldc, beta,
                                (double *)C, ldc);
        if (dt == OMX_F32 && prec == OMX_PREC_F32 && (ctx->gemm_cfg < 0 || ctx->gemm_cfg == 7))
            return launch_sgemm(ctx, false, false, 2, m, n, k, alpha, (const float *)A1, (const float *)A2, lda,
                                (const float *)B1, (const float *)B2, ldb, beta0, (const float *)C0, beta, (float *)C, ldc);
        return OMX_ERR_UNSUPPORTED;
    }
    if (dt == OMX_F64) {
        const double *a1 = (const double *)A1, *a2 = (const double *)A2, *b1 = (const double *)B1,
                     *b2 = (const double *)B2, *c0 = (const double *)C0;
        if (prec == OMX_PREC_F64)
            return run_gemm<double, OMX_PREC_F64, false, false, 2>(ctx, m, n, k, alpha, a1, a2, lda, b1, b2, ldb,
                                                                   beta0, c0, beta, (double *)C, ldc);
        if (prec == OMX_PREC_F32)
            return run_gemm<double, OMX_PREC_F32, false, false, 2>(ctx, m, n, k, alpha, a1, a2, lda, b1, b2, ldb,
                                                                   beta0, c0, beta, (double *)C, ldc);
        if (prec == OMX_PREC_BF16)
            return run_gemm<double, OMX_PREC_BF16, false, false, 2>(ctx, m, n, k, alpha, a1, a2, lda, b1, b2, ldb,
                                                                    beta0, c0, beta, (double *)C, ldc);
    } else if (dt == OMX_F32) {
        const float *a1 = (const float *)A1, *a2 = (const float *)A2, *b1 = (const float *)B1,
                    *b2 = (const float *)B2, *c0 = (const float *)C0;
        if (prec == OMX_PREC_F32)
            return run_gemm<float, OMX_PREC_F32, false, false, 2>(ctx, m, n, k, alpha, a1, a2, lda, b1, b2, ldb, beta0,
                                                                  c0, beta, (float *)C, ldc);
        if (prec == OMX_PREC_BF16)
            return run_gemm<float, OMX_PREC_BF16, false, false, 2>(ctx, m, n, k, alpha, a1, a2, lda, b1, b2, ldb,
                                                                   beta0, c0, beta, (float *)C, ldc);
    }
    set_error("calc_G: unsupported (dt=%d, prec=%d)", dt, prec);
    return OMX_ERR_UNSUPPORTED;
}

// C(i, j) := C(j, i) for i < j (n x n, ld ldc): copies the lower triangle onto the upper one.  One
// 64 x 64 tile pair per workgroup (the upper tile and the lower one it mirrors, the diagonal tiles
// on themselves), through an LDS transpose so that reads and writes run along columns.
template <typename TS>
__global__ __launch_bounds__(256) void k_sym_mirror(int n, TS *__restrict__ C, int64_t ldc,
                                                    const int *__restrict__ mask) {
    constexpr int T = 64;
    __shared__ TS tile[T][T + 1];
    if (mask && !*mask) return;  // system masked off (whole workgroup, before the barrier)
    int a, b;  // lower tile (a, b), a >= b; it fills the upper tile (b, a)
    tile_of_lower(blockIdx.x, (n + T - 1) / T, a, b);
    const int r0 = a * T, c0 = b * T;  // lower tile origin (rows r0.., columns c0..)
    for (int q = threadIdx.x; q < T * T; q += 256) {
        const int r = q % T, c = q / T;  // r fastest: along a column
        if (r0 + r < n && c0 + c < n) tile[c][r] = C[(int64_t)(r0 + r) + (int64_t)(c0 + c) * ldc];
    }
    __syncthreads();
    for (int q = threadIdx.x; q < T * T; q += 256) {
        const int i = q % T, j = q / T;  // upper element (c0 + i, r0 + j), i fastest: along a column
        const int gi = c0 + i, gj = r0 + j;
        if (gi < gj && gj < n) C[(int64_t)gi + (int64_t)gj * ldc] = tile[i][j];
    }
}

// C := alpha * A * B^T for a product known to be symmetric (n x n; A, B n x k, 'n' and 't'), as
// AW = (C*H)*C^T with H symmetric in omm()'s calc_AW (omm_ops.F90:44-64).  The kernels compute the
// lower-triangle tiles only where they can (ctx->gemm_sym), otherwise the full product; the lower
// triangle is then mirrored, so C is exactly symmetric.
int launch_gemm_sym(omx_ctx ctx, int prec, int dt, int n, int k, double alpha, const void *A, int64_t lda,
                    const void *B, int64_t ldb, void *C, int64_t ldc) {
    ctx->gemm_sym = 2;
    int rc = launch_gemm(ctx, prec, dt, false, true, n, n, k, alpha, A, lda, B, ldb, 0.0, C, ldc);
    const bool whole = ctx->gemm_sym == 3;  // the product wrote the upper triangle too
    ctx->gemm_sym = 0;
    if (rc || whole) return rc;
    const int nt = (n + 63) / 64;
    const unsigned grid = (unsigned)(nt * (nt + 1) / 2);
    if (dt == OMX_F64)
        hipLaunchKernelGGL(k_sym_mirror<double>, dim3(grid), dim3(256), 0, ctx->stream, n, (double *)C, ldc,
                           ctx->launch_mask);
    else
        hipLaunchKernelGGL(k_sym_mirror<float>, dim3(grid), dim3(256), 0, ctx->stream, n, (float *)C, ldc,
                           ctx->launch_mask);
    OMX_CHECK_HIP(hipGetLastError());
    return OMX_OK;
}

}  // namespace omx

using namespace omx;

extern "C" int omx_gemm(omx_ctx ctx, int prec, int dt, char opA, char opB, int m, int n, int k, double alpha,
                        const void *A, int64_t lda, const void *B, int64_t ldb, double beta, void *C, int64_t ldc) {
    OMX_REQUIRE(ctx, "omx_gemm: null context");
    OMX_REQUIRE(valid_op(opA) && valid_op(opB), "omx_gemm: invalid op ('%c','%c')", opA, opB);
    OMX_REQUIRE(m >= 0 && n >= 0 && k >= 0, "omx_gemm: negative dimension");
    bool trA = is_trans(opA), trB = is_trans(opB);
    OMX_REQUIRE(lda >= std::max(1, trA ? k : m) && ldb >= std::max(1, trB ? n : k) && ldc >= std::max(1, m),
                "omx_gemm: leading dimension too small");
    if (m == 0 || n == 0) return OMX_OK;
    if (k == 0) return omx_scale(ctx, dt, m, n, beta, C, ldc);
    OMX_REQUIRE(A && B && C, "omx_gemm: null operand");
    if (dt == OMX_C128 || dt == OMX_C64)  // complex: FP64 / FP32 MFMA by element type
        return launch_zgemm(ctx, dt, opA, opB, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
    return launch_gemm(ctx, prec, dt, trA, trB, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
}

extern "C" int omx_omm_search(omx_ctx ctx, int prec, int dt, int n, int k, const void *HC, const void *SC, const void *HG,
                              const void *SG, int64_t ldx, const void *D, int64_t ldd, void *HWd, void *SWd, void *HWdd,
                              void *SWdd, int64_t ldw) {
    OMX_REQUIRE(ctx && n >= 0 && k >= 0, "omx_omm_search: bad arguments");
    OMX_REQUIRE(ldx >= std::max(1, n) && ldd >= std::max(1, n) && ldw >= std::max(1, n),
                "omx_omm_search: leading dimension too small");
    OMX_REQUIRE(dt == OMX_F64 || dt == OMX_F32, "omx_omm_search: unsupported element type %d", dt);
    if (n == 0) return OMX_OK;
    OMX_REQUIRE(HC && SC && HG && SG && D && HWd && SWd && HWdd && SWdd, "omx_omm_search: null operand");
    const void *const A[4] = {HC, SC, HG, SG};
    void *const C[4] = {HWd, SWd, HWdd, SWdd};
    // The tuner has no say in it, and a forced tile gets the one launch's order of adding, so that neither
    // changes a bit.
    const bool one = prec == (dt == OMX_F64 ? OMX_PREC_F64 : OMX_PREC_F32) && search_in_one(ctx, dt, n, k, ldx, ldd);
    if (one && (ctx->gemm_cfg < 0 || ctx->gemm_cfg == 7)) return launch_search(ctx, dt, n, k, A, ldx, D, ldd, C, ldw);
    int rc = OMX_OK;
    ctx->one_part = one;
    for (int q = 0; q < 4 && !rc; ++q)
        rc = q < 2 ? omx_gemm(ctx, prec, dt, 'n', 't', n, n, k, 1.0, A[q], ldx, D, ldd, 0.0, C[q], ldw)
                   : omx_gemm_sym(ctx, prec, dt, n, k, 1.0, A[q], ldx, D, ldd, C[q], ldw);
    ctx->one_part = false;
    return rc;
}

extern "C" int omx_gemm_sym(omx_ctx ctx, int prec, int dt, int n, int k, double alpha, const void *A, int64_t lda,
                            const void *B, int64_t ldb, void *C, int64_t ldc) {
    OMX_REQUIRE(ctx, "omx_gemm_sym: null context");
    OMX_REQUIRE(n >= 0 && k >= 0, "omx_gemm_sym: negative dimension");
    OMX_REQUIRE(lda >= std::max(1, n) && ldb >= std::max(1, n) && ldc >= std::max(1, n),
                "omx_gemm_sym: leading dimension too small");
    OMX_REQUIRE(dt == OMX_F64 || dt == OMX_F32 || dt == OMX_C128 || dt == OMX_C64,
                "omx_gemm_sym: unsupported element type %d", dt);
    if (n == 0) return OMX_OK;
    if (k == 0) return omx_scale(ctx, dt, n, n, 0.0, C, ldc);
    OMX_REQUIRE(A && B && C, "omx_gemm_sym: null operand");
    if (dt == OMX_C128 || dt == OMX_C64)  // Hermitian: C = alpha A B^H
        return launch_zgemm_herm(ctx, dt, n, k, alpha, A, lda, B, ldb, C, ldc);
    return launch_gemm_sym(ctx, prec, dt, n, k, alpha, A, lda, B, ldb, C, ldc);
}

extern "C" int omx_gemm_set_tile(omx_ctx ctx, int cfg) {
    OMX_REQUIRE(ctx && cfg >= -1 && cfg < kNumCfg, "omx_gemm_set_tile: configuration %d not in [-1, %d)", cfg,
                kNumCfg);
    ctx->gemm_cfg = cfg;
    return OMX_OK;
}

extern "C" int omx_omm_calc_G(omx_ctx ctx, int prec, int dt, int n, int m, const void *HW, const void *SW,
                              int64_t ldw, const void *HC, const void *SC, void *G, int64_t ldc) {
    OMX_REQUIRE(ctx && HW && SW && HC && SC && G, "omx_omm_calc_G: null argument");
    OMX_REQUIRE(n > 0 && m > 0 && ldw >= n && ldc >= n, "omx_omm_calc_G: bad shape");
    OMX_REQUIRE(G != HC && G != SC, "omx_omm_calc_G: G must not alias HC or SC");
    const bool cplx = (dt == OMX_C128 || dt == OMX_C64);
    // G = 4*HC - 2*(SW*HC + HW*SC): pair product with the 4*HC term folded into the epilogue.
    int rc = cplx ? launch_zgemm_pair(ctx, dt, n, m, n, -2.0, SW, HW, ldw, HC, SC, ldc, 4.0, HC, 0.0, G, ldc)
                  : launch_gemm_pair(ctx, prec, dt, n, m, n, -2.0, SW, HW, ldw, HC, SC, ldc, 4.0, HC, 0.0, G, ldc);
    if (rc != OMX_ERR_UNSUPPORTED) return rc;
    // Unaligned n: three passes (G = 4HC; G -= 2 SW HC; G -= 2 HW SC), as calc_G in omm_ops.F90:35-37.
    rc = omx_add(ctx, dt, 'n', n, m, 4.0, HC, ldc, 0.0, G, ldc);
    if (rc) return rc;
    if (cplx) {
        rc = launch_zgemm(ctx, dt, 'n', 'n', n, m, n, -2.0, SW, ldw, HC, ldc, 1.0, G, ldc);
        if (rc) return rc;
        return launch_zgemm(ctx, dt, 'n', 'n', n, m, n, -2.0, HW, ldw, SC, ldc, 1.0, G, ldc);
    }
    rc = launch_gemm(ctx, prec, dt, false, false, n, m, n, -2.0, SW, ldw, HC, ldc, 1.0, G, ldc);
    if (rc) return rc;
    return launch_gemm(ctx, prec, dt, false, false, n, m, n, -2.0, HW, ldw, SC, ldc, 1.0, G, ldc);
}

// FP64 products C := alpha * sum_p op(A_p) op(B_p) + beta0*C0 + beta*C on the FP64 matrix cores, and FP32
// ones of FP32 operands on the FP32 ones, with the operands loaded straight into LDS, for every m, n, k and
// every leading dimension up to 2^20 (NPAIR = 2: calc_G's two products back to back along K).
//
// Staging.  K is taken in slices of 16 (FP32: 32), 128 bytes.  An operand whose row index is contiguous (A
// 'n', B 't') lands k-major: ROWS elements per k-row, several k-rows per wave load (FP32: with the 16-byte
// chunks rotated by k-row, dl_rot).  One whose k is contiguous (A 't', B 'n') lands row-major: 128 bytes
// per row, 8 rows per wave load, logical 16-byte chunk c of row r at physical chunk c ^ ((r >> 1) & 7).  A wave load is one buffer_load_dwordx4 ... lds, 16 bytes
// per lane, lane l landing at byte 16*l.  The descriptors are rebased at every slice, so a lane's byte
// offset is the same for every slice, and they end exactly where the matrix ends: the hardware's range
// check is per dword, so anything past the last element arrives as zero and an odd size, an odd leading
// dimension or an 8-byte aligned operand needs no other path.  Rows past m or n inside the matrix only
// feed results that are not stored.  k past the end of a k-contiguous row would be the next row's
// values; the last slice clears those in LDS before they are read.
//
// What bounds it: the FP64 matrix core (64 cycles per 16x16x4 step and SIMD), except where the result has
// fewer tiles than the chip has CUs; there it is the serial chain of slices of one tile, and below that
// the launch.  Before, only m, n % 128 == 0 with k % 16 == 0 took this path and everything else was staged
// through registers in 128x128 tiles: 54 x 54 x 108 22 us (now 4.3), 432 x 432 x 864 about 35 us (14),
// 1458 x 1458 x 2916 340 us (225), 4394 x 4394 x 8788 5.84 ms (5.14), gradient of 2662 x 5324 2.96 ms (2.30).
// FP32: an FP32 step takes half the time of an FP64 one, so a slice of 32 takes as long as an FP64 slice of
// 16 and the same tiles and model serve.  Before, only Grams of whole 128 tiles that fill the chip were
// loaded this way: 54 x 54 x 108 21 us (now 4.2), 250 x 250 x 500 30 (6.1), 1458 x 1458 x 2916 242 (124;
// symmetric 252, now 76; pair 512, now 239), 4394 x 4394 x 8788 4.14 ms (2.93; symmetric 2.61, now 1.35), pair
// of 4394 x 8788 8.64 ms (5.24), 4096 x 4096 x 8192 1.90 (1.86).  Errors against FP64 (relative, Gram): 250 x
// 500 2.4e-7 (2.1e-7), 1458 x 2916 4.9e-7 (2.1e-7), as before where K is one chain (see carries); the carry
// costs 2 %.
//
// Tiles.  Three tile sizes with the same K chain per element (K in order, so the results do not depend
// on the tile): 128x128 (8 waves of 32x64, two stages), 64x64 (4 waves of 32x32, three stages) and 32x32
// (4 waves of 16x16, two stages of four slices: a lone tile's slice takes 0.16 us, with one-slice stages
// 0.34 us, because the barrier and the first LDS read are paid once per stage).  Stage s+NST-1 is issued while stage s feeds the MFMAs, one barrier
// per slice; waves whose sub-tile lies outside the result (or, for a symmetric product, above the
// diagonal) take part in the loads and barriers only.
#include <algorithm>

#include "omx_internal.h"
#include "omx_mfma.h"

namespace omx {

// Per element type: a slice of K is 128 bytes of a k-contiguous row, one matrix-core step is 16x16x4.
template <typename R>
struct DlT;
template <>
struct DlT<double> {
    typedef d4v acc;
    static constexpr int DK = 16, CH = 2;  // K slice; elements of a 16-byte chunk
    __device__ static inline acc mfma(double a, double b, acc c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    __device__ static inline int row(int lq, int v) { return lq + 4 * v; }  // of a result register
};
template <>
struct DlT<float> {
    typedef f4v acc;
    static constexpr int DK = 32, CH = 4;
    __device__ static inline acc mfma(float a, float b, acc c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    __device__ static inline int row(int lq, int v) { return 4 * lq + v; }
};

// XOR of the 16-byte chunks of FP32 k-row kk of a k-major tile: a step reads 16 consecutive floats from each
// of four consecutive k-rows, which would share their banks.
template <typename R, int ROWS>
__device__ inline int dl_rot(int kk) {
    return sizeof(R) == 8 ? 0 : ROWS == 32 ? (kk & 2) << 1 : (kk & 3) << 2;
}
// Byte offset of lane `lane` of wave load `ins` of an operand tile (ROWS rows x DK) from the slice's
// descriptor base.  KC: k contiguous.
template <typename R, int ROWS, bool KC>
__device__ inline int dl_voff(int ins, int lane, int ld) {
    constexpr int ES = sizeof(R);
    if constexpr (KC) {
        const int r = ins * 8 + (lane >> 3);
        return ES * r * ld + 16 * ((lane & 7) ^ dl_swz(r));
    } else {
        constexpr int LPR = ROWS * ES / 16;  // lanes per k-row
        const int kk = ins * (64 / LPR) + lane / LPR;
        return ES * kk * ld + 16 * ((lane % LPR) ^ dl_rot<R, ROWS>(kk));
    }
}
// The element (row r, k kk) of a staged tile; dl_at: its place in a k-contiguous one.
template <typename R>
__device__ inline int dl_at(int r, int kk) {
    constexpr int CH = DlT<R>::CH;
    return r * DlT<R>::DK + ((kk / CH) ^ dl_swz(r)) * CH + kk % CH;
}
template <typename R, int ROWS, bool KC>
__device__ inline R dl_elem(const R *t, int r, int kk) {
    return t[KC ? dl_at<R>(r, kk) : kk * ROWS + (r ^ dl_rot<R, ROWS>(kk) * DlT<R>::CH)];
}
// Start of an operand tile (row i0, k 0), and the bytes from there to the end of the operand (extent rows
// x k, leading dimension ld).
template <typename R, bool KC>
__device__ inline const char *dl_base(const R *P, int i0, int64_t ld) {
    return (const char *)(P + (KC ? (int64_t)i0 * ld : i0));
}
template <typename R, bool KC>
__device__ inline int64_t dl_left(int extent, int k, int i0, int64_t ld) {
    return (int64_t)sizeof(R) * (KC ? (int64_t)(extent - 1 - i0) * ld + k : (int64_t)(k - 1) * ld + (extent - i0));
}

// Batched products: blockIdx.y selects the product, its operands and result offset by these strides
// (elements; single products only, no split of K).
struct DlBatch {
    int64_t sA = 0, sB = 0, sC = 0;
    // with `four`: the line-search products A[y] B^T into C[y], the last two of them symmetric
    int four = 0;
    const void *A[4] = {nullptr, nullptr, nullptr, nullptr};
    void *C[4] = {nullptr, nullptr, nullptr, nullptr};
};

// EXACT: m, n are multiples of the tile and k of the slice, so nothing needs the descriptors' end, a
// cleared tail or guarded stores; the 128x128 tile is faster without them (8192 x 8192 x 16384 Gram 29.8
// against 29.9 ms, gradient 60.4 against 61.6 ms).
// CY: the sums are carried every `carry` slices, not at all for 0 (FP32 products, the FP64 ones of carries64 and masked
// pairs (see seam); the FP64 ones take the 64 and 32 tiles: the 128 tile has no registers for a second set of sums).
template <typename R, class CF, bool TRA, bool TRB, int NPAIR, bool EXACT, bool CY>
__global__ __launch_bounds__(CF::NT, CF::MINW) void k_dgemm_dl(int m, int n, int k, double alpha,
                                                               const R *__restrict__ A1,
                                                               const R *__restrict__ A2, int64_t lda,
                                                               const R *__restrict__ B1,
                                                               const R *__restrict__ B2, int64_t ldb,
                                                               double beta0, const R *__restrict__ C0,
                                                               int64_t ldc0, double beta, R *__restrict__ C,
                                                               int64_t ldc, int sym, int tbase, int nsplit, int sps,
                                                               R *__restrict__ partial,
                                                               const int *__restrict__ mask, int carry, DlBatch bat) {
    constexpr int BM = CF::BM, BN = CF::BN, NST = CF::NST, NW = CF::WGM * CF::WGN;
    constexpr int DK = DlT<R>::DK, LD = 1024 / sizeof(R);  // K slice, elements of a wave load
    constexpr int INS = DK * (BM + BN) / LD, LPW = INS / NW, U = CF::U;
    constexpr int SLICE = DK * (BM + BN), STAGE = U * SLICE;
    constexpr bool KCA = TRA, KCB = !TRB;
    static_assert(LPW * NW == INS && BM == BN && NW % 2 == 0, "each wave loads one operand");
    __shared__ __align__(16) R smem[NST * STAGE];
    if (mask && !*mask) return;  // system masked off (grouped solver; whole workgroup, before any barrier)
    if (bat.four) {
        const int T = (m + BM - 1) / BM;
        A1 = (const R *)bat.A[blockIdx.y];
        C = (R *)bat.C[blockIdx.y];
        if (blockIdx.y < 2)
            sym = 0;
        else if ((int)blockIdx.x >= T * (T + 1) / 2)
            return;  // the tiles above the diagonal
    } else {
        A1 += blockIdx.y * bat.sA;
        B1 += blockIdx.y * bat.sB;
        C += blockIdx.y * bat.sC;
    }
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wm = wave / CF::WGN, wn = wave % CF::WGN;
    // tile w of the launch's tile order and the part z of K it takes
    const int w = tbase + (int)blockIdx.x / nsplit, z = (int)blockIdx.x % nsplit;
    int tm, tn;
    if (sym)
        tile_of_lower(w, (m + BM - 1) / BM, tm, tn);
    else
        tile_of(w, (m + BM - 1) / BM, (n + BN - 1) / BN, tm, tn);
    const int i0 = tm * BM, j0 = tn * BN;
    const int wi = i0 + wm * CF::WM, wj = j0 + wn * CF::WN;
    const bool live = wi < m && wj < n && !(sym && wj > wi + CF::WM - 1);
    const int nsl = (k + DK - 1) / DK;  // slices of one product
    const int sb = z * sps, ns = min(NPAIR * nsl, sb + sps) - sb;

    typename DlT<R>::acc acc[CF::FBM][CF::FBN];
#pragma unroll
    for (int a = 0; a < CF::FBM; ++a)
#pragma unroll
        for (int b = 0; b < CF::FBN; ++b) acc[a][b] = typename DlT<R>::acc{0, 0, 0, 0};
    typename DlT<R>::acc tot[CY ? CF::FBM : 1][CY ? CF::FBN : 1];  // (see carry_sums)
    if constexpr (CY) {
#pragma unroll
        for (int a = 0; a < CF::FBM; ++a)
#pragma unroll
            for (int b = 0; b < CF::FBN; ++b) tot[a][b] = typename DlT<R>::acc{0, 0, 0, 0};
    }
    // The first half of the waves loads A, the second half B.  Slices are issued in order: the wave's
    // descriptor advances by one slice each time, and starts over at the second product of a pair.
    const bool on_b = wave >= NW / 2;
    const int ins0 = (on_b ? wave - NW / 2 : wave) * LPW;
    int voff[LPW];
#pragma unroll
    for (int q = 0; q < LPW; ++q)
        voff[q] = on_b ? dl_voff<R, BN, KCB>(ins0 + q, lane, (int)ldb) : dl_voff<R, BM, KCA>(ins0 + q, lane, (int)lda);
    const int64_t step = (int64_t)sizeof(R) * (on_b ? (KCB ? DK : DK * ldb) : (KCA ? DK : DK * lda));
    const int64_t all = on_b ? dl_left<R, KCB>(n, k, j0, ldb) : dl_left<R, KCA>(m, k, i0, lda);
    const char *const first = on_b ? dl_base<R, KCB>(B1, j0, ldb) : dl_base<R, KCA>(A1, i0, lda);
    const char *const second = on_b ? dl_base<R, KCB>(B2, j0, ldb) : dl_base<R, KCA>(A2, i0, lda);
    const int sb_in = NPAIR == 2 && sb >= nsl ? sb - nsl : sb;
    const char *pos = (NPAIR == 2 && sb >= nsl ? second : first) + sb_in * step;
    int64_t left = all - sb_in * step;
    // slice (of this part) where the second product starts; the last slice of each product if it is partial
    const int sw = nsl - sb, t1 = k % DK ? sw - 1 : -1, t2 = NPAIR == 2 && k % DK ? sw + nsl - 1 : -1;
    auto issue = [&](int s) {  // the U slices of stage s
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int sl = s * U + u;
            if (U > 1 && sl >= ns) break;
            R *st = smem + (s % NST) * STAGE + u * SLICE + wave * LPW * LD;
            if (NPAIR == 2 && sl == sw) {
                pos = second;
                left = all;
            }
            const __amdgpu_buffer_rsrc_t r = raw_rsrc(pos, EXACT || (uint32_t)((uint64_t)left >> 31) ? 0x7ffffff8 : (int)left);
            pos += step;
            left -= step;
#pragma unroll
            for (int q = 0; q < LPW; ++q) {
                const int vo = voff[q];  // (a local: see k_bgemm_tn)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void *)(st + q * LD), 16, vo, 0, 0, 0);
            }
        }
    };
    const int li = lane & 15, lk = lane >> 4;
    // one slice: the fragments of k step ks + 4 are read before the MFMAs of step ks
    auto slice = [&](const R *As, const R *Bs) {
        R a[2][CF::FBM], b[2][CF::FBN];
        auto frag = [&](int ks, R (&fa)[CF::FBM], R (&fb)[CF::FBN]) {
            const int kk = ks + lk;
#pragma unroll
            for (int f = 0; f < CF::FBM; ++f) fa[f] = dl_elem<R, BM, KCA>(As, wm * CF::WM + f * 16 + li, kk);
#pragma unroll
            for (int f = 0; f < CF::FBN; ++f) fb[f] = dl_elem<R, BN, KCB>(Bs, wn * CF::WN + f * 16 + li, kk);
        };
        frag(0, a[0], b[0]);
#pragma unroll
        for (int ks = 0; ks < DK; ks += 4) {
            const int cur = (ks / 4) & 1;
            if (ks + 4 < DK) frag(ks + 4, a[cur ^ 1], b[cur ^ 1]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int fm = 0; fm < CF::FBM; ++fm)
#pragma unroll
                for (int fn = 0; fn < CF::FBN; ++fn)  // (b, a): the result's columns run along i
                    acc[fm][fn] = DlT<R>::mfma(b[cur][fn], a[cur][fm], acc[fm][fn]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    const int nst = (ns + U - 1) / U, nfull = ns / U;  // stages, and those with all their slices
#pragma unroll
    for (int s = 0; s < NST - 1; ++s)
        if (s < nst) issue(s);
    auto march = [&](auto work) {  // waves outside the result only load, clear and wait
        for (int s = 0; s < nst; ++s) {
            // this wave's loads of stage s have landed (the NST - 2 later stages stay in flight)
            if (NST > 2 && s + NST - 2 < nfull)
                __builtin_amdgcn_s_waitcnt(waitcnt_vmcnt(LPW * U * (NST - 2)));
            else
                __builtin_amdgcn_s_waitcnt(waitcnt_vmcnt(0));
            wg_barrier();  // everyone's have; stage s-1 is no longer read
            if (s + NST - 1 < nst) issue(s + NST - 1);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int sl = s * U + u;
                if (U > 1 && sl >= ns) break;
                R *As = smem + (s % NST) * STAGE + u * SLICE, *Bs = As + DK * BM;
                if (!EXACT && (KCA || KCB) && (sl == t1 || (NPAIR == 2 && sl == t2))) {  // k-contiguous rows end at k
                    if (KCA)
                        for (int e = t; e < BM * DK; e += CF::NT)
                            if (e % DK >= k % DK) As[dl_at<R>(e / DK, e % DK)] = (R)0;
                    if (KCB)
                        for (int e = t; e < BN * DK; e += CF::NT)
                            if (e % DK >= k % DK) Bs[dl_at<R>(e / DK, e % DK)] = (R)0;
                    wg_barrier();
                }
                if (decltype(work)::value) {
                    slice(As, Bs);
                    if constexpr (CY) {
                        // (a period of 4 slices or more ends with a stage of 4)
                        if (carry && ((u == U - 1 && (sl & (carry - 1)) == carry - 1) || (NPAIR == 2 && sl + 1 == sw)))
                            carry_sums(acc, tot);
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
    if constexpr (CY) {
#pragma unroll
        for (int a = 0; a < CF::FBM; ++a)
#pragma unroll
            for (int b = 0; b < CF::FBN; ++b) acc[a][b] = tot[a][b] + acc[a][b];
    }
    const int lq = lane >> 4;
    if (partial) {  // a K part of a split tile: the raw sums, reduced in part order later
        R *pt = partial + (int64_t)blockIdx.x * (BM * BN);
#pragma unroll
        for (int fm = 0; fm < CF::FBM; ++fm)
#pragma unroll
            for (int fn = 0; fn < CF::FBN; ++fn)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    pt[(wm * CF::WM + fm * 16 + li) + (wn * CF::WN + fn * 16 + DlT<R>::row(lq, v)) * BM] = acc[fm][fn][v];
        return;
    }
#pragma unroll
    for (int fm = 0; fm < CF::FBM; ++fm)
#pragma unroll
        for (int fn = 0; fn < CF::FBN; ++fn) {
            const int i = wi + fm * 16 + li;
            if (!EXACT && i >= m) continue;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int j = wj + fn * 16 + DlT<R>::row(lq, v);
                if ((!EXACT && j >= n) || (sym && j > i)) continue;
                double r = alpha * (double)acc[fm][fn][v];
                if (C0) r += beta0 * (double)C0[(int64_t)i + (int64_t)j * ldc0];
                if (beta != 0.0) r += beta * (double)C[(int64_t)i + (int64_t)j * ldc];
                C[(int64_t)i + (int64_t)j * ldc] = (R)r;
                if (sym == 2 && j < i) C[(int64_t)j + (int64_t)i * ldc] = (R)r;
            }
        }
}

// C tile := alpha * (sum of its nsplit K parts, in part order) + beta0*C0 + beta*C for the tiles tbase..
// of the launch's tile order (blockIdx.x: tile, blockIdx.y: a 1024-element slice of it).
template <typename R, int BM, int BN>
__global__ __launch_bounds__(256) void k_dl_split_reduce(int m, int n, int sym, int tbase, int nsplit,
                                                         const R *__restrict__ partial, double alpha,
                                                         double beta0, const R *__restrict__ C0, int64_t ldc0,
                                                         double beta, R *__restrict__ C, int64_t ldc) {
    int tm, tn;
    if (sym)
        tile_of_lower(tbase + (int)blockIdx.x, (m + BM - 1) / BM, tm, tn);
    else
        tile_of(tbase + (int)blockIdx.x, (m + BM - 1) / BM, (n + BN - 1) / BN, tm, tn);
    const R *pt = partial + (int64_t)blockIdx.x * nsplit * (BM * BN);
    const int e0 = blockIdx.y * 1024;
    for (int e = e0 + threadIdx.x; e < e0 + 1024; e += 256) {
        const int i = tm * BM + e % BM, j = tn * BN + e / BM;
        if (i >= m || j >= n || (sym && j > i)) continue;  // (parts above the diagonal are not written)
        R sum = (R)0;
        for (int zz = 0; zz < nsplit; ++zz) sum += pt[(int64_t)zz * (BM * BN) + e];
        const int64_t off = (int64_t)i + (int64_t)j * ldc;
        double r = alpha * (double)sum;
        if (C0) r += beta0 * (double)C0[(int64_t)i + (int64_t)j * ldc0];
        if (beta != 0.0) r += beta * (double)C[off];
        C[off] = (R)r;
        if (sym == 2 && j < i) C[(int64_t)j + (int64_t)i * ldc] = (R)r;
    }
}

template <int BM_, int BN_, int WGM_, int WGN_, int MINW_, int NST_, int U_>
struct DlCfg {
    static constexpr int BM = BM_, BN = BN_, WGM = WGM_, WGN = WGN_, NST = NST_, MINW = MINW_, U = U_;
    static constexpr int NT = 64 * WGM * WGN, WM = BM / WGM, WN = BN / WGN, FBM = WM / 16, FBN = WN / 16;
};
typedef DlCfg<128, 128, 4, 2, 4, 2, 1> Dl128;
typedef DlCfg<64, 64, 2, 2, 2, 3, 1> Dl64;
typedef DlCfg<32, 32, 2, 2, 2, 2, 4> Dl32;

static int tiles_of(int m, int n, int b, bool sym) {
    const int tm = (m + b - 1) / b, tn = (n + b - 1) / b;
    return sym ? tm * (tm + 1) / 2 : tm * tn;
}

// dl_time, dl_cost: time of a product by tile and by the parts K is split into, in microseconds: rounds of workgroups over
// the CUs (workgroups that share a CU share its matrix cores) times the slices of a part, plus what a launch,
// a round and the reduction of the parts cost.  The constants are a least-squares fit to 60 shapes (54 x 54
// x 108 to 4394 x 4394 x 8788, Grams, symmetric Grams and pairs; every tile and 1 to 12 parts): 11 % rms, and
// the choices they lead to are within 1.6 % of the fastest of all on average.
//
// dl_tail_parts: a symmetric product in 128x128 tiles whose last round of resident workgroups (two per CU) is not full:
// the parts along K that each tile of that round is split into (1: it is not split).  Only for orders
// that are multiples of 128; elsewhere the symmetric form adds exactly as the full product does.
static int dl_tail_parts(omx_ctx ctx, int m, int tiles, bool sym, int nsl) {
    const int slots = 2 * ctx->num_cus, rest = tiles % slots;
    if (!sym || m % 128 || ctx->launch_mask || ctx->one_part || tiles < slots || !rest) return 1;
    int parts = std::max(1, std::min(16, slots / rest));
    while (parts > 1 && nsl % parts) --parts;
    return parts;
}
static const int kDlEdge[3] = {128, 64, 32};
// units workgroups of tile q and sps slices each
static double dl_time(omx_ctx ctx, int q, int64_t units, int sps) {
    const double slice[3] = {1.90, 0.515, 0.172};  // a CU's time for one 16-wide slice of a tile
    const double alone[3] = {2.15, 0.69, 0.172};   // the same with a single workgroup on the CU
    const int64_t rounds = (units + ctx->num_cus - 1) / ctx->num_cus;
    // 64: three workgroups share a CU, so a last one alone costs more; with many rounds the CUs drift apart
    // and the last is half empty on average.
    double per = std::max(slice[q] * rounds, alone[q]);
    if (q == 1 && rounds % 3 == 1 && rounds < 6) per = slice[q] * (rounds - 1) + alone[q];
    if (q == 1 && rounds >= 6) per = slice[q] * 0.5 * (rounds + (double)units / ctx->num_cus);
    return 4.5 + 0.55 * rounds + per * sps;
}
static double dl_cost(omx_ctx ctx, int q, bool sym, int m, int n, int nsl, int splits, int nbatch, int es) {
    const int units = tiles_of(m, n, kDlEdge[q], sym) * splits * nbatch, rounds = (units + ctx->num_cus - 1) / ctx->num_cus;
    const int sps = (nsl + splits - 1) / splits;
    const int tail = dl_tail_parts(ctx, q == 0 && splits == 1 && nbatch == 1 && es == 8 ? m : 1, units, sym, nsl);
    if (tail > 1) {
        const int whole = units / (2 * ctx->num_cus) * 2;  // two workgroups of every round share a CU
        return 9.8 + 0.55 * whole + 1.90 * (whole * sps + 2.0 * sps / tail);
    }
    double t = dl_time(ctx, q, units, sps);
    // 128: two workgroups share a CU, and the parts of most of a third round land in pairs.  (Reached by FP32 products;
    // FP32 Grams of 1410 to 1440 states 123 us instead of 146, 1474 to 1520 130 to 133 instead of 135, 2114 to 2176 335
    // to 340 instead of 340 to 350, gradients of 1058 to 1088 states 110 instead of 123: all that it changes.)
    if (q == 0 && splits > 1 && rounds == 3 && 2 * units > 5 * ctx->num_cus && units < 3 * ctx->num_cus)
        t += 0.1 * 1.90 * 3 * sps;
    return t + (splits > 1 ? 5.3 + 1e-6 * es * (splits + 1) * m * n / 4.9 : 0.0);
}
static int dl_tile(omx_ctx ctx, bool sym, int m, int n, int nsl, int splits, int nbatch, int es, double *cost = nullptr,
                   bool carried = false) {
    int best = 0;
    double c = 0.0;
    const int first = es == 8 && (carried || carries64(ctx, m, n));
    for (int q = first; q < 3; ++q) {
        const double t = dl_cost(ctx, q, sym, m, n, nsl, splits, nbatch, es);
        if (q == first || t < c) {
            best = q;
            c = t;
        }
    }
    if (cost) *cost = c;
    return best;
}

// The number of parts with the least time; for a square result that of the full and the symmetric form
// together, so that both add the same parts.
int dgemm_k_splits(omx_ctx ctx, int m, int n, int nsl, int es) {
    if (ctx->launch_mask || ctx->one_part || (es == 4 && !carries(ctx, m, n))) return 1;
    int best = 1;
    double cost = 0.0;
    for (int s : {1, 2, 3, 4, 5, 6, 8, 12}) {
        if (s > 1 && nsl < 2 * s) break;
        double t, u = 0.0;
        dl_tile(ctx, false, m, n, nsl, s, 1, es, &t);
        if (m == n) dl_tile(ctx, true, m, n, nsl, s, 1, es, &u);
        if (s == 1 || t + u < cost) {
            best = s;
            cost = t + u;
        }
    }
    return best;
}

constexpr int kSeam = 1 << 30;  // a carry period that no product reaches: carried at a pair's seam only
// Carry period of an FP64 product: by the parts that 128 tiles were split into, two workgroups per CU, 64 values at
// the least.
static int dl_period(omx_ctx ctx, int m, int n, int nsl) {
    if (ctx->carry64) return 4;
    const int64_t tiles = tiles_of(m, n, 128, false);
    return carry_period(nsl, std::min<int64_t>((2 * ctx->num_cus + tiles - 1) / tiles, nsl / 4));
}

template <typename R, class CF, bool TRA, bool TRB, int NPAIR>
static int run_tile(omx_ctx ctx, int sym, int splits, int sps, int m, int n, int k, double alpha, const R *A1,
                    const R *A2, int64_t lda, const R *B1, const R *B2, int64_t ldb, double beta0,
                    const R *C0, int64_t ldc0, double beta, R *C, int64_t ldc, int nbatch,
                    const DlBatch &bat, bool seam) {
    constexpr int DK = DlT<R>::DK;
    const int tiles = tiles_of(m, n, CF::BM, sym != 0);
    const int nsl = NPAIR * ((k + DK - 1) / DK);
    int whole = tiles, rest = 0, rsplit = 1;
    if (splits > 1) {
        whole = 0;
        rest = tiles;
        rsplit = splits;
    } else if (CF::BM == 128 && sizeof(R) == 8 && (rsplit = dl_tail_parts(ctx, m, tiles, sym != 0, nsl)) > 1) {
        rest = tiles % (2 * ctx->num_cus);
        whole = tiles - rest;
        sps = nsl / rsplit;
    }
    if (rest) {
        const int rc = ensure_ws(ctx, sizeof(R) * (size_t)rest * rsplit * CF::BM * CF::BN);
        if (rc == OMX_ERR_NOMEM) {  // no room for the parts: K whole, which needs none
            clear_error();
            whole = tiles;
            rest = 0;
        } else if (rc) {
            return rc;
        }
    }
    constexpr bool single = sizeof(R) == 4;
    auto launch = [&](int grid, int tbase, int parts, int per, R *partial, const int *mask) {
#define OMX_DL_LAUNCH(EX, CY, CARRY)                                                                                       \
    hipLaunchKernelGGL((k_dgemm_dl<R, CF, TRA, TRB, NPAIR, EX, CY>), dim3(grid, nbatch), dim3(CF::NT), 0, ctx->stream, m, n, k, \
                       alpha, A1, A2, lda, B1, B2, ldb, beta0, C0, ldc0, beta, C, ldc, sym, tbase, parts, per, partial, mask, \
                       CARRY, bat)
        if constexpr (single) {
            const int carry = carries(ctx, m, n) ? 4 : seam ? kSeam : 0;
            if (CF::BM == 128 && m % 128 == 0 && n % 128 == 0 && k % DK == 0)
                OMX_DL_LAUNCH(CF::BM == 128, true, carry);
            else
                OMX_DL_LAUNCH(false, true, carry);
        } else if (CF::BM == 128 && m % 128 == 0 && n % 128 == 0 && k % DK == 0) {
            OMX_DL_LAUNCH(CF::BM == 128, false, 0);
        } else if (CF::BM != 128 && (seam || carries64(ctx, m, n))) {
            OMX_DL_LAUNCH(false, CF::BM != 128, seam ? kSeam : dl_period(ctx, m, n, nsl));
        } else {
            OMX_DL_LAUNCH(false, false, 0);
        }
#undef OMX_DL_LAUNCH
    };
    if (whole) launch(whole, 0, 1, nsl, nullptr, ctx->launch_mask);
    if (rest) {
        launch(rest * rsplit, whole, rsplit, sps, (R *)ctx->ws, nullptr);
        hipLaunchKernelGGL((k_dl_split_reduce<R, CF::BM, CF::BN>), dim3(rest, CF::BM * CF::BN / 1024), dim3(256), 0,
                           ctx->stream, m, n, sym, whole, rsplit, (const R *)ctx->ws, alpha, beta0, C0,
                           ldc0, beta, C, ldc);
    }
    OMX_CHECK_HIP(hipGetLastError());
    return OMX_OK;
}

template <typename R, bool TRA, bool TRB, int NPAIR>
static int run_ops(omx_ctx ctx, int m, int n, int k, double alpha, const R *A1, const R *A2, int64_t lda,
                   const R *B1, const R *B2, int64_t ldb, double beta0, const R *C0, int64_t ldc0,
                   double beta, R *C, int64_t ldc, int nbatch = 1, const DlBatch &bat = DlBatch()) {
    const int sym = (m == n && NPAIR == 1 && !TRA && TRB) ? ctx->gemm_sym : 0;
    const int nsl = NPAIR * ((k + DlT<R>::DK - 1) / DlT<R>::DK);
    int splits = nbatch > 1 ? 1 : dgemm_k_splits(ctx, m, n, nsl, sizeof(R));
    // The two products of a pair whose K is no multiple of the slice used to be made in separate passes, and in one chain
    // over both they are rounded 1.4 times as much.  Their sums are kept apart: carried at the seam (FP32, and
    // masked launches, in 64 and 32 tiles), or in two parts of K where the model splits none (pairs against 80 bits,
    // separate passes, one chain, now: FP64 2001 states 1.42e-15, 2.01e-15, 1.42e-15, 1.15 -> 1.21 ms, 4001 2.23e-15,
    // 2.90e-15, 2.23e-15, 7.78 -> 8.01 ms; FP32 2662 9.2e-7, 1.31e-6, 9.2e-7).
    bool seam = NPAIR == 2 && k % DlT<R>::DK != 0 && !(sizeof(R) == 4 ? carries(ctx, m, n) : carries64(ctx, m, n));
    if (seam && sizeof(R) == 8 && !ctx->launch_mask) {
        splits = std::max(splits, 2);
        seam = false;
    }
    const int sps = (nsl + splits - 1) / splits;
    splits = (nsl + sps - 1) / sps;
    const int cls = NPAIR == 2 ? OMX_K_GEMM_PAIR : OMX_K_GEMM;
    const int tile = dl_tile(ctx, sym != 0, m, n, nsl, splits, nbatch, sizeof(R), nullptr, seam);
    hipEvent_t ev;
    prof_begin(ctx, cls, &ev);
    prof_work(ctx, cls, 2.0 * (sym ? sym_area(m, kDlEdge[tile]) : (double)m * n) * (double)NPAIR * k,
              sizeof(R) * ((double)NPAIR * ((double)m * k + (double)k * n) +
                                (double)m * n * (1 + (C0 ? 1 : 0) + (beta != 0.0 ? 1 : 0))));
    int rc;
#define OMX_DL_RUN(CF) \
    run_tile<R, CF, TRA, TRB, NPAIR>(ctx, sym, splits, sps, m, n, k, alpha, A1, A2, lda, B1, B2, ldb, beta0, C0, ldc0, beta, C, ldc, \
                                  nbatch, bat, seam)
    if (tile == 0)
        rc = OMX_DL_RUN(Dl128);
    else if (tile == 1)
        rc = OMX_DL_RUN(Dl64);
    else
        rc = OMX_DL_RUN(Dl32);
#undef OMX_DL_RUN
    prof_end(ctx, cls, ev);
    if (!rc && sym == 2) ctx->gemm_sym = 3;  // the upper triangle is written too
    return rc;
}

template <typename R>
static int launch_dl(omx_ctx ctx, bool trA, bool trB, int npair, int m, int n, int k, double alpha, const R *A1, const R *A2,
                     int64_t lda, const R *B1, const R *B2, int64_t ldb, double beta0, const R *C0, int64_t ldc0, double beta,
                     R *C, int64_t ldc) {
    if (m <= 0 || n <= 0 || k <= 0 || lda > (1 << 20) || ldb > (1 << 20))  // 32-bit lane offsets
        return OMX_ERR_UNSUPPORTED;
#define OMX_DL_OPS(TA, TB, NP) \
    run_ops<R, TA, TB, NP>(ctx, m, n, k, alpha, A1, A2, lda, B1, B2, ldb, beta0, C0, ldc0, beta, C, ldc)
    if (npair == 2) return OMX_DL_OPS(false, false, 2);
    if (!trA && !trB) return OMX_DL_OPS(false, false, 1);
    if (!trA && trB) return OMX_DL_OPS(false, true, 1);
    if (trA && !trB) return OMX_DL_OPS(true, false, 1);
    return OMX_DL_OPS(true, true, 1);
#undef OMX_DL_OPS
}

// The line-search products of one CG step in one launch (see DlBatch), where the model finds that faster than
// one by one: small results leave most of the chip idle each, larger ones are split along K to fill it
// (twelve steps of omm() at 54 x 108 1.65 -> 1.33 ms, four at 1458 x 2916 6.48 -> 6.26 ms).  search_tile: its tile and
// time; search_in_one: whether it is taken.
static int search_tile(omx_ctx ctx, int n, int nsl, int es, double &time) {
    const int first = es == 8 && carries64(ctx, n, n);
    int tile = first;
    for (int q = first; q < 3; ++q) {
        const double t = dl_time(ctx, q, 2LL * (tiles_of(n, n, kDlEdge[q], false) + tiles_of(n, n, kDlEdge[q], true)), nsl);
        if (q == first || t < time) {
            tile = q;
            time = t;
        }
    }
    return tile;
}
bool search_in_one(omx_ctx ctx, int dt, int n, int k, int64_t lda, int64_t ldb) {
    if (n <= 0 || k <= 0 || lda > (1 << 20) || ldb > (1 << 20)) return false;
    const int es = dt == OMX_F64 ? 8 : 4, dk = 128 / es, nsl = (k + dk - 1) / dk, splits = dgemm_k_splits(ctx, n, n, nsl, es);
    double four = 0.0, full = 0.0, lower = 0.0;
    search_tile(ctx, n, nsl, es, four);
    dl_tile(ctx, false, n, n, nsl, splits, 1, es, &full);
    dl_tile(ctx, true, n, n, nsl, splits, 1, es, &lower);
    return four < 2.0 * (full + lower);
}

template <typename R>
static int run_search(omx_ctx ctx, int n, int k, const R *const A[4], int64_t lda, const R *B, int64_t ldb, R *const C[4],
                      int64_t ldc) {
    const int nsl = (k + DlT<R>::DK - 1) / DlT<R>::DK;
    double time = 0.0;
    const int tile = search_tile(ctx, n, nsl, sizeof(R), time);
    DlBatch bat;
    bat.four = 1;
    for (int q = 0; q < 4; ++q) {
        bat.A[q] = A[q];
        bat.C[q] = C[q];
    }
    hipEvent_t ev;
    prof_begin(ctx, OMX_K_GEMM, &ev);
    prof_work(ctx, OMX_K_GEMM, 4.0 * ((double)n * n + sym_area(n, kDlEdge[tile])) * k,
              sizeof(R) * (5.0 * n * k + 4.0 * (double)n * n));
    const dim3 grid(tiles_of(n, n, kDlEdge[tile], false), 4);
    const int carry = sizeof(R) == 4 ? (carries(ctx, n, n) ? 4 : 0) : carries64(ctx, n, n) ? dl_period(ctx, n, n, nsl) : 0;
#define OMX_DL_FOUR(CF, EX, CY)                                                                                            \
    hipLaunchKernelGGL((k_dgemm_dl<R, CF, false, true, 1, EX, CY>), grid, dim3(CF::NT), 0, ctx->stream, n, n, k, 1.0, A[0], \
                       A[0], lda, B, B, ldb, 0.0, (const R *)nullptr, (int64_t)0, 0.0, C[0], ldc, 2, 0, 1, nsl,             \
                       (R *)nullptr, ctx->launch_mask, carry, bat)
    constexpr bool single = sizeof(R) == 4;
    if (tile == 0 && n % 128 == 0 && k % DlT<R>::DK == 0)
        OMX_DL_FOUR(Dl128, true, single);
    else if (tile == 0)
        OMX_DL_FOUR(Dl128, false, single);
    else if (tile == 1 && carry)
        OMX_DL_FOUR(Dl64, false, true);
    else if (tile == 1)
        OMX_DL_FOUR(Dl64, false, single);
    else if (carry)
        OMX_DL_FOUR(Dl32, false, true);
    else
        OMX_DL_FOUR(Dl32, false, single);
#undef OMX_DL_FOUR
    prof_end(ctx, OMX_K_GEMM, ev);
    OMX_CHECK_HIP(hipGetLastError());
    return OMX_OK;
}

int launch_search(omx_ctx ctx, int dt, int n, int k, const void *const A[4], int64_t lda, const void *B, int64_t ldb,
                  void *const C[4], int64_t ldc) {
    if (dt == OMX_F64) {
        const double *const a[4] = {(const double *)A[0], (const double *)A[1], (const double *)A[2], (const double *)A[3]};
        double *const c[4] = {(double *)C[0], (double *)C[1], (double *)C[2], (double *)C[3]};
        return run_search(ctx, n, k, a, lda, (const double *)B, ldb, c, ldc);
    }
    const float *const a[4] = {(const float *)A[0], (const float *)A[1], (const float *)A[2], (const float *)A[3]};
    float *const c[4] = {(float *)C[0], (float *)C[1], (float *)C[2], (float *)C[3]};
    return run_search(ctx, n, k, a, lda, (const float *)B, ldb, c, ldc);
}

int launch_dgemm(omx_ctx ctx, bool trA, bool trB, int npair, int m, int n, int k, double alpha, const double *A1,
                 const double *A2, int64_t lda, const double *B1, const double *B2, int64_t ldb, double beta0,
                 const double *C0, int64_t ldc0, double beta, double *C, int64_t ldc) {
    return launch_dl(ctx, trA, trB, npair, m, n, k, alpha, A1, A2, lda, B1, B2, ldb, beta0, C0, ldc0, beta, C, ldc);
}

int launch_sgemm(omx_ctx ctx, bool trA, bool trB, int npair, int m, int n, int k, double alpha, const float *A1,
                 const float *A2, int64_t lda, const float *B1, const float *B2, int64_t ldb, double beta0, const float *C0,
                 double beta, float *C, int64_t ldc) {
    return launch_dl(ctx, trA, trB, npair, m, n, k, alpha, A1, A2, lda, B1, B2, ldb, beta0, C0, ldc, beta, C, ldc);
}

int launch_dgemm_batched(omx_ctx ctx, int m, int n, int k, double alpha, const double *A, int64_t lda, int64_t sA,
                         const double *B, int64_t ldb, int64_t sB, double *C, int64_t ldc, int64_t sC, int nbatch) {
    if (m <= 0 || n <= 0 || k <= 0 || lda > (1 << 20) || ldb > (1 << 20) || nbatch > 65535) return OMX_ERR_UNSUPPORTED;
    DlBatch bat;
    bat.sA = sA;
    bat.sB = sB;
    bat.sC = sC;
    return run_ops<double, false, false, 1>(ctx, m, n, k, alpha, A, A, lda, B, B, ldb, 0.0, nullptr, 0, 0.0, C, ldc, nbatch, bat);
}

}  // namespace omx

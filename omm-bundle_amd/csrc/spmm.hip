// Dense x block-sparse product Y := alpha*X*A + beta*Y on CDNA4 (the H*C and S*C products of
// the OMM loop; MatrixSwitch/src/MatrixSwitch_mm_multiply.F90:263-327 and
// pspBLAS/src/pspLevel3/pspMspm_nn.F90:58-212 compute the same product from CSC).
//
// X, Y: no x nb column-major; a basis column X(:,k) is a contiguous vector of `no` state
// coefficients.  A: BSR-4 by block columns.  Output column 4J+c is
//     Y(:,4J+c) = sum over blocks (I,J), r = 0..3 of X(:,4I+r) * A_IJ(r,c),
// summed in ascending (I, r), the order of the reference's CSC loop.
//
// Mapping: a workgroup of four waves owns a chunk of RC = 64*VEC*WPG consecutive states (WPG waves
// stacked in rows, each lane loading one 8- or 16-byte vector per basis column; the other waves take
// the neighbouring block columns) and a run of jper block columns per wave, taken in walk order (the
// identity, or an order attached to the operator that keeps the basis columns a block column gathers
// close in time to their other uses, e.g. the lattice in x-y tiles).  Each lane keeps 4*VEC
// accumulators and issues the loads of a whole batch of NB blocks before using them (memory-level
// parallelism); the 16 block values are wave-uniform and come through the scalar cache.  Workgroup
// ids are dealt round-robin over the 8 XCDs, and the id -> (row chunk, block-column run) map is
// XCD-aware:
//   mode 0: XCD x owns a contiguous eighth of the row chunks and cycles through them for one
//           block-column run before the next, so the chip reads whole basis columns at once;
//   mode 1: XCD x owns chunks x, x+8, ... and walks every block column of one chunk before the
//           next, so an XCD's L2 holds the neighbourhood of the current block columns of a
//           single chunk.
// Of the chunks left over (their number mod 8) every XCD walks an eighth of the block columns.
//
// What mattered is how often a basis column crosses from memory into an L2: a column is gathered by
// seven block columns (a lattice operator), up to two lattice planes apart.  The default is therefore
// the narrowest chunk (WPG = 1: 1 KB per basis column, so three planes of 256 sites are 3 MB of a 4 MB
// L2) in mode 1, with large results stored past the L2 (spmm_nt); no load is predicated, and any number
// of states, leading dimension and alignment takes 16-byte vectors.  Measured, default shapes, us
// (before: WPG = 4, chunk counts that 8 does not divide spread over all L2s, predicated loads, scalar
// access unless everything divides and aligns):
//   FP64  8192 x 16384  797 -> 590    4394 x 8788  332 -> 182    2611 x 5280  128 -> 62   54 x 108  6.5 -> 4.9
//   FP32  8192 x 16384  427 -> 300    4394 x 8788  179 -> 107    2611 x 5280   72 -> 39   250 x 500 5.1 -> 5.0
// The copy rate of the card allows 419 and 209 us at the largest size.  There, FP64, 2.8 GB cross
// the L2s' memory side (1.3 times X and Y; 4.4 GB with 512-state chunks) at 4.6 TB/s, a copy at 5.9, and 9.4 GB are
// requested of the L2s.  Which of the two binds is not established: a band of +-3 block columns takes the same time
// with 13 % more of the one and 9 % less of the other.
// A zero entry stored inside a block contributes an exact zero, so the per-element sum equals
// the reference's CSC sum over its stored entries.
#include <algorithm>
#include <utility>

#include "omx_internal.h"
#include "omx_mfma.h"

namespace omx {

template <typename T, int VEC>
struct VecT;
template <>
struct VecT<double, 2> {
    typedef double2 type;
};
template <>
struct VecT<double, 1> {
    typedef double type;
};
template <>
struct VecT<float, 4> {
    typedef float4 type;
};
template <>
struct VecT<float, 1> {
    typedef float type;
};
template <>
struct VecT<float, 2> {
    typedef float2 type;
};

template <typename T, int VEC>
__device__ inline void vload(const T *p, T (&out)[VEC]) {
    typedef typename VecT<T, VEC>::type V;
    V v = *reinterpret_cast<const V *>(p);
    const T *s = reinterpret_cast<const T *>(&v);
#pragma unroll
    for (int q = 0; q < VEC; ++q) out[q] = s[q];
}
template <typename T, int VEC>
__device__ inline void vstore(T *p, const T (&in)[VEC]) {
    typedef typename VecT<T, VEC>::type V;
    V v;
    T *d = reinterpret_cast<T *>(&v);
#pragma unroll
    for (int q = 0; q < VEC; ++q) d[q] = in[q];
    *reinterpret_cast<V *>(p) = v;
}

// The same for vectors aligned only to their elements: one 8- or 16-byte access all the same.
template <typename T, int VEC>
struct UVec {
    typedef T type __attribute__((ext_vector_type(VEC), aligned(sizeof(T))));
};
template <typename T>
struct UVec<T, 1> {
    typedef T type;
};
template <typename T, int VEC>
__device__ inline void uload(const T *p, T (&out)[VEC]) {
    const typename UVec<T, VEC>::type u = *reinterpret_cast<const typename UVec<T, VEC>::type *>(p);
    __builtin_memcpy(out, &u, sizeof out);
}
// nt: past the caches (spmm_nt)
template <typename T, int VEC>
__device__ inline void ustore(T *p, const T (&in)[VEC], int nt) {
    typename UVec<T, VEC>::type u;
    __builtin_memcpy(&u, in, sizeof in);
    typename UVec<T, VEC>::type *q = reinterpret_cast<typename UVec<T, VEC>::type *>(p);
    if (nt) {  // the empty statements keep the compiler from merging the two stores into a plain one
        asm volatile("");
        __builtin_nontemporal_store(u, q);
        asm volatile("");
    } else {
        *q = u;
    }
}

// y := alpha*acc + beta*y_old in FP64 with one explicit rounding sequence (product, then a fused
// multiply-add), so that every SpMM kernel rounds the epilogue identically whatever the compiler's
// contraction choices.
template <typename T>
__device__ inline T spmm_out(double alpha, T acc, double beta, T old) {
    const double p = alpha * (double)acc;
    return (T)(beta != 0.0 ? __builtin_fma(beta, (double)old, p) : p);
}

template <typename T, int VEC, int NB, int WPG>
__global__ __launch_bounds__(256) void k_spmm_bsr4(int no, int nb, int nbc, double alpha,
                                                 const T *__restrict__ X, int64_t ldx,
                                                 const int *__restrict__ colptr, const int *__restrict__ rowidx,
                                                 const double *__restrict__ val, double beta,
                                                 T *__restrict__ Y, int64_t ldy, int nrc, int njg, int jper,
                                                 int mode, int nt, const int *__restrict__ walk,
                                                 const int *__restrict__ mask) {
    constexpr int RC = 64 * VEC * WPG, WJ = 4 / WPG;
    if (mask && !*mask) return;
    const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;  // dispatch is round-robin over 8 XCDs
    const int per = nrc >> 3, rest = nrc & 7;
    int rc, jg;
    if (local < per * njg) {
        if (mode == 0) {
            rc = xcd * per + local % per;
            jg = local / per;
        } else {
            rc = (local / njg) * 8 + xcd;
            jg = local % njg;
        }
    } else {  // the last nrc % 8 chunks: an eighth of the block columns of each on every XCD
        const int e = local - per * njg, eighth = (njg + 7) >> 3;
        rc = per * 8 + e / eighth;
        jg = xcd * eighth + e % eighth;
        if (rc >= nrc || jg >= njg) return;  // whole workgroup
    }
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform block columns
    const int i0 = rc * RC + (threadIdx.x & 63) * VEC + (wave % WPG) * 64 * VEC;
    // Every lane loads a whole vector (no >= VEC): one that would end past the last state is moved back to
    // end there, so no load is predicated; of such a vector the first `skip` states belong to the lane
    // before and are not stored.
    const int at = min(i0, no - VEC), skip = i0 - at;
    const bool any = (i0 < no);
    X += at;
    Y += at;
    const int jbeg = jg * jper * WJ, jend = min(nbc, jbeg + jper * WJ);

    for (int jj = jbeg + wave / WPG; jj < jend; jj += WJ) {
        const int J = walk ? walk[jj] : jj;
        T acc[4][VEC];
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int q = 0; q < VEC; ++q) acc[c][q] = (T)0;
        const int lb = colptr[J], le = colptr[J + 1];
        // Blocks are taken in batches of up to NB: all their basis columns are requested before
        // any is used, so each lane keeps 4*NB vector loads in flight; the accumulation then runs
        // in ascending (block, r) order.
        for (int l0 = lb; l0 < le; l0 += NB) {
            const int nblk = min(NB, le - l0);
            T x[NB][4][VEC];
            int I[NB];
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                if (b < nblk) {
                    I[b] = rowidx[l0 + b];
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        uload<T, VEC>(X + (int64_t)min(4 * I[b] + r, nb - 1) * ldx, x[b][r]);
                }
            }
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                if (b < nblk) {
                    if (4 * I[b] + 4 > nb) {  // the last block row ends at nb: no basis columns past it
#pragma unroll
                        for (int r = 1; r < 4; ++r)
#pragma unroll
                            for (int q = 0; q < VEC; ++q) x[b][r][q] = 4 * I[b] + r < nb ? x[b][r][q] : (T)0;
                    }
                    const double *v = val + 16 * (int64_t)(l0 + b);
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
#pragma unroll
                        for (int c = 0; c < 4; ++c) {
                            const T a = (T)v[r + 4 * c];
#pragma unroll
                            for (int q = 0; q < VEC; ++q) acc[c][q] = fma(x[b][r][q], a, acc[c][q]);
                        }
                    }
                }
            }
        }
        if (!any) continue;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int jcol = 4 * J + c;
            if (jcol >= nb) break;
            T *dst = Y + (int64_t)jcol * ldy;
            T out[VEC];
            if (beta != 0.0) {
                T old[VEC];
                uload<T, VEC>(dst, old);
#pragma unroll
                for (int q = 0; q < VEC; ++q) out[q] = spmm_out(alpha, acc[c][q], beta, old[q]);
            } else {
#pragma unroll
                for (int q = 0; q < VEC; ++q) out[q] = spmm_out(alpha, acc[c][q], 0.0, (T)0);
            }
            if (skip == 0) {
                ustore<T, VEC>(dst, out, nt);
            } else {
#pragma unroll
                for (int q = 1; q < VEC; ++q)
                    if (q >= skip) dst[q] = out[q];
            }
        }
    }
}

// ---- 2.5-D kernel for lattice operators ------------------------------------------------------
// An operator whose pattern is the periodic 7-point stencil of an Lx x Ly x Lz lattice of 4x4
// blocks (block column J = site x + Lx*(y + Ly*z) holds exactly the blocks of J, x+-1, y+-1,
// z+-1; recognised at upload, omx_bsr_s::lat) gathers each basis column 7 times.  Here a
// workgroup owns one row chunk (RW = 64*VEC states) of a 4x4 tile of sites and marches through
// the tile's z-planes: wave w owns site w of the tile and keeps its own basis columns of planes
// z-1, z, z+1 in registers (z+2 in flight); the plane-z columns of the tile and of its 16-site halo
// (x-1, x+4, y-1, y+4 edges, one site per wave) are in LDS, double-buffered by plane parity, where
// the in-plane neighbours are read.  Each basis column then crosses from L2 about twice (own +
// halo) instead of 7 times.  The 7 blocks of a column are taken in stored order with the FMA
// sequence of k_spmm_bsr4, so the results are the same bits.
// Measured at n = 16384 (FP64): 1.2x the algorithmic HBM bytes (2.6 GB per launch against 2.8 GB
// for k_spmm_bsr4), but 0.89 ms against 0.59 ms (FP32: 0.57 against 0.30 ms): one
// workgroup per CU (128 KB of LDS) and a barrier per plane.  The block values come through the
// scalar cache (broadcast with v_readlane they cost 2.6x the VALU instructions of k_spmm_bsr4 and
// the kernel 1.08 ms).  It is therefore opt-in (omx_spmm_stencil).
constexpr int ST_TX = 4, ST_TY = 4, ST_WAVES = ST_TX * ST_TY, ST_SLOTS = ST_WAVES + 2 * (ST_TX + ST_TY);
constexpr int ST_VBYTES = 8;  // bytes per lane and basis column: 64 FP64 or 128 FP32 states per wave

// Workgroup barrier for LDS traffic only: this wave's LDS operations complete (lgkmcnt(0)), then
// s_barrier.  Global loads in flight (the prefetch of later planes into registers) are not waited
// for; the compiler waits for them where their registers are used.  The signal fences keep the
// compiler from moving LDS accesses across the barrier.
__device__ inline void lds_barrier() {
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0xc07f);  // gfx9 encoding: vmcnt 63, expcnt 7, lgkmcnt 0
    __builtin_amdgcn_s_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// Sorts the 7 (key, tag) pairs by key: a 16-comparator network, checked on all 0/1 inputs.
__device__ inline void sort7(int (&k)[7], int (&d)[7]) {
    constexpr int P[16][2] = {{0, 6}, {2, 3}, {4, 5}, {0, 2}, {1, 4}, {3, 6}, {0, 1}, {2, 5},
                              {3, 4}, {1, 2}, {4, 6}, {2, 3}, {4, 5}, {1, 2}, {3, 4}, {5, 6}};
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        const int a = P[q][0], b = P[q][1];
        const bool sw = k[a] > k[b];
        const int ka = sw ? k[b] : k[a], kb = sw ? k[a] : k[b];
        const int da = sw ? d[b] : d[a], db = sw ? d[a] : d[b];
        k[a] = ka;
        k[b] = kb;
        d[a] = da;
        d[b] = db;
    }
}

// f(z0 + k, integral_constant<k>) for k = 0.. while z0 + k < Lz: the march unrolled so that every
// register-ring slot index is a compile-time constant.
template <typename F, int... Ks>
__device__ inline void unroll_steps(F &f, int z0, int Lz, std::integer_sequence<int, Ks...>) {
    ((z0 + Ks < Lz ? f(z0 + Ks, std::integral_constant<int, Ks>{}) : void()), ...);
}

template <typename T, int MINB>
__global__ __launch_bounds__(64 * ST_WAVES, MINB) void k_spmm_stencil(int no, int Lx, int Ly, int Lz, double alpha,
                                                                 const T *__restrict__ X, int64_t ldx,
                                                                 const int *__restrict__ colptr,
                                                                 const int *__restrict__ rowidx,
                                                                 const double *__restrict__ val, double beta,
                                                                 T *__restrict__ Y, int64_t ldy, int nrc, int ntx,
                                                                 int ntiles, const int *__restrict__ mask) {
    constexpr int VEC = ST_VBYTES / sizeof(T);
    constexpr int RW = 64 * VEC;
    __shared__ __align__(16) T lds[2][ST_SLOTS][4][RW];
    if (mask && !*mask) return;
    const int wid = blockIdx.x;
    int rc, t;
    if ((nrc & 7) == 0) {
        // dispatch is round-robin over the 8 XCDs: the tiles of one row chunk run on one XCD, so the
        // halo columns a tile reads are the plane its neighbours are loading into that XCD's L2
        const int xcd = wid & 7, local = wid >> 3;
        rc = (local / ntiles) * 8 + xcd;
        t = local % ntiles;
    } else {
        rc = wid / ntiles;
        t = wid % ntiles;
    }
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int bx = (t % ntx) * ST_TX, by = (t / ntx) * ST_TY;
    const int tx = w % ST_TX, ty = w / ST_TX;
    const int ox = bx + tx, oy = by + ty;  // own site of wave w
    // halo site of wave w: edges x = bx-1, x = bx+4 (k = y offset), y = by-1, y = by+4 (k = x offset)
    const int side = w / 4, k = w % 4;
    int hx, hy;
    if (side == 0) {
        hx = bx - 1; hy = by + k;
    } else if (side == 1) {
        hx = bx + ST_TX; hy = by + k;
    } else if (side == 2) {
        hx = bx + k; hy = by - 1;
    } else {
        hx = bx + k; hy = by + ST_TY;
    }
    hx = (hx + Lx) % Lx;
    hy = (hy + Ly) % Ly;
    const int plane = Lx * Ly;
    const int own_xy = ox + Lx * oy, halo_xy = hx + Lx * hy;
    const int i0 = rc * RW + lane * VEC;
    const bool full = (i0 + VEC <= no);
    const bool any = (i0 < no);
    // in-plane neighbours of the own site: their LDS slots (own tile or halo edge)
    const int slot_xm = (tx > 0) ? w - 1 : ST_WAVES + 0 * 4 + ty;
    const int slot_xp = (tx < ST_TX - 1) ? w + 1 : ST_WAVES + 1 * 4 + ty;
    const int slot_ym = (ty > 0) ? w - ST_TX : ST_WAVES + 2 * 4 + tx;
    const int slot_yp = (ty < ST_TY - 1) ? w + ST_TX : ST_WAVES + 3 * 4 + tx;
    const int xy_xm = (ox + Lx - 1) % Lx + Lx * oy, xy_xp = (ox + 1) % Lx + Lx * oy;
    const int xy_ym = ox + Lx * ((oy + Ly - 1) % Ly), xy_yp = ox + Lx * ((oy + 1) % Ly);

    auto load = [&](int site, T (&x)[4][VEC]) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const T *src = X + (int64_t)(4 * site + r) * ldx + i0;
            if (full) {
                vload<T, VEC>(src, x[r]);
            } else {
#pragma unroll
                for (int q = 0; q < VEC; ++q) x[r][q] = (any && i0 + q < no) ? src[q] : (T)0;
            }
        }
    };
    auto to_lds = [&](int buf, int slot, const T (&x)[4][VEC]) {
#pragma unroll
        for (int r = 0; r < 4; ++r) vstore<T, VEC>(&lds[buf][slot][r][lane * VEC], x[r]);
    };
    auto fma_block = [&](const T (&x)[4][VEC], const double *__restrict__ v, T (&acc)[4][VEC]) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const T a = (T)v[r + 4 * c];
#pragma unroll
                for (int q = 0; q < VEC; ++q) acc[c][q] = fma(x[r][q], a, acc[c][q]);
            }
    };
    // plane z of the march: xm, xc, xp hold the own site's planes z-1, z, z+1, hc the halo of plane
    // z+1 and buffer z&1 plane z of the tile and halo.  The step loads the own plane z+2 into xn and
    // the halo of plane z+2 into hn (a step ahead of their use), computes plane z, then stages plane
    // z+1 (xp, hc) into the other buffer.
    // Register rings, slots fixed at compile time (plane p of the own site in own[p % 5], halo plane
    // p in halo[p % 3]): the step of plane z computes from planes z-1, z, z+1, stages plane z+1 and
    // the halo of plane z+1 into the other LDS buffer, and loads the own plane z+3 and the halo of
    // plane z+3, two steps before their use.
    T own[5][4][VEC], halo[3][4][VEC];
    auto step = [&](int z, auto K) {
        constexpr int k = decltype(K)::value;  // z % 15
        T (&xm)[4][VEC] = own[(k + 4) % 5];
        T (&xc)[4][VEC] = own[k % 5];
        T (&xp)[4][VEC] = own[(k + 1) % 5];
        T (&hc)[4][VEC] = halo[(k + 1) % 3];
        const bool more = (z + 1 < Lz);
        if (z + 2 < Lz) load(own_xy + plane * ((z + 3) % Lz), own[(k + 3) % 5]);
        if (z + 3 < Lz) load(halo_xy + plane * (z + 3), halo[k % 3]);
        const int buf = z & 1;
        const int zo = plane * z;
        const int J = own_xy + zo;
        const int Jzm = own_xy + plane * ((z + Lz - 1) % Lz), Jzp = own_xy + plane * ((z + 1) % Lz);
        T acc[4][VEC];
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int q = 0; q < VEC; ++q) acc[c][q] = (T)0;
        // the stored (ascending block row) order of the 7 blocks: sort the neighbour sites, each
        // tagged with where its basis columns are (0 self, 1 z-1, 2 z+1, 3..6 the LDS slots of x-1,
        // x+1, y-1, y+1)
        int key[7] = {J, Jzm, Jzp, xy_xm + zo, xy_xp + zo, xy_ym + zo, xy_yp + zo};
        int dir[7] = {0, 1, 2, 3, 4, 5, 6};
        sort7(key, dir);
        int dpack = 0;
#pragma unroll
        for (int b = 0; b < 7; ++b) dpack |= dir[b] << (3 * b);
        // The 7 blocks of block column J are stored at 7J..7J+6 (every column of a recognised
        // lattice holds exactly 7), so their 112 values are contiguous at val + 112 J; J is
        // wave-uniform, so a block's 16 values come through the scalar cache.  A loop, not
        // unrolled: one block's values (32 scalar registers) live at a time.
        const double *vals = val + 112 * (int64_t)J;
#pragma unroll 1
        for (int b = 0; b < 7; ++b) {
            const double *a = vals + 16 * b;
            const int d = (dpack >> (3 * b)) & 7;
            if (d == 0) {
                fma_block(xc, a, acc);
            } else if (d == 1) {
                fma_block(xm, a, acc);
            } else if (d == 2) {
                fma_block(xp, a, acc);
            } else {
                const int slot = (d == 3) ? slot_xm : (d == 4) ? slot_xp : (d == 5) ? slot_ym : slot_yp;
                T x[4][VEC];
#pragma unroll
                for (int r = 0; r < 4; ++r) vload<T, VEC>(&lds[buf][slot][r][lane * VEC], x[r]);
                fma_block(x, a, acc);
            }
        }
        if (any) {
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                T *dst = Y + (int64_t)(4 * J + c) * ldy + i0;
                T out[VEC];
                if (full) {
                    if (beta != 0.0) {
                        T old[VEC];
                        vload<T, VEC>(dst, old);
#pragma unroll
                        for (int q = 0; q < VEC; ++q) out[q] = spmm_out(alpha, acc[c][q], beta, old[q]);
                    } else {
#pragma unroll
                        for (int q = 0; q < VEC; ++q) out[q] = spmm_out(alpha, acc[c][q], 0.0, (T)0);
                    }
                    vstore<T, VEC>(dst, out);
                } else {
#pragma unroll
                    for (int q = 0; q < VEC; ++q)
                        if (i0 + q < no) dst[q] = spmm_out(alpha, acc[c][q], beta, beta != 0.0 ? dst[q] : (T)0);
                }
            }
        }
        if (more) {
            // buffer (z+1)&1 was last read in the step of plane z-1, which every wave finished
            // before the barrier that ended it
            to_lds(buf ^ 1, w, xp);
            to_lds(buf ^ 1, ST_WAVES + w, hc);
        }
        lds_barrier();
    };

    load(own_xy + plane * (Lz - 1), own[4]);
    load(own_xy, own[0]);
    load(own_xy + plane, own[1]);
    load(own_xy + plane * 2, own[2]);
    load(halo_xy, halo[0]);
    load(halo_xy + plane, halo[1]);
    if (Lz > 2) load(halo_xy + plane * 2, halo[2]);
    to_lds(0, w, own[0]);
    to_lds(0, ST_WAVES + w, halo[0]);
    lds_barrier();
    for (int z0 = 0; z0 < Lz; z0 += 15) unroll_steps(step, z0, Lz, std::make_integer_sequence<int, 15>{});
}

template <typename T>
static void launch_spmm_stencil(omx_ctx ctx, int no, double alpha, const T *X, int64_t ldx, omx_bsr A, double beta,
                                T *Y, int64_t ldy) {
    constexpr int RW = 64 * (ST_VBYTES / sizeof(T));
    const int nrc = (no + RW - 1) / RW;
    const int ntx = A->lat[0] / ST_TX, nty = A->lat[1] / ST_TY;
    const unsigned grid = (unsigned)((int64_t)nrc * ntx * nty);
    hipLaunchKernelGGL((k_spmm_stencil<T, 2>), dim3(grid), dim3(64 * ST_WAVES), 0, ctx->stream, no, A->lat[0], A->lat[1],
                       A->lat[2], alpha, X, ldx, A->d_colptr, A->d_rowidx, A->d_val, beta, Y, ldy, nrc, ntx,
                       ntx * nty, ctx->launch_mask);
}

// The stencil kernel applies to a recognised lattice with Lx, Ly multiples of the 4x4 tile, with
// its 8-byte vectors aligned (FP32: no, the leading dimensions and the base addresses even).
template <typename T>
static bool stencil_applies(const omx_ctx ctx, const omx_bsr A, int no, const T *X, int64_t ldx, const T *Y,
                            int64_t ldy) {
    constexpr int V = ST_VBYTES / sizeof(T);
    const bool aligned = (no % V == 0) && (ldx % V == 0) && (ldy % V == 0) &&
                         ((uintptr_t)X % ST_VBYTES == 0) && ((uintptr_t)Y % ST_VBYTES == 0);
    return A->lat[0] > 0 && A->lat[0] % ST_TX == 0 && A->lat[1] % ST_TY == 0 && A->lat[2] >= 3 && !A->d_walk &&
           A->group == 0 && !ctx->spmm_forced && ctx->spmm_stencil && aligned && A->nb == 4 * A->nbc &&
           (int64_t)((no + 64 * V - 1) / (64 * V)) * (A->lat[0] / ST_TX) * (A->lat[1] / ST_TY) < (1LL << 31);
}

typedef omx_spmm_shape_s SpmmShape;

// Results go past the caches where they are more than the memory-side cache holds (256 MB), so that the
// L2s keep the basis columns that later block columns gather (FP64, same run, 8192 x 16384: 535 us instead of 566
// with results kept in the caches, 4394 x 8788: 171 instead of 195); smaller results stay for the product that reads them next (complex128,
// 2000 x 4000, SpMM and Gram: 1168 us against 1200).
static int spmm_nt(double bytes) { return bytes > 256e6; }

template <typename T, int VEC, int NB>
static void launch_spmm(omx_ctx ctx, const SpmmShape &sh, int no, int nb, double alpha, const T *X, int64_t ldx,
                        omx_bsr A, double beta, T *Y, int64_t ldy) {
    const int nrc = (no + 64 * VEC * sh.wpg - 1) / (64 * VEC * sh.wpg);
    const int jg = sh.jper * (4 / sh.wpg), njg = (A->nbc + jg - 1) / jg;
    const unsigned grid = (unsigned)(8 * ((int64_t)(nrc >> 3) * njg + (nrc & 7) * ((njg + 7) >> 3)));
#define OMX_SPMM_LAUNCH(W)                                                                                       \
    hipLaunchKernelGGL((k_spmm_bsr4<T, VEC, NB, W>), dim3(grid), dim3(256), 0, ctx->stream, no, nb, A->nbc, \
                       alpha, X, ldx, A->d_colptr, A->d_rowidx, A->d_val, beta, Y, ldy, nrc, njg, sh.jper,   \
                       sh.mode, spmm_nt(sizeof(T) * (double)no * nb), A->d_walk, ctx->launch_mask)
    if (sh.wpg == 1)
        OMX_SPMM_LAUNCH(1);
    else if (sh.wpg == 2)
        OMX_SPMM_LAUNCH(2);
    else
        OMX_SPMM_LAUNCH(4);
#undef OMX_SPMM_LAUNCH
}

template <typename T, int VEC>
static void launch_spmm_shape(omx_ctx ctx, const SpmmShape &sh, int no, int nb, double alpha, const T *X,
                              int64_t ldx, omx_bsr A, double beta, T *Y, int64_t ldy) {
    if (sh.batch >= 8)
        launch_spmm<T, VEC, 8>(ctx, sh, no, nb, alpha, X, ldx, A, beta, Y, ldy);
    else if (sh.batch >= 4)
        launch_spmm<T, VEC, 4>(ctx, sh, no, nb, alpha, X, ldx, A, beta, Y, ldy);
    else
        launch_spmm<T, VEC, 1>(ctx, sh, no, nb, alpha, X, ldx, A, beta, Y, ldy);
}

static int64_t spmm_grid(const SpmmShape &sh, int rows_per_wave, int no, int nbc) {
    const int64_t nrc = (no + (int64_t)rows_per_wave * sh.wpg - 1) / ((int64_t)rows_per_wave * sh.wpg);
    return (nrc + 8) * ((nbc + sh.jper - 1) / sh.jper + 8);
}

// Autotuner for the SpMM launch shape: the first time an operator shape is seen with tuning on,
// the candidate shapes are timed into a scratch result (one warm-up and one timed launch each)
// and the fastest is remembered.
template <typename T, int VEC>
static int tuned_spmm_shape(omx_ctx ctx, int no, int nb, const T *X, int64_t ldx, omx_bsr A, SpmmShape &out) {
    char key[160];
    snprintf(key, sizeof key, "spmm es=%d vec=%d no=%d nb=%d nnzb=%lld walk=%d", (int)sizeof(T), VEC, no, nb,
             (long long)A->nnzb, A->d_walk ? 1 : 0);
    auto it = ctx->tune_spmm.find(key);
    if (it != ctx->tune_spmm.end()) {
        out = it->second.first;
        return OMX_OK;
    }
    std::vector<SpmmShape> cands;
    for (int mode : {0, 1})
        for (int w : {1, 2, 4})
            for (int b : {4, 8})
                for (int jp : {1, 4}) {
                    SpmmShape sh;
                    sh.batch = b;
                    sh.wpg = w;
                    sh.jper = jp;
                    sh.mode = mode;
                    if (spmm_grid(sh, 64 * VEC, no, A->nbc) < (1LL << 31)) cands.push_back(sh);
                }
    OMX_REQUIRE(!cands.empty(), "omx_spmm: grid too large");
    T *tmp = nullptr;
    OMX_CHECK_HIP(dev_malloc((void **)&tmp, sizeof(T) * (size_t)no * nb));
    hipEvent_t e0, e1;
    OMX_CHECK_HIP(hipEventCreate(&e0));
    OMX_CHECK_HIP(hipEventCreate(&e1));
    SpmmShape best = cands[0];
    float best_ms = -1.0f;
    for (const SpmmShape &sh : cands) {
        float ms = 0.0f;
        for (int rep = 0; rep < 2; ++rep) {
            (void)hipEventRecord(e0, ctx->stream);
            launch_spmm_shape<T, VEC>(ctx, sh, no, nb, 1.0, X, ldx, A, 0.0, tmp, no);
            (void)hipEventRecord(e1, ctx->stream);
            (void)hipEventSynchronize(e1);
            (void)hipEventElapsedTime(&ms, e0, e1);
        }
        if (best_ms < 0.0f || ms < best_ms) {
            best = sh;
            best_ms = ms;
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    (void)hipFree(tmp);
    OMX_CHECK_HIP(hipGetLastError());
    ctx->tune_spmm[key] = {best, (double)best_ms};
    out = best;
    return OMX_OK;
}

// LDS-staged gathers (the operator carries a group plan, omx_bsr_set_walk_groups).  The work
// items are (chunk of PR = 64 states, group of block columns consecutive in walk order).  For an
// item, a workgroup loads the distinct basis-column blocks the whole group gathers, for its 64
// states, into LDS (16-byte loads along the states); then each wave computes block columns of the
// group from LDS with one state per lane.  Each block column's blocks are taken in ascending
// (block, r) order with the same FMAs as k_spmm_bsr4, so the results are bitwise equal; what
// changes is that a block shared by several block columns of the group crosses from L2 once.
// The grid is persistent: 8*K workgroups, workgroup (x, i) on XCD x (dispatch is round-robin over
// the 8 XCDs) takes the items of that XCD's state chunks (x, x+8, ...) with stride K, so the K
// workgroups of an XCD walk neighbouring groups of one chunk together and share its L2.  The next
// item's gathers are loaded into registers while the current item computes from LDS.
constexpr int PATCH_ROWS = 64, PATCH_UMAX = 40, PATCH_NT = 256;

template <typename T>
__global__ __launch_bounds__(PATCH_NT, 2) void k_spmm_patch(int no, int nb, int nbc, double alpha,
                                                            const T *__restrict__ X, int64_t ldx,
                                                            const int *__restrict__ colptr,
                                                            const double *__restrict__ val,
                                                            const int *__restrict__ walk, int group, int ngroups,
                                                            const int *__restrict__ gptr,
                                                            const int *__restrict__ uidx,
                                                            const unsigned char *__restrict__ slot, double beta,
                                                            T *__restrict__ Y, int64_t ldy, int nrc,
                                                            const int *__restrict__ mask) {
    constexpr int PR = PATCH_ROWS;
    constexpr int VEC = 16 / sizeof(T);
    constexpr int VPC = PR / VEC;                               // vectors per block column of a chunk
    constexpr int NV = PATCH_UMAX * 4 * VPC / PATCH_NT;         // vectors per thread at most
    static_assert(NV * PATCH_NT == PATCH_UMAX * 4 * VPC, "LDS tile not divisible");
    typedef typename VecT<T, VEC>::type V;
    __shared__ V xs[PATCH_UMAX * 4 * VPC];
    if (mask && !*mask) return;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const bool xcd_map = (nrc & 7) == 0 && (gridDim.x & 7) == 0;
    const int K = xcd_map ? (int)gridDim.x >> 3 : (int)gridDim.x;
    const int x = xcd_map ? (int)blockIdx.x & 7 : 0, first = xcd_map ? (int)blockIdx.x >> 3 : (int)blockIdx.x;
    const int64_t nitems = xcd_map ? (int64_t)(nrc >> 3) * ngroups : (int64_t)nrc * ngroups;
    auto decode = [&](int64_t k, int &rc, int &g) {
        if (xcd_map) {
            rc = (int)(k / ngroups) * 8 + x;
            g = (int)(k % ngroups);
        } else {
            rc = (int)(k / ngroups);
            g = (int)(k % ngroups);
        }
    };
    const bool xal = (ldx % VEC == 0) && ((reinterpret_cast<uintptr_t>(X) & 15) == 0);
    V regs[NV];
    auto fetch = [&](int rc, int g) {
        const int r0 = rc * PR, u0 = gptr[g], nv = (gptr[g + 1] - u0) * 4 * VPC;
        const bool full = xal && (r0 + PR <= no);
#pragma unroll
        for (int q = 0; q < NV; ++q) {
            const int e = tid + PATCH_NT * q;
            if (e < nv) {
                const int rv = (e % VPC) * VEC, uc = e / VPC;
                const int col = 4 * uidx[u0 + (uc >> 2)] + (uc & 3);
                const T *src = X + (int64_t)col * ldx + r0 + rv;
                if (col < nb && full) {
                    regs[q] = *reinterpret_cast<const V *>(src);
                } else {
                    T t[VEC];
#pragma unroll
                    for (int h = 0; h < VEC; ++h) t[h] = (col < nb && r0 + rv + h < no) ? src[h] : (T)0;
                    regs[q] = *reinterpret_cast<const V *>(t);
                }
            }
        }
    };
    int64_t k = first;
    int rc = 0, g = 0;
    if (k < nitems) {
        decode(k, rc, g);
        fetch(rc, g);
    }
    while (k < nitems) {
        const int nv = (gptr[g + 1] - gptr[g]) * 4 * VPC;
        __syncthreads();  // the previous item's reads of xs are done
#pragma unroll
        for (int q = 0; q < NV; ++q) {
            const int e = tid + PATCH_NT * q;
            if (e < nv) xs[e] = regs[q];
        }
        __syncthreads();
        const int crc = rc, cg = g;
        const int64_t kn = k + K;
        if (kn < nitems) {  // next item's gathers in flight while this one computes
            decode(kn, rc, g);
            fetch(rc, g);
        }
        const T *xt = reinterpret_cast<const T *>(xs);
        const int i = crc * PR + lane;
        const int jb = cg * group, je = min(nbc, jb + group);
        for (int jj = jb + wv; jj < je; jj += PATCH_NT / 64) {
            const int J = walk ? walk[jj] : jj;
            T acc[4] = {(T)0, (T)0, (T)0, (T)0};
            const int lb = colptr[J], le = colptr[J + 1];
            // blocks in batches of 8: their slots and LDS reads are issued together, then the FMAs
            // run in ascending (block, r) order
            for (int l0 = lb; l0 < le; l0 += 8) {
                const int nblk = min(8, le - l0);
                int sl[8];
#pragma unroll
                for (int b = 0; b < 8; ++b) sl[b] = b < nblk ? (int)slot[l0 + b] : 0;
                T xr[8][4];
#pragma unroll
                for (int b = 0; b < 8; ++b)
#pragma unroll
                    for (int r = 0; r < 4; ++r) xr[b][r] = b < nblk ? xt[(sl[b] * 4 + r) * PR + lane] : (T)0;
#pragma unroll
                for (int b = 0; b < 8; ++b) {
                    if (b < nblk) {
                        const double *v = val + 16 * (int64_t)(l0 + b);
#pragma unroll
                        for (int r = 0; r < 4; ++r)
#pragma unroll
                            for (int c = 0; c < 4; ++c) acc[c] = fma(xr[b][r], (T)v[r + 4 * c], acc[c]);
                    }
                }
            }
            if (i >= no) continue;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int jcol = 4 * J + c;
                if (jcol >= nb) break;
                T *dst = Y + (int64_t)jcol * ldy + i;
                *dst = spmm_out(alpha, acc[c], beta, beta != 0.0 ? *dst : (T)0);
            }
        }
        k = kn;
    }
}

template <typename T>
static void launch_spmm_patch(omx_ctx ctx, int no, int nb, double alpha, const T *X, int64_t ldx, omx_bsr A,
                              double beta, T *Y, int64_t ldy) {
    const int nrc = (no + PATCH_ROWS - 1) / PATCH_ROWS;
    const int64_t items = (int64_t)nrc * A->ngroups;
    // two workgroups per CU, all resident; fewer when there are fewer items
    const int64_t want = 8LL * std::max(1, 2 * ctx->num_cus / 8);
    const unsigned grid = (unsigned)std::max<int64_t>(1, std::min<int64_t>(want, items));
    hipLaunchKernelGGL(k_spmm_patch<T>, dim3(grid), dim3(PATCH_NT), 0, ctx->stream, no, nb, A->nbc, alpha, X, ldx,
                       A->d_colptr, A->d_val, A->d_walk, A->group, A->ngroups, A->d_gptr, A->d_uidx, A->d_slot, beta,
                       Y, ldy, nrc, ctx->launch_mask);
}

template <typename T, int VEC>
static int run_spmm(omx_ctx ctx, int no, int nb, double alpha, const T *X, int64_t ldx, omx_bsr A, double beta, T *Y,
                    int64_t ldy) {
    if (A->group > 0 && !ctx->spmm_forced) {
        OMX_REQUIRE((int64_t)((no + PATCH_ROWS - 1) / PATCH_ROWS) * A->ngroups < (1LL << 31), "omx_spmm: grid too large");
        hipEvent_t ev;
        prof_begin(ctx, OMX_K_SPMM, &ev);
        prof_work(ctx, OMX_K_SPMM, 2.0 * 16.0 * A->nnzb * no,
                  sizeof(T) * 2.0 * (double)no * nb * (beta != 0.0 ? 1.5 : 1.0) + A->nnzb * (16.0 * 8 + 4) +
                      4.0 * (A->nbc + 1));
        launch_spmm_patch<T>(ctx, no, nb, alpha, X, ldx, A, beta, Y, ldy);
        prof_end(ctx, OMX_K_SPMM, ev);
        OMX_CHECK_HIP(hipGetLastError());
        return OMX_OK;
    }
    if (stencil_applies<T>(ctx, A, no, X, ldx, Y, ldy)) {
        hipEvent_t ev;
        prof_begin(ctx, OMX_K_SPMM, &ev);
        prof_work(ctx, OMX_K_SPMM, 2.0 * 16.0 * A->nnzb * no,
                  sizeof(T) * 2.0 * (double)no * nb * (beta != 0.0 ? 1.5 : 1.0) + A->nnzb * (16.0 * 8 + 4) +
                      4.0 * (A->nbc + 1));
        launch_spmm_stencil<T>(ctx, no, alpha, X, ldx, A, beta, Y, ldy);
        prof_end(ctx, OMX_K_SPMM, ev);
        OMX_CHECK_HIP(hipGetLastError());
        return OMX_OK;
    }
    SpmmShape sh;
    if (ctx->spmm_forced) {
        sh = ctx->spmm_shape;  // forced (omx_spmm_set_tile)
    } else if (ctx->autotune) {
        int rc = tuned_spmm_shape<T, VEC>(ctx, no, nb, X, ldx, A, sh);
        if (rc) return rc;
    }
    OMX_REQUIRE(spmm_grid(sh, 64 * VEC, no, A->nbc) < (1LL << 31), "omx_spmm: grid too large");
    hipEvent_t ev;
    prof_begin(ctx, OMX_K_SPMM, &ev);
    prof_work(ctx, OMX_K_SPMM, 2.0 * 16.0 * A->nnzb * no,
              sizeof(T) * 2.0 * (double)no * nb * (beta != 0.0 ? 1.5 : 1.0) + A->nnzb * (16.0 * 8 + 4) + 4.0 * (A->nbc + 1));
    launch_spmm_shape<T, VEC>(ctx, sh, no, nb, alpha, X, ldx, A, beta, Y, ldy);
    prof_end(ctx, OMX_K_SPMM, ev);
    OMX_CHECK_HIP(hipGetLastError());
    return OMX_OK;
}

// Complex operator and complex X, Y (interleaved (re, im), element type R per part): each lane holds
// VEC complex states, the workgroup's waves take neighbouring block columns of one 64*VEC-state band;
// DUAL: the products with two operators of one block pattern, X read once.  Measured, complex128:
// 2000 x 4000 165 -> 75 us (copy rate: 50), 701 x 1512 32 -> 13; complex64 2000 x 4000 83 -> 47 (before:
// the block values loaded by every lane, since the block column came from the thread id, and loads
// predicated).
template <typename R, int VEC, int WPG, bool DUAL>
__global__ __launch_bounds__(64 * WPG) void k_spmm_bsr4_z(int no, int nb, int nbc, double alpha,
                                                        const R *__restrict__ X, int64_t ldx,
                                                        const int *__restrict__ colptr, const int *__restrict__ rowidx,
                                                        const double *__restrict__ val, double beta,
                                                        R *__restrict__ Y, int64_t ldy, int nbands, int jgroups, int nt,
                                                        int64_t sX, int64_t sY, int64_t sV, int nbatch,
                                                        const int *__restrict__ active,
                                                        const double *__restrict__ val2, R *__restrict__ Y2) {
    constexpr int ROWS = 64 * VEC;
    constexpr int NB = 4, NO = DUAL ? 2 : 1;
    // ids are dealt round-robin over the 8 XCDs: a system of a batch (operator values, X and Y offset by
    // its strides), else a row band, stays on one XCD
    int w = blockIdx.x, band, jg, sys = 0;
    if (nbatch > 1) {
        const int per = nbands * jgroups;
        if ((nbatch & 7) == 0) {
            sys = (w >> 3) / per * 8 + (w & 7);
            w = (w >> 3) % per;
        } else {
            sys = w / per;
            w = w % per;
        }
        band = w / jgroups;
        jg = w % jgroups;
    } else {  // as in k_spmm_bsr4, mode 1 (spmm_z_grid launches what each map needs)
        const int xcd = w & 7, local = w >> 3, whole = (nbands >> 3) * jgroups, eighth = (jgroups + 7) >> 3;
        if (local < whole) {
            band = (local / jgroups) * 8 + xcd;
            jg = local % jgroups;
        } else {
            band = (nbands & ~7) + (local - whole) / eighth;
            jg = xcd * eighth + (local - whole) % eighth;
            if (band >= nbands || jg >= jgroups) return;
        }
    }
    if (active && !active[sys]) return;
    // wave-uniform, so that the block values come through the scalar cache
    const int J = jg * WPG + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (J >= nbc) return;  // whole wave; the kernel has no barriers
    // as in k_spmm_bsr4: a vector that would end past the last state is moved back
    const int i0 = band * ROWS + (threadIdx.x & 63) * VEC, at = min(i0, no - VEC), skip = i0 - at;
    X += sys * sX + 2 * at;
    const double *const vals[2] = {val + sys * sV, DUAL ? val2 + sys * sV : nullptr};
    R *const out[2] = {Y + sys * sY + 2 * at, DUAL ? Y2 + sys * sY + 2 * at : nullptr};
    R ar[NO][4][VEC], ai[NO][4][VEC];
#pragma unroll
    for (int o = 0; o < NO; ++o)
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int q = 0; q < VEC; ++q) ar[o][c][q] = ai[o][c][q] = (R)0;
    const int lb = colptr[J], le = colptr[J + 1];
    for (int l0 = lb; l0 < le; l0 += NB) {
        const int nblk = min(NB, le - l0);
        R x[NB][4][2 * VEC];
        int I[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            if (b < nblk) {
                I[b] = rowidx[l0 + b];
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    uload<R, 2 * VEC>(X + 2 * (int64_t)min(4 * I[b] + r, nb - 1) * ldx, x[b][r]);
            }
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            if (b < nblk) {
                if (4 * I[b] + 4 > nb) {  // the last block row ends at nb: no basis columns past it
#pragma unroll
                    for (int r = 1; r < 4; ++r)
#pragma unroll
                        for (int q = 0; q < 2 * VEC; ++q) x[b][r][q] = 4 * I[b] + r < nb ? x[b][r][q] : (R)0;
                }
#pragma unroll
                for (int o = 0; o < NO; ++o) {
                    const double *v = vals[o] + 32 * (int64_t)(l0 + b);
#pragma unroll
                    for (int r = 0; r < 4; ++r)
#pragma unroll
                        for (int c = 0; c < 4; ++c) {
                            const R vr = (R)v[2 * (r + 4 * c)], vi = (R)v[2 * (r + 4 * c) + 1];
#pragma unroll
                            for (int q = 0; q < VEC; ++q) {
                                const R xr = x[b][r][2 * q], xi = x[b][r][2 * q + 1];
                                ar[o][c][q] = fma(xr, vr, ar[o][c][q]);
                                ar[o][c][q] = fma(-xi, vi, ar[o][c][q]);
                                ai[o][c][q] = fma(xr, vi, ai[o][c][q]);
                                ai[o][c][q] = fma(xi, vr, ai[o][c][q]);
                            }
                        }
                }
            }
        }
    }
    if (i0 >= no) return;
#pragma unroll
    for (int o = 0; o < NO; ++o)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int jcol = 4 * J + c;
            if (jcol >= nb) break;
            R *dst = out[o] + 2 * (int64_t)jcol * ldy;
            R res[2 * VEC], old[2 * VEC];
            if (beta != 0.0) uload<R, 2 * VEC>(dst, old);
#pragma unroll
            for (int q = 0; q < VEC; ++q) {
                double orr = alpha * (double)ar[o][c][q], oii = alpha * (double)ai[o][c][q];
                if (beta != 0.0) {
                    orr += beta * (double)old[2 * q];
                    oii += beta * (double)old[2 * q + 1];
                }
                res[2 * q] = (R)orr;
                res[2 * q + 1] = (R)oii;
            }
            if (skip == 0) {
                ustore<R, 2 * VEC>(dst, res, nt);
            } else {
#pragma unroll
                for (int q = 1; q < VEC; ++q)
                    if (q >= skip) {
                        dst[2 * q] = res[2 * q];
                        dst[2 * q + 1] = res[2 * q + 1];
                    }
            }
        }
}

// Workgroups of k_spmm_bsr4_z's map: a batch's systems one after another; a single system (of an operator
// or of a batch of one) in the eight-XCD map, whose left-over bands end in whole eighths.
static int64_t spmm_z_grid(int nbands, int jgroups, int nbatch) {
    if (nbatch > 1) return (int64_t)nbands * jgroups * nbatch;
    return 8 * ((int64_t)(nbands >> 3) * jgroups + (int64_t)(nbands & 7) * ((jgroups + 7) >> 3));
}

template <typename R, int VEC>
static int run_spmm_z(omx_ctx ctx, int no, int nb, double alpha, const R *X, int64_t ldx, omx_bsr A, double beta,
                      R *Y, int64_t ldy) {
    constexpr int ROWS = 64 * VEC, WPG = 4;
    const int nbands = (no + ROWS - 1) / ROWS;
    const int jgroups = (A->nbc + WPG - 1) / WPG;
    const int64_t total = spmm_z_grid(nbands, jgroups, 1);
    OMX_REQUIRE(total < (1LL << 31), "omx_spmm: grid too large");
    hipEvent_t ev;
    prof_begin(ctx, OMX_K_SPMM, &ev);
    prof_work(ctx, OMX_K_SPMM, 8.0 * 16.0 * A->nnzb * no,
              2.0 * sizeof(R) * 2.0 * (double)no * nb * (beta != 0.0 ? 1.5 : 1.0) + A->nnzb * (32.0 * 8 + 4) +
                  4.0 * (A->nbc + 1));
    hipLaunchKernelGGL((k_spmm_bsr4_z<R, VEC, WPG, false>), dim3((unsigned)total), dim3(64 * WPG), 0, ctx->stream, no,
                       nb, A->nbc, alpha, X, ldx, A->d_colptr, A->d_rowidx, A->d_val, beta, Y, ldy, nbands, jgroups,
                       spmm_nt(2.0 * sizeof(R) * no * nb), (int64_t)0, (int64_t)0, (int64_t)0, 1, (const int *)nullptr, (const double *)nullptr,
                       (R *)nullptr);
    prof_end(ctx, OMX_K_SPMM, ev);
    OMX_CHECK_HIP(hipGetLastError());
    return OMX_OK;
}

template <typename R, int VEC>
static int run_spmm_z_batched(omx_ctx ctx, int no, int nb, int nbc, const int *colptr, const int *rowidx, const double *val,
                              const double *val2, int64_t sV, const void *X, int64_t ldx, int64_t sX, void *Y, void *Y2,
                              int64_t ldy, int64_t sY, int nbatch, const int *active) {
    constexpr int ROWS = 64 * VEC, WPG = 4;
    const int nbands = (no + ROWS - 1) / ROWS, jgroups = (nbc + WPG - 1) / WPG;
    const int64_t total = spmm_z_grid(nbands, jgroups, nbatch);
    OMX_REQUIRE(total < (1LL << 31), "batched spmm: grid too large");
    hipLaunchKernelGGL((k_spmm_bsr4_z<R, VEC, WPG, true>), dim3((unsigned)total), dim3(64 * WPG), 0, ctx->stream, no, nb, nbc,
                       1.0, (const R *)X, ldx, colptr, rowidx, val, 0.0, (R *)Y, ldy, nbands, jgroups, 0, 2 * sX, 2 * sY, sV,
                       nbatch, active, val2, (R *)Y2);
    OMX_CHECK_HIP(hipGetLastError());
    return OMX_OK;
}

// Batched complex SpMM (complex128, or complex64 with the FP64 operator values rounded to FP32) of two
// operators over nbatch systems sharing one block pattern: Y_s := X_s * A_s, Y2_s := X_s * B_s, the
// values of A_s and B_s at val + s*sV, val2 + s*sV (doubles), X_s, Y_s and Y2_s at s*sX, s*sY (complex
// elements).
int launch_spmm_z_batched(omx_ctx ctx, int dt, int no, int nb, int nbc, const int *colptr, const int *rowidx,
                          const double *val, const double *val2, int64_t sV, const void *X, int64_t ldx, int64_t sX,
                          void *Y, void *Y2, int64_t ldy, int64_t sY, int nbatch, const int *active) {
    if (dt == OMX_C128)
        return run_spmm_z_batched<double, 1>(ctx, no, nb, nbc, colptr, rowidx, val, val2, sV, X, ldx, sX, Y, Y2, ldy, sY,
                                             nbatch, active);
    return run_spmm_z_batched<float, 1>(ctx, no, nb, nbc, colptr, rowidx, val, val2, sV, X, ldx, sX, Y, Y2, ldy, sY, nbatch,
                                        active);
}

}  // namespace omx

using namespace omx;

extern "C" int omx_spmm_stencil(omx_ctx ctx, int enable) {
    OMX_REQUIRE(ctx, "omx_spmm_stencil: null context");
    ctx->spmm_stencil = (enable != 0);
    return OMX_OK;
}

extern "C" int omx_spmm_set_tile(omx_ctx ctx, int batch, int wpg, int jper, int mode) {
    OMX_REQUIRE(ctx, "omx_spmm_set_tile: null context");
    if (batch == 0) {
        ctx->spmm_forced = false;
        return OMX_OK;
    }
    OMX_REQUIRE((batch == 1 || batch == 4 || batch == 8) && (wpg == 1 || wpg == 2 || wpg == 4) && jper >= 1 &&
                    jper <= 4096 && (mode == 0 || mode == 1),
                "omx_spmm_set_tile: bad shape (batch %d, wpg %d, jper %d, mode %d)", batch, wpg, jper, mode);
    ctx->spmm_shape.batch = batch;
    ctx->spmm_shape.wpg = wpg;
    ctx->spmm_shape.jper = jper;
    ctx->spmm_shape.mode = mode;
    ctx->spmm_forced = true;
    return OMX_OK;
}

static void clear_patch_plan(omx_bsr A) {
    if (A->d_gptr) (void)hipFree(A->d_gptr);
    if (A->d_uidx) (void)hipFree(A->d_uidx);
    if (A->d_slot) (void)hipFree(A->d_slot);
    A->d_gptr = A->d_uidx = nullptr;
    A->d_slot = nullptr;
    A->group = A->ngroups = 0;
}

extern "C" int omx_bsr_set_walk(omx_bsr A, const int *order) {
    OMX_REQUIRE(A, "omx_bsr_set_walk: null operator");
    omx_ctx ctx = A->ctx;
    OMX_CHECK_HIP(hipStreamSynchronize(ctx->stream));
    clear_patch_plan(A);
    if (!order) {
        if (A->d_walk) OMX_CHECK_HIP(hipFree(A->d_walk));
        A->d_walk = nullptr;
        return OMX_OK;
    }
    std::vector<char> seen(A->nbc, 0);
    for (int j = 0; j < A->nbc; ++j) {
        OMX_REQUIRE(order[j] >= 0 && order[j] < A->nbc && !seen[order[j]],
                    "omx_bsr_set_walk: order is not a permutation of the %d block columns (entry %d)", A->nbc, j);
        seen[order[j]] = 1;
    }
    if (!A->d_walk) OMX_CHECK_HIP(dev_malloc((void **)&A->d_walk, sizeof(int) * std::max(A->nbc, 1)));
    OMX_CHECK_HIP(hipMemcpyAsync(A->d_walk, order, sizeof(int) * A->nbc, hipMemcpyHostToDevice, ctx->stream));
    OMX_CHECK_HIP(hipStreamSynchronize(ctx->stream));
    return OMX_OK;
}

// 16-byte vectors once they make more than two waves per CU; below that a lane with one state has the
// shorter chain (FP32, 250 x 500: 5.0 us against 5.9; 432 x 864: 5.2 and 5.9; 686 x 1372, four waves per
// CU: 7.4 and 6.8.  FP64: 250 x 500 4.8 and 5.1, 432 x 864 5.6 and 5.4).
static bool spmm_wide(omx_ctx ctx, int no, int vec, omx_bsr A) {
    return no >= vec && (int64_t)((no + 64 * vec - 1) / (64 * vec)) * A->nbc > 2 * ctx->num_cus;
}

extern "C" int omx_spmm(omx_ctx ctx, int dt, int no, int nb, double alpha, const void *X, int64_t ldx, omx_bsr A,
                        double beta, void *Y, int64_t ldy) {
    OMX_REQUIRE(ctx && A, "omx_spmm: null argument");
    OMX_REQUIRE(nb == A->nb, "omx_spmm: operator is %d x %d but X has %d columns", A->nb, A->nb, nb);
    OMX_REQUIRE(no >= 0 && ldx >= std::max(1, no) && ldy >= std::max(1, no), "omx_spmm: bad leading dimension");
    const bool zdt = (dt == OMX_C128 || dt == OMX_C64);
    OMX_REQUIRE(!A->is_complex || zdt, "omx_spmm: complex operator needs a complex element type");
    if (no == 0) return OMX_OK;
    OMX_REQUIRE(X && Y, "omx_spmm: null operand");
    OMX_REQUIRE(X != Y, "omx_spmm: X and Y must not alias");
    if (zdt) {
        OMX_REQUIRE(A->is_complex, "omx_spmm: complex X needs a complex operator");
        if (dt == OMX_C128) return run_spmm_z<double, 1>(ctx, no, nb, alpha, (const double *)X, ldx, A, beta, (double *)Y, ldy);
        if (no >= 2) return run_spmm_z<float, 2>(ctx, no, nb, alpha, (const float *)X, ldx, A, beta, (float *)Y, ldy);
        return run_spmm_z<float, 1>(ctx, no, nb, alpha, (const float *)X, ldx, A, beta, (float *)Y, ldy);
    }
    if (dt == OMX_F64) {
        if (spmm_wide(ctx, no, 2, A)) return run_spmm<double, 2>(ctx, no, nb, alpha, (const double *)X, ldx, A, beta, (double *)Y, ldy);
        return run_spmm<double, 1>(ctx, no, nb, alpha, (const double *)X, ldx, A, beta, (double *)Y, ldy);
    }
    if (dt == OMX_F32) {
        if (spmm_wide(ctx, no, 4, A)) return run_spmm<float, 4>(ctx, no, nb, alpha, (const float *)X, ldx, A, beta, (float *)Y, ldy);
        return run_spmm<float, 1>(ctx, no, nb, alpha, (const float *)X, ldx, A, beta, (float *)Y, ldy);
    }
    set_error("omx_spmm: unsupported element type %d", dt);
    return OMX_ERR_UNSUPPORTED;
}

// =============================================================================================
// Dense x dense -> block-sparse pattern (SDDMM): Cp := alpha * (A^T B) restricted to the stored
// blocks of Cp + beta * Cp, with A, B no x nb column-major.  Block (I,J), entry (r,c) is the dot
// product over the state index of basis columns 4I+r of A and 4J+c of B.  This is the
// reference's dense*dense -> CSC product (MatrixSwitch/src/MatrixSwitch_mm_multiply.F90:334-398,
// op = 'c','n'), used for the density matrix D = C^T (QW C) on the pattern of H
// (libOMM/src/omm_ops.F90:104-124 with a sparse D_min) and for dE/dH.
//
// Mapping: a wave owns one block column J and a chunk of states.  The 4 x 4 result of a stored block is a
// sum over states, so it runs on v_mfma_f64_4x4x4 (four independent 4x4x4 products): lane l holds column
// l & 3 of the block at the VEC consecutive states that l >> 2 numbers, and the sum over states needs no
// shuffles until the chunk's end, where two add the four products.  A step is 16*VEC states: one load of
// 1 KB straight into LDS for B's columns and one for every stored block's, four runs of 256 bytes each
// (loaded in the matrix core's own layout, neighbouring lanes fall into different lines, and the L1 takes
// 64 cycles per load: 0.92 ms instead of 0.66 at 8192 x 16384).  The tiles' 16-byte vectors are swizzled
// by column (no bank conflicts), and a wave has only one set of them: with 8 KB per wave 20 waves fit on a
// CU and hide each other's waits (two sets, 8 waves: 0.70 ms; three: 1.02).
// Sums are kept short: a block's two accumulators take turns and are added up apart every two steps, the parts of the
// chunks in four sums.  Against 80 bits, FP64, 1458 and 8192 states 1.75e-16 and 2.2e-16 off, as with sums by thread and
// wave (1.74e-16, 2.2e-16); in one chain per chunk and over the chunks 2.4e-16 and 3.4e-16, at the same time (FP32
// 359 us instead of 375).  A block's vectors are read right before their products: all of them at once take the
// registers of a fifth workgroup per CU.
// The block's partial result goes to the workspace, and a second kernel adds the chunks in a
// fixed order.  The id -> (chunk, block columns) map is that of k_spmm_bsr4, mode 1.
//
// Bound by what crosses the L2s' memory side: 4.5 GB are read there per launch at 8192 x 16384, twice the operands
// (probably the waves that gather one basis column run apart and miss each other's lines), at 6.8 TB/s; the matrix cores
// are busy 14 % of the time, and no LDS read conflicts.  Measured, us, before (a thread per state, 17 shuffles per
// block, wave and chunk) and after:
//   FP64  8192 x 16384   976 -> 654   4394 x 8788  337 -> 244   1458 x 2916  34 -> 31   54 x 108  15 -> 9
//   FP32  8192 x 16384  1610 -> 375   4394 x 8788  548 -> 127    250 x 500  20 -> 10
// =============================================================================================
namespace omx {

constexpr int SD_NBK = 7;           // stored blocks taken together (a lattice column's)
constexpr int64_t SD_LD = 1 << 26;  // leading dimensions whose block columns 32-bit offsets reach

template <typename T>
__global__ __launch_bounds__(256, 5) void k_sddmm_bsr4_partial(int no, int nb, int nbc, const T *__restrict__ A, int64_t lda,
                                                          const T *__restrict__ B, int64_t ldb,
                                                          const int *__restrict__ colptr, const int *__restrict__ rowidx,
                                                          int chunk, int nrc, int njg, int64_t nnzb,
                                                          double *__restrict__ partial) {
    constexpr int VEC = 16 / sizeof(T), SV = 16 * VEC, TILE = 4 * SV;  // states of a step, elements of its tile
    __shared__ __align__(16) T smem[4 * (SD_NBK + 1) * TILE];
    const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3, whole = (nrc >> 3) * njg, eighth = (njg + 7) >> 3;
    int rc, jg;
    if (local < whole) {
        rc = (local / njg) * 8 + xcd;
        jg = local % njg;
    } else {
        rc = (nrc & ~7) + (local - whole) / eighth;
        jg = xcd * eighth + (local - whole) % eighth;
        if (rc >= nrc || jg >= njg) return;
    }
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int J = jg * 4 + wave;
    if (J >= nbc) return;  // whole wave; the kernel has no barriers, each wave has its own tiles
    T *const tb = smem + wave * (SD_NBK + 1) * TILE, *const ta = tb + TILE;
    const int lane = threadIdx.x & 63;
    // loads: lane l brings vector (l & 15) ^ 4 c of column c = l >> 4; reads: lane l takes vector l >> 2 of column l & 3
    const int lc = lane >> 4, lv = ((lane & 15) ^ (4 * lc)) * VEC;
    const int col = lane & 3, rv = lane >> 2, at = (col * 16 + (rv ^ (4 * col))) * VEC;
    const int beg = rc * chunk, len = min(no - beg, chunk);
    const int nfull = max(lda, ldb) < SD_LD ? len / SV : 0;  // steps through LDS (32-bit offsets in a block)
    const T *const pb = B + (int64_t)4 * J * ldb + beg;
    const int ob = (min(lc, nb - 1 - 4 * J) * (int)ldb + lv) * (int)sizeof(T);
    const bool jin = 4 * J + col < nb;
    const int le = colptr[J + 1];
    for (int l0 = colptr[J]; l0 < le; l0 += SD_NBK) {
        const int nblk = min(SD_NBK, le - l0);
        int I[SD_NBK];
        int oa[SD_NBK];
        double acc[SD_NBK][2], tot[SD_NBK];
#pragma unroll
        for (int b = 0; b < SD_NBK; ++b) {
            I[b] = rowidx[l0 + min(b, nblk - 1)];
            oa[b] = (min(lc, nb - 1 - 4 * I[b]) * (int)lda + lv) * (int)sizeof(T);
            acc[b][0] = acc[b][1] = tot[b] = 0.0;
        }
        // products of one step: xb and the xa(b) are this lane's vectors of B and of A's block b
        auto products = [&](T (&xb)[VEC], auto xa) {
            if (4 * J + 4 > nb) {  // no basis columns past nb: their results are zero
#pragma unroll
                for (int q = 0; q < VEC; ++q) xb[q] = jin ? xb[q] : (T)0;
            }
#pragma unroll
            for (int b = 0; b < SD_NBK; ++b)
                if (b < nblk) {
                    T x[VEC];
                    xa(b, x);
                    if (4 * I[b] + 4 > nb) {
#pragma unroll
                        for (int q = 0; q < VEC; ++q) x[q] = 4 * I[b] + col < nb ? x[q] : (T)0;
                    }
#pragma unroll
                    for (int q = 0; q < VEC; ++q)
                        acc[b][q & 1] = __builtin_amdgcn_mfma_f64_4x4x4f64((double)x[q], (double)xb[q], acc[b][q & 1], 0, 0, 0);
                }
        };
        auto carry = [&]() {
#pragma unroll
            for (int b = 0; b < SD_NBK; ++b) {
                tot[b] += acc[b][0] + acc[b][1];
                acc[b][0] = acc[b][1] = 0.0;
            }
        };
        auto load = [&](const T *p, T *to, int o) {
            const __amdgpu_buffer_rsrc_t r = raw_rsrc(p);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void *)to, 16, o, 0, 0, 0);
        };
        for (int st = 0; st < nfull; ++st) {
            __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt 0: the tiles of the step before are read
            __atomic_signal_fence(__ATOMIC_SEQ_CST);
            load(pb + st * SV, tb, ob);
#pragma unroll
            for (int b = 0; b < SD_NBK; ++b)
                if (b < nblk) load(A + (int64_t)4 * I[b] * lda + beg + st * SV, ta + b * TILE, oa[b]);
            __builtin_amdgcn_s_waitcnt(waitcnt_vmcnt(0));
            __atomic_signal_fence(__ATOMIC_SEQ_CST);
            T xb[VEC];
            uload<T, VEC>(tb + at, xb);
            products(xb, [&](int b, T (&x)[VEC]) { uload<T, VEC>(ta + b * TILE + at, x); });
            if (st & 1) carry();
        }
        carry();
        for (int st = nfull; st * SV < len; ++st) {  // the last states
            const int s = st * SV + rv * VEC;
            auto tail = [&](const T *p, T (&x)[VEC]) {
#pragma unroll
                for (int q = 0; q < VEC; ++q) x[q] = s + q < len ? p[beg + s + q] : (T)0;
            };
            T xb[VEC];
            tail(B + (int64_t)min(4 * J + col, nb - 1) * ldb, xb);
            products(xb, [&](int b, T (&x)[VEC]) { tail(A + (int64_t)min(4 * I[b] + col, nb - 1) * lda, x); });
        }
#pragma unroll
        for (int b = 0; b < SD_NBK; ++b)
            if (b < nblk) {  // lane j + 4 g + 16 i holds entry (i, j) of product g
                double t = tot[b] + (acc[b][0] + acc[b][1]);
                t += __shfl_xor(t, 4, 64);
                t += __shfl_xor(t, 8, 64);
                if ((lane & 12) == 0) partial[((int64_t)rc * nnzb + l0 + b) * 16 + (lane >> 4) + 4 * col] = t;
            }
    }
}

__global__ void k_sddmm_bsr4_final(int64_t nnzb, int nparts, const double *__restrict__ partial, double alpha,
                                   double beta, double *__restrict__ vals) {
    const int64_t total = nnzb * 16;
    for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < total; q += (int64_t)gridDim.x * blockDim.x) {
        double t[4] = {0.0, 0.0, 0.0, 0.0};  // every fourth part, then the four: shorter chains
        int p = 0;
        for (; p + 4 <= nparts; p += 4)
#pragma unroll
            for (int h = 0; h < 4; ++h) t[h] += partial[(int64_t)(p + h) * total + q];
#pragma unroll
        for (int h = 0; h < 3; ++h)
            if (p + h < nparts) t[h] += partial[(int64_t)(p + h) * total + q];
        const double s = (t[0] + t[1]) + (t[2] + t[3]);
        vals[q] = (beta == 0.0) ? alpha * s : alpha * s + beta * vals[q];
    }
}

template <typename T>
static int run_sddmm(omx_ctx ctx, int no, int nb, double alpha, const T *A, int64_t lda, const T *B, int64_t ldb,
                     double beta, omx_bsr C) {
    // chunks of 512 states (more of them cost partial results), shorter ones while that leaves less than
    // eight waves per CU (432 x 864: 128 states 10 us, 256 12, 512 18; 1458 x 2916: 31, 32, 30)
    int chunk = 512;
    while (chunk > 128 && (int64_t)((no + chunk - 1) / chunk) * C->nbc < 8 * ctx->num_cus) chunk /= 2;
    const int nparts = (no + chunk - 1) / chunk, njg = (C->nbc + 3) / 4;
    const int64_t grid = 8 * ((int64_t)(nparts >> 3) * njg + (nparts & 7) * ((njg + 7) >> 3));
    OMX_REQUIRE(grid < (1LL << 31), "omx_sddmm_bsr: grid too large");
    const size_t bytes = sizeof(double) * 16 * (size_t)C->nnzb * nparts;
    int rc = ensure_ws(ctx, bytes);
    if (rc) return rc;
    double *partial = (double *)ctx->ws;
    hipEvent_t ev;
    prof_begin(ctx, OMX_K_SPMM, &ev);
    prof_work(ctx, OMX_K_SPMM, 2.0 * 16.0 * C->nnzb * no, sizeof(T) * 2.0 * (double)no * nb + C->nnzb * (16.0 * 8 + 4));
    hipLaunchKernelGGL(k_sddmm_bsr4_partial<T>, dim3((unsigned)grid), dim3(256), 0, ctx->stream, no, nb, C->nbc, A, lda, B,
                       ldb, C->d_colptr, C->d_rowidx, chunk, nparts, njg, C->nnzb, partial);
    const int64_t total = C->nnzb * 16;
    const int g2 = (int)std::max<int64_t>(1, std::min<int64_t>((total + 255) / 256, 8192));
    hipLaunchKernelGGL(k_sddmm_bsr4_final, dim3(g2), dim3(256), 0, ctx->stream, C->nnzb, nparts, partial, alpha, beta,
                       C->d_val);
    prof_end(ctx, OMX_K_SPMM, ev);
    OMX_CHECK_HIP(hipGetLastError());
    return OMX_OK;
}

}  // namespace omx

extern "C" int omx_sddmm_bsr(omx_ctx ctx, int dt, int no, int nb, double alpha, const void *A, int64_t lda,
                             const void *B, int64_t ldb, double beta, omx_bsr C) {
    OMX_REQUIRE(ctx && C, "omx_sddmm_bsr: null argument");
    OMX_REQUIRE(nb == C->nb && !C->is_complex, "omx_sddmm_bsr: pattern does not match nb");
    OMX_REQUIRE(no >= 0 && lda >= std::max(1, no) && ldb >= std::max(1, no), "omx_sddmm_bsr: bad leading dimension");
    if (C->nnzb == 0) return OMX_OK;
    if (no == 0) {  // empty contraction: Cp := beta * Cp
        const int g2 = (int)std::max<int64_t>(1, std::min<int64_t>((C->nnzb * 16 + 255) / 256, 8192));
        hipLaunchKernelGGL(k_sddmm_bsr4_final, dim3(g2), dim3(256), 0, ctx->stream, C->nnzb, 0, (const double *)nullptr,
                           alpha, beta, C->d_val);
        OMX_CHECK_HIP(hipGetLastError());
        return OMX_OK;
    }
    OMX_REQUIRE(A && B, "omx_sddmm_bsr: null operand");
    if (dt == OMX_F64) return run_sddmm<double>(ctx, no, nb, alpha, (const double *)A, lda, (const double *)B, ldb, beta, C);
    if (dt == OMX_F32) return run_sddmm<float>(ctx, no, nb, alpha, (const float *)A, lda, (const float *)B, ldb, beta, C);
    set_error("omx_sddmm_bsr: unsupported element type %d", dt);
    return OMX_ERR_UNSUPPORTED;
}

extern "C" int omx_bsr_set_walk_groups(omx_bsr A, const int *order, int group) {
    OMX_REQUIRE(A && group >= 0, "omx_bsr_set_walk_groups: bad arguments");
    int rc = omx_bsr_set_walk(A, order);
    if (rc || group == 0) return rc;
    OMX_REQUIRE(!A->is_complex, "omx_bsr_set_walk_groups: real operators only");
    omx_ctx ctx = A->ctx;
    const int nbc = A->nbc;
    std::vector<int> colptr(nbc + 1), rowidx(std::max<int64_t>(A->nnzb, 1));
    OMX_CHECK_HIP(hipMemcpy(colptr.data(), A->d_colptr, sizeof(int) * (nbc + 1), hipMemcpyDeviceToHost));
    if (A->nnzb) OMX_CHECK_HIP(hipMemcpy(rowidx.data(), A->d_rowidx, sizeof(int) * A->nnzb, hipMemcpyDeviceToHost));
    const int ngroups = (nbc + group - 1) / group;
    std::vector<int> gptr(ngroups + 1, 0), uidx;
    std::vector<unsigned char> slot(std::max<int64_t>(A->nnzb, 1), 0);
    std::vector<int> where(nbc, -1);
    for (int g = 0; g < ngroups; ++g) {
        const int jb = g * group, je = std::min(nbc, jb + group);
        std::vector<int> u;
        for (int jj = jb; jj < je; ++jj) {
            const int J = order ? order[jj] : jj;
            for (int l = colptr[J]; l < colptr[J + 1]; ++l) u.push_back(rowidx[l]);
        }
        std::sort(u.begin(), u.end());
        u.erase(std::unique(u.begin(), u.end()), u.end());
        if ((int)u.size() > PATCH_UMAX) {
            (void)omx_bsr_set_walk(A, order);  // keep the walk, without the plan
            set_error("omx_bsr_set_walk_groups: group %d gathers %d distinct blocks (at most %d)", g, (int)u.size(),
                      PATCH_UMAX);
            return OMX_ERR_ARG;
        }
        for (size_t q = 0; q < u.size(); ++q) where[u[q]] = (int)q;
        for (int jj = jb; jj < je; ++jj) {
            const int J = order ? order[jj] : jj;
            for (int l = colptr[J]; l < colptr[J + 1]; ++l) slot[l] = (unsigned char)where[rowidx[l]];
        }
        uidx.insert(uidx.end(), u.begin(), u.end());
        gptr[g + 1] = (int)uidx.size();
    }
    bool ok = dev_malloc((void **)&A->d_gptr, sizeof(int) * (ngroups + 1)) == hipSuccess &&
              dev_malloc((void **)&A->d_uidx, sizeof(int) * std::max<size_t>(uidx.size(), 1)) == hipSuccess &&
              dev_malloc((void **)&A->d_slot, slot.size()) == hipSuccess;
    if (!ok) {
        clear_patch_plan(A);
        set_error("omx_bsr_set_walk_groups: device allocation failed");
        return OMX_ERR_NOMEM;
    }
    OMX_CHECK_HIP(hipMemcpy(A->d_gptr, gptr.data(), sizeof(int) * (ngroups + 1), hipMemcpyHostToDevice));
    if (!uidx.empty())
        OMX_CHECK_HIP(hipMemcpy(A->d_uidx, uidx.data(), sizeof(int) * uidx.size(), hipMemcpyHostToDevice));
    OMX_CHECK_HIP(hipMemcpy(A->d_slot, slot.data(), slot.size(), hipMemcpyHostToDevice));
    A->group = group;
    A->ngroups = ngroups;
    (void)ctx;
    return OMX_OK;
}

// Workgroup reductions shared by the element-wise kernels and the batched solver (EW_NT threads).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace omx {

constexpr int EW_NT = 256;

// The workgroup's sums of v into out[0..NV-1].  Many values are summed over a wave by recursive halving: at
// offset 32 a lane keeps half of the (sixteen) values and adds its partner's copies of that half, then at 16,
// 8 and 4; two more steps add the four lanes that share a value: 17 shuffles instead of 6 per value (the
// coefficient kernel at 54 x 54 7.5 -> 5.5 us, at 1458 x 1458 33 -> 28).  Few or many, a wave's values are added
// in one order, lanes 32 apart first, then 16, 8, 4, 2 and 1: a CG trajectory hangs on the last bit of these sums.
template <int NV>
__device__ inline void block_reduce_store(double (&v)[NV], double *__restrict__ out) {
    static_assert(NV <= 16, "sixteen values at most");
    __shared__ double red[NV][EW_NT / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if constexpr (NV > 4) {
        double w[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) w[q] = q < NV ? v[q] : 0.0;
#pragma unroll
        for (int half = 8; half >= 1; half >>= 1) {
            const int off = 4 * half;  // 32, 16, 8, 4
            const bool up = lane & off;
#pragma unroll
            for (int q = 0; q < half; ++q) {
                const double keep = up ? w[q + half] : w[q], send = up ? w[q] : w[q + half];
                w[q] = keep + __shfl_xor(send, off, 64);
            }
        }
        double s = w[0];
        s += __shfl_xor(s, 2, 64);
        s += __shfl_xor(s, 1, 64);
        const int q = lane >> 2;  // the value this lane holds
        if ((lane & 3) == 0 && q < NV) red[q][wave] = s;
    } else {
#pragma unroll
        for (int q = 0; q < NV; ++q) {
            double s = v[q];
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
            if (lane == 0) red[q][wave] = s;
        }
    }
    __syncthreads();
    if (threadIdx.x < NV) {
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < EW_NT / 64; ++w) s += red[threadIdx.x][w];
        out[threadIdx.x] = s;
    }
}

// Sums of nblocks groups of NV partial values each, ascending, into out.
template <int NV>
__device__ inline void reduce_partials(int nblocks, const double *__restrict__ partial, double *__restrict__ out) {
    double v[NV];
#pragma unroll
    for (int q = 0; q < NV; ++q) v[q] = 0.0;
    for (int b = threadIdx.x; b < nblocks; b += EW_NT)
#pragma unroll
        for (int q = 0; q < NV; ++q) v[q] += partial[(int64_t)b * NV + q];
    block_reduce_store<NV>(v, out);
}

// True in every thread of the last of the launch's workgroups to get here, once the others' global stores from
// before their calls are visible to it; the ticket is back at 0 then.  (A workgroup's values are stored by
// threads that fence; the release and acquire at device scope cover the L2s of the other XCDs.)
__device__ inline bool last_workgroup(unsigned *ticket) {
    __shared__ bool last;
    __threadfence();
    __syncthreads();
    if (threadIdx.x == 0) {
        last = atomicAdd(ticket, 1u) == gridDim.x - 1;
        if (last) atomicExch(ticket, 0u);
    }
    __syncthreads();
    __threadfence();
    return last;
}

// The line-search coefficients and then their thirteen sums (k_coeff_partial's order) into out[0..17]:
// deterministic per-term sums, then the closed forms, written by thread 0.
__device__ inline void coeff_final(int nblocks, const double *__restrict__ partial, double *__restrict__ out) {
    __shared__ double tr[13];
    reduce_partials<13>(nblocks, partial, tr);
    __syncthreads();
    if (threadIdx.x == 0) {
        const double TrH = tr[0], TrHS = tr[1], TrHd = tr[2], TrHdS = tr[3], TrHSd = tr[4], TrHdd = tr[5],
                     TrHddS = tr[6], TrHSdd = tr[7], TrHdSd = tr[8], TrHdSdH = tr[9], TrHddSd = tr[10],
                     TrHdSdd = tr[11], TrHddSdd = tr[12];
        out[0] = 2.0 * TrH - TrHS;
        out[1] = 2.0 * (2.0 * TrHd - TrHdS - TrHSd);
        out[2] = 2.0 * (TrHdd - TrHdSd - TrHdSdH) - TrHddS - TrHSdd;
        out[3] = -2.0 * (TrHddSd + TrHdSdd);
        out[4] = -TrHddSdd;
        for (int q = 0; q < 13; ++q) out[5 + q] = tr[q];
    }
}

}  // namespace omx

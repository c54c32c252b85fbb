// Device pieces shared by the matrix-core products: vector types, raw buffer descriptors for loads
// straight into LDS, and the waits and barriers those loads need.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

namespace omx {

typedef double d4v __attribute__((ext_vector_type(4)));
typedef float f4v __attribute__((ext_vector_type(4)));
typedef __bf16 bf8v __attribute__((ext_vector_type(8)));

typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(1))) void glb_void;
// s_waitcnt immediate (gfx9 encoding): vmcnt(vm), expcnt and lgkmcnt left at their maxima
constexpr int waitcnt_vmcnt(int vm) { return (vm & 0xF) | ((vm >> 4) << 14) | (7 << 4) | (0xF << 8); }
// Swizzle of the 16-byte chunks of a k-contiguous FP64 tile row (16 k values, 128 bytes)
__device__ inline int dl_swz(int j) { return (j >> 1) & 7; }
// Raw (unstrided) buffer descriptor over `bytes` bytes from p, for the buffer loads into LDS of
// the direct-to-LDS products; word 3 is gfx9's for 32-bit data without swizzling.  Dwords at or
// past `bytes` read as zero instead of touching memory (checked dword by dword).
template <typename T>
__device__ inline __amdgpu_buffer_rsrc_t raw_rsrc(const T *p, int bytes = 0x7fffffff) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<T *>(p), (short)0, bytes, 0x00020000);
}
// Workgroup barrier that waits for nothing but this wave's own LDS reads: global loads into LDS stay
// in flight (the caller waits for the ones it needs with s_waitcnt vmcnt first).
__device__ inline void wg_barrier() {
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0xc07f);  // gfx9 encoding: vmcnt 63, expcnt 7, lgkmcnt 0
    __builtin_amdgcn_s_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// Carried sums: a few slices of K (FP32 128 values, FP64 64 to 256) are accumulated at a time and these sums added up
// apart (restarting at a pair's second product too).  FP32 and FP64 products of small results do (carries): one
// FP32 chain over all of K would be three times less accurate at 700 x 700 x 1500 than the parts of about 160 that
// such a product used to be split into.  So do the FP64 products of the factorisations (dense_la.hip).
template <typename AV, int FM, int FN>
__device__ inline void carry_sums(AV (&acc)[FM][FN], AV (&tot)[FM][FN]) {
#pragma unroll
    for (int a = 0; a < FM; ++a)
#pragma unroll
        for (int b = 0; b < FN; ++b) {
            tot[a][b] = tot[a][b] + acc[a][b];
            acc[a][b] = AV{0, 0, 0, 0};
        }
}

}  // namespace omx

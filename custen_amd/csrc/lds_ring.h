// lds_ring.h -- building blocks of kernels whose workgroup splits into waves
// that move rows between memory and an LDS ring and one wave that computes.
//
// The waves meet only through progress counters in LDS.  A wave's LDS
// operations take effect in issue order, so a counter written after data (or
// after the reads of a slot) is seen only once those are done, and neither
// side drains its queues for it.  Every wave of the workgroup is resident and
// each wait is for a step another wave reaches unconditionally.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "stencil_band.h"  // LDS-typed pointers, waitVmcnt

namespace custen {
namespace dev {

__device__ __forceinline__ void post(int& f, int v)
{
    __asm__ __volatile__("" ::: "memory");
    __hip_atomic_store(&f, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    __asm__ __volatile__("" ::: "memory");
}

__device__ __forceinline__ int peek(const int& f)
{
    return __builtin_amdgcn_readfirstlane(
        __hip_atomic_load(&f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
}

__device__ __forceinline__ void waitFor(const int& f, int v)
{
    while (peek(f) < v) __builtin_amdgcn_s_sleep(1);
    __asm__ __volatile__("" ::: "memory");
}

// Barrier of the workgroup with every memory operation complete (between two
// sweeps of which the second reads what the first stored).
__device__ __forceinline__ void sweepBarrier()
{
    __asm__ __volatile__("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_s_barrier();
    __asm__ __volatile__("" ::: "memory");
}

// Rows of an array as a buffer: p is the first row, the same for all lanes.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rowBuffer(const void* p)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, 0x7fffffff,
                                             0x00020000);
}

// BYTES (16 or 4) per lane from rs + voff + soff to LDS at l + lane * BYTES.
template <int BYTES>
__device__ __forceinline__ void rowDma(__amdgpu_buffer_rsrc_t rs, Lds<char>* l, uint32_t voff,
                                       uint32_t soff)
{
    static_assert(BYTES == 16 || BYTES == 4, "16 or 4 bytes per lane");
    if constexpr (BYTES == 16)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (LdsVoid*)l, 16, voff, soff, 0, 0);
    else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (LdsVoid*)l, 4, voff, soff, 0, 0);
}

__device__ __forceinline__ double rowLoad(__amdgpu_buffer_rsrc_t rs, uint32_t voff)
{
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rs, voff, 0, 0));
}

__device__ __forceinline__ void rowStore(__amdgpu_buffer_rsrc_t rs, double v, uint32_t voff,
                                         uint32_t soff)
{
    typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), rs, voff, soff, 0);
}

}  // namespace dev
}  // namespace custen

// Device code shared by the matrix-core kernels: vector types, direct-to-LDS
// loads, explicit waits and barriers, fp4 expansion.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>
#include <utility>

#include "fiu_device.h"

namespace fiu {

// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>), inline.
template <class F, int... I>
__device__ __forceinline__ void static_for_impl(F &&f, std::integer_sequence<int, I...>)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F> __device__ __forceinline__ void static_for(F &&f)
{
    static_for_impl(f, std::make_integer_sequence<int, N>{});
}

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));

// Direct-to-LDS buffer load of 16 bytes per lane from byte offset voff of
// the resource: lane l's bytes land at lds_group + 16 l (lds_group
// wave-uniform).  The per-lane offsets stay fixed while the resource base
// moves (scalar arithmetic only).
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t r, uint32_t voff, int8_t *lds_group)
{
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void *)lds_group, 16, voff, 0, 0,
                                            0);
}

// Wait until at most N vector-memory operations of this wave are pending
// (vmcnt N; lgkm and exp counters not waited on).
template <int N> __device__ __forceinline__ void wait_vmcnt()
{
    static_assert(N >= 0 && N < 64, "vmcnt immediate");   // bits 3:0 and 15:14
    __builtin_amdgcn_s_waitcnt(0x0f70 | (N & 15) | N >> 4 << 14);
}

// wait_vmcnt<L * s>() for a runtime, wave-uniform s (clamped to 0 .. S).
template <int S, int L> __device__ __forceinline__ void wait_stages(int s)
{
    if constexpr (S > 0) {
        if (s >= S) {
            wait_vmcnt<L * S>();
            return;
        }
        wait_stages<S - 1, L>(s);
    } else {
        wait_vmcnt<0>();
    }
}

// Workgroup barrier with no memory fence (a fence would drain every pending
// direct-to-LDS load, including the ones meant to stay in flight); the
// waits are explicit, the empty asm statements keep the compiler from moving
// memory accesses across the barrier.
__device__ __forceinline__ void stage_barrier()
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// Eight bits (b < 256) as eight e2m1 nibbles, bit i -> nibble i = 0x2 (1.0)
// or 0x0: the bits are spread 4 apart by three shift-or-mask steps, then
// moved to bit 1 of each nibble.
__device__ __forceinline__ uint32_t byte_fp4(uint32_t b)
{
    b = (b | (b << 12)) & 0x000F000Fu;
    b = (b | (b << 6)) & 0x03030303u;
    b = (b | (b << 3)) & 0x11111111u;
    return b << 1;
}

typedef float v4f __attribute__((ext_vector_type(4)));

}  // namespace fiu

// buffer.hpp -- global loads and stores through buffer descriptors.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace ostft {

// A buffer descriptor over `bytes` bytes from a wave-uniform address: a load
// or store then takes one 32-bit lane offset and a scalar offset, where the
// 64-bit addresses of 32 loads would cost two vector instructions each.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer(const void* p, uint32_t bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00027000);
}

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float2 load2(__amdgpu_buffer_rsrc_t r, uint32_t lane_off, uint32_t off)
{
    return __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(r, lane_off, off, 0));
}
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float4 load4(__amdgpu_buffer_rsrc_t r, uint32_t lane_off, uint32_t off)
{
    return __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r, lane_off, off, 0));
}
__device__ __forceinline__ void store1(__amdgpu_buffer_rsrc_t r, uint32_t lane_off, uint32_t off, float v)
{
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), r, lane_off, off, 0);
}
__device__ __forceinline__ void store2(__amdgpu_buffer_rsrc_t r, uint32_t lane_off, uint32_t off, float2 v)
{
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, lane_off, off, 0);
}

}  // namespace ostft

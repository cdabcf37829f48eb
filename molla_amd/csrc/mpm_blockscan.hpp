// mpm_blockscan.hpp -- wave and block prefix sums shared by the sort and the
// layout kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mpm {

__device__ __forceinline__ uint32_t shfl_up_bits(uint32_t v, int o) { return (uint32_t)__shfl_up((int)v, o, 64); }
__device__ __forceinline__ uint64_t shfl_up_bits(uint64_t v, int o) {
    return (uint64_t(shfl_up_bits(uint32_t(v >> 32), o)) << 32) | shfl_up_bits(uint32_t(v), o);
}

// Inclusive prefix sum over the wave's 64 lanes (all active).
template <class T>
__device__ __forceinline__ T wave_incl_scan(T v) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const T t = shfl_up_bits(v, o);
        if (lane >= o) v += t;
    }
    return v;
}

// Exclusive prefix sum over the block (a multiple of 64, at most 1024
// threads); s_wave: 64 entries of LDS.  `total` (may be null) receives the
// block's sum.  Every thread calls it; s_wave is free again on return.
template <class T>
__device__ __forceinline__ T block_excl_scan(T v, T* s_wave, T* total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    const T incl = wave_incl_scan(v);
    if (lane == 63) s_wave[wave] = incl;
    __syncthreads();
    if (wave == 0) {
        const T w = lane < nw ? s_wave[lane] : T(0);
        const T wi = wave_incl_scan(w);
        if (lane < nw) s_wave[lane] = wi - w;
        if (lane == nw - 1) s_wave[63] = wi;
    }
    __syncthreads();
    const T r = incl - v + s_wave[wave];
    if (total) *total = s_wave[63];
    __syncthreads();
    return r;
}

// Counter `i` of a table of u16 counters goes up by the lanes of `same` (the
// wave's lanes with this counter) and every one of them gets the word that
// holds it after that; counter_half takes it out.  The wave's LDS accesses
// stay in program order, so rounds can be issued one after the other without
// waiting for the words.
__device__ __forceinline__ uint32_t counter_add(uint16_t* table, uint32_t i, uint64_t same, uint64_t lt) {
    uint32_t* w = reinterpret_cast<uint32_t*>(table) + i / 2u;
    if ((same & lt) == 0ull)
        __hip_atomic_fetch_add(w, (uint32_t)__popcll(same) << (16u * (i & 1u)), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_WORKGROUP);
    __builtin_amdgcn_wave_barrier();
    return __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ uint32_t counter_half(uint32_t word, uint32_t i) {
    return (word >> (16u * (i & 1u))) & 0xffffu;
}

}  // namespace mpm

// Device helpers shared by the step kernels of the time loop.
#pragma once
#include "sfg_internal.h"

namespace sfg {

template <bool EXACT, class T>
__device__ __forceinline__ T mac(T acc, T a, T x)
{
    if constexpr (EXACT) return acc + a * x;
    else return __builtin_fmaf(a, x, acc);
}

// Loads and stores of data no other lane of this step touches again (a row's
// own accelerations, the Kahan terms, every output) may carry the streaming
// (nontemporal) hint, so the lines they occupy do not push the neighbours'
// fields, which nine rows gather, out of L2.
template <bool NT, class T>
__device__ __forceinline__ T ld_once(const T *p)
{
    if constexpr (NT) return __builtin_nontemporal_load(p);
    else return *p;
}

template <bool NT, class T>
__device__ __forceinline__ void st_once(T *p, T v)
{
    if constexpr (NT) __builtin_nontemporal_store(v, p);
    else *p = v;
}

// bfloat16 halves of a 32-bit word (precision 3 keeps the Kahan terms of two
// displacement fields per word): the low half is field 2k, the high half 2k+1.
__device__ __forceinline__ float bf16_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
// round to nearest even (the terms are finite: a Kahan term is the rounding
// error of an FP32 sum)
__device__ __forceinline__ uint32_t bf16_bits(float f)
{
    const uint32_t u = __float_as_uint(f);
    return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
}

// Read-only arrays of a step (pattern, values, coefficients, schedules) are
// read through the constant address space: they do not change during a
// launch, which lets wave-uniform reads (one row per wave) go through the
// scalar unit instead of the vector-memory path the gathers saturate.
template <class T>
__device__ __forceinline__ const __attribute__((address_space(4))) T *ro(const T *p)
{
    return (const __attribute__((address_space(4))) T *)p;
}

// Workgroups are dispatched round-robin over the 8 XCDs; this map makes each
// XCD walk one contiguous range of logical blocks (shot chunk, row block), so
// neighbouring rows share that XCD's L2.  A bijection on [0, nb) for any nb.
__device__ __forceinline__ unsigned int xcd_contiguous(unsigned int bid, unsigned int nb)
{
    const unsigned int q = nb / 8, r = nb % 8;
    const unsigned int x = bid % 8, l = bid / 8;
    return x * q + (x < r ? x : r) + l;
}

// Stripes: tiles are taken in runs of 8*Q; within a run XCD x (workgroup ids
// x, x+8, ...) steps tiles x*Q .. x*Q+Q-1.  All XCDs then sweep the rows
// together, each keeping one stripe of consecutive row blocks, so a row's
// neighbours on the adjacent grid lines were fetched into the same XCD's L2.
// A bijection on [0, nb): the ids past the last whole run map to themselves.
__device__ __forceinline__ unsigned int xcd_striped(unsigned int bid, unsigned int nb, unsigned int q)
{
    const unsigned int span = 8u * q;
    if (bid >= (nb / span) * span) return bid;
    const unsigned int x = bid % 8, k = bid / 8;
    return (k / q) * span + x * q + k % q;
}

// Step number of a launch with the given slot; the first thread of the grid
// hands t + 1 to the next launch (the other slot).  One store per launch: a
// per-block completion count on one address serialises tens of thousands of
// atomics per step at one L2 channel.
__device__ __forceinline__ int begin_step(Ctrl *ctrl, int slot)
{
    const int t = __hip_atomic_load(&ctrl->step[slot], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0)
        __hip_atomic_store(&ctrl->step[slot ^ 1], t + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return t;
}

} // namespace sfg

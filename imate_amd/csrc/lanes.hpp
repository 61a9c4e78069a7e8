// Sums over neighbouring lanes of a wavefront (device code).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace slq {

// Lane l's value from the lane that Ctrl names (row operations within 16
// lanes; every lane of the row is read, so all of its lanes must be active).
template <int Ctrl>
__device__ __forceinline__ int dpp(int x)
{
    return __builtin_amdgcn_update_dpp(0, x, Ctrl, 0xf, 0xf, true);
}

template <int Ctrl>
__device__ __forceinline__ float dpp(float x)
{
    return __builtin_bit_cast(float, dpp<Ctrl>(__builtin_bit_cast(int, x)));
}

template <int Ctrl>
__device__ __forceinline__ double dpp(double x)
{
    const uint64_t u = __builtin_bit_cast(uint64_t, x);
    const uint32_t lo = (uint32_t) dpp<Ctrl>((int) (uint32_t) u);
    const uint32_t hi = (uint32_t) dpp<Ctrl>((int) (uint32_t) (u >> 32));
    return __builtin_bit_cast(double, ((uint64_t) hi << 32) | lo);
}

// Sum over P = 1, 2, 4, 8 or 16 neighbouring lanes, the same value in each:
// lane ^ 1, ^ 2 (quad permutes), then the mirrored half row and row, whose
// lanes already agree within quads and halves; 32 and 64 by shuffles.
template <int P, typename T>
__device__ __forceinline__ T lanes_sum(T x)
{
    if constexpr (P > 1) x += dpp<0xB1>(x);
    if constexpr (P > 2) x += dpp<0x4E>(x);
    if constexpr (P > 4) x += dpp<0x141>(x);
    if constexpr (P > 8) x += dpp<0x140>(x);
    if constexpr (P > 16) x += __shfl_xor(x, 16);
    if constexpr (P > 32) x += __shfl_xor(x, 32);
    return x;
}

template <int P>
__device__ __forceinline__ double lanes_product(double x)
{
    if constexpr (P > 1) x *= dpp<0xB1>(x);
    if constexpr (P > 2) x *= dpp<0x4E>(x);
    if constexpr (P > 4) x *= dpp<0x141>(x);
    if constexpr (P > 8) x *= dpp<0x140>(x);
    return x;
}

}  // namespace slq

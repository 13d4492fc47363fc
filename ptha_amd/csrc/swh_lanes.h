// Neighbour values across a wavefront, for the kernels whose lanes are columns.
//
// A shift by one lane is a data-parallel-primitive move (wave_shl / wave_shr), a VALU
// operation that the compiler can fold into its consumer, where __shfl_up / __shfl_down
// are permutes through LDS (ds_bpermute: an LDS round trip on the chain of every level of
// a row). Rows of the two-step kernel at 2048 x 2048 took
// 49 permutes each; the finite-volume step of 2000 x 1000 went from 341 to 321 us with the
// moves and with scalar_load below.
#pragma once
#include <hip/hip_runtime.h>

namespace swh {

constexpr int kDppWaveShl1 = 0x130;   // lane i takes lane i + 1
constexpr int kDppWaveShr1 = 0x138;   // lane i takes lane i - 1

// ctrl applied to the 32-bit halves of v; the lane at the open end takes 0. Every lane of
// the wavefront must execute it.
template <int ctrl, typename T>
__device__ __forceinline__ T lane_shift(T v)
{
    if constexpr (sizeof(T) == 4) {
        return __builtin_bit_cast(T, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), ctrl, 0xf, 0xf, true));
    } else {
        const long long b = __builtin_bit_cast(long long, v);
        const int lo = __builtin_amdgcn_mov_dpp((int)(b & 0xffffffff), ctrl, 0xf, 0xf, true);
        const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), ctrl, 0xf, 0xf, true);
        return __builtin_bit_cast(T, ((long long)hi << 32) | (unsigned int)lo);
    }
}

// A value of the same address on every lane, through the scalar cache (the tables are not
// written by any kernel that reads them here). As a vector load it would be waited for
// behind the state's loads, which return in order: each row then pays a trip to memory.
template <typename T>
__device__ __forceinline__ T scalar_load(const T *p)
{
    return *(const __attribute__((address_space(4))) T *)p;
}

// the value of the lane to the east (lane + 1), to the west (lane - 1)
template <typename T>
__device__ __forceinline__ T lane_east(T v) { return lane_shift<kDppWaveShl1>(v); }
template <typename T>
__device__ __forceinline__ T lane_west(T v) { return lane_shift<kDppWaveShr1>(v); }

// the value of the lane to the west; lane 0 takes 'edge' instead
__device__ __forceinline__ float lane_west_or(float v, float edge)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, edge),
                                                                 __builtin_bit_cast(int, v), kDppWaveShr1, 0xf, 0xf,
                                                                 false));
}
__device__ __forceinline__ double lane_west_or(double v, double edge)
{
    const long long b = __builtin_bit_cast(long long, v), e = __builtin_bit_cast(long long, edge);
    const int lo = __builtin_amdgcn_update_dpp((int)(e & 0xffffffff), (int)(b & 0xffffffff), kDppWaveShr1, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp((int)(e >> 32), (int)(b >> 32), kDppWaveShr1, 0xf, 0xf, false);
    return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned int)lo);
}

// The tile of workgroup b of the B of a grid. Workgroups go round the 8 XCDs (each with its own
// L2) by their linear index; this gives each XCD a contiguous range of the tiles, in order, so
// that tiles that share rows or cache lines meet in one L2.
__device__ __forceinline__ unsigned xcd_tile(unsigned b, unsigned B)
{
    const unsigned xcd = b % 8u, slot = b / 8u, n8 = B / 8u, rem = B % 8u;
    return xcd < rem ? xcd * (n8 + 1u) + slot : rem * (n8 + 1u) + (xcd - rem) * n8 + slot;
}

}  // namespace swh

// device_common.h - wavefront reductions, the wavefront key sort and the
// sample-point lookup shared by the kernels of the library.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace hase {

// written by earlier kernels only, indexed uniformly: read through the scalar cache
typedef const __attribute__((address_space(4))) uint32_t ConstU32;

struct SampleGeom {
    float px, py;
    int plane;   // level of the sample point (its height in layer units)
    uint32_t p;  // mesh point under the sample
};

__device__ __forceinline__ SampleGeom sample_point(const float2* pts, uint32_t np, uint32_t sample)
{
    uint32_t p = sample % np, lv = sample / np;
    float2 xy = pts[p];
    return SampleGeom{xy.x, xy.y, (int)lv, p};
}

__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

__device__ __forceinline__ unsigned long long wave_sum_u64(unsigned long long v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Adds the work-group's sum of v to *counter with one atomic (every thread of
// the work-group calls it; red holds one word per wavefront).  Atomics of all
// wavefronts on one address take ~4 ns each, one after the other: 8192 of them
// at the end of a launch kept it open for ~33 us.
__device__ __forceinline__ void block_count(unsigned long long v, unsigned long long* red, unsigned long long* counter)
{
    v = wave_sum_u64(v);
    if ((threadIdx.x & 63u) == 0u) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0u) {
        unsigned long long s = 0;
        for (uint32_t i = 0; i < (blockDim.x + 63u) / 64u; ++i) s += red[i];
        if (s) atomicAdd(counter, s);
    }
}

// v of the lane that DPP control kCtrl names, 0.0 where it names none
template <int kCtrl, int kRowMask>
__device__ __forceinline__ double dpp_or_zero(double v)
{
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, kCtrl, kRowMask, 0xF, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), kCtrl, kRowMask, 0xF, false);
    return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}

// Inclusive scans of N values within a 64-lane wavefront, side by side so
// that each hides the others' latency: shifts by 1, 2, 4 and 8 within rows of
// 16 lanes, then the row ends broadcast to the next row (rows 1 and 3) and the
// second row's end to the upper half.
template <int N>
__device__ __forceinline__ void wave_inclusive_scan(double (&v)[N])
{
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] += dpp_or_zero<0x111, 0xF>(v[i]);
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] += dpp_or_zero<0x112, 0xF>(v[i]);
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] += dpp_or_zero<0x114, 0xF>(v[i]);
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] += dpp_or_zero<0x118, 0xF>(v[i]);
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] += dpp_or_zero<0x142, 0xA>(v[i]);
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] += dpp_or_zero<0x143, 0xC>(v[i]);
}

// Lane 63's value in every lane
__device__ __forceinline__ double wave_last(double v)
{
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, 63);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), 63);
    return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}

// Bitonic sort of a wavefront's 256 keys, ascending, key r * 64 + lane in
// v[r] of that lane.  Every lane of the wavefront takes part (the exchanges
// read the partner lane's register).
__device__ __forceinline__ void wave_sort256(uint32_t (&v)[4], int lane)
{
#pragma unroll
    for (uint32_t k = 2u; k <= 256u; k <<= 1) {
#pragma unroll
        for (uint32_t d = k >> 1; d > 0u; d >>= 1) {
            if (d >= 64u) {
                // partners in the same lane: registers r and r + d / 64
                const uint32_t rd = d >> 6;
#pragma unroll
                for (uint32_t r = 0; r < 4u; ++r) {
                    if (r & rd) continue;
                    const bool asc = ((r * 64u + (uint32_t)lane) & k) == 0u;
                    const uint32_t a = v[r], b = v[r | rd];
                    const uint32_t lo = a < b ? a : b, hi = a < b ? b : a;
                    v[r] = asc ? lo : hi;
                    v[r | rd] = asc ? hi : lo;
                }
            } else {
#pragma unroll
                for (uint32_t r = 0; r < 4u; ++r) {
                    const uint32_t w = (uint32_t)__shfl_xor((int)v[r], (int)d, 64);
                    const bool lower = ((uint32_t)lane & d) == 0u;
                    const bool asc = ((r * 64u + (uint32_t)lane) & k) == 0u;
                    const uint32_t lo = v[r] < w ? v[r] : w, hi = v[r] < w ? w : v[r];
                    v[r] = lower == asc ? lo : hi;
                }
            }
        }
    }
}

}  // namespace hase

// lane_sums.h -- sums of many values over the 64 lanes of a wavefront.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#ifndef DEVI
#define DEVI __device__ __forceinline__
#endif

namespace {

// ---- sums over the 64 lanes of many values at once ------------------------------------------
// Each of the six butterfly steps adds pairs of lanes and halves the number of values a lane
// holds (a lane keeps one half of the values and gives the other to its partner), so V values
// take about V + 6 additions instead of 6 V.  Value i of the remaining ceil(V / 64) in a lane is
// the total number lane_value<V>(lane, i), or -1.
template <int CTRL>
DEVI double dpp_mov(double x)
{
    const uint64_t b = __builtin_bit_cast(uint64_t, x);
    const uint32_t lo = __builtin_amdgcn_mov_dpp((int)(uint32_t)b, CTRL, 0xf, 0xf, true);
    const uint32_t hi = __builtin_amdgcn_mov_dpp((int)(uint32_t)(b >> 32), CTRL, 0xf, 0xf, true);
    return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}

// exchanges the upper half of a with the lower half of b (halves of 32 lanes, or of 16 in each 32)
template <int W>
DEVI void swap_halves(double &a, double &b)
{
    const uint64_t ua = __builtin_bit_cast(uint64_t, a), ub = __builtin_bit_cast(uint64_t, b);
    if constexpr (W == 32) {
        const auto lo = __builtin_amdgcn_permlane32_swap((uint32_t)ua, (uint32_t)ub, false, false);
        const auto hi = __builtin_amdgcn_permlane32_swap((uint32_t)(ua >> 32), (uint32_t)(ub >> 32), false, false);
        a = __builtin_bit_cast(double, (uint64_t)hi[0] << 32 | lo[0]);
        b = __builtin_bit_cast(double, (uint64_t)hi[1] << 32 | lo[1]);
    } else {
        const auto lo = __builtin_amdgcn_permlane16_swap((uint32_t)ua, (uint32_t)ub, false, false);
        const auto hi = __builtin_amdgcn_permlane16_swap((uint32_t)(ua >> 32), (uint32_t)(ub >> 32), false, false);
        a = __builtin_bit_cast(double, (uint64_t)hi[0] << 32 | lo[0]);
        b = __builtin_bit_cast(double, (uint64_t)hi[1] << 32 | lo[1]);
    }
}

// partner lane (lane ^ W) within a row of 16: rotation by 8, mirror of 8 with mirror of 4, quad permutations
template <int W>
DEVI double row_partner(double x)
{
    if constexpr (W == 8) return dpp_mov<0x128>(x);        // row_ror:8
    else if constexpr (W == 4) return dpp_mov<0x1b>(dpp_mov<0x141>(x));   // row_half_mirror, quad_perm [3,2,1,0]
    else if constexpr (W == 2) return dpp_mov<0x4e>(x);    // quad_perm [2,3,0,1]
    else return dpp_mov<0xb1>(x);                          // quad_perm [1,0,3,2]
}

template <int V, int W>
DEVI void lane_halve(double *v, int lane)
{
    constexpr int h = (V + 1) / 2;
    const bool up = lane & W;
#pragma unroll
    for (int i = 0; i < h; ++i) {
        double a = v[i], b = i + h < V ? v[i + h] : 0.0;
        if constexpr (W >= 16) {
            swap_halves<W>(a, b);
            v[i] = a + b;
        } else {
            v[i] = (up ? b : a) + row_partner<W>(up ? a : b);
        }
    }
    if constexpr (W > 1) lane_halve<h, W / 2>(v, lane);
}

template <int V>
DEVI void lane_sums(double *v, int lane)
{
    lane_halve<V, 32>(v, lane);
}

// The total held as value i by `lane` after lane_sums<V>: bit by bit, from the last step back.
template <int V, int W = 32>
DEVI int lane_value(int lane, int i)
{
    constexpr int h = (V + 1) / 2;
    if constexpr (W > 1) {
        i = lane_value<h, W / 2>(lane, i);
        if (i < 0) return -1;
    } else if (i >= h) {
        return -1;
    }
    const int j = lane & W ? i + h : i;
    return j < V ? j : -1;
}

}  // namespace

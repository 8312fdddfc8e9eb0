// lane_sum.h -- sums over lanes whose numbers differ in their high bits
// (device code only).
//
// The reductions give 64 / T bodies T lanes each and add over the lane bits 32,
// 16, 8, 4 down to 64 / T.  A shuffle through LDS (ds_bpermute, two for an
// FP64 value) waits for LDS at every level; gfx950 exchanges lane halves and
// rows in registers instead: v_permlane32_swap and v_permlane16_swap of a
// value with itself leave both partners side by side, and a row rotation by 8
// is lane ^ 8.  A rotation by 4 gives lane ^ 4 or lane ^ 12, which hold the
// same sum once the bit-8 level is done.  Every level adds the same two
// values as v + __shfl_xor(v, bit), so the sums are the same bits.
// Small-system steps on MI355X, mixed: 1000 bodies 3.71 us (4.00 with shuffles,
// 3.54 without the sums), 2048 4.92 (5.12), 6001 16.1 (16.4); the reductions of
// the symmetric kernels are bound by their loads and do not change.
#pragma once

#include <hip/hip_runtime.h>

namespace utcnb {

// The pair (a, b) whose sum is v + (v of lane ^ BIT), BIT = 32, 16, 8 or (after
// the level of bit 8) 4.
template <int BIT>
__device__ __forceinline__ void lane_partners(unsigned v, unsigned& a, unsigned& b)
{
    static_assert(BIT == 32 || BIT == 16 || BIT == 8 || BIT == 4, "lane bit");
    if constexpr (BIT == 32) {
        const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
        a = r[0];
        b = r[1];
    } else if constexpr (BIT == 16) {
        const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
        a = r[0];
        b = r[1];
    } else {
        a = v;
        b = (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x120 | BIT /* row_ror */, 0xF, 0xF, false);
    }
}

template <int BIT>
__device__ __forceinline__ float lane_add(float v)
{
    unsigned a, b;
    lane_partners<BIT>(__float_as_uint(v), a, b);
    return __uint_as_float(a) + __uint_as_float(b);
}

template <int BIT>
__device__ __forceinline__ double lane_add(double v)
{
    const unsigned long long u = (unsigned long long)__double_as_longlong(v);
    unsigned al, ah, bl, bh;
    lane_partners<BIT>((unsigned)u, al, bl);
    lane_partners<BIT>((unsigned)(u >> 32), ah, bh);
    return __longlong_as_double((long long)(((unsigned long long)ah << 32) | al)) +
           __longlong_as_double((long long)(((unsigned long long)bh << 32) | bl));
}

// v summed over the lane bits LOW .. 32 (LOW = 4 .. 64; 64: v itself), in every lane.
template <int LOW, typename T>
__device__ __forceinline__ T lane_sum(T v)
{
    static_assert(LOW >= 4 && LOW <= 64, "lowest lane bit");
    if constexpr (LOW <= 32)
        v = lane_add<32>(v);
    if constexpr (LOW <= 16)
        v = lane_add<16>(v);
    if constexpr (LOW <= 8)
        v = lane_add<8>(v);
    if constexpr (LOW <= 4)
        v = lane_add<4>(v);
    return v;
}

}  // namespace utcnb

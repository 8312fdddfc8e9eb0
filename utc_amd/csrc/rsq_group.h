// rsq_group.h -- reciprocal square roots of a group of pairs (device code only).
//
// What bounds the FP32 pair kernels is how the SIMD shares its issue slots
// between two waves.  Measured on MI355X (profiles/probe_valu_pairing.txt): one
// wave alone issues a plain FP32 instruction every 4.4 cycles, but two waves
// that are both in plain VGPR arithmetic issue two at a time, 2.2-2.25 cycles
// each.  v_rsq_f32 takes 7.75 cycles and pairs with nothing, and while one
// wave is in its roots the other runs its FMAs unpaired: with equal priorities
// 14 FMAs and a root cost two waves 58 cycles (8 roots in a row, then their
// 112 FMAs), of which 39 are needed.  Raising the wave's priority for its
// roots lets it finish them at once, so the waves fall back into step: 40
// cycles with two waves per SIMD, 39 with four, 40 and 40 with groups of 4,
// 42 and 40 with single roots.  (Lower priority for the roots costs 64, a
// barrier before them 71.)  So the kernels compute the distances of a group of
// pairs first and take their roots here, together: 8 pairs, or 4 where the
// registers of 8 would cost a wave.
//
// The asm block ends with two scalar instructions, more than the one wait
// state a transcendental result needs before a plain VALU instruction may
// read it.
#pragma once

#include <hip/hip_runtime.h>

namespace utcnb {

// y[i] = v_rsq_f32(d[i]), i < N.
template <int N>
__device__ __forceinline__ void rsq_group(const float* d, float* y)
{
    static_assert(N >= 1, "group size");
    if constexpr (N >= 8) {
        asm volatile("s_setprio 3\n\t"
                     "v_rsq_f32 %0, %8\n\tv_rsq_f32 %1, %9\n\tv_rsq_f32 %2, %10\n\tv_rsq_f32 %3, %11\n\t"
                     "v_rsq_f32 %4, %12\n\tv_rsq_f32 %5, %13\n\tv_rsq_f32 %6, %14\n\tv_rsq_f32 %7, %15\n\t"
                     "s_setprio 0\n\ts_nop 0"
                     : "=&v"(y[0]), "=&v"(y[1]), "=&v"(y[2]), "=&v"(y[3]), "=&v"(y[4]), "=&v"(y[5]), "=&v"(y[6]),
                       "=&v"(y[7])
                     : "v"(d[0]), "v"(d[1]), "v"(d[2]), "v"(d[3]), "v"(d[4]), "v"(d[5]), "v"(d[6]), "v"(d[7]));
        if constexpr (N > 8)
            rsq_group<N - 8>(d + 8, y + 8);
    } else if constexpr (N >= 4) {
        asm volatile("s_setprio 3\n\t"
                     "v_rsq_f32 %0, %4\n\tv_rsq_f32 %1, %5\n\tv_rsq_f32 %2, %6\n\tv_rsq_f32 %3, %7\n\t"
                     "s_setprio 0\n\ts_nop 0"
                     : "=&v"(y[0]), "=&v"(y[1]), "=&v"(y[2]), "=&v"(y[3])
                     : "v"(d[0]), "v"(d[1]), "v"(d[2]), "v"(d[3]));
        if constexpr (N > 4)
            rsq_group<N - 4>(d + 4, y + 4);
    } else if constexpr (N >= 2) {
        asm volatile("s_setprio 3\n\tv_rsq_f32 %0, %2\n\tv_rsq_f32 %1, %3\n\ts_setprio 0\n\ts_nop 0"
                     : "=&v"(y[0]), "=&v"(y[1])
                     : "v"(d[0]), "v"(d[1]));
        if constexpr (N > 2)
            rsq_group<1>(d + 2, y + 2);
    } else {
        asm volatile("s_setprio 3\n\tv_rsq_f32 %0, %1\n\ts_setprio 0\n\ts_nop 0" : "=&v"(y[0]) : "v"(d[0]));
    }
}

}  // namespace utcnb

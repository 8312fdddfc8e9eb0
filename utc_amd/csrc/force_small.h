// force_small.h -- one-kernel steps for small systems (device code; included
// by force_tmpl.h).
//
// Below about 8192 bodies a step is bound by latency, not by issue rate: the
// symmetric kernels need a second kernel to add their partial sums, and the
// one-pass kernels give every wave 64 targets, so a small system has too few
// waves to fill the chip and each wave waits on its scalar source loads.
// Here a workgroup of W waves owns TW = TL * A targets and all sources:
//  * the workgroup copies the n source bodies into LDS once, with padding
//    after them to a whole number of the splits' root groups (256 to 1024
//    bodies; at most CAP);
//  * lane l = t + TL * g of wave w holds targets t, t + TL, ..., t + (A-1) TL
//    of the workgroup and sums sources split, split + SPL, split + 2 SPL, ...
//    with split = w * G + g, G = 64 / TL source groups per wave and SPL =
//    G * W source splits per workgroup: the TL lanes of a group read the same
//    LDS record (a broadcast), the G groups consecutive ones;
//  * the G lanes of a target meet in registers (lane_sum.h), the W
//    waves in LDS, in a fixed order (bitwise repeatable), and TW threads run
//    the integrator epilogue: one launch per step, nothing in HBM between.
// COMP: sums of up to BLOCK sources are Kahan-added per lane (as the 64-source
// partials of the other kernels) and the lanes and waves are combined in FP64;
// otherwise plain FP32 throughout (the plain FP32 path).  BLOCK is 32, but 8 for
// the 64 splits of TL = 8, W = 8: they serve 1025 to 2048 bodies in place of
// 128 splits, whose sums are half as long (the field's error there, 2048
// bodies in a cube, Newton: 4.1e-8 with 128 splits, 5.0e-8 with 64 and blocks of
// 32, 3.7e-8 with blocks of 8, which take 4.6 us per step for 4.5).
// Pair arithmetic as in stream_sources: 12 VALU instructions and a root per
// ordered pair, the roots of 8 pairs together (rsq_group.h), plus one LDS read
// per source shared by the lane's A targets.  Per step, mixed: N = 8192 22.1 us
// (27.3 with a root per pair), 6001 15.1 (21.2; 18.3 with 32 targets per
// workgroup instead of 24), 4096 8.2 (9.6), 2000 4.7, 1000 3.4.  Up to 2048
// bodies the launch, the copy into LDS and the ends of the sums bound it: lane
// sums by shuffles took 4.0 at 1000, and the copy through registers, a load and
// its store in turn, 3.7 at 1000, 8.8 at 4096 and 23.3 at 8192 (all loads into
// registers first, in a run-time number, went through scratch: 4.7, 13.0, 32.3).
// Padding to whole root groups instead of to 1024 bodies: 1100 4.6 to 4.0, 4200
// 13.3 to 12.1, 7200 22.0 to 20.5.
#pragma once

#include <type_traits>

#include "lane_sum.h"

namespace utcnb {

template <int A, int TL, int W, int CAP, bool COMP, bool NEWTON, class Epi>
__global__ __launch_bounds__(64 * W) void small_force_kernel(const float4* __restrict__ src, int i0, int nt,
                                                             int n, float eps2, Epi epi)
{
    constexpr int G = 64 / TL, TW = TL * A, SPL = G * W;
    constexpr int J = A == 1 ? 8 : A == 2 ? 4 : 2;  // sources per group of reciprocal roots
    constexpr int BLOCK = TL == 8 && W == 8 ? 8 : 32;  // sources per plain partial of a lane
    // the same number of sources for every split, whole groups: padding after n
    const int iters = (n + SPL * J - 1) / (SPL * J) * J, fill = iters * SPL;
    using Acc = typename std::conditional<COMP, double, float>::type;
    __shared__ float4 sh[CAP];
    __shared__ Acc red[W][TW][3];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int t = lane % TL, g = lane / TL;
    const int tgt0 = blockIdx.x * TW;
    // the epilogue's state loads, issued before the pair work (thread j < TW
    // updates target tgt0 + j)
    typename Epi::State pre{};
    if (threadIdx.x < TW && tgt0 + (int)threadIdx.x < nt)
        pre = epi.load(i0 + tgt0 + threadIdx.x);

    float px[A], py[A], pz[A], hx[A], hy[A], hz[A], cx[A], cy[A], cz[A];
#pragma unroll
    for (int a = 0; a < A; ++a) {
        const int tt = tgt0 + a * TL + t;
        const float4 p = src[i0 + (tt < nt ? tt : nt - 1)];  // clamped lanes compute but never store
        px[a] = p.x; py[a] = p.y; pz[a] = p.z;
        hx[a] = hy[a] = hz[a] = cx[a] = cy[a] = cz[a] = 0.f;
    }
    // every load of the copy in flight at once, past the registers: a wave
    // fills 64 consecutive LDS slots with one load
    for (int k = wave * 64; k < fill; k += 64 * W) {
        if (k + lane < n)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src + k + lane),
                                             (__attribute__((address_space(3))) void*)&sh[k], 16, 0, 0);
        else
            sh[k + lane] = make_float4(kPadCoord, kPadCoord, kPadCoord, 0.f);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();

    const int split = wave * G + g;
    for (int b0 = 0; b0 < iters; b0 += BLOCK) {
        const int b1 = b0 + BLOCK < iters ? b0 + BLOCK : iters;
        float ax[A], ay[A], az[A];
#pragma unroll
        for (int a = 0; a < A; ++a) {
            if constexpr (COMP) {
                ax[a] = ay[a] = az[a] = 0.f;
            } else {
                ax[a] = hx[a]; ay[a] = hy[a]; az[a] = hz[a];
            }
        }
#pragma unroll 1
        for (int i = b0; i < b1; i += J) {
            float rx[J * A], ry[J * A], rz[J * A], d2[J * A], y[J * A], m[J];
#pragma unroll
            for (int u = 0; u < J; ++u) {
                const float4 b = sh[split + (i + u) * SPL];
                m[u] = b.w;
#pragma unroll
                for (int a = 0; a < A; ++a) {
                    const int q = u * A + a;
                    rx[q] = b.x - px[a]; ry[q] = b.y - py[a]; rz[q] = b.z - pz[a];
                    d2[q] = __builtin_fmaf(rx[q], rx[q],
                                           __builtin_fmaf(ry[q], ry[q], __builtin_fmaf(rz[q], rz[q], eps2)));
                }
            }
            rsq_group<J * A>(d2, y);
#pragma unroll
            for (int u = 0; u < J; ++u)
#pragma unroll
                for (int a = 0; a < A; ++a) {
                    const int q = u * A + a;
                    const float s = pair_scale<NEWTON>(d2[q], y[q], m[u]);
                    ax[a] = __builtin_fmaf(rx[q], s, ax[a]);
                    ay[a] = __builtin_fmaf(ry[q], s, ay[a]);
                    az[a] = __builtin_fmaf(rz[q], s, az[a]);
                }
        }
#pragma unroll
        for (int a = 0; a < A; ++a) {
            if constexpr (COMP) {
                kahan_add(hx[a], cx[a], ax[a]);
                kahan_add(hy[a], cy[a], ay[a]);
                kahan_add(hz[a], cz[a], az[a]);
            } else {
                hx[a] = ax[a]; hy[a] = ay[a]; hz[a] = az[a];
            }
        }
    }

    // lanes t, t + TL, ..., t + 64 - TL hold the same targets
#pragma unroll
    for (int a = 0; a < A; ++a) {
        Acc v[3];
        if constexpr (COMP) {  // Kahan keeps the running error as -c: the sum is hi - c
            v[0] = (double)hx[a] - (double)cx[a];
            v[1] = (double)hy[a] - (double)cy[a];
            v[2] = (double)hz[a] - (double)cz[a];
        } else {
            v[0] = hx[a]; v[1] = hy[a]; v[2] = hz[a];
        }
#pragma unroll
        for (int c = 0; c < 3; ++c)
            v[c] = lane_sum<TL>(v[c]);
        if (g == 0) {
#pragma unroll
            for (int c = 0; c < 3; ++c)
                red[wave][a * TL + t][c] = v[c];
        }
    }
    __syncthreads();
    if (threadIdx.x < TW) {
        const int j = threadIdx.x;
        Acc s[3] = {red[0][j][0], red[0][j][1], red[0][j][2]};
#pragma unroll
        for (int w = 1; w < W; ++w)
#pragma unroll
            for (int c = 0; c < 3; ++c)
                s[c] += red[w][j][c];
        const int tt = tgt0 + j;
        if (tt < nt) {
            if constexpr (COMP) {  // split the FP64 sum exactly into (hi, c) with hi - c = s
                const float h0 = (float)s[0], h1 = (float)s[1], h2 = (float)s[2];
                epi.store(i0 + tt, pre, h0, h1, h2, (float)((double)h0 - s[0]), (float)((double)h1 - s[1]),
                          (float)((double)h2 - s[2]));
            } else {
                epi.store(i0 + tt, pre, s[0], s[1], s[2], 0.f, 0.f, 0.f);
            }
        }
    }
}

// Targets [i0, i0 + nt) of a system whose n sources, padded, fit the tile's
// LDS capacity CAP.
template <int A, int TL, int W, int CAP, bool COMP, bool NEWTON, class Epi>
hipError_t launch_small_tile(const float4* src, int i0, int nt, int n, float eps2, const Epi& epi,
                             hipStream_t st)
{
    static_assert(A <= 3 && 64 % TL == 0 && kPadJ / 8 % ((64 / TL) * W) == 0,
                  "each split takes a multiple of 8 sources, in groups of 8 / A");

    if (n < 1 || pad_j(n) > CAP)
        return hipErrorInvalidValue;
    constexpr int TW = TL * A;
    const int blocks = (nt + TW - 1) / TW;
    hipLaunchKernelGGL((small_force_kernel<A, TL, W, CAP, COMP, NEWTON, Epi>), dim3(blocks), dim3(64 * W), 0, st,
                       src, i0, nt, n, eps2, epi);
    return hipGetLastError();
}

}  // namespace utcnb

// force_part.h -- one-pass force with the sources split over separate waves
// (device code; included by force_tmpl.h).
//
// The one-pass kernel (force_kernel) keeps the waves that share a target tile
// in one workgroup, so its grid has as many workgroups as target tiles, each
// a large piece of work: when they do not fill a whole number of rounds of the
// chip the last round is nearly empty (32769 targets: 257 workgroups of 128
// targets on 256 CUs take as long as 512).  Here every wave is on its own: wave
// (tile, part) sums the source chunks of one of P parts for 64 K targets and
// writes its sums to HBM, P records per target, and a second kernel adds a
// target's records in FP64 (compensated paths) or FP32 in a fixed order and
// runs the epilogue.  A target's sums depend on P and n_pad alone, not on the
// range of targets, so slices give the bits of the whole field.
// 12 VALU instructions and a root per ordered pair bound it, as in
// force_kernel; the records are 12 P bytes per target each way.
#pragma once

#include "sym_reduce.h"

namespace utcnb {

// part: [P][nt] records of three floats.
template <int K, bool COMP, bool NEWTON>
__global__ __launch_bounds__(256) void part_force_kernel(const float4* __restrict__ src, int i0, int nt, int n_pad,
                                                         int P, float eps2, float* __restrict__ part)
{
    const int lane = threadIdx.x & 63;
    const int tile = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), p = blockIdx.y;
    if (tile * 64 * K >= nt)
        return;  // whole waves only
    float px[K], py[K], pz[K], hx[K], hy[K], hz[K], cx[K], cy[K], cz[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int t = tile * 64 * K + k * 64 + lane;
        const float4 b = src[i0 + (t < nt ? t : nt - 1)];  // clamped lanes compute but never store
        px[k] = b.x; py[k] = b.y; pz[k] = b.z;
        hx[k] = hy[k] = hz[k] = cx[k] = cy[k] = cz[k] = 0.f;
    }
    const int chunks = n_pad / kChunk;  // a part may be empty when P > chunks
    const int c0 = (int)((long long)chunks * p / P), c1 = (int)((long long)chunks * (p + 1) / P);
    stream_sources<K, COMP, NEWTON>(src, c0 * kChunk, c1 * kChunk, eps2, px, py, pz, hx, hy, hz, cx, cy, cz);
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int t = tile * 64 * K + k * 64 + lane;
        if (t < nt) {
            float* o = part + ((size_t)p * nt + t) * 3;
            o[0] = hx[k] - cx[k];
            o[1] = hy[k] - cy[k];
            o[2] = hz[k] - cz[k];
        }
    }
}

// Target j's P records summed by T lanes (lane t takes records t, t + T, ...;
// lane_sum.h combines them, as in sym_reduce.h), then the epilogue.
template <int T, typename Acc, class Epi>
__global__ __launch_bounds__(256) void part_reduce_kernel(const float* __restrict__ part, int i0, int nt, int P,
                                                          Epi epi)
{
    int j, t;
    sym_reduce_lane<T>(j, t);
    const int jj = j < nt ? j : nt - 1;
    Acc s[3] = {Acc(0), Acc(0), Acc(0)};
#pragma unroll 4
    for (int p = t; p < P; p += T)
        part_add(s, ((const Part3*)part)[(size_t)p * nt + jj]);
#pragma unroll
    for (int c = 0; c < 3; ++c)
        s[c] = lane_sum<64 / T>(s[c]);
    if (j < nt && t == 0)
        sum_epilogue(epi, i0 + j, s);
}

template <int K, bool COMP, bool NEWTON, class Epi>
hipError_t launch_part_tile(int P, const float4* src, int i0, int nt, int n_pad, float eps2, float* part,
                            const Epi& epi, hipStream_t st)
{
    if (!part || P < 1 || P > 65535)
        return hipErrorInvalidValue;
    const int tiles = (nt + 64 * K - 1) / (64 * K);
    hipLaunchKernelGGL((part_force_kernel<K, COMP, NEWTON>), dim3((tiles + 3) / 4, P), dim3(256), 0, st, src, i0, nt,
                       n_pad, P, eps2, part);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess)
        return e;
    using Acc = typename std::conditional<COMP, double, float>::type;
    const int T = sym_reduce_lanes(nt);
    const dim3 grid((unsigned)(((long long)nt * T + 255) / 256));
#define PART_REDUCE(TT) \
    hipLaunchKernelGGL((part_reduce_kernel<TT, Acc, Epi>), grid, dim3(256), 0, st, part, i0, nt, P, epi)
    switch (T) {
    case 1: PART_REDUCE(1); break;
    case 2: PART_REDUCE(2); break;
    case 4: PART_REDUCE(4); break;
    case 8: PART_REDUCE(8); break;
    default: PART_REDUCE(16); break;
    }
#undef PART_REDUCE
    return hipGetLastError();
}

}  // namespace utcnb

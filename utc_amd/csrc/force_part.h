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
// runs the epilogue.  Both tiles, K = 1 with P = 128 and K = 2 with P = 64, add
// the same kSourceParts = 128 partial sums in the same order: with P = 64 a wave
// takes two of them in turn and adds the second to the first, with P = 128 the
// second kernel does, and its lanes per target are a constant.  So a target's
// sums depend on n_pad alone, not on the range of targets or the tile that its
// size selects, and slices give the bits of the whole field.
// 12 VALU instructions and a root per ordered pair bound it, as in
// force_kernel; the records are 12 P bytes per target each way.
#pragma once

#include "sym_reduce.h"

namespace utcnb {

constexpr int kSourceParts = 128;  // parts the sources are summed in
constexpr int kPartLanes = 16;     // lanes per target in the second kernel

// part: [P][nt] records of three floats, P = kSourceParts / H.
template <int K, int H, bool COMP, bool NEWTON>
__global__ __launch_bounds__(256) void part_force_kernel(const float4* __restrict__ src, int i0, int nt, int n_pad,
                                                         float eps2, float* __restrict__ part)
{
    const int lane = threadIdx.x & 63;
    const int tile = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), p = blockIdx.y;
    if (tile * 64 * K >= nt)
        return;  // whole waves only
    float px[K], py[K], pz[K], sx[K], sy[K], sz[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int t = tile * 64 * K + k * 64 + lane;
        const float4 b = src[i0 + (t < nt ? t : nt - 1)];  // clamped lanes compute but never store
        px[k] = b.x; py[k] = b.y; pz[k] = b.z;
    }
    const int chunks = n_pad / kChunk;  // a part may be empty when there are fewer chunks than parts
#pragma unroll 1
    for (int h = 0; h < H; ++h) {
        const int c0 = (int)((long long)chunks * (p * H + h) / kSourceParts);
        const int c1 = (int)((long long)chunks * (p * H + h + 1) / kSourceParts);
        float hx[K], hy[K], hz[K], cx[K], cy[K], cz[K];
#pragma unroll
        for (int k = 0; k < K; ++k)
            hx[k] = hy[k] = hz[k] = cx[k] = cy[k] = cz[k] = 0.f;
        stream_sources<K, COMP, NEWTON>(src, c0 * kChunk, c1 * kChunk, eps2, px, py, pz, hx, hy, hz, cx, cy, cz);
#pragma unroll
        for (int k = 0; k < K; ++k) {
            sx[k] = h == 0 ? hx[k] - cx[k] : sx[k] + (hx[k] - cx[k]);
            sy[k] = h == 0 ? hy[k] - cy[k] : sy[k] + (hy[k] - cy[k]);
            sz[k] = h == 0 ? hz[k] - cz[k] : sz[k] + (hz[k] - cz[k]);
        }
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int t = tile * 64 * K + k * 64 + lane;
        if (t < nt) {
            float* o = part + ((size_t)p * nt + t) * 3;
            o[0] = sx[k];
            o[1] = sy[k];
            o[2] = sz[k];
        }
    }
}

// Target j's kSourceParts / 2 pairs of parts summed by kPartLanes lanes (lane t
// takes pairs t, t + kPartLanes, ...; lane_sum.h combines them, as in
// sym_reduce.h), then the epilogue.  H = 2: a record is a pair.
template <int H, typename Acc, class Epi>
__global__ __launch_bounds__(256) void part_reduce_kernel(const float* __restrict__ part, int i0, int nt, Epi epi)
{
    int j, t;
    sym_reduce_lane<kPartLanes>(j, t);
    const int jj = j < nt ? j : nt - 1;
    const Part3* rec = (const Part3*)part;
    Acc s[3] = {Acc(0), Acc(0), Acc(0)};
#pragma unroll
    for (int p = t; p < kSourceParts / 2; p += kPartLanes) {
        Part3 r = rec[(size_t)(H == 2 ? p : 2 * p) * nt + jj];
        if constexpr (H == 1) {
            const Part3 q = rec[(size_t)(2 * p + 1) * nt + jj];
            r.x += q.x; r.y += q.y; r.z += q.z;
        }
        part_add(s, r);
    }
#pragma unroll
    for (int c = 0; c < 3; ++c)
        s[c] = lane_sum<64 / kPartLanes>(s[c]);
    if (j < nt && t == 0)
        sum_epilogue(epi, i0 + j, s);
}

// Targets [i0, i0 + nt), as many per launch as the workspace holds.
template <int K, int H, bool COMP, bool NEWTON, class Epi>
hipError_t launch_part_tile(const float4* src, int i0, int nt, int n_pad, float eps2, const PartWs& ws, const Epi& epi,
                            hipStream_t st)
{
    constexpr int P = kSourceParts / H;
    using Acc = typename std::conditional<COMP, double, float>::type;
    const size_t most = ws.p ? ws.floats / (3 * P) : 0;
    if (most < 1)
        return hipErrorInvalidValue;
    for (int a = 0; a < nt;) {
        const int c = most < (size_t)(nt - a) ? (int)most : nt - a;
        const int tiles = (c + 64 * K - 1) / (64 * K);
        hipLaunchKernelGGL((part_force_kernel<K, H, COMP, NEWTON>), dim3((tiles + 3) / 4, P), dim3(256), 0, st, src,
                           i0 + a, c, n_pad, eps2, ws.p);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess)
            return e;
        const dim3 grid((unsigned)(((long long)c * kPartLanes + 255) / 256));
        hipLaunchKernelGGL((part_reduce_kernel<H, Acc, Epi>), grid, dim3(256), 0, st, ws.p, i0 + a, c, epi);
        e = hipGetLastError();
        if (e != hipSuccess)
            return e;
        a += c;
    }
    return hipSuccess;
}

}  // namespace utcnb

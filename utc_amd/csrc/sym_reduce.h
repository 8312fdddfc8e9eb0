// sym_reduce.h -- per-body sums of the symmetric kernels' partials (device
// code only), shared by the force (sym.hip) and VJP (sym_vjp.hip) reductions.
//
// Body b of a system with NW wave blocks of 64K bodies has R target-side
// partials, row r of ipart (n_pad records) from wave r of its wave block, and
// the reactions from the NW/2 wave blocks before its own, d + 1 = 1 .. NW/2
// places below, the one half way round only where the upper half did not skip
// it.  Undivided sub-units (RS = 1): one record per wave block and d, jpart
// [NW][NW/2][64K].  Divided ones (sym_split.h): each of the waves that share
// a sub-unit left a record of 64 bodies, jpart [NW][R][J][64].
// T lanes share a body: lane t adds rows t, t + T, ... of ipart, then the
// reactions from d = t, t + T, ..., in that order (in FP64 on the compensated
// paths, in FP32 on the plain one), then the T sums are combined over the lane
// bits (lane_sum.h).  The order depends only on (T, R, RS, NW), in batches on
// (R, NW) (sym_batch_sum), so results are bitwise repeatable; with T = 1 it is the
// plain sequential order.  Lane
// layout in a wave: lane = t * (64/T) + j for the wave's j-th body, so the 64/T
// lanes of one t read 64/T consecutive records.
#pragma once

#include <hip/hip_runtime.h>

#include "lane_sum.h"
#include "sym_split.h"

namespace utcnb {

struct Part3 {
    float x, y, z;
};

template <typename Acc>
__device__ __forceinline__ void part_add(Acc (&s)[3], const Part3& p)
{
    s[0] += p.x; s[1] += p.y; s[2] += p.z;
}
__device__ __forceinline__ void part_add(double (&s)[4], const float4& p)
{
    s[0] += p.x; s[1] += p.y; s[2] += p.z; s[3] += p.w;
}

// Lanes per body: the fewest (1..16) that give the reduction about 2^19
// threads, enough waves to keep HBM requests in flight at small N.
inline int sym_reduce_lanes(long long bodies)
{
    int T = 1;
    while (T < 16 && bodies * T < (1LL << 19))
        T *= 2;
    return T;
}

// (body, t) of this thread for T lanes per body; bodies are numbered from the
// first body of the launch.
template <int T>
__device__ __forceinline__ void sym_reduce_lane(int& body, int& t)
{
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    const int lane = g & 63;
    t = lane / (64 / T);
    body = (g >> 6) * (64 / T) + lane % (64 / T);
}

// All 64 lanes of the wave must call this (it exchanges lanes); b must be a
// valid body of the system for every lane.
template <int T, bool SPLIT, typename P, typename Acc, int C>
__device__ __forceinline__ void sym_split_sum(const P* __restrict__ ipart, const P* __restrict__ jpart, int b,
                                              int NW, int R, int K, int t, Acc (&s)[C], int rs = 1)
{
    const int n_pad = NW * 64 * K;
    const int half = NW / 2, v = b / (64 * K), loc = b - v * (64 * K);
#pragma unroll
    for (int c = 0; c < C; ++c)
        s[c] = Acc(0);
    if constexpr (!SPLIT) {
        const int Q = R + half;
#pragma unroll 4
        for (int q = t; q < Q; q += T) {
            const P* p;
            if (q < R) {
                p = ipart + (size_t)q * n_pad + b;
            } else {
                const int d = q - R;
                int w = v - 1 - d;
                if (w < 0)
                    w += NW;
                if (2 * (d + 1) == NW && w >= half)
                    continue;
                p = jpart + ((size_t)w * half + d) * (64 * K) + loc;
            }
            part_add(s, *p);
        }
    } else {
#pragma unroll 4
        for (int r = t; r < R; r += T)
            part_add(s, ipart[(size_t)r * n_pad + b]);
        const int J = SymSplit::records(NW, K, R, rs), kb = loc >> 6, lane = loc & 63;
        for (int d = t; d < half; d += T) {
            int w = v - 1 - d;
            if (w < 0)
                w += NW;
            if (2 * (d + 1) == NW && w >= half)
                continue;
            const SymSplit sp(NW, w, K, R, rs);
            const int q = (d + 1) * K + kb, r0 = sp.wave(q * rs), r1 = sp.wave((q + 1) * rs - 1);
            // the waves after the first began inside the sub-unit: it is their
            // record 0.  Four records in flight (one at a time, each with its
            // division: the VJP's reduction at N = 4096 6.3 us, now 5.4).
            const P* p = jpart + (((size_t)w * R + r0) * J) * 64 + lane;
            const int first = (q - sp.first(r0) / rs) * 64;
            for (int r = 0; r <= r1 - r0; r += 4) {
                P x[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const int i = r + k < r1 - r0 ? r + k : r1 - r0;
                    x[k] = p[(size_t)i * J * 64 + (i == 0 ? first : 0)];
                }
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (r + k <= r1 - r0)
                        part_add(s, x[k]);
            }
        }
    }
#pragma unroll
    for (int c = 0; c < C; ++c)
        s[c] = lane_sum<64 / T>(s[c]);
}

// The same sums of undivided sub-units in batches, in an order that does not
// depend on T, which follows the batch's size, so that a system's bits are its
// own: always 16 interleaved sums, 16 / T to a lane, which meet in the order of
// lane_sum's levels for T = 16.
template <int T, typename P, int C>
__device__ __forceinline__ void sym_batch_sum(const P* __restrict__ ipart, const P* __restrict__ jpart, int b, int NW,
                                              int R, int K, int t, double (&s)[C])
{
    constexpr int U = 16 / T;
    const int n_pad = NW * 64 * K, half = NW / 2, v = b / (64 * K), loc = b - v * (64 * K);
    // the last record is the block half way round's, which a lower half's body
    // does not have: the upper half skipped it
    const int Q = R + half - (NW % 2 == 0 && v < half);
    const auto record = [&](int q) {
        const int d = q - R;
        int w = v - 1 - d;
        if (w < 0)
            w += NW;
        return *(q < R ? ipart + (size_t)q * n_pad + b : jpart + ((size_t)w * half + d) * (64 * K) + loc);
    };
    double a[U][C];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
        for (int c = 0; c < C; ++c)
            a[u][c] = 0.0;
    int q = t;
#pragma unroll(U >= 4 ? 1 : 4 / U)
    for (; q + T * (U - 1) < Q; q += 16)
#pragma unroll
        for (int u = 0; u < U; ++u)
            part_add(a[u], record(q + T * u));
#pragma unroll
    for (int u = 0; u < U - 1; ++u)
        if (q + T * u < Q)
            part_add(a[u], record(q + T * u));
#pragma unroll
    for (int m = U / 2; m >= 1; m /= 2)
#pragma unroll
        for (int u = 0; u < m; ++u)
#pragma unroll
            for (int c = 0; c < C; ++c)
                a[u][c] += a[u + m][c];
#pragma unroll
    for (int c = 0; c < C; ++c)
        s[c] = lane_sum<64 / T>(a[0][c]);
}

}  // namespace utcnb

// force_tmpl.h -- all-pairs softened-gravity kernels for gfx950 (CDNA4).
//
// Mapping.  A wavefront owns K target bodies per lane (64*K targets) and
// streams a contiguous range of source bodies.  The source index is uniform
// across the wave: with K = 1 or S = 1 source bodies come through scalar loads
// (s_load_dwordx16 = four float4 bodies) into SGPRs and every VALU op takes
// its source operand straight from an SGPR, else through vector loads of one
// address (at the kernel): no LDS traffic and no broadcast instructions in the
// inner loop.  S waves of a workgroup split the source
// range of one target tile; their partial sums meet in LDS at the end.
//
// Arithmetic per pair (the reference's pair, benchapps/nbody/seq/bodysystem.h:70-96,
// rewritten for the VALU): r = pj - pi (3 sub), d2 = r.r + eps2 (3 fma),
// y = v_rsq_f32(d2) (transcendental), s = mj*y*y*y (3 mul), acc += r*s
// (3 fma): 12 VALU instructions and a root per pair.  The roots of 8 pairs are
// taken together (rsq_group.h): k2s8 at N = 262144 18.6 ms/step, 20.8 with a
// root per pair; k2s16 20.8, was 23.7.  Replacing y^3 by rsq(d2)*rcp(d2) (11
// instructions, two transcendentals) is slower.  The NEWTON
// variant applies one Newton-Raphson step to y, carried into the cube: with
// e = 1 - d2*y^2 the refined y1 = y (1 + e/2) has y1^3 = y^3 (1 + 3e/2) +
// O(e^2) y^3, and |e| ~ 2^-22 leaves the e^2 terms far below FP32 rounding,
// so y1^3 = fma(y^3 * e, 1.5, y^3): three slots more than y^3 alone (15 per
// pair).  Refining y first and cubing it (e, y/2, fma, then the cube) costs
// four, and y*(1.5 - 0.5*d2*y*y) five.
//
// Compensation.  Each target keeps (hi, c) per component: 64 sources are
// summed plainly into a partial, which is added to hi with Kahan's
// compensated summation (Kahan 1965).  Cost: 12 ops per 64 pairs.
#pragma once

#include "internal.h"
#include "rsq_group.h"

namespace utcnb {

// m d2^{-3/2} from d2 and y = rsq(d2).
template <bool NEWTON>
__device__ __forceinline__ float pair_scale(float d2, float y, float m)
{
    if constexpr (NEWTON) {
        const float y2 = y * y;
        const float e = __builtin_fmaf(-d2, y2, 1.0f);
        const float y3 = y2 * y;
        return m * __builtin_fmaf(y3 * e, 1.5f, y3);
    } else {
        return m * y * y * y;
    }
}

// Kahan step: add partial p into (s, c).
__device__ __forceinline__ void kahan_add(float& s, float& c, float p)
{
    float y = p - c;
    float t = s + y;
    c = (t - s) - y;
    s = t;
}

// Stream sources [j0, j1) (multiple of kChunk) against K targets per lane.
template <int K, bool COMP, bool NEWTON>
__device__ __forceinline__ void stream_sources(const float4* __restrict__ src, int j0, int j1,
                                               float eps2, const float (&px)[K],
                                               const float (&py)[K], const float (&pz)[K],
                                               float (&hx)[K], float (&hy)[K], float (&hz)[K],
                                               float (&cx)[K], float (&cy)[K], float (&cz)[K])
{
    for (int jc = j0; jc < j1; jc += kChunk) {
        float ax[K], ay[K], az[K];
#pragma unroll
        for (int k = 0; k < K; ++k) {
            if constexpr (COMP) {
                ax[k] = 0.f; ay[k] = 0.f; az[k] = 0.f;
            } else {
                ax[k] = hx[k]; ay[k] = hy[k]; az[k] = hz[k];
            }
        }
        constexpr int J = K >= 4 ? 4 : 8 / K;  // sources (one or two scalar loads) per group of roots
#pragma unroll 1
        for (int j = jc; j < jc + kChunk; j += J) {
            float rx[J][K], ry[J][K], rz[J][K], d2[J * K], y[J * K], bw[J];
#pragma unroll
            for (int u = 0; u < J; ++u) {
                const float4 b = src[j + u];
                bw[u] = b.w;
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    rx[u][k] = b.x - px[k];
                    ry[u][k] = b.y - py[k];
                    rz[u][k] = b.z - pz[k];
                    d2[u * K + k] = __builtin_fmaf(rx[u][k], rx[u][k],
                                                   __builtin_fmaf(ry[u][k], ry[u][k],
                                                                  __builtin_fmaf(rz[u][k], rz[u][k], eps2)));
                }
            }
            rsq_group<J * K>(d2, y);
#pragma unroll
            for (int u = 0; u < J; ++u)
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    const float s = pair_scale<NEWTON>(d2[u * K + k], y[u * K + k], bw[u]);
                    ax[k] = __builtin_fmaf(rx[u][k], s, ax[k]);
                    ay[k] = __builtin_fmaf(ry[u][k], s, ay[k]);
                    az[k] = __builtin_fmaf(rz[u][k], s, az[k]);
                }
        }
#pragma unroll
        for (int k = 0; k < K; ++k) {
            if constexpr (COMP) {
                kahan_add(hx[k], cx[k], ax[k]);
                kahan_add(hy[k], cy[k], ay[k]);
                kahan_add(hz[k], cz[k], az[k]);
            } else {
                hx[k] = ax[k]; hy[k] = ay[k]; hz[k] = az[k];
            }
        }
    }
}

// ---- epilogues ---------------------------------------------------------------
// Called once per target i < n with the summed field a = hi + c' where c' is
// the compensation term (zero for plain sums).  load(i) reads the state the
// update needs and store(i, state, ...) applies it, so a kernel can issue the
// loads early; operator() does both.

// Plain FP32 state, the reference's damped kick-drift
// (benchapps/nbody/seq/bodysystem.cc:161-172) with kick factor pos.w or 1.
struct EpiFP32 {
    const float4* pos_old;
    float4* pos_new;
    float4* vel;
    float dt, damping;
    int kick;
    struct State {
        float4 p, v;
    };
    __device__ __forceinline__ State load(int i) const { return {pos_old[i], vel[i]}; }
    __device__ __forceinline__ void store(int i, State st, float hx, float hy, float hz, float, float,
                                          float) const
    {
        float4 p = st.p;
        float4 v = st.v;
        float w = kick == UTCNB_KICK_REFERENCE ? p.w : 1.0f;
        v.x = (v.x + (hx * w) * dt) * damping;
        v.y = (v.y + (hy * w) * dt) * damping;
        v.z = (v.z + (hz * w) * dt) * damping;
        p.x += v.x * dt;
        p.y += v.y * dt;
        p.z += v.z * dt;
        pos_new[i] = p;
        vel[i] = v;
    }
    __device__ __forceinline__ void operator()(int i, float hx, float hy, float hz, float cx, float cy,
                                               float cz) const
    {
        store(i, load(i), hx, hy, hz, cx, cy, cz);
    }
};

// FP64 state updated in place, new FP32 snapshot written for the next step and
// once more to keep (or null; the adjoint's trajectory).
struct EpiMixed {
    double4* pos;
    double4* vel;
    float4* snap_new;
    double dt, damping;
    int kick;
    float4* keep = nullptr;
    struct State {
        double4 p, v;
    };
    __device__ __forceinline__ State load(int i) const { return {pos[i], vel[i]}; }
    __device__ __forceinline__ void store(int i, State st, float hx, float hy, float hz, float cx, float cy,
                                          float cz) const
    {
        // Kahan keeps the running error as -c; the sum is hi - c.
        double ax = (double)hx - (double)cx;
        double ay = (double)hy - (double)cy;
        double az = (double)hz - (double)cz;
        double4 p = st.p;
        double4 v = st.v;
        double w = kick == UTCNB_KICK_REFERENCE ? p.w : 1.0;
        v.x = (v.x + (ax * w) * dt) * damping;
        v.y = (v.y + (ay * w) * dt) * damping;
        v.z = (v.z + (az * w) * dt) * damping;
        p.x += v.x * dt;
        p.y += v.y * dt;
        p.z += v.z * dt;
        pos[i] = p;
        vel[i] = v;
        const float4 s = make_float4((float)p.x, (float)p.y, (float)p.z, (float)p.w);
        snap_new[i] = s;
        if (keep)
            keep[i] = s;
    }
    __device__ __forceinline__ void operator()(int i, float hx, float hy, float hz, float cx, float cy,
                                               float cz) const
    {
        store(i, load(i), hx, hy, hz, cx, cy, cz);
    }
};

// Field only, as FP64 [3n]; body i goes to row i - off (off = the first
// target of a slice, 0 for all bodies).
struct EpiAccel {
    double* acc3;
    int off = 0;
    struct State {};
    __device__ __forceinline__ State load(int) const { return {}; }
    __device__ __forceinline__ void store(int i, State, float hx, float hy, float hz, float cx, float cy,
                                          float cz) const
    {
        const size_t r = 3 * (size_t)(i - off);
        acc3[r + 0] = (double)hx - (double)cx;
        acc3[r + 1] = (double)hy - (double)cy;
        acc3[r + 2] = (double)hz - (double)cz;
    }
    __device__ __forceinline__ void operator()(int i, float hx, float hy, float hz, float cx, float cy,
                                               float cz) const
    {
        store(i, load(i), hx, hy, hz, cx, cy, cz);
    }
};

// The epilogues take (hi, c) with value hi - c; split an FP64 sum exactly.
template <class Epi>
__device__ __forceinline__ void sum_epilogue(const Epi& epi, int i, const double (&s)[3])
{
    const float h0 = (float)s[0], h1 = (float)s[1], h2 = (float)s[2];
    epi(i, h0, h1, h2, (float)((double)h0 - s[0]), (float)((double)h1 - s[1]), (float)((double)h2 - s[2]));
}

// Plain FP32 sums go to the epilogue as they are (no compensation term).
template <class Epi>
__device__ __forceinline__ void sum_epilogue(const Epi& epi, int i, const float (&s)[3])
{
    epi(i, s[0], s[1], s[2], 0.f, 0.f, 0.f);
}

}  // namespace utcnb

#include "force_part.h"   // use the pieces above
#include "force_small.h"

namespace utcnb {

// ---- the kernel --------------------------------------------------------------
// W waves per workgroup; S of them split the sources of one target tile, so a
// workgroup holds W/S target tiles of 64*K bodies.  `src` holds n_pad bodies
// (multiple of kPadJ); the targets are bodies [i0, i0 + nt) (all n bodies, or
// one slice of them, against every source).
template <int K, int S, int W, bool COMP, bool NEWTON, class Epi>
__global__ __launch_bounds__(64 * W) void force_kernel(const float4* __restrict__ src, int i0, int nt,
                                                       int n_pad, float eps2, Epi epi)
{
    constexpr int T = W / S;  // target tiles per workgroup
    const int lane = threadIdx.x & 63;
    // K = 1: in a scalar register, so that the sources come through scalar loads;
    // 16 waves of vector loads, 1 KiB each, were bound by the L1 with a source for
    // one pair per lane (N = 16384: k1s16 143 us, now 87, k1s8 124 and 114; 131072:
    // k1s4 8.9 and 4.5 ms).  With K = 2 and 4 the vector loads are faster up to
    // 40000 bodies, as scalar ones leave one group of them in flight (k2s2 at 16384
    // 736 us, scalar 879; k2s8 196 and 215).
    const int w0 = threadIdx.x >> 6, wave = K == 1 ? __builtin_amdgcn_readfirstlane(w0) : w0;
    const int tile = blockIdx.x * T + wave / S;
    const int part = wave % S;

    float px[K], py[K], pz[K];
    float hx[K], hy[K], hz[K], cx[K], cy[K], cz[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        int t = tile * 64 * K + k * 64 + lane;
        int il = i0 + (t < nt ? t : nt - 1);  // clamp: lanes past the last target compute but never store
        float4 p = src[il];
        px[k] = p.x; py[k] = p.y; pz[k] = p.z;
        hx[k] = hy[k] = hz[k] = 0.f;
        cx[k] = cy[k] = cz[k] = 0.f;
    }
    const int len = n_pad / S;
    stream_sources<K, COMP, NEWTON>(src, part * len, part * len + len, eps2, px, py, pz, hx, hy,
                                    hz, cx, cy, cz);

    if constexpr (S > 1) {
        // Partials of the S waves meet in LDS; wave part 0 combines them in
        // part order (deterministic).
        __shared__ float red[W][K][6][64];
#pragma unroll
        for (int k = 0; k < K; ++k) {
            red[wave][k][0][lane] = hx[k];
            red[wave][k][1][lane] = hy[k];
            red[wave][k][2][lane] = hz[k];
            red[wave][k][3][lane] = cx[k];
            red[wave][k][4][lane] = cy[k];
            red[wave][k][5][lane] = cz[k];
        }
        __syncthreads();
        if (part != 0)
            return;
#pragma unroll
        for (int q = 1; q < S; ++q) {
#pragma unroll
            for (int k = 0; k < K; ++k) {
                if constexpr (COMP) {
                    // fold the other wave's (hi, c): hi - c is its value
                    kahan_add(hx[k], cx[k], red[wave + q][k][0][lane] - red[wave + q][k][3][lane]);
                    kahan_add(hy[k], cy[k], red[wave + q][k][1][lane] - red[wave + q][k][4][lane]);
                    kahan_add(hz[k], cz[k], red[wave + q][k][2][lane] - red[wave + q][k][5][lane]);
                } else {
                    hx[k] += red[wave + q][k][0][lane];
                    hy[k] += red[wave + q][k][1][lane];
                    hz[k] += red[wave + q][k][2][lane];
                }
            }
        }
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
        int t = tile * 64 * K + k * 64 + lane;
        if (t < nt)
            epi(i0 + t, hx[k], hy[k], hz[k], cx[k], cy[k], cz[k]);
    }
}

template <int K, int S, bool COMP, bool NEWTON, class Epi>
hipError_t launch_force_tile(const float4* src, int i0, int nt, int n_pad, float eps2, const Epi& epi,
                             hipStream_t st)
{
    constexpr int W = S < 4 ? 4 : S;
    constexpr int T = W / S;
    const int tiles = (nt + 64 * K - 1) / (64 * K);
    const int blocks = (tiles + T - 1) / T;
    hipLaunchKernelGGL((force_kernel<K, S, W, COMP, NEWTON, Epi>), dim3(blocks), dim3(64 * W), 0,
                       st, src, i0, nt, n_pad, eps2, epi);
    return hipGetLastError();
}

// Dispatch over the tile table (must match tile_get()); targets [i0, i0 + nt).
// part: workspace of the tiles with source parts.
// n: the system's bodies (the small-system tiles read no more of src, the
// others the n_pad padded ones).
template <bool COMP, bool NEWTON, class Epi>
hipError_t launch_force_range(int tile, const float4* src, int i0, int nt, int n, int n_pad, float eps2,
                              const PartWs& part, const Epi& epi, hipStream_t st)
{
    if (nt < 1)
        return hipErrorInvalidValue;
    switch (tile) {
    case kTilePart128: return launch_part_tile<1, 1, COMP, NEWTON>(src, i0, nt, n_pad, eps2, part, epi, st);
    case kTilePart64: return launch_part_tile<2, 2, COMP, NEWTON>(src, i0, nt, n_pad, eps2, part, epi, st);
    case 0: return launch_force_tile<1, 1, COMP, NEWTON>(src, i0, nt, n_pad, eps2, epi, st);
    case 1: return launch_force_tile<2, 1, COMP, NEWTON>(src, i0, nt, n_pad, eps2, epi, st);
    case 2: return launch_force_tile<4, 1, COMP, NEWTON>(src, i0, nt, n_pad, eps2, epi, st);
    case 3: return launch_force_tile<1, 2, COMP, NEWTON>(src, i0, nt, n_pad, eps2, epi, st);
    case 4: return launch_force_tile<2, 2, COMP, NEWTON>(src, i0, nt, n_pad, eps2, epi, st);
    case 5: return launch_force_tile<1, 4, COMP, NEWTON>(src, i0, nt, n_pad, eps2, epi, st);
    case 6: return launch_force_tile<2, 4, COMP, NEWTON>(src, i0, nt, n_pad, eps2, epi, st);
    case 7: return launch_force_tile<1, 8, COMP, NEWTON>(src, i0, nt, n_pad, eps2, epi, st);
    case 8: return launch_force_tile<2, 8, COMP, NEWTON>(src, i0, nt, n_pad, eps2, epi, st);
    case 9: return launch_force_tile<1, 16, COMP, NEWTON>(src, i0, nt, n_pad, eps2, epi, st);
    case 28: return launch_small_tile<1, 4, 8, 2048, COMP, NEWTON>(src, i0, nt, n, eps2, epi, st);
    case 29: return launch_small_tile<1, 8, 8, 2048, COMP, NEWTON>(src, i0, nt, n, eps2, epi, st);
    // 8 targets per workgroup, 24 where 8 would take 3 rounds of the 256 CUs
    // and 24 one: 4097 to 6144 bodies (6001: 15.1 us for 19.2; 6500: 31.7 for 27.1)
    case 30:
        if (n > 4096 && n <= 6144)
            return launch_small_tile<3, 8, 16, 8192, COMP, NEWTON>(src, i0, nt, n, eps2, epi, st);
        return launch_small_tile<1, 8, 16, 8192, COMP, NEWTON>(src, i0, nt, n, eps2, epi, st);
    case 31: return launch_small_tile<1, 16, 16, 4096, COMP, NEWTON>(src, i0, nt, n, eps2, epi, st);
    case 32: return launch_small_tile<1, 16, 16, 8192, COMP, NEWTON>(src, i0, nt, n, eps2, epi, st);
    case 33: return launch_small_tile<2, 16, 16, 8192, COMP, NEWTON>(src, i0, nt, n, eps2, epi, st);
    case 34: return launch_force_tile<2, 16, COMP, NEWTON>(src, i0, nt, n_pad, eps2, epi, st);
    case 35: return launch_force_tile<4, 8, COMP, NEWTON>(src, i0, nt, n_pad, eps2, epi, st);
    case 36: return launch_force_tile<4, 16, COMP, NEWTON>(src, i0, nt, n_pad, eps2, epi, st);
    default: return hipErrorInvalidValue;
    }
}

// All n bodies as targets.
template <bool COMP, bool NEWTON, class Epi>
hipError_t launch_force(int tile, const float4* src, int n, int n_pad, float eps2, const PartWs& part,
                        const Epi& epi, hipStream_t st)
{
    return launch_force_range<COMP, NEWTON>(tile, src, 0, n, n, n_pad, eps2, part, epi, st);
}

}  // namespace utcnb

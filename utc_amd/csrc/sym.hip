// sym.hip -- all-pairs force evaluating every unordered pair once.
//
// The field on body i from body j and the reaction on j from i share r, d^2
// and y^3 = (|r|^2 + eps2)^{-3/2}: a_i += m_j y^3 r, a_j -= m_i y^3 r.  The
// one-pass kernels (force_tmpl.h) spend 12 VALU instructions and a root per
// ordered pair; here an unordered pair costs 16 (3 sub, 3 fma, 2 mul for y^3,
// 2 mul for the two mass factors, 6 fma for the two accumulations) and a
// root, 8 and half a root per ordered pair.  When the wave's targets and the
// block's sources all have one mass m (the reference's initial conditions
// give every body mass 1), both sides use y^3 r directly and the block
// partials are scaled by m once: 14 instructions.  For m a power of two the
// two forms are bitwise equal; otherwise they differ by the rounding of one
// product per partial.
//
// Mapping.  Bodies form wave blocks of 64*K (lane l holds K targets).  Wave
// block w takes (a) its own K blocks of 64 sources: block kb both sides
// against target slots k < kb and target side only against slot kb (K <= 4;
// at K = 8, target side only against every slot), and (b) the source blocks
// of wave blocks v = w+1 .. w+NW/2 (mod NW), both sides; for even NW the
// block half way round is taken by the lower half only, so every unordered
// pair of wave blocks is visited exactly once.  A block of 64
// sources lies in the wave's own LDS, twice in a row; at step t = 0 .. 63 lane
// l meets source (l + t) mod 64, at slot l + t, and adds its K reactions to
// the source's sum in LDS at the same slot (slots s and s + 64 are one source
// and meet at the end), so after 64 steps every target has met every source.
// No two lanes touch one slot in a step and the steps of a wave run in order,
// so the sums need no atomics and are the same on every run.
// R waves split a wave block's work into sub-units (u, kb): source block kb of
// unit u, where unit 0 is the wave block's own sources and unit 1 + d the wave
// block d + 1 places round; wave r takes sub-units [Q*r/R, Q*(r+1)/R) of
// Q = K (NW/2 + 1).  The waves' target-side partials and the reaction
// partials go to HBM, and a second kernel adds them per body in a fixed order
// (deterministic) and applies the integrator epilogue.
// Smaller systems have few sub-units per wave: one more or less is a large part
// of a wave's work, and while the longer waves finish the SIMD's others are
// gone (a wave alone issues half as fast).  Tiles with a rotation split RS
// (SPLIT kernels) cut each sub-unit's 64 rotation steps into RS chunks of 64/RS
// steps, and the R waves of a wave block share its Q * RS chunks in a row;
// a sub-unit that two waves share has a reaction record from each.  N = 16384
// 61.5 us per step against 67.5 with whole sub-units of K = 4, 32768 195 against
// 211, 9001 33.2 against 38.7 (sweeps at tile_default in force_fp32.hip).
//
// What bounds it: FP32 issue and, at large N, the power the FMAs draw.  A step
// issues one 16-byte and three 4-byte LDS reads and three LDS writes beside
// its K pairs; carrying the source and its sums round the wave in registers
// instead (7 DPP moves per step, which pair with nothing), as launches of few
// waves do (sym_block_reg), and taking each root as it comes cost 55 cycles per
// pair and wave where this takes 44 (N = 262144, equal masses: 23.2e6 clocks for
// 28.9e6; the clock drops from 2383 to 2113 MHz meanwhile, so the time falls
// less).  Per step, mixed, same
// device: N = 262144 10.7-10.9 ms (12.3 before), log-uniform masses 11.8
// (14.0), N = 65536 0.716 ms (0.829), plain FP32 0.700 (0.819), N = 16384
// (sym4r64) 68 us (75).  The roots are taken 4 at a time: with 8 the K = 8
// kernel needs 202 VGPRs (two waves per SIMD) and runs 3-10% slower; held to
// 128 VGPRs it spills and runs 8-10% slower.
#include "force_tmpl.h"
#include "sym_items.h"
#include "sym_reduce.h"

namespace utcnb {

// Adds a block partial p into the running target sum: Kahan-compensated
// (COMP) or plain FP32.
template <bool COMP>
__device__ __forceinline__ void block_add(float& a, float& c, float p)
{
    if constexpr (COMP)
        kahan_add(a, c, p);
    else
        a += p;
}

// A wave's source block and its reaction sums in LDS (wave private).  Slots are
// read and written up to 127 = 63 + 64.
struct SymLds {
    float4 s[128];    // the block's 64 sources, twice
    float g[3][128];  // reaction sums of source (slot mod 64)
};

// LDS written by other lanes of the wave is read after this (the wave's LDS
// operations run in order; this keeps the compiler from moving them).
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// A block of 64 sources (lane l's source s) into the wave's LDS, its reaction
// sums zeroed (N2 > 0).
template <int N2>
__device__ __forceinline__ void sym_fill(SymLds& L, int lane, float4 s)
{
    wave_lds_fence();
    L.s[lane] = s;
    L.s[lane + 64] = s;
    if constexpr (N2 > 0) {
#pragma unroll
        for (int c = 0; c < 3; ++c)
            L.g[c][lane] = L.g[c][lane + 64] = 0.f;
    }
    wave_lds_fence();
}

// Rotation steps [t0, t0 + steps) of the block in L against target slots
// 0 .. N-1 of each lane: at step t lane l meets source (l + t) mod 64.  Slots
// k < N2 are two-sided; the others collect the target side only.  Target-side
// sums are added to p, the reactions to the sources' sums in L.
// UNI: every target mass mi[k] and source mass is the same, and the sums lack
// that factor.  STEPSUM: a step's N2 reactions on a source are summed by
// themselves before they meet its sum, which so takes 64 additions, not 64 N2.
template <int K, int N, int N2, bool NEWTON, bool UNI, bool STEPSUM>
__device__ __forceinline__ void sym_rotate(SymLds& L, int lane, int t0, int steps, const float (&xi)[K],
                                           const float (&yi)[K], const float (&zi)[K], const float (&mi)[K],
                                           float eps2, float (&px)[N], float (&py)[N], float (&pz)[N])
{
    const float4* sp = &L.s[lane + t0];
    float* gp = &L.g[0][lane + t0];
    float4 cur = *sp;
    // a loop with the LDS fences and a run-time trip count is not unrolled
    // otherwise; steps is a multiple of 4
    for (int t4 = 0; t4 < steps; t4 += 4)
#pragma unroll
    for (int t = t4; t < t4 + 4; ++t) {
        const float4 nxt = sp[t + 1];  // the next step's source: at most L.s[127]
        float ox = 0.f, oy = 0.f, oz = 0.f;
        if constexpr (N2 > 0) {
            ox = gp[t]; oy = gp[128 + t]; oz = gp[256 + t];
        }
        float gx = STEPSUM ? 0.f : ox, gy = STEPSUM ? 0.f : oy, gz = STEPSUM ? 0.f : oz;
        constexpr int GK = N < 4 ? N : 4;  // pairs per group of reciprocal roots
#pragma unroll
        for (int k0 = 0; k0 < N; k0 += GK) {
            float rx[GK], ry[GK], rz[GK], d2[GK], y[GK];
#pragma unroll
            for (int q = 0; q < GK; ++q) {
                const int k = k0 + q;
                rx[q] = cur.x - xi[k]; ry[q] = cur.y - yi[k]; rz[q] = cur.z - zi[k];
                d2[q] = __builtin_fmaf(rx[q], rx[q], __builtin_fmaf(ry[q], ry[q], __builtin_fmaf(rz[q], rz[q], eps2)));
            }
            rsq_group<GK>(d2, y);
#pragma unroll
            for (int q = 0; q < GK; ++q) {
                const int k = k0 + q;
                const float y3 = pair_scale<NEWTON>(d2[q], y[q], 1.0f);
                const float si = UNI ? y3 : cur.w * y3;
                px[k] = __builtin_fmaf(rx[q], si, px[k]);
                py[k] = __builtin_fmaf(ry[q], si, py[k]);
                pz[k] = __builtin_fmaf(rz[q], si, pz[k]);
                if (k < N2) {
                    const float cj = UNI ? y3 : mi[k] * y3;
                    gx = __builtin_fmaf(-rx[q], cj, gx);
                    gy = __builtin_fmaf(-ry[q], cj, gy);
                    gz = __builtin_fmaf(-rz[q], cj, gz);
                }
            }
        }
        if constexpr (N2 > 0) {
            gp[t] = STEPSUM ? ox + gx : gx;
            gp[128 + t] = STEPSUM ? oy + gy : gy;
            gp[256 + t] = STEPSUM ? oz + gz : gz;
        }
        wave_lds_fence();
        cur = nxt;
    }
}

// Lane l receives lane l-1's value (lane 0 lane 63's).  Every lane has a source
// under wave_ror:1, so the "old" operand is never used; passing v rotates in
// place (K = 2, 7.7% faster there), 0 writes a new register (K = 8, 3%).
template <int K>
__device__ __forceinline__ float wave_ror1(float v)
{
    const int x = __float_as_int(v);
    return __int_as_float(__builtin_amdgcn_update_dpp(K <= 2 ? x : 0, x, 0x13C /* wave_ror:1 */, 0xF, 0xF, false));
}

// sym_block (below) with the block and its reaction sums carried round the wave
// in registers: at step t lane l meets source (l - t) mod 64.  The DPP moves pair
// with nothing, but a wave that has a SIMD to itself waits longer for the LDS of
// sym_rotate than it issues them.
template <int K, int N, int N2, bool NEWTON, bool COMP, bool UNI, int SPLIT>
__device__ __forceinline__ void sym_block_reg(int lane, int t0, int steps, int len, float4 s, const float (&xi)[K],
                                              const float (&yi)[K], const float (&zi)[K], const float (&mi)[K],
                                              float m, float eps2, float (&ax)[K], float (&ay)[K], float (&az)[K],
                                              float (&cx)[K], float (&cy)[K], float (&cz)[K], float (&g)[3])
{
    float sx = s.x, sy = s.y, sz = s.z, sm = s.w;
    if (SPLIT != 0 && t0 != 0) {  // wave-uniform
        const int from = (lane - t0) & 63;
        sx = __shfl(sx, from, 64); sy = __shfl(sy, from, 64); sz = __shfl(sz, from, 64); sm = __shfl(sm, from, 64);
    }
    for (int t = t0;;) {
        float px[N], py[N], pz[N], gx = 0.f, gy = 0.f, gz = 0.f;
#pragma unroll
        for (int k = 0; k < N; ++k)
            px[k] = py[k] = pz[k] = 0.f;
        const int n = SPLIT != 0 ? len : 64;  // a multiple of 4
        for (int i4 = 0; i4 < n; i4 += 4)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                constexpr int GK = N < 4 ? N : 4;  // pairs per group of reciprocal roots
#pragma unroll
                for (int k0 = 0; k0 < N; k0 += GK) {
                    float rx[GK], ry[GK], rz[GK], d2[GK], y[GK];
#pragma unroll
                    for (int q = 0; q < GK; ++q) {
                        const int k = k0 + q;
                        rx[q] = sx - xi[k]; ry[q] = sy - yi[k]; rz[q] = sz - zi[k];
                        d2[q] = __builtin_fmaf(rx[q], rx[q],
                                               __builtin_fmaf(ry[q], ry[q], __builtin_fmaf(rz[q], rz[q], eps2)));
                        if constexpr (K == 2)
                            y[q] = __builtin_amdgcn_rsqf(d2[q]);
                    }
                    if constexpr (K != 2)
                        rsq_group<GK>(d2, y);
#pragma unroll
                    for (int q = 0; q < GK; ++q) {
                        const int k = k0 + q;
                        const float y3 = pair_scale<NEWTON>(d2[q], y[q], 1.0f);
                        const float si = UNI ? y3 : sm * y3;
                        px[k] = __builtin_fmaf(rx[q], si, px[k]);
                        py[k] = __builtin_fmaf(ry[q], si, py[k]);
                        pz[k] = __builtin_fmaf(rz[q], si, pz[k]);
                        if (k < N2) {
                            const float cj = UNI ? y3 : mi[k] * y3;
                            gx = __builtin_fmaf(-rx[q], cj, gx);
                            gy = __builtin_fmaf(-ry[q], cj, gy);
                            gz = __builtin_fmaf(-rz[q], cj, gz);
                        }
                    }
                }
                sx = wave_ror1<K>(sx); sy = wave_ror1<K>(sy); sz = wave_ror1<K>(sz);
                if constexpr (!UNI)
                    sm = wave_ror1<K>(sm);
                if constexpr (N2 > 0) {
                    gx = wave_ror1<K>(gx); gy = wave_ror1<K>(gy); gz = wave_ror1<K>(gz);
                }
            }
#pragma unroll
        for (int k = 0; k < N; ++k) {
            if constexpr (UNI) {
                px[k] *= m; py[k] *= m; pz[k] *= m;
            }
            block_add<COMP>(ax[k], cx[k], px[k]);
            block_add<COMP>(ay[k], cy[k], py[k]);
            block_add<COMP>(az[k], cz[k], pz[k]);
        }
        if constexpr (N2 > 0) {
            const int home = (t + n) & 63;  // lane l holds the sums of source l - home
            if (SPLIT != 0 && home != 0) {
                const int from = (lane + home) & 63;
                gx = __shfl(gx, from, 64); gy = __shfl(gy, from, 64); gz = __shfl(gz, from, 64);
            }
            g[0] = t == t0 ? gx : g[0] + gx;
            g[1] = t == t0 ? gy : g[1] + gy;
            g[2] = t == t0 ? gz : g[2] + gz;
        }
        t += n;
        if (SPLIT == 0 || t >= t0 + steps)
            break;
    }
    if constexpr (UNI && N2 > 0) {
#pragma unroll
        for (int c = 0; c < 3; ++c)
            g[c] *= m;
    }
}

// Rotation steps [t0, t0 + steps) of a block of 64 sources against the lanes'
// target slots (sym_rotate): target-side partials are added into (a, c) by
// block_add<COMP>, the reaction sums of lane l's own source come back in g
// (N2 > 0), all of it scaled by the mass m (UNI).
// SPLIT 1, K <= 4: partials and reaction sums are taken up after every len
// steps, a chunk, so that no chain of plain FP32 additions is longer than a
// chunk's pairs.  SPLIT 2: STEPSUM (K = 8, for the sizes whose K = 2 and 4 tiles
// had chains a quarter as long).  Field's error against 64 bits, N = 16384 in a
// cube, Newton: sym4r64x2 3.71e-8 without and 3.00e-8 with, sym8r128 5.04e-8
// without and 2.80e-8 with (59.3 and 61.1 us per step; 24575 4.18e-8 and
// 2.34e-8).
template <int K, int N, int N2, bool NEWTON, bool COMP, bool UNI, int SPLIT, bool REG>
__device__ __forceinline__ void sym_block(SymLds& L, int lane, int t0, int steps, int len, float4 s,
                                          const float (&xi)[K], const float (&yi)[K], const float (&zi)[K],
                                          const float (&mi)[K], float m, float eps2, float (&ax)[K], float (&ay)[K],
                                          float (&az)[K], float (&cx)[K], float (&cy)[K], float (&cz)[K], float (&g)[3])
{
    if constexpr (REG) {
        sym_block_reg<K, N, N2, NEWTON, COMP, UNI, SPLIT>(lane, t0, steps, len, s, xi, yi, zi, mi, m, eps2, ax, ay, az,
                                                          cx, cy, cz, g);
        return;
    }
    constexpr bool CHUNKS = SPLIT == 1 && K <= 4;
    sym_fill<N2>(L, lane, s);
    for (int t = t0;;) {
        float px[N], py[N], pz[N];
#pragma unroll
        for (int k = 0; k < N; ++k)
            px[k] = py[k] = pz[k] = 0.f;
        sym_rotate<K, N, N2, NEWTON, UNI, SPLIT == 2>(L, lane, t, CHUNKS ? len : steps, xi, yi, zi, mi, eps2, px,
                                                            py, pz);
#pragma unroll
        for (int k = 0; k < N; ++k) {
            if constexpr (UNI) {
                px[k] *= m; py[k] *= m; pz[k] *= m;
            }
            block_add<COMP>(ax[k], cx[k], px[k]);
            block_add<COMP>(ay[k], cy[k], py[k]);
            block_add<COMP>(az[k], cz[k], pz[k]);
        }
        if constexpr (N2 > 0) {
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const float r = L.g[c][lane] + L.g[c][lane + 64];
                g[c] = t == t0 ? r : g[c] + r;
            }
        }
        if constexpr (!CHUNKS)
            break;
        t += len;
        if (t >= t0 + steps)
            break;
        if constexpr (N2 > 0) {
            wave_lds_fence();
#pragma unroll
            for (int c = 0; c < 3; ++c)
                L.g[c][lane] = L.g[c][lane + 64] = 0.f;
            wave_lds_fence();
        }
    }
    if constexpr (UNI && N2 > 0) {
#pragma unroll
        for (int c = 0; c < 3; ++c)
            g[c] *= m;
    }
}

// Own source block KB of the wave's block (K <= 4): target slots k < KB meet
// it two-sided (the pairs of blocks k and KB, each unordered pair once), slot
// KB one-sided (the block with itself: each ordered pair once, the self pair
// adds r = 0); slots k > KB take these sources when their own block is the
// source.  The reaction sums belong to slot KB.
template <int K, bool NEWTON, bool COMP, int SPLIT, bool REG, int KB = 0>
__device__ __forceinline__ void sym_own_at(int kb, bool uni, SymLds& L, int lane, int t0, int steps, int len, float4 s,
                                           const float (&xi)[K], const float (&yi)[K], const float (&zi)[K],
                                           const float (&mi)[K], float m, float eps2, float (&ax)[K], float (&ay)[K],
                                           float (&az)[K], float (&cx)[K], float (&cy)[K], float (&cz)[K])
{
    if (kb == KB) {
        float g[3];
        if (uni)
            sym_block<K, KB + 1, KB, NEWTON, COMP, true, SPLIT, REG>(L, lane, t0, steps, len, s, xi, yi, zi, mi, m, eps2, ax,
                                                                ay, az, cx, cy, cz, g);
        else
            sym_block<K, KB + 1, KB, NEWTON, COMP, false, SPLIT, REG>(L, lane, t0, steps, len, s, xi, yi, zi, mi, m, eps2, ax,
                                                                 ay, az, cx, cy, cz, g);
        if constexpr (KB > 0) {
            block_add<COMP>(ax[KB], cx[KB], g[0]);
            block_add<COMP>(ay[KB], cy[KB], g[1]);
            block_add<COMP>(az[KB], cz[KB], g[2]);
            // keeps the compiler from merging the K branches' adds into one
            // through a pointer to slot KB, which would put the sums in memory
            asm volatile("; own block %0" : : "n"(KB));
        }
    } else if constexpr (KB + 1 < K) {
        sym_own_at<K, NEWTON, COMP, SPLIT, REG, KB + 1>(kb, uni, L, lane, t0, steps, len, s, xi, yi, zi, mi, m, eps2, ax, ay,
                                                   az, cx, cy, cz);
    }
}

// The work of wave r of wave block w of one system: src = the system's
// padded bodies (NW wave blocks of 64K); ipart: [R][n_pad][3] target-side
// sums; jpart: [NW][NW/2][64K][3] reactions, or the rows of wave blocks
// jbase, jbase + 1, ... only (a chunk of a step).  ipart may also hold a
// range of bodies only: body b of row r is record r * istride + b - ibody0
// (istride < 0: n_pad, the whole system).  COMP: the target-side block
// partials are Kahan-added (the compensated paths); otherwise plain FP32 sums.
// nr: the wave does the work of waves r .. r + nr - 1 in turn (not SPLIT).
// SPLIT (1 or 2, sym_block): the waves share the sub-units by chunks of 64 / rs
// rotation steps (rs divides 16) and the reactions take a record per wave and sub-unit: jpart is
// [NW][R][J][64][3] (SymSplit, sym_split.h).
template <int K, bool NEWTON, bool COMP, int SPLIT = 0, bool REG = false>
__device__ __forceinline__ void sym_wave(const float4* __restrict__ src, int NW, int R, int w, int r,
                                         float eps2, float* __restrict__ ipart,
                                         float* __restrict__ jpart, SymLds& L, int lane, int jbase = 0,
                                         long long istride = -1, int ibody0 = 0, int rs = 1, int nr = 1)
{
    const int half = NW / 2;
    const int n_pad = NW * 64 * K;
    float xi[K], yi[K], zi[K], mi[K], ax[K], ay[K], az[K], cx[K], cy[K], cz[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const float4 p = src[w * 64 * K + k * 64 + lane];
        xi[k] = p.x; yi[k] = p.y; zi[k] = p.z; mi[k] = p.w;
    }
    // one mass for every target of the wave?
    const float m0 = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(mi[0])));
    bool tuni = true;
#pragma unroll
    for (int k = 0; k < K; ++k)
        tuni = tuni && mi[k] == m0;
    for (const int r1 = r + nr; r < r1; ++r) {
#pragma unroll
        for (int k = 0; k < K; ++k)
            ax[k] = ay[k] = az[k] = cx[k] = cy[k] = cz[k] = 0.f;
        // sub-unit q = (unit u, source block kb): u = 0 is the wave block's own
        // sources, u = 1 + d the wave block d + 1 places round
        int qf, ql, c0 = 0, c1 = 0, J = 0;
        const int len = SPLIT != 0 ? 64 / rs : 64;
        if constexpr (SPLIT != 0) {
            const SymSplit sp(NW, w, K, R, rs);
            c0 = sp.first(r);
            c1 = sp.first(r + 1);
            qf = c0 / rs;
            ql = (c1 + rs - 1) / rs;
            J = SymSplit::records(NW, K, R, rs);
        } else {
            const int Q = (half + 1) * K;
            qf = (int)((long long)Q * r / R);
            ql = (int)((long long)Q * (r + 1) / R);
        }
        for (int q = qf; q < ql; ++q) {
            // rotation steps [t0, t0 + steps): all but for the first and last sub-unit
            int t0 = 0, steps = 64;
            if constexpr (SPLIT != 0) {
                const int a = q == qf ? c0 - q * rs : 0, e = q + 1 == ql ? c1 - q * rs : rs;
                t0 = a * len;
                steps = (e - a) * len;
            }
            const int u = q / K, kb = q - u * K;
            if (u == 0) {
                const float4 s = src[w * 64 * K + kb * 64 + lane];
                const bool uni = __ballot(tuni && s.w == m0) == ~0ull;
                if constexpr (K <= 4) {
                    // own block kb: two-sided against the lower target slots
                    sym_own_at<K, NEWTON, COMP, SPLIT, REG>(kb, uni, L, lane, t0, steps, len, s, xi, yi, zi, mi, m0, eps2, ax, ay,
                                                       az, cx, cy, cz);
                } else {
                    // own block kb (K = 8, where own blocks are a small share and
                    // eight variants of sym_own_at would crowd the instruction cache):
                    // target side only (each ordered pair once, self pair gives 0)
                    float g[3];
                    sym_block<K, K, 0, NEWTON, COMP, false, SPLIT, REG>(L, lane, t0, steps, len, s, xi, yi, zi, mi, m0, eps2, ax,
                                                                   ay, az, cx, cy, cz, g);
                }
                continue;
            }
            const int d = u - 1;
            if (2 * (d + 1) == NW && w >= half)
                continue;  // the block half way round: taken by the lower half
            int v = w + 1 + d;
            if (v >= NW)
                v -= NW;
            const float4 s = src[v * 64 * K + kb * 64 + lane];
            float g[3];
            if (__ballot(tuni && s.w == m0) == ~0ull)
                sym_block<K, K, K, NEWTON, COMP, true, SPLIT, REG>(L, lane, t0, steps, len, s, xi, yi, zi, mi, m0, eps2, ax, ay,
                                                              az, cx, cy, cz, g);
            else
                sym_block<K, K, K, NEWTON, COMP, false, SPLIT, REG>(L, lane, t0, steps, len, s, xi, yi, zi, mi, m0, eps2, ax, ay,
                                                               az, cx, cy, cz, g);
            const size_t o = SPLIT != 0 ? ((((size_t)w * R + r) * J + (q - qf)) * 64 + lane) * 3
                                   : (((size_t)(w - jbase) * half + d) * (64 * K) + kb * 64 + lane) * 3;
            jpart[o + 0] = g[0];
            jpart[o + 1] = g[1];
            jpart[o + 2] = g[2];
        }
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const size_t o = ((size_t)r * (size_t)(istride < 0 ? n_pad : istride) + (w * 64 * K - ibody0) + k * 64 +
                              lane) * 3;
            ipart[o + 0] = ax[k] - cx[k];
            ipart[o + 1] = ay[k] - cy[k];
            ipart[o + 2] = az[k] - cz[k];
        }
    }
}

// One system: wave gw = w * R + r.  SPLIT: rs rotation chunks per sub-unit.
template <int K, bool NEWTON, bool COMP, int SPLIT, bool REG>
__global__ __launch_bounds__(256, 2) void sym_force_kernel(const float4* __restrict__ src, int NW, int R,
                                                        float eps2, float* __restrict__ ipart,
                                                        float* __restrict__ jpart, int rs)
{
    __shared__ SymLds lds[REG ? 1 : 4];
    int gw = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6);
    // whole sub-units: the schedule in scalar registers, 1 to 3% from 65536
    // bodies (717 to 704 us); split, the same within 0.7% either way
    if constexpr (SPLIT == 0)
        gw = __builtin_amdgcn_readfirstlane(gw);
    if (gw >= NW * R)
        return;  // whole waves only
    sym_wave<K, NEWTON, COMP, SPLIT, REG>(src, NW, R, gw / R, gw % R, eps2, ipart, jpart,
                                          lds[REG ? 0 : threadIdx.x >> 6], threadIdx.x & 63, 0, -1, 0, rs);
}

// Batched systems: each wave runs items (system, wave block, split), a system
// laid out as for one system.
template <int K>
__global__ __launch_bounds__(256) void batch_sym_kernel(BatchSymGeom g, int nwaves, const float4* __restrict__ snap,
                                                        float eps2, float* __restrict__ ipart,
                                                        float* __restrict__ jpart)
{
    __shared__ SymLds lds[4];
    const int gw = __builtin_amdgcn_readfirstlane((int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6));
    if (gw >= nwaves)
        return;  // whole waves only
    const int lane = threadIdx.x & 63;
    int pos = 0;
    for (int it = batch_next_item(g, gw, pos, lane); it >= 0; it = batch_next_item(g, gw, pos, lane)) {
        const int4 item = g.items[it];  // (system, wave block, splits)
        const int s = item.x;
        sym_wave<K, false, true>(snap + g.off[s], g.nw[s], item.w, item.y, item.z & 0xffff, eps2, ipart + g.ipo[s],
                                 jpart + g.jpo[s], lds[threadIdx.x >> 6], lane, 0, -1, 0, 1, item.z >> 16);
    }
}

// Zeroes the dynamic schedule's work counter before a launch (a kernel, not a
// memset, so the step can sit in a captured graph).
__global__ void batch_counter_reset_kernel(int* counter)
{
    if (threadIdx.x == 0)
        *counter = 0;
}

// Body b's partials summed by T lanes (sym_reduce.h) in FP64 (Acc = double,
// the compensated paths) or plain FP32 (Acc = float), then the epilogue.
template <int T, bool SPLIT, typename Acc, class Epi>
__global__ __launch_bounds__(256) void sym_reduce_kernel(const float* __restrict__ ipart,
                                                         const float* __restrict__ jpart, int n, int NW,
                                                         int R, int K, int rs, Epi epi)
{
    int b, t;
    sym_reduce_lane<T>(b, t);
    Acc s[3];
    sym_split_sum<T, SPLIT>((const Part3*)ipart, (const Part3*)jpart, b < n ? b : n - 1, NW, R, K, t, s, rs);
    if (b < n && t == 0)
        sum_epilogue(epi, b, s);
}

// Batched systems: body b of the concatenated padded layout (systems start on
// multiples of kBatchSymAlign, so block b / kBatchSymAlign names the system).
template <int T>
__global__ __launch_bounds__(256) void batch_sym_reduce_kernel(BatchSymGeom g, int total, int K,
                                                               const float* __restrict__ ipart,
                                                               const float* __restrict__ jpart, EpiMixed epi)
{
    int j, t;
    sym_reduce_lane<T>(j, t);
    const int b = g.body0 + j, bb = g.body0 + (j < total ? j : total - 1);
    const int s = g.sys_of_block[bb / kBatchSymAlign];
    const int loc = bb - g.off[s];  // padding bodies are summed too (their records exist)
    double sum[3];
    sym_batch_sum<T>((const Part3*)(ipart + g.ipo[s]), (const Part3*)(jpart + g.jpo[s]), loc, g.nw[s], g.rs[s], K, t,
                     sum);
    if (j < total && loc < g.n[s] && t == 0)
        sum_epilogue(epi, b, sum);  // padding bodies keep their far-away zero-mass records
}

// K = 8 tiles divide the sub-units of smaller systems: up to 46080 bodies
// sym8r64, below 40960 sym8r128, there with the waves that make 2048 in all
// (sweeps at tile_default, force_fp32.hip; undivided sym8r128 at 28672 161 us for
// 153).  Divided sym8r64 would be faster up to 65535 bodies (49152 406 us for
// 427), but its reaction records, one more per wave, no longer fit the 64 MiB
// of utcnb_accel_noalloc from 46081, where the undivided ones do up to 49152, and
// a tile's bits are the same with a handle and without.
int sym_tile_r(const Tile& t, int n_pad)
{
    if (t.k != 8 || t.s != 128 || n_pad >= 40960)
        return t.s;
    const int R = 2048 / (n_pad / (64 * t.k));
    return R < t.s ? R : t.s;
}

int sym_tile_rs(const Tile& t, int n_pad)
{
    return t.k == 8 && ((t.s == 64 && n_pad <= 46080) || (t.s == 128 && n_pad < 40960)) ? 8 : t.rs;
}

size_t sym_ipart_floats(int n_pad, int K, int R) { (void)K; return (size_t)R * n_pad * 3; }
size_t sym_jpart_floats(int n_pad, const Tile& t)
{
    const int NW = n_pad / (64 * t.k);
    const int rs = sym_tile_rs(t, n_pad);
    if (rs == 1)
        return (size_t)NW * (NW / 2) * 64 * t.k * 3;
    const int R = sym_tile_r(t, n_pad);
    return (size_t)NW * R * SymSplit::records(NW, t.k, R, rs) * 64 * 3;
}

// The form of the divided kernels (sym_block): to 24576 bodies K = 8 serves
// sizes that K = 2 and 4 did; above it has no longer chains than undivided, and
// summing by steps takes 3.7% at 32768.
static int sym_split_form(const Tile& t, int n_pad)
{
    if (sym_tile_rs(t, n_pad) == 1)
        return 0;
    return t.k == 8 && n_pad <= 24576 ? 2 : 1;
}

// Launches of at most this many waves carry the sources in registers
// (sym_block_reg): a wave to a SIMD, for K = 2 two.  Per step, mixed, us,
// registers and LDS: sym2r32 at 1024 bodies (256 waves) 10.8 and 13.8, 4096 (1024)
// 15.8 and 21.2, 8192 (2048) 29.4 and 31.2, 9001 (2304) 41.3 and 37.7; sym4r4 at
// 8192 (128) 165 and 186, sym4r64 at 4096 (1024) 17.7 and 18.9, sym4r16 at 20480
// (1280) 182 and 143; sym8r4 at 8192 (64) 309 and 327, sym8r32 at 20480 (1280) 170
// and 135; divided, sym2r64x2 at 2048 (1024) 9.8 and 11.5, sym4r64x2 at 4096 (1024)
// 16.9 and 18.3, at 8192 (2048) 26.8 and 26.0.  Shares: 3 of 8 of 9001 bodies (666)
// 30.1 and 32.8, of 12288 (1176) 35.2 and 34.3, of 16384 (1056) 42.6 and 39.1.
constexpr int kRegWaves = 1024, kRegWavesK2 = 2048;

template <int K, bool COMP, int SPLIT, bool REG>
static void launch_sym_pairs_as(bool newton, int rs, dim3 grid, const float4* src, int NW, int R, float eps2,
                                float* ipart, float* jpart, hipStream_t st)
{
    if (newton)
        hipLaunchKernelGGL((sym_force_kernel<K, true, COMP, SPLIT, REG>), grid, dim3(256), 0, st, src, NW, R, eps2,
                           ipart, jpart, rs);
    else
        hipLaunchKernelGGL((sym_force_kernel<K, false, COMP, SPLIT, REG>), grid, dim3(256), 0, st, src, NW, R, eps2,
                           ipart, jpart, rs);
}

template <int K, bool COMP>
static void launch_sym_pairs(bool newton, int split, int rs, dim3 grid, const float4* src, int NW, int R, float eps2,
                             float* ipart, float* jpart, hipStream_t st)
{
#define SYM_PAIRS(SPLIT, REG) launch_sym_pairs_as<K, COMP, SPLIT, REG>(newton, rs, grid, src, NW, R, eps2, ipart, jpart, st)
    const bool reg = NW * R <= (K == 2 ? kRegWavesK2 : kRegWaves);
    if constexpr (K == 8) {
        if (split == 2)
            return SYM_PAIRS(2, false);
        if (split == 1)
            return SYM_PAIRS(1, false);
    } else {
        if (split == 1 && reg)
            return SYM_PAIRS(1, true);
        if (split == 1)
            return SYM_PAIRS(1, false);
    }
    if (reg)
        SYM_PAIRS(0, true);
    else
        SYM_PAIRS(0, false);
#undef SYM_PAIRS
}

template <bool SPLIT, typename Acc, class Epi>
static void launch_sym_reduce(int T, const float* ipart, const float* jpart, int n, int NW, int R, int K, int rs,
                              const Epi& epi, hipStream_t st)
{
    const dim3 rgrid((unsigned)(((long long)n * T + 255) / 256));
#define SYM_REDUCE(TT) \
    hipLaunchKernelGGL((sym_reduce_kernel<TT, SPLIT, Acc, Epi>), rgrid, dim3(256), 0, st, ipart, jpart, n, NW, R, K, rs, \
                       epi)
    switch (T) {
    case 1: SYM_REDUCE(1); break;
    case 2: SYM_REDUCE(2); break;
    case 4: SYM_REDUCE(4); break;
    case 8: SYM_REDUCE(8); break;
    default: SYM_REDUCE(16); break;
    }
#undef SYM_REDUCE
}

// comp: Kahan-added block partials and an FP64 reduction (the MIXED step and
// the field of a MIXED handle); otherwise plain FP32 sums throughout
// (PREC_FP32).
template <class Epi>
hipError_t launch_sym(const Tile& t, bool newton, bool comp, const float4* src, int n, int n_pad, float eps2,
                      float* ipart, float* jpart, const Epi& epi, hipStream_t st)
{
    const int K = t.k, R = sym_tile_r(t, n_pad), rs = sym_tile_rs(t, n_pad), split = sym_split_form(t, n_pad);
    if (n_pad % (128 * K) != 0 || !ipart || !jpart || rs < 1 || 16 % rs != 0)
        return hipErrorInvalidValue;
    const int NW = n_pad / (64 * K);
    const int waves = NW * R;
    const dim3 grid((waves + 3) / 4);
    if (K == 2)
        comp ? launch_sym_pairs<2, true>(newton, split, rs, grid, src, NW, R, eps2, ipart, jpart, st)
             : launch_sym_pairs<2, false>(newton, split, rs, grid, src, NW, R, eps2, ipart, jpart, st);
    else if (K == 4)
        comp ? launch_sym_pairs<4, true>(newton, split, rs, grid, src, NW, R, eps2, ipart, jpart, st)
             : launch_sym_pairs<4, false>(newton, split, rs, grid, src, NW, R, eps2, ipart, jpart, st);
    else if (K == 8)
        comp ? launch_sym_pairs<8, true>(newton, split, rs, grid, src, NW, R, eps2, ipart, jpart, st)
             : launch_sym_pairs<8, false>(newton, split, rs, grid, src, NW, R, eps2, ipart, jpart, st);
    else
        return hipErrorInvalidValue;
    hipError_t e = hipGetLastError();
    if (e != hipSuccess)
        return e;
    const int T = sym_reduce_lanes(n);
    if (rs > 1 && comp)
        launch_sym_reduce<true, double>(T, ipart, jpart, n, NW, R, K, rs, epi, st);
    else if (rs > 1)
        launch_sym_reduce<true, float>(T, ipart, jpart, n, NW, R, K, rs, epi, st);
    else if (comp)
        launch_sym_reduce<false, double>(T, ipart, jpart, n, NW, R, K, rs, epi, st);
    else
        launch_sym_reduce<false, float>(T, ipart, jpart, n, NW, R, K, rs, epi, st);
    return hipGetLastError();
}

// ---- one share of a system sharded over targets by wave blocks -----------------
// Share g of G owns wave blocks [w0, w1) (the first NW % G shares one block
// more) and evaluates, for each of them, the same sub-units as sym_wave does
// in a full step: its own blocks and the half ring after it.  Its target-side
// partials go to ipart (R_share rows: the whole system's row layout, or the
// share's own contiguous region of the buffer); its reaction partials (for bodies of the wave blocks after each of its blocks,
// mostly owned by other shares) are summed per destination body into react3,
// which a sharded run adds up over the shares (a reduce-scatter); the share
// then adds its bodies' target-side partials to the summed reactions and
// integrates them.  On one device, running every share and summing the react3
// arrays gives the full step's sums in another FP64 order.

// jbase: the first wave block whose reaction rows jpart holds (0 for a
// whole-system buffer, w0 for a buffer of the share's rows only).
// ipart: rows of istride bodies starting at body ibody0 (see sym_wave).
template <int K, bool NEWTON, bool REG>
__global__ __launch_bounds__(256) void sym_share_kernel(const float4* __restrict__ src, int NW, int R, int w0,
                                                        int nwaves, float eps2, float* __restrict__ ipart,
                                                        float* __restrict__ jpart, int jbase, long long istride,
                                                        int ibody0)
{
    __shared__ SymLds lds[REG ? 1 : 4];
    const int gw = __builtin_amdgcn_readfirstlane((int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6));
    if (gw >= nwaves)
        return;  // whole waves only
    sym_wave<K, NEWTON, true, 0, REG>(src, NW, R, w0 + gw / R, gw % R, eps2, ipart, jpart,
                                      lds[REG ? 0 : threadIdx.x >> 6], threadIdx.x & 63, jbase, istride, ibody0);
}

// react3[b] (FP64, bodies b < n) = the reactions on body b from the wave
// blocks [w0, w1), in increasing block order; 0 where none of them reaches b.
// With accumulate, the previous react3[b] plus that sum.
__global__ __launch_bounds__(256) void sym_react_kernel(const float* __restrict__ jpart, int n, int NW, int K,
                                                        int w0, int w1, int jbase, bool accumulate,
                                                        double* __restrict__ react3)
{
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= n)
        return;
    const int half = NW / 2, B = 64 * K;
    const int v = b / B, loc = b - v * B;
    double s0 = 0.0, s1 = 0.0, s2 = 0.0;
    // four blocks' records in flight, a block that does not reach b adds 0 (a
    // branch around each load took them one by one: share 3 of 8 of 131072
    // bodies 14.6 us, now 9.0)
#pragma unroll 4
    for (int w = w0; w < w1; ++w) {
        int d = v - 1 - w;
        if (d < 0)
            d += NW;
        // v in w's half ring, and not skipped by w's upper half?
        const bool in = d < half && !(2 * (d + 1) == NW && w >= half);
        const Part3 p = ((const Part3*)jpart)[((size_t)(w - jbase) * half + (in ? d : 0)) * B + loc];
        s0 += in ? p.x : 0.f;
        s1 += in ? p.y : 0.f;
        s2 += in ? p.z : 0.f;
    }
    double* o = react3 + 3 * (size_t)b;
    if (accumulate) {
        o[0] += s0;
        o[1] += s1;
        o[2] += s2;
    } else {
        o[0] = s0;
        o[1] = s1;
        o[2] = s2;
    }
}

// Bodies [start, start + count): their R target-side partials (rows of
// istride bodies from body ibody0) summed in FP64 by T lanes per body (lane t
// takes rows t, t + T, ...; lane_sum.h combines the lanes, as in
// sym_reduce.h), plus react_sum3[j] (the reactions summed over the shares),
// then the epilogue.
template <int T, class Epi>
__global__ __launch_bounds__(256) void sym_share_finish_kernel(const float* __restrict__ ipart, long long istride,
                                                               int ibody0, int R, int start, int count,
                                                               const double* __restrict__ react_sum3, Epi epi)
{
    int j, t;
    sym_reduce_lane<T>(j, t);
    const int b = start + (j < count ? j : count - 1);
    double s[3] = {0.0, 0.0, 0.0};
#pragma unroll 4
    for (int r = t; r < R; r += T)
        part_add(s, ((const Part3*)ipart)[(size_t)r * (size_t)istride + (b - ibody0)]);
#pragma unroll
    for (int c = 0; c < 3; ++c)
        s[c] = lane_sum<64 / T>(s[c]);
    if (j < count && t == 0) {
        s[0] += react_sum3[3 * (size_t)j + 0];
        s[1] += react_sum3[3 * (size_t)j + 1];
        s[2] += react_sum3[3 * (size_t)j + 2];
        sum_epilogue(epi, b, s);
    }
}

void sym_share_blocks(int NW, int shares, int share, int* w0, int* w1)
{
    const int per = NW / shares, extra = NW % shares;
    *w0 = share < extra ? share * (per + 1) : share * per + extra;
    *w1 = *w0 + (share < extra ? per + 1 : per);
}

int sym_share_splits(int nw_share, int K, int NW)
{
    // about 12288 waves (four rounds of the chip's 256 CUs x 4 SIMDs x 3 waves
    // of this kernel), every wave with the same number u of the Q sub-units
    // of its wave block (the last one of a block fewer): u = Q nw / 12288,
    // R_share = ceil(Q / u).  Fewer waves leave a longer end, more leave more
    // target-side records for the finish to read.  Pairs and finish, us, by
    // waves:         4096   6144   8192  12288  16384  32768
    //   131072, 1/8   459    420    425    412    415    432
    //   131072, 1/2  1729   1587   1545   1406   1457   1446
    //   262144, 1/8  1712   1579   1532   1393   1444   1437
    //    65536, 1/4   251    235    235    236    237    239
    const long long Q = (long long)K * (NW / 2 + 1);
    long long u = Q * nw_share / 12288;
    if (u < 1)
        u = 1;
    return (int)((Q + u - 1) / u);
}

// The target-side partials of share `share` in a buffer of Rs x n_pad
// records: the whole system's rows (compact = false: body b of row r at
// r * n_pad + b) or the share's own region (compact: Rs rows of the share's
// bodies, contiguous, at record Rs * w0 * 64K; the shares' regions tile the
// buffer).
static void share_ipart_layout(int n_pad, int K, int Rs, int w0, int w1, bool compact, size_t* base,
                               long long* istride, int* ibody0)
{
    const int B = 64 * K;
    *base = compact ? (size_t)Rs * w0 * B * 3 : 0;
    *istride = compact ? (long long)(w1 - w0) * B : n_pad;
    *ibody0 = compact ? w0 * B : 0;
}

hipError_t launch_sym_share_pairs(const Tile& t, bool newton, const float4* src, int n, int n_pad, float eps2,
                                  int shares, int share, int Rs, float* ipart, bool compact_ipart, float* jpart,
                                  bool jpart_share_rows, double* react3, bool accumulate, hipStream_t st)
{
    const int K = t.k;
    if (n_pad % (128 * K) != 0 || !ipart || !jpart)
        return hipErrorInvalidValue;
    const int NW = n_pad / (64 * K);
    int w0, w1;
    sym_share_blocks(NW, shares, share, &w0, &w1);
    const int nwaves = (w1 - w0) * Rs;
    const int jbase = jpart_share_rows ? w0 : 0;
    size_t ibase;
    long long istride;
    int ibody0;
    share_ipart_layout(n_pad, K, Rs, w0, w1, compact_ipart, &ibase, &istride, &ibody0);
    if (nwaves > 0) {
        const dim3 grid((nwaves + 3) / 4), block(256);
        const bool reg = nwaves <= kRegWaves;
#define SHARE_AS(KK, NEWTON, REG)                                                                                \
    hipLaunchKernelGGL((sym_share_kernel<KK, NEWTON, REG>), grid, block, 0, st, src, NW, Rs, w0, nwaves, eps2, \
                       ipart + ibase, jpart, jbase, istride, ibody0)
#define SHARE_LAUNCH(KK)              \
    if (newton && reg)                \
        SHARE_AS(KK, true, true);     \
    else if (newton)                  \
        SHARE_AS(KK, true, false);    \
    else if (reg)                     \
        SHARE_AS(KK, false, true);    \
    else                              \
        SHARE_AS(KK, false, false);
        if (K == 2) {
            SHARE_LAUNCH(2)
        } else if (K == 4) {
            SHARE_LAUNCH(4)
        } else if (K == 8) {
            SHARE_LAUNCH(8)
        } else {
            return hipErrorInvalidValue;
        }
#undef SHARE_AS
#undef SHARE_LAUNCH
        hipError_t e = hipGetLastError();
        if (e != hipSuccess)
            return e;
    }
    hipLaunchKernelGGL(sym_react_kernel, dim3((n + 255) / 256), dim3(256), 0, st, jpart, n, NW, K, w0, w1, jbase,
                       accumulate, react3);
    return hipGetLastError();
}

template <class Epi>
static hipError_t launch_sym_finish(const float* ipart, long long istride, int ibody0, int Rs, int start, int count,
                                    const double* react_sum3, const Epi& epi, hipStream_t st)
{
    const int T = sym_reduce_lanes(count);
    const dim3 grid((unsigned)(((long long)count * T + 255) / 256)), block(256);
#define FINISH(TT) hipLaunchKernelGGL((sym_share_finish_kernel<TT, Epi>), grid, block, 0, st, ipart, istride, ibody0, \
                                      Rs, start, count, react_sum3, epi)
    switch (T) {
    case 1: FINISH(1); break;
    case 2: FINISH(2); break;
    case 4: FINISH(4); break;
    case 8: FINISH(8); break;
    default: FINISH(16); break;
    }
#undef FINISH
    return hipGetLastError();
}

// A whole step of the symmetric tile evaluated in `chunks` chunks of wave
// blocks, one after the other: each chunk's pair work (target-side partials
// into ipart, R_share rows; its reactions into jchunk, a buffer of one chunk's
// rows) and the reactions summed per body into react3, accumulated over the
// chunks in order; then every body's target-side partials plus react3 and
// the epilogue.  The same pair work as one launch of the symmetric kernel
// with partial-sum memory for one chunk's reactions.
template <class Epi>
hipError_t launch_sym_chunked(const Tile& t, bool newton, const float4* src, int n, int n_pad, float eps2,
                              int chunks, int Rs, float* ipart, float* jchunk, double* react3, const Epi& epi,
                              hipStream_t st)
{
    for (int g = 0; g < chunks; ++g) {
        hipError_t e = launch_sym_share_pairs(t, newton, src, n, n_pad, eps2, chunks, g, Rs, ipart, false, jchunk,
                                              true, react3, g > 0, st);
        if (e != hipSuccess)
            return e;
    }
    return launch_sym_finish(ipart, n_pad, 0, Rs, 0, n, react3, epi, st);
}

template hipError_t launch_sym_chunked<EpiMixed>(const Tile&, bool, const float4*, int, int, float, int, int, float*,
                                                 float*, double*, const EpiMixed&, hipStream_t);
template hipError_t launch_sym_chunked<EpiAccel>(const Tile&, bool, const float4*, int, int, float, int, int, float*,
                                                 float*, double*, const EpiAccel&, hipStream_t);

hipError_t launch_sym_share_finish_mixed(const StepArgs& a, int shares, int share, int Rs, int start, int count,
                                         const float* ipart, const double* react_sum3, float4* snap_new,
                                         double4* pos, double4* vel, hipStream_t st)
{
    const Tile& t = tile_get(a.share_tile);
    const int NW = a.n_pad / (64 * t.k);
    int w0, w1;
    sym_share_blocks(NW, shares, share, &w0, &w1);
    size_t ibase;
    long long istride;
    int ibody0;
    share_ipart_layout(a.n_pad, t.k, Rs, w0, w1, true, &ibase, &istride, &ibody0);
    EpiMixed epi{pos, vel, snap_new, a.dt, a.damping, a.kick};
    return launch_sym_finish(ipart + ibase, istride, ibody0, Rs, start, count, react_sum3, epi, st);
}

hipError_t launch_batch_counter_reset(int* counter, hipStream_t st)
{
    hipLaunchKernelGGL(batch_counter_reset_kernel, dim3(1), dim3(64), 0, st, counter);
    return hipGetLastError();
}

hipError_t launch_batch_sym_step(const BatchSymGeom& g, int nwaves, int total, const float4* snap_old,
                                 float4* snap_new, double4* pos, double4* vel, float eps2, double dt,
                                 double damping, int kick, float* ipart, float* jpart, hipStream_t st,
                                 float4* keep)
{
    hipError_t e;
    if (g.counter && (e = launch_batch_counter_reset(g.counter, st)) != hipSuccess)
        return e;
    hipLaunchKernelGGL((batch_sym_kernel<kBatchSymK>), dim3((nwaves + 3) / 4), dim3(256), 0, st, g, nwaves,
                       snap_old, eps2, ipart, jpart);
    e = hipGetLastError();
    if (e != hipSuccess)
        return e;
    EpiMixed epi{pos, vel, snap_new, dt, damping, kick, keep};
    const int T = sym_reduce_lanes(total);
    const dim3 rgrid((unsigned)(((long long)total * T + 255) / 256));
    switch (T) {
    case 1: hipLaunchKernelGGL(batch_sym_reduce_kernel<1>, rgrid, dim3(256), 0, st, g, total, kBatchSymK, ipart, jpart, epi); break;
    case 2: hipLaunchKernelGGL(batch_sym_reduce_kernel<2>, rgrid, dim3(256), 0, st, g, total, kBatchSymK, ipart, jpart, epi); break;
    case 4: hipLaunchKernelGGL(batch_sym_reduce_kernel<4>, rgrid, dim3(256), 0, st, g, total, kBatchSymK, ipart, jpart, epi); break;
    case 8: hipLaunchKernelGGL(batch_sym_reduce_kernel<8>, rgrid, dim3(256), 0, st, g, total, kBatchSymK, ipart, jpart, epi); break;
    default: hipLaunchKernelGGL(batch_sym_reduce_kernel<16>, rgrid, dim3(256), 0, st, g, total, kBatchSymK, ipart, jpart, epi); break;
    }
    return hipGetLastError();
}

template hipError_t launch_sym<EpiFP32>(const Tile&, bool, bool, const float4*, int, int, float, float*, float*,
                                        const EpiFP32&, hipStream_t);
template hipError_t launch_sym<EpiMixed>(const Tile&, bool, bool, const float4*, int, int, float, float*, float*,
                                         const EpiMixed&, hipStream_t);
template hipError_t launch_sym<EpiAccel>(const Tile&, bool, bool, const float4*, int, int, float, float*, float*,
                                         const EpiAccel&, hipStream_t);

}  // namespace utcnb

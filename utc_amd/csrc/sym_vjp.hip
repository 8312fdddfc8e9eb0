// sym_vjp.hip -- the adjoint pair sum (VJP) evaluating every unordered pair once.
//
// With alpha the per-body kick adjoint, r = x_j - x_i, d^2 = |r|^2 + eps2,
// y = d^-1, J(r) = y^3 I - 3 y^5 r r^T and w = m_i alpha_j - m_j alpha_i, the
// pair (i, j) adds
//   xb_i += J w,            xb_j -= J w            (J is even in r, w odd in i<->j)
//   mb_i -= y^3 alpha_j.r,  mb_j += y^3 alpha_i.r
// so both bodies' terms come from one evaluation.  Written as
// J w = y^3 (w - 3 y^2 (r.w) r) with r.w = m_i (a_j.r) - m_j (a_i.r), reusing
// the two dot products the mass terms need, an unordered pair costs 36 VALU
// instructions (3 sub, 3 fma for d^2, 2 mul for y^2 and y^3, 6 for the two dot
// products, 2 for r.w, 2 mul for -3 y^2 r.w, 6 for w, 3 fma for the bracket,
// 6 fma for the two position terms, 2 fma for the two mass terms) and a root,
// against 31 per ordered pair in the one-pass VJP.  When the targets of the
// wave and the sources of a block all have one mass m, w = m (alpha_j -
// alpha_i) and r.w = m (a_j.r - a_i.r): the pair works with the differences
// alone and the block's position partials are scaled by m once (31).
//
// As in the force kernel a source block and its reaction sums rotate through
// the wave's LDS and the roots of a step's 4 pairs are taken together.  FP32
// issue bounds it: per VJP step (pair sum, reduction and the adjoint's
// per-body work), same device, N = 65536 1.59 ms (2.09 with the block carried
// round the wave in 10 DPP moves per step and one root at a time), N = 16384
// with log-uniform masses 162 us (200); 96 systems of 256 to 8192 bodies, 20
// steps forward and adjoint 16.7 ms (20.9).  Roots 2 at a time, an unroll of 4
// and 128 VGPRs (four waves per SIMD, for three) are the same within
// 1%; without unrolling it is 8% slower at N = 65536.
//
// The mapping is the symmetric force kernel's (sym.hip): wave blocks of 64*K
// bodies, unit 0 = own blocks (source block kb two-sided against target slots
// k < kb, one-sided against slot kb), unit 1 + d = the wave block d + 1 places
// round (both sides), R waves per wave block split the K (NW/2+1) (unit,
// source block) sub-units: in chunks of 4 rotation steps (SymSplit,
// sym_split.h), or whole ones in batches.
// Partials go to HBM (float4 per body: x, y, z, m) and a second kernel adds
// them per body in FP64, in a fixed order, into xbar and mbar.
#include "internal.h"
#include "rsq_group.h"
#include "sym_items.h"
#include "sym_reduce.h"
#include "vjp_pair.h"

namespace utcnb {

namespace {

__device__ __forceinline__ void kahan1(float& s, float& c, float p)
{
    const float y = p - c;
    const float t = s + y;
    c = (t - s) - y;
    s = t;
}

}  // namespace

// A wave's source block and its reaction sums in LDS (wave private), as in
// sym.hip: source s in slots s and s + 64.
struct SymVjpLds {
    float4 p[128], a[128];
    float h[4][128];
};

__device__ __forceinline__ void vjp_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// A block of 64 sources (lane l's source: position/mass sp, alpha sa; wave
// private LDS L) against target slots 0 .. N-1 of each lane: at step t in
// [t0, t0 + steps) lane l meets source (l + t) mod 64.  Slots k < N2 are two-sided; slot N2 < N is the
// block with itself (self pairs included, so w is exact: vjp_pair.h), target
// side only.  The target-side block partials are Kahan-added into (g, c); the
// reaction sums of lane l's own source come back in h (N2 > 0).
// UNI: every target mass mi[k] and source mass equals m (two-sided slots).
template <int K, int N, int N2, bool UNI>
__device__ __forceinline__ void sym_vjp_block(SymVjpLds& L, int lane, int t0, int steps, float4 sp, float4 sa, const float (&xi)[K],
                                              const float (&yi)[K], const float (&zi)[K], const float (&mi)[K],
                                              const float (&bx)[K], const float (&by)[K], const float (&bz)[K],
                                              float m, float eps2, float (&g)[K][4], float (&c)[K][4], float4& h)
{
    float p[N][4];
#pragma unroll
    for (int k = 0; k < N; ++k)
        p[k][0] = p[k][1] = p[k][2] = p[k][3] = 0.f;
    vjp_lds_fence();
    L.p[lane] = L.p[lane + 64] = sp;
    L.a[lane] = L.a[lane + 64] = sa;
    if constexpr (N2 > 0) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
            L.h[q][lane] = L.h[q][lane + 64] = 0.f;
    }
    vjp_lds_fence();
    const float4* pp = &L.p[lane];
    const float4* pa = &L.a[lane];
    float* ph = &L.h[0][lane];
    float4 cp = pp[t0], ca = pa[t0];
    // a loop with the LDS fences and a run-time trip count is not unrolled
    // otherwise; steps is even
    for (int t2 = t0; t2 < t0 + steps; t2 += 2)
#pragma unroll
    for (int t = t2; t < t2 + 2; ++t) {
        const float4 np = pp[t + 1], na = pa[t + 1];  // the next step's source: at most slot 127
        float hx = 0.f, hy = 0.f, hz = 0.f, hm = 0.f;
        if constexpr (N2 > 0) {
            hx = ph[t]; hy = ph[128 + t]; hz = ph[256 + t]; hm = ph[384 + t];
        }
        float rx[N], ry[N], rz[N], d2[N], yy[N];
#pragma unroll
        for (int k = 0; k < N; ++k) {
            rx[k] = cp.x - xi[k]; ry[k] = cp.y - yi[k]; rz[k] = cp.z - zi[k];
            d2[k] = __builtin_fmaf(rx[k], rx[k], __builtin_fmaf(ry[k], ry[k], __builtin_fmaf(rz[k], rz[k], eps2)));
        }
        rsq_group<N>(d2, yy);
#pragma unroll
        for (int k = 0; k < N; ++k) {
            const float y = yy[k], y2 = y * y, y3 = y2 * y;
            const float arj = __builtin_fmaf(ca.x, rx[k], __builtin_fmaf(ca.y, ry[k], ca.z * rz[k]));
            if (k < N2) {
                // J w = y^3 (w - 3 y^2 (r.w) r), r.w = m_i (a_j.r) - m_j (a_i.r)
                const float ari = __builtin_fmaf(bx[k], rx[k], __builtin_fmaf(by[k], ry[k], bz[k] * rz[k]));
                float s3, wx, wy, wz;
                if constexpr (UNI) {  // w / m and r.w / m
                    s3 = (-3.f * y2) * (arj - ari);
                    wx = ca.x - bx[k]; wy = ca.y - by[k]; wz = ca.z - bz[k];
                } else {
                    s3 = (-3.f * y2) * __builtin_fmaf(mi[k], arj, -(cp.w * ari));
                    wx = w_fast(mi[k], ca.x, cp.w, bx[k]);
                    wy = w_fast(mi[k], ca.y, cp.w, by[k]);
                    wz = w_fast(mi[k], ca.z, cp.w, bz[k]);
                }
                const float tx = __builtin_fmaf(s3, rx[k], wx);
                const float ty = __builtin_fmaf(s3, ry[k], wy);
                const float tz = __builtin_fmaf(s3, rz[k], wz);
                p[k][0] = __builtin_fmaf(y3, tx, p[k][0]);
                p[k][1] = __builtin_fmaf(y3, ty, p[k][1]);
                p[k][2] = __builtin_fmaf(y3, tz, p[k][2]);
                hx = __builtin_fmaf(-y3, tx, hx);
                hy = __builtin_fmaf(-y3, ty, hy);
                hz = __builtin_fmaf(-y3, tz, hz);
                hm = __builtin_fmaf(y3, ari, hm);
            } else {
                const float y5m3 = (-3.f * y2) * y3;
                const float wx = w_exact(mi[k], ca.x, cp.w, bx[k]);
                const float wy = w_exact(mi[k], ca.y, cp.w, by[k]);
                const float wz = w_exact(mi[k], ca.z, cp.w, bz[k]);
                const float e = y5m3 * __builtin_fmaf(rx[k], wx, __builtin_fmaf(ry[k], wy, rz[k] * wz));
                p[k][0] = __builtin_fmaf(e, rx[k], __builtin_fmaf(y3, wx, p[k][0]));
                p[k][1] = __builtin_fmaf(e, ry[k], __builtin_fmaf(y3, wy, p[k][1]));
                p[k][2] = __builtin_fmaf(e, rz[k], __builtin_fmaf(y3, wz, p[k][2]));
            }
            p[k][3] = __builtin_fmaf(-y3, arj, p[k][3]);
        }
        if constexpr (N2 > 0) {
            ph[t] = hx; ph[128 + t] = hy; ph[256 + t] = hz; ph[384 + t] = hm;
        }
        vjp_lds_fence();
        cp = np;
        ca = na;
    }
#pragma unroll
    for (int k = 0; k < N; ++k) {
        if constexpr (UNI) {
            if (k < N2) {
                p[k][0] *= m; p[k][1] *= m; p[k][2] *= m;
            }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
            kahan1(g[k][q], c[k][q], p[k][q]);
    }
    if constexpr (N2 > 0) {
        h = make_float4(L.h[0][lane] + L.h[0][lane + 64], L.h[1][lane] + L.h[1][lane + 64],
                        L.h[2][lane] + L.h[2][lane + 64], L.h[3][lane] + L.h[3][lane + 64]);
        if constexpr (UNI) {
            h.x *= m; h.y *= m; h.z *= m;
        }
    }
}

// Own source block KB of the wave's block, for the wave-uniform kb: target
// slots k < KB meet it two-sided, slot KB one-sided (the block with itself);
// slots k > KB take these sources when their own block is the source.  The
// reaction sums belong to slot KB.
template <int K, int KB = 0>
__device__ __forceinline__ void sym_vjp_own_at(int kb, bool uni, SymVjpLds& L, int lane, int t0, int steps, float4 sp, float4 sa,
                                               const float (&xi)[K], const float (&yi)[K], const float (&zi)[K],
                                               const float (&mi)[K], const float (&bx)[K], const float (&by)[K],
                                               const float (&bz)[K], float m, float eps2, float (&g)[K][4],
                                               float (&c)[K][4])
{
    if (kb == KB) {
        float4 h;
        if (uni)
            sym_vjp_block<K, KB + 1, KB, true>(L, lane, t0, steps, sp, sa, xi, yi, zi, mi, bx, by, bz, m, eps2, g, c, h);
        else
            sym_vjp_block<K, KB + 1, KB, false>(L, lane, t0, steps, sp, sa, xi, yi, zi, mi, bx, by, bz, m, eps2, g, c, h);
        if constexpr (KB > 0) {
            kahan1(g[KB][0], c[KB][0], h.x);
            kahan1(g[KB][1], c[KB][1], h.y);
            kahan1(g[KB][2], c[KB][2], h.z);
            kahan1(g[KB][3], c[KB][3], h.w);
        }
        // keeps the compiler from merging the K branches' adds into one
        // through a pointer to slot KB, which would put the sums in memory
        asm volatile("; own block %0" : : "n"(KB));
    } else if constexpr (KB + 1 < K) {
        sym_vjp_own_at<K, KB + 1>(kb, uni, L, lane, t0, steps, sp, sa, xi, yi, zi, mi, bx, by, bz, m, eps2, g, c);
    }
}

// The work of wave r of wave block w of one system.  jrec: two float4 per
// body {x,y,z,m} {ax,ay,az,0}, n_pad = NW*64*K bodies; nr: it does that of
// waves r .. r + nr - 1 in turn (not SPLIT); ipart: [R][n_pad]
// float4; jpart: [NW][NW/2][64K] float4, SPLIT: [NW][R][J][64] (SymSplit).
template <int K, bool SPLIT>
__device__ __forceinline__ void sym_vjp_wave(const float4* __restrict__ jrec, int NW, int R, int w, int r,
                                             float eps2, float4* __restrict__ ipart,
                                             float4* __restrict__ jpart, SymVjpLds& L, int lane, int rs = 1,
                                             int nr = 1)
{
    const int half = NW / 2;
    const int n_pad = NW * 64 * K;
    float xi[K], yi[K], zi[K], mi[K], bx[K], by[K], bz[K];
    float g[K][4], c[K][4];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int b = w * 64 * K + k * 64 + lane;
        const float4 p = jrec[2 * b], a = jrec[2 * b + 1];
        xi[k] = p.x; yi[k] = p.y; zi[k] = p.z; mi[k] = p.w;
        bx[k] = a.x; by[k] = a.y; bz[k] = a.z;
    }
    // one mass m0 for every target of the wave?
    const float m0 = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(mi[0])));
    bool tuni = true;
#pragma unroll
    for (int k = 0; k < K; ++k)
        tuni = tuni && mi[k] == m0;
    for (const int r1 = r + nr; r < r1; ++r) {
#pragma unroll
        for (int k = 0; k < K; ++k)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                g[k][q] = c[k][q] = 0.f;
        // sub-unit su = (unit u, source block kb): u = 0 is the wave block's own
        // sources, u = 1 + d the wave block d + 1 places round
        int qf, ql, c0 = 0, c1 = 0, J = 0;
        if constexpr (SPLIT) {
            const SymSplit split(NW, w, K, R, rs);
            c0 = split.first(r);
            c1 = split.first(r + 1);
            qf = c0 / rs;
            ql = (c1 + rs - 1) / rs;
            J = SymSplit::records(NW, K, R, rs);
        } else {
            const int Q = (half + 1) * K;
            qf = (int)((long long)Q * r / R);
            ql = (int)((long long)Q * (r + 1) / R);
        }
        for (int su = qf; su < ql; ++su) {
            // rotation steps [t0, t0 + steps): all but for the first and last sub-unit
            int t0 = 0, steps = 64;
            if constexpr (SPLIT) {
                const int a = su == qf ? c0 - su * rs : 0, e = su + 1 == ql ? c1 - su * rs : rs;
                t0 = a * (64 / rs);
                steps = (e - a) * (64 / rs);
            }
            const int u = su / K, kb = su - u * K;
            if (u == 0) {
                // own block kb: two-sided against the lower target slots
                const int b = w * 64 * K + kb * 64 + lane;
                const float4 sp = jrec[2 * b], sa = jrec[2 * b + 1];
                const bool uni = __ballot(tuni && sp.w == m0) == ~0ull;
                sym_vjp_own_at<K>(kb, uni, L, lane, t0, steps, sp, sa, xi, yi, zi, mi, bx, by, bz, m0, eps2, g, c);
                continue;
            }
            const int d = u - 1;
            if (2 * (d + 1) == NW && w >= half)
                continue;  // the block half way round: taken by the lower half
            int v = w + 1 + d;
            if (v >= NW)
                v -= NW;
            const int b = v * 64 * K + kb * 64 + lane;
            const float4 sp = jrec[2 * b], sa = jrec[2 * b + 1];
            float4 h;
            if (__ballot(tuni && sp.w == m0) == ~0ull)
                sym_vjp_block<K, K, K, true>(L, lane, t0, steps, sp, sa, xi, yi, zi, mi, bx, by, bz, m0, eps2, g, c, h);
            else
                sym_vjp_block<K, K, K, false>(L, lane, t0, steps, sp, sa, xi, yi, zi, mi, bx, by, bz, m0, eps2, g, c, h);
            jpart[SPLIT ? (((size_t)w * R + r) * J + (su - qf)) * 64 + lane
                        : ((size_t)w * half + d) * (64 * K) + kb * 64 + lane] = h;
        }
#pragma unroll
        for (int k = 0; k < K; ++k)
            ipart[(size_t)r * n_pad + w * 64 * K + k * 64 + lane] =
                make_float4(g[k][0] - c[k][0], g[k][1] - c[k][1], g[k][2] - c[k][2], g[k][3] - c[k][3]);
    }
}

// One system: wave gw = w * R + r.
template <int K>
__global__ __launch_bounds__(256, 2) void sym_vjp_kernel(const float4* __restrict__ jrec, int NW, int R,
                                                      float eps2, float4* __restrict__ ipart,
                                                      float4* __restrict__ jpart, int rs)
{
    __shared__ SymVjpLds lds[4];
    const int gw = __builtin_amdgcn_readfirstlane((int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6));
    if (gw >= NW * R)
        return;  // whole waves only
    sym_vjp_wave<K, true>(jrec, NW, R, gw / R, gw % R, eps2, ipart, jpart, lds[threadIdx.x >> 6], threadIdx.x & 63,
                          rs);
}

// Batched systems: each wave runs items in the schedule of batch_next_item
// (sym_items.h).
template <int K>
__global__ __launch_bounds__(256, 2) void batch_sym_vjp_kernel(BatchSymGeom g, int nwaves,
                                                            const float4* __restrict__ jrec, float eps2,
                                                            float4* __restrict__ ipart,
                                                            float4* __restrict__ jpart)
{
    __shared__ SymVjpLds lds[4];
    const int gw = __builtin_amdgcn_readfirstlane((int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6));
    if (gw >= nwaves)
        return;  // whole waves only
    const int lane = threadIdx.x & 63;
    int pos = 0;
    for (int it = batch_next_item(g, gw, pos, lane); it >= 0; it = batch_next_item(g, gw, pos, lane)) {
        const int4 item = g.items[it];  // (system, wave block, splits)
        const int s = item.x;
        sym_vjp_wave<K, false>(jrec + 2 * (size_t)g.off[s], g.nw[s], item.w, item.y, item.z & 0xffff, eps2,
                               ipart + g.vipo[s], jpart + g.vjpo[s], lds[threadIdx.x >> 6], lane, 1, item.z >> 16);
    }
}

// Body b's position adjoint after the VJP, and the record of the step before:
// the work of adjoint_pre_kernel (adjoint.hip), the same operations, on values
// still in registers.  Adjoint of 20 steps, ms: N = 1000 0.51 (0.55 with a
// launch of its own), 4096 0.70 (0.73), 16384 3.62 (3.71).
__device__ __forceinline__ void adjoint_next(const AdjointNext& next, size_t b, const double (&s)[4],
                                             double* __restrict__ xbar3, double* __restrict__ mbar)
{
    double x[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        x[k] = xbar3[3 * b + k] + s[k];
        xbar3[3 * b + k] = x[k];
    }
    mbar[b] += s[3];
    if (!next.pos)
        return;
    double al[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const double ub = next.vbar3[3 * b + k] + x[k] * next.dt;
        next.vbar3[3 * b + k] = next.damping * ub;
        al[k] = next.damping * next.dt * ub;
    }
    next.jrec[2 * b] = next.pos[b];
    next.jrec[2 * b + 1] = make_float4((float)al[0], (float)al[1], (float)al[2], 0.f);
}

// xbar_b += the sum of body b's partials, mbar_b likewise (T lanes per body,
// sym_reduce.h), then adjoint_next.
template <int T>
__global__ __launch_bounds__(256) void sym_vjp_reduce_kernel(const float4* __restrict__ ipart,
                                                             const float4* __restrict__ jpart, int n,
                                                             int NW, int R, int K, int rs,
                                                             double* __restrict__ xbar3,
                                                             double* __restrict__ mbar, AdjointNext next)
{
    int b, t;
    sym_reduce_lane<T>(b, t);
    double s[4];
    sym_split_sum<T, true>(ipart, jpart, b < n ? b : n - 1, NW, R, K, t, s, rs);
    if (b < n && t == 0)
        adjoint_next(next, b, s, xbar3, mbar);
}

// Batched systems: body b of the concatenated padded layout.
template <int T>
__global__ __launch_bounds__(256) void batch_sym_vjp_reduce_kernel(BatchSymGeom g, int total, int K,
                                                                   const float4* __restrict__ ipart,
                                                                   const float4* __restrict__ jpart,
                                                                   double* __restrict__ xbar3,
                                                                   double* __restrict__ mbar, AdjointNext next)
{
    int j, t;
    sym_reduce_lane<T>(j, t);
    const int b = g.body0 + j, bb = g.body0 + (j < total ? j : total - 1);
    const int s = g.sys_of_block[bb / kBatchSymAlign];
    const int loc = bb - g.off[s];
    double sum[4];
    sym_batch_sum<T>(ipart + g.vipo[s], jpart + g.vjpo[s], loc, g.nw[s], g.rs[s], K, t, sum);
    if (j < total && loc < g.n[s] && t == 0)
        adjoint_next(next, b, sum, xbar3, mbar);
}

constexpr int kSymVjpK = 4;
constexpr int kSymVjpRs = 16;  // rotation chunks per sub-unit, single systems

int sym_vjp_splits(int n_pad, int cu_count)
{
    // Two waves for every SIMD, that start together and end together but for a
    // chunk of 4 steps (a third wave on a SIMD runs unpaired); at most
    // 128, whose target-side records the reduction reads for each body, and at
    // least 3 chunks each.  From 40960 bodies 32: there the waves drift apart
    // over the chip and shorter ones, several in turn, fill its end.  Adjoint
    // of 20 steps, ms, against 32 waves of whole sub-units: N = 4096 0.79
    // (1.22), 8192 1.40 (1.93), 16384 3.48 (3.85), 32768 11.55 (12.37); 10
    // steps at 65536 21.75 (21.85; with R = 16 22.4).  Chunks of 8 steps are
    // the same within 2%, 4096 and 6144 waves up to 10% slower at 8192.
    const int NW = n_pad / (64 * kSymVjpK);
    int R = (cu_count > 0 ? cu_count : 256) * 8 / NW;
    if (R < 16)
        R = 32;
    const int most = SymSplit(NW, 0, kSymVjpK, 1, kSymVjpRs).chunks / 3;
    return R < most ? (R < 128 ? R : 128) : (most < 128 ? most : 128);
}

size_t sym_vjp_ipart_float4s(int n_pad, int R) { return (size_t)R * n_pad; }
size_t sym_vjp_jpart_float4s(int n_pad, int R)
{
    const int NW = n_pad / (64 * kSymVjpK);
    return (size_t)NW * R * SymSplit::records(NW, kSymVjpK, R, kSymVjpRs) * 64;
}
bool sym_vjp_applies(int n_pad) { return n_pad % (128 * kSymVjpK) == 0; }

hipError_t launch_sym_vjp(const float4* jrec, int n, int n_pad, float eps2, int R, float4* ipart,
                          float4* jpart, double* xbar3, double* mbar, const AdjointNext& next, hipStream_t st)
{
    if (!sym_vjp_applies(n_pad) || R < 1 || !ipart || !jpart)
        return hipErrorInvalidValue;
    const int NW = n_pad / (64 * kSymVjpK);
    const int waves = NW * R;
    hipLaunchKernelGGL((sym_vjp_kernel<kSymVjpK>), dim3((waves + 3) / 4), dim3(256), 0, st, jrec, NW, R,
                       eps2, ipart, jpart, kSymVjpRs);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess)
        return e;
    const int T = sym_reduce_lanes(n);
    const dim3 rgrid((unsigned)(((long long)n * T + 255) / 256));
    switch (T) {
    case 1: hipLaunchKernelGGL(sym_vjp_reduce_kernel<1>, rgrid, dim3(256), 0, st, ipart, jpart, n, NW, R, kSymVjpK, kSymVjpRs, xbar3, mbar, next); break;
    case 2: hipLaunchKernelGGL(sym_vjp_reduce_kernel<2>, rgrid, dim3(256), 0, st, ipart, jpart, n, NW, R, kSymVjpK, kSymVjpRs, xbar3, mbar, next); break;
    case 4: hipLaunchKernelGGL(sym_vjp_reduce_kernel<4>, rgrid, dim3(256), 0, st, ipart, jpart, n, NW, R, kSymVjpK, kSymVjpRs, xbar3, mbar, next); break;
    case 8: hipLaunchKernelGGL(sym_vjp_reduce_kernel<8>, rgrid, dim3(256), 0, st, ipart, jpart, n, NW, R, kSymVjpK, kSymVjpRs, xbar3, mbar, next); break;
    default: hipLaunchKernelGGL(sym_vjp_reduce_kernel<16>, rgrid, dim3(256), 0, st, ipart, jpart, n, NW, R, kSymVjpK, kSymVjpRs, xbar3, mbar, next); break;
    }
    return hipGetLastError();
}

hipError_t launch_batch_sym_vjp(const BatchSymGeom& g, int nwaves, int total, const float4* jrec,
                                float eps2, float4* ipart, float4* jpart, double* xbar3, double* mbar,
                                const AdjointNext& next, hipStream_t st)
{
    static_assert(kBatchSymK == kSymVjpK, "batched and single-system symmetric VJP share K");
    hipError_t e;
    if (g.counter && (e = launch_batch_counter_reset(g.counter, st)) != hipSuccess)
        return e;
    hipLaunchKernelGGL((batch_sym_vjp_kernel<kBatchSymK>), dim3((nwaves + 3) / 4), dim3(256), 0, st, g,
                       nwaves, jrec, eps2, ipart, jpart);
    e = hipGetLastError();
    if (e != hipSuccess)
        return e;
    const int T = sym_reduce_lanes(total);
    const dim3 rgrid((unsigned)(((long long)total * T + 255) / 256));
    switch (T) {
    case 1: hipLaunchKernelGGL(batch_sym_vjp_reduce_kernel<1>, rgrid, dim3(256), 0, st, g, total, kBatchSymK, ipart, jpart, xbar3, mbar, next); break;
    case 2: hipLaunchKernelGGL(batch_sym_vjp_reduce_kernel<2>, rgrid, dim3(256), 0, st, g, total, kBatchSymK, ipart, jpart, xbar3, mbar, next); break;
    case 4: hipLaunchKernelGGL(batch_sym_vjp_reduce_kernel<4>, rgrid, dim3(256), 0, st, g, total, kBatchSymK, ipart, jpart, xbar3, mbar, next); break;
    case 8: hipLaunchKernelGGL(batch_sym_vjp_reduce_kernel<8>, rgrid, dim3(256), 0, st, g, total, kBatchSymK, ipart, jpart, xbar3, mbar, next); break;
    default: hipLaunchKernelGGL(batch_sym_vjp_reduce_kernel<16>, rgrid, dim3(256), 0, st, g, total, kBatchSymK, ipart, jpart, xbar3, mbar, next); break;
    }
    return hipGetLastError();
}

}  // namespace utcnb

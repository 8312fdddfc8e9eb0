// ref.hip -- the reference's own arithmetic on gfx950, bit for bit.
//
// One thread per body sums every source in index order 0..n-1 with exactly
// the operations of benchapps/nbody/seq/bodysystem.h:70-96 (sqrt_T, then a
// DOUBLE division 1.0/sqrt even for T=float, then inv*inv*inv), and then
// applies the damped kick-drift of benchapps/nbody/seq/bodysystem.cc:135-181.
// This file is compiled with -ffp-contract=off so that no multiply-add is
// fused; sqrtf and the FP64 division are IEEE correctly rounded on this
// target, so every rounding matches the reference's CPU path.
//
// Source bodies are uniform across the wave and arrive through scalar loads.
// For eps2 >= 2^-96 the FP32 kernels take ref_inv_dist and ref_inv_dist_group
// (ref_inv.h): the same correctly rounded sqrtf and division, without the
// generic rescaling; for
// eps2 >= 2^-600 the FP64 kernels take ref_inv_dist64 on every group of four
// sources whose d2 stay below 2^600 (the same operations as the generic FP64
// sqrt and division there).
#include "internal.h"
#include "ref_inv.h"

namespace utcnb {

#pragma clang fp contract(off)

template <typename T, bool FAST>
__device__ __forceinline__ T inv_dist(T d2);

template <>
__device__ __forceinline__ float inv_dist<float, false>(float d2)
{
    // (float)(1.0 / (double)sqrtf(d2)) -- the literal 1.0 makes the division FP64.
    return (float)(1.0 / (double)sqrtf(d2));
}

template <>
__device__ __forceinline__ float inv_dist<float, true>(float d2)
{
    return ref_inv_dist(d2);  // d2 >= eps2 >= kRefInvMin
}

template <>
__device__ __forceinline__ double inv_dist<double, false>(double d2)
{
    return 1.0 / sqrt(d2);
}

template <>
__device__ __forceinline__ double inv_dist<double, true>(double d2)
{
    // d2 >= eps2 >= kRefInv64Min; beyond kRefInv64Max (or NaN) the generic path
    if (d2 <= kRefInv64Max)
        return ref_inv_dist64(d2);
    return 1.0 / sqrt(d2);
}

// One source j in the reference's order of operations: the geometry (r and
// d2 = ((rx rx + ry ry) + rz rz) + eps2), then the sums with inv = 1/sqrt(d2).
template <typename T, typename T4>
__device__ __forceinline__ T ref_geom(const T4& pj, const T4& pi, T eps2, T& r0, T& r1, T& r2)
{
    r0 = pj.x - pi.x;
    r1 = pj.y - pi.y;
    r2 = pj.z - pi.z;
    T d2 = r0 * r0 + r1 * r1 + r2 * r2;
    d2 += eps2;
    return d2;
}

template <typename T>
__device__ __forceinline__ void ref_accum(T mj, T inv, T r0, T r1, T r2, T& a0, T& a1, T& a2)
{
    T inv3 = inv * inv * inv;
    T s = mj * inv3;
    a0 += r0 * s;
    a1 += r1 * s;
    a2 += r2 * s;
}

template <typename T, typename T4, bool FAST>
__device__ __forceinline__ void ref_pair(const T4& pj, const T4& pi, T eps2, T& a0, T& a1, T& a2)
{
    T r0, r1, r2;
    const T d2 = ref_geom(pj, pi, eps2, r0, r1, r2);
    ref_accum(pj.w, inv_dist<T, FAST>(d2), r0, r1, r2, a0, a1, a2);
}

// G FP64 sources with one wave-uniform choice: ref_inv_dist64 when every
// lane's G d2 lie within its range (always, short of coordinates 1e90
// apart), else the generic sqrt and division.  Sums in j order as ref_pair.
template <int G>
__device__ __forceinline__ void ref_group64(const double4 (&q)[G], const double4& pi, double eps2,
                                            double& a0, double& a1, double& a2)
{
    double r[G][3], d2[G], inv[G];
    bool ok = true;
#pragma unroll
    for (int k = 0; k < G; ++k) {
        d2[k] = ref_geom(q[k], pi, eps2, r[k][0], r[k][1], r[k][2]);
        ok = ok && d2[k] <= kRefInv64Max;
    }
    if (__ballot(!ok) == 0) {
#pragma unroll
        for (int k = 0; k < G; ++k)
            inv[k] = ref_inv_dist64(d2[k]);
    } else {
#pragma unroll
        for (int k = 0; k < G; ++k)
            inv[k] = 1.0 / sqrt(d2[k]);
    }
#pragma unroll
    for (int k = 0; k < G; ++k)
        ref_accum(q[k].w, inv[k], r[k][0], r[k][1], r[k][2], a0, a1, a2);
}

// Sources in index order, eight per trip: their loads (one s_load_dwordx16 per
// four FP32 or two FP64 bodies) and inverse distances are independent, so they
// overlap, while the sums still take j = 0, 1, 2, ... in turn (no
// reassociation in this file).  FP32 takes the eight inverse distances from
// one group of v_rsq_f32 (ref_inv_dist_group): n = 262144 35.0 ms, 131072 11.4
// (47.8 and 13.5 with a square root and a reciprocal per pair, sixteen per
// trip).  Eight FP64 sources ran 5% faster than four at 262144 and 20% at
// 16384..65536 (two VGPRs spill to scratch; sixteen spill SGPRs and ran
// slower).
template <typename T, typename T4, bool FAST>
__device__ __forceinline__ void ref_field(const T4* __restrict__ pos, int n, T eps2, const T4& pi,
                                          T& a0, T& a1, T& a2)
{
    a0 = 0; a1 = 0; a2 = 0;
    int j = 0;
    if constexpr (sizeof(T) == 4 && FAST) {
        for (; j + 8 <= n; j += 8) {
            T4 q[8];
#pragma unroll
            for (int k = 0; k < 8; ++k)
                q[k] = pos[j + k];
            T r[8][3], d2[8], inv[8];
#pragma unroll
            for (int k = 0; k < 8; ++k)
                d2[k] = ref_geom(q[k], pi, eps2, r[k][0], r[k][1], r[k][2]);
            ref_inv_dist_group<8>(d2, inv);
#pragma unroll
            for (int k = 0; k < 8; ++k)
                ref_accum(q[k].w, inv[k], r[k][0], r[k][1], r[k][2], a0, a1, a2);
        }
    } else if constexpr (FAST) {
        for (; j + 8 <= n; j += 8) {
            T4 q[8];
#pragma unroll
            for (int k = 0; k < 8; ++k)
                q[k] = pos[j + k];
            ref_group64<8>(q, pi, eps2, a0, a1, a2);
        }
    }
    for (; j + 4 <= n; j += 4) {
        const T4 q0 = pos[j], q1 = pos[j + 1], q2 = pos[j + 2], q3 = pos[j + 3];
        if constexpr (FAST && sizeof(T) == 8) {
            const T4 q[4] = {q0, q1, q2, q3};
            ref_group64<4>(q, pi, eps2, a0, a1, a2);
        } else {
            ref_pair<T, T4, FAST>(q0, pi, eps2, a0, a1, a2);
            ref_pair<T, T4, FAST>(q1, pi, eps2, a0, a1, a2);
            ref_pair<T, T4, FAST>(q2, pi, eps2, a0, a1, a2);
            ref_pair<T, T4, FAST>(q3, pi, eps2, a0, a1, a2);
        }
    }
    for (; j < n; ++j)
        ref_pair<T, T4, FAST>(pos[j], pi, eps2, a0, a1, a2);
}

// The damped kick-drift of a body p with field a (pos_new: the result; v: in place).
template <typename T, typename T4>
__device__ __forceinline__ void ref_update(T4 p, T a0, T a1, T a2, T dt, T damping, T4& pos_new, T4& vel)
{
    T w = p.w;  // the reference's "invMass" (holds m_i), seq/bodysystem.cc:149
    T4 v = vel;
    v.x += (a0 * w) * dt;
    v.y += (a1 * w) * dt;
    v.z += (a2 * w) * dt;
    v.x *= damping;
    v.y *= damping;
    v.z *= damping;
    p.x += v.x * dt;
    p.y += v.y * dt;
    p.z += v.z * dt;
    pos_new = p;
    vel = v;
}

// Fused force + integrate; the twin of the reference's
// _integrateNBodySystem_kernel<T> (benchapps/nbody/cuda/bodysystem_kernel.cu:87-138)
// and of its multi-GPU form that takes a slice of targets
// (benchapps/nbody/utc-snode-mgpu/mgpu/bodysystem_kernel.cu:88-140): targets
// i0 + t for t < cnt against all n sources of pos_old; the new position and
// velocity of target i0 + t are pos_new[t] and vel[t] (the caller offsets
// full-size arrays by i0).
template <typename T, typename T4, bool FAST>
__global__ void ref_step_kernel(const T4* __restrict__ pos_old, T4* __restrict__ pos_new,
                                T4* __restrict__ vel, int n, int i0, int cnt, T dt, T eps2, T damping)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= cnt)
        return;
    T4 p = pos_old[i0 + t];
    T a0, a1, a2;
    ref_field<T, T4, FAST>(pos_old, n, eps2, p, a0, a1, a2);
    ref_update(p, a0, a1, a2, dt, damping, pos_new[t], vel[t]);
}

// Field of targets i0 + t, t < cnt, into acc3[3t .. 3t+2].
template <typename T, typename T4, bool FAST>
__global__ void ref_accel_kernel(const T4* __restrict__ pos, int n, int i0, int cnt, T eps2,
                                 double* __restrict__ acc3)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= cnt)
        return;
    T a0, a1, a2;
    ref_field<T, T4, FAST>(pos, n, eps2, pos[i0 + t], a0, a1, a2);
    acc3[3 * (size_t)t + 0] = (double)a0;
    acc3[3 * (size_t)t + 1] = (double)a1;
    acc3[3 * (size_t)t + 2] = (double)a2;
}

// ---- few targets: terms by many waves, sums by one ------------------------------
//
// With one thread per body the order of the sums leaves n / 64 waves: 256 of
// them at n = 16384, each waiting on its own pairs.  But only the additions
// are bound to the order; the terms r s of different sources are independent.
// Here a workgroup owns 16 A targets: W waves compute the terms (lane t + 16 g
// of wave w: targets t, t + 16, ..., the four sources of quad 4 w + g of each
// batch of 16 W sources) and leave them in LDS, and A further waves (lane
// 16 c + t: component c of target t), at raised priority, add them to the sums
// in source order, one batch behind: two batches of LDS, one barrier per
// batch.  Sources past the end leave terms of +0, which change no sum (a sum
// that starts at +0 is never -0).  The chain of dependent additions, 9 clocks
// per source, bounds small n; the terms (about 34 VALU instructions and a root
// per pair, twice the issue time that leaves) and the waits at the barrier
// bound larger n, and from n = 131072 one thread per body, without the LDS
// traffic, is faster.  Per step on MI355X, FP32 / FP64 state, one thread per
// body before: n = 1024 11.6 / 19.3 us (87 / 120), 4096 29.6 / 57 (336 / 474),
// 16384 250 / 602 (1325 / 1882), 32768 0.87 / 2.05 ms (2.65 / 3.73), 65536
// 3.2 / - (5.3 / 8.0); 131072: 12.2 for 11.4 with one thread.
template <typename T>
struct RefQuad;
template <>
struct RefQuad<float> {
    using type = float4;
};
template <>
struct RefQuad<double> {
    using type = double4;
};

// The inverse distances of G pairs.
template <typename T, bool FAST, int G>
__device__ __forceinline__ void ref_inv_group(const T (&d2)[G], T (&inv)[G])
{
    if constexpr (FAST && sizeof(T) == 8) {
        bool ok = true;
#pragma unroll
        for (int k = 0; k < G; ++k)
            ok = ok && d2[k] <= kRefInv64Max;
        if (__ballot(!ok) == 0) {
#pragma unroll
            for (int k = 0; k < G; ++k)
                inv[k] = ref_inv_dist64(d2[k]);
        } else {
#pragma unroll
            for (int k = 0; k < G; ++k)
                inv[k] = 1.0 / sqrt(d2[k]);
        }
    } else if constexpr (FAST) {
        ref_inv_dist_group<G>(d2, inv);
    } else {
#pragma unroll
        for (int k = 0; k < G; ++k)
            inv[k] = inv_dist<T, false>(d2[k]);
    }
}

// STEP: the fused step as ref_step_kernel; else the field as ref_accel_kernel.
template <typename T, typename T4, bool FAST, int A, int W, bool STEP>
__global__ __launch_bounds__(64 * (W + A)) void ref_split_kernel(const T4* __restrict__ pos_old,
                                                                 T4* __restrict__ pos_new, T4* __restrict__ vel,
                                                                 int n, int i0, int cnt, T dt, T eps2, T damping,
                                                                 double* __restrict__ acc3)
{
    constexpr int Q = 4 * W;  // quads of sources per batch
    using V = typename RefQuad<T>::type;
    __shared__ V term[2][Q][A][48];  // [batch parity][quad][target group][16 c + t]: 4 sources
    // the wave index as a scalar: the two roles are a uniform branch, each with
    // one barrier per batch
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int t = lane & 15;
    const int tile0 = blockIdx.x * 16 * A;
    const int batches = (n + 4 * Q - 1) / (4 * Q);
    if (wave < W) {
        const int quad = 4 * wave + (lane >> 4);
        T4 p[A];
#pragma unroll
        for (int a = 0; a < A; ++a) {
            const int tt = tile0 + 16 * a + t;
            p[a] = pos_old[i0 + (tt < cnt ? tt : cnt - 1)];  // clamped targets are summed but not stored
        }
        T4 q[4], nx[4];
        // the four sources of this lane's quad in batch b (past the end: the last)
        const auto fetch = [&](int b) {
            if ((b + 1) * (4 * Q) <= n) {
                const T4* src = pos_old + b * (4 * Q);
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    nx[k] = src[(unsigned)(4 * quad + k)];
            } else {
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const int j = (b * Q + quad) * 4 + k;
                    nx[k] = pos_old[j < n ? j : n - 1];
                }
            }
        };
        fetch(0);
        for (int b = 0; b < batches; ++b) {
#pragma unroll
            for (int k = 0; k < 4; ++k)
                q[k] = nx[k];
            if (b + 1 < batches)
                fetch(b + 1);  // while this batch's terms are computed
            T r[4 * A][3], d2[4 * A], inv[4 * A];
#pragma unroll
            for (int a = 0; a < A; ++a)
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    d2[4 * a + k] = ref_geom(q[k], p[a], eps2, r[4 * a + k][0], r[4 * a + k][1], r[4 * a + k][2]);
            ref_inv_group<T, FAST, 4 * A>(d2, inv);
#pragma unroll
            for (int a = 0; a < A; ++a) {
                T o[3][4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const T inv3 = inv[4 * a + k] * inv[4 * a + k] * inv[4 * a + k];
                    const T s = q[k].w * inv3;
#pragma unroll
                    for (int c = 0; c < 3; ++c)
                        o[c][k] = r[4 * a + k][c] * s;
                }
                if (b + 1 == batches) {
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        if ((b * Q + quad) * 4 + k >= n)
                            o[0][k] = o[1][k] = o[2][k] = T(0);
                }
#pragma unroll
                for (int c = 0; c < 3; ++c)
                    term[b & 1][quad][a][16 * c + t] = V{o[c][0], o[c][1], o[c][2], o[c][3]};
            }
            __syncthreads();
        }
        return;
    }
    __builtin_amdgcn_s_setprio(3);
    const int a = wave - W;
    const int slot = lane < 48 ? lane : 47;  // lanes 48..63 repeat lane 47 and store nothing
    T s = 0;
    for (int b = 0; b < batches; ++b) {
        __syncthreads();
#pragma unroll 8
        for (int k = 0; k < Q; ++k) {
            const V v = term[b & 1][k][a][slot];
            s += v.x;
            s += v.y;
            s += v.z;
            s += v.w;
        }
    }
    const T a0 = s, a1 = __shfl(s, 16 + t, 64), a2 = __shfl(s, 32 + t, 64);
    const int tt = tile0 + 16 * a + t;
    if (lane >= 16 || tt >= cnt)
        return;
    if constexpr (STEP) {
        ref_update(pos_old[i0 + tt], a0, a1, a2, dt, damping, pos_new[tt], vel[tt]);
    } else {
        acc3[3 * (size_t)tt + 0] = (double)a0;
        acc3[3 * (size_t)tt + 1] = (double)a1;
        acc3[3 * (size_t)tt + 2] = (double)a2;
    }
}

template <typename T, typename T4, bool FAST, int A, int W, bool STEP>
static void launch_ref_split(const T4* pos_old, T4* pos_new, T4* vel, int n, int i0, int cnt, T dt, T eps2, T damping,
                             double* acc3, hipStream_t st)
{
    hipLaunchKernelGGL((ref_split_kernel<T, T4, FAST, A, W, STEP>), dim3((cnt + 16 * A - 1) / (16 * A)),
                       dim3(64 * (W + A)), 0, st, pos_old, pos_new, vel, n, i0, cnt, dt, eps2, damping, acc3);
}

// The kernel by the number of targets (the figures: per step at n = cnt,
// MI355X).  FP32: up to 4096 targets the 16-target workgroups fill the CUs
// once (<1, 8> 29.6 us at 4096, <2, 12> 36.4, <1, 4> 45.3); up to 16384 the
// 32-target ones do in two rounds (<2, 12> 68.7 us at 8192, <1, 8> 74.4, <2, 6>
// 86; at 16384 all are within 3%); beyond, several smaller workgroups per CU
// (<2, 6> 3.21 ms at 65536, <2, 12> 3.42).  FP64, whose terms take twice the
// LDS: <1, 6> 178 us at 8192, <1, 3> 200; <1, 3> 602 us at 16384, <1, 6> 629.
// Above the last bound one thread per body is faster.
template <typename T, typename T4, bool FAST, bool STEP>
static void launch_ref(const T4* pos_old, T4* pos_new, T4* vel, int n, int i0, int cnt, T dt, T eps2, T damping,
                       double* acc3, int block, hipStream_t st)
{
    if constexpr (sizeof(T) == 4) {
        if (cnt <= 4096)
            return launch_ref_split<T, T4, FAST, 1, 8, STEP>(pos_old, pos_new, vel, n, i0, cnt, dt, eps2, damping,
                                                             acc3, st);
        if (cnt <= 16384)
            return launch_ref_split<T, T4, FAST, 2, 12, STEP>(pos_old, pos_new, vel, n, i0, cnt, dt, eps2, damping,
                                                              acc3, st);
        if (cnt <= 98304)
            return launch_ref_split<T, T4, FAST, 2, 6, STEP>(pos_old, pos_new, vel, n, i0, cnt, dt, eps2, damping,
                                                             acc3, st);
    } else {
        if (cnt <= 8192)
            return launch_ref_split<T, T4, FAST, 1, 6, STEP>(pos_old, pos_new, vel, n, i0, cnt, dt, eps2, damping,
                                                             acc3, st);
        if (cnt <= 49152)
            return launch_ref_split<T, T4, FAST, 1, 3, STEP>(pos_old, pos_new, vel, n, i0, cnt, dt, eps2, damping,
                                                             acc3, st);
    }
    if constexpr (STEP) {
        if (block <= 0)
            block = 256;
        hipLaunchKernelGGL((ref_step_kernel<T, T4, FAST>), dim3((unsigned)((cnt + block - 1) / block)), dim3(block), 0,
                           st, pos_old, pos_new, vel, n, i0, cnt, dt, eps2, damping);
    } else {
        hipLaunchKernelGGL((ref_accel_kernel<T, T4, FAST>), dim3((unsigned)((cnt + 255) / 256)), dim3(256), 0, st,
                           pos_old, n, i0, cnt, eps2, acc3);
    }
}

hipError_t launch_ref_step_slice_f32(const float4* pos_old, float4* pos_new, float4* vel, int n, int i0, int cnt,
                                     float dt, float eps2, float damping, int block, hipStream_t st)
{
    if (eps2 >= kRefInvMin && eps2 <= 3.0e38f)
        launch_ref<float, float4, true, true>(pos_old, pos_new, vel, n, i0, cnt, dt, eps2, damping, nullptr, block, st);
    else
        launch_ref<float, float4, false, true>(pos_old, pos_new, vel, n, i0, cnt, dt, eps2, damping, nullptr, block,
                                               st);
    return hipGetLastError();
}

hipError_t launch_ref_step_slice_f64(const double4* pos_old, double4* pos_new, double4* vel, int n, int i0,
                                     int cnt, double dt, double eps2, double damping, int block, hipStream_t st)
{
    if (eps2 >= kRefInv64Min)
        launch_ref<double, double4, true, true>(pos_old, pos_new, vel, n, i0, cnt, dt, eps2, damping, nullptr, block,
                                                st);
    else
        launch_ref<double, double4, false, true>(pos_old, pos_new, vel, n, i0, cnt, dt, eps2, damping, nullptr, block,
                                                 st);
    return hipGetLastError();
}

hipError_t launch_ref_step_f32(const float4* pos_old, float4* pos_new, float4* vel, int n,
                               float dt, float eps2, float damping, int block, hipStream_t st)
{
    return launch_ref_step_slice_f32(pos_old, pos_new, vel, n, 0, n, dt, eps2, damping, block, st);
}

hipError_t launch_ref_step_f64(const double4* pos_old, double4* pos_new, double4* vel, int n,
                               double dt, double eps2, double damping, int block,
                               hipStream_t st)
{
    return launch_ref_step_slice_f64(pos_old, pos_new, vel, n, 0, n, dt, eps2, damping, block, st);
}

hipError_t launch_ref_accel_slice_f32(const float4* src, int n, int i0, int cnt, float eps2, double* acc3,
                                      hipStream_t st)
{
    if (eps2 >= kRefInvMin && eps2 <= 3.0e38f)
        launch_ref<float, float4, true, false>(src, nullptr, nullptr, n, i0, cnt, 0.f, eps2, 0.f, acc3, 0, st);
    else
        launch_ref<float, float4, false, false>(src, nullptr, nullptr, n, i0, cnt, 0.f, eps2, 0.f, acc3, 0, st);
    return hipGetLastError();
}

hipError_t launch_ref_accel_slice_f64(const double4* src, int n, int i0, int cnt, double eps2, double* acc3,
                                      hipStream_t st)
{
    if (eps2 >= kRefInv64Min)
        launch_ref<double, double4, true, false>(src, nullptr, nullptr, n, i0, cnt, 0.0, eps2, 0.0, acc3, 0, st);
    else
        launch_ref<double, double4, false, false>(src, nullptr, nullptr, n, i0, cnt, 0.0, eps2, 0.0, acc3, 0, st);
    return hipGetLastError();
}

hipError_t launch_ref_accel_f32(const float4* src, int n, float eps2, double* acc3,
                                hipStream_t st)
{
    return launch_ref_accel_slice_f32(src, n, 0, n, eps2, acc3, st);
}

hipError_t launch_ref_accel_f64(const double4* src, int n, double eps2, double* acc3,
                                hipStream_t st)
{
    return launch_ref_accel_slice_f64(src, n, 0, n, eps2, acc3, st);
}

}  // namespace utcnb

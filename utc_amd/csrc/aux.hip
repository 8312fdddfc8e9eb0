// aux.hip -- O(N) helper kernels (padding, snapshots, conversions) and the
// FP64 energy / momentum diagnostics.
#include "internal.h"
#include "ref_inv.h"

namespace utcnb {

__global__ void pad_f32_kernel(float4* p, int n, int n_pad)
{
    int i = n + blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n_pad)
        p[i] = make_float4(kPadCoord, kPadCoord, kPadCoord, 0.0f);
}

__global__ void pad_f64_kernel(double4* p, int n, int n_pad)
{
    int i = n + blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n_pad)
        p[i] = make_double4(kPadCoord, kPadCoord, kPadCoord, 0.0);
}

hipError_t launch_pad_f32(float4* p, int n, int n_pad, hipStream_t st)
{
    if (n_pad <= n)
        return hipSuccess;
    int cnt = n_pad - n;
    hipLaunchKernelGGL(pad_f32_kernel, dim3((cnt + 255) / 256), dim3(256), 0, st, p, n, n_pad);
    return hipGetLastError();
}

hipError_t launch_pad_f64(double4* p, int n, int n_pad, hipStream_t st)
{
    if (n_pad <= n)
        return hipSuccess;
    int cnt = n_pad - n;
    hipLaunchKernelGGL(pad_f64_kernel, dim3((cnt + 255) / 256), dim3(256), 0, st, p, n, n_pad);
    return hipGetLastError();
}

__global__ void snapshot_kernel(const double4* __restrict__ pos, float4* __restrict__ snap, int n)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        double4 p = pos[i];
        snap[i] = make_float4((float)p.x, (float)p.y, (float)p.z, (float)p.w);
    }
}

hipError_t launch_snapshot(const double4* pos, float4* snap, int n, hipStream_t st)
{
    hipLaunchKernelGGL(snapshot_kernel, dim3((n + 255) / 256), dim3(256), 0, st, pos, snap, n);
    return hipGetLastError();
}

__global__ void f32_to_f64_kernel(const float4* __restrict__ s, double4* __restrict__ d, int n)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        float4 v = s[i];
        d[i] = make_double4(v.x, v.y, v.z, v.w);
    }
}

hipError_t launch_f32_to_f64(const float4* src, double4* dst, int n, hipStream_t st)
{
    hipLaunchKernelGGL(f32_to_f64_kernel, dim3((n + 255) / 256), dim3(256), 0, st, src, dst, n);
    return hipGetLastError();
}

hipError_t launch_f64_to_f32(const double4* src, float4* dst, int n, hipStream_t st)
{
    return launch_snapshot(src, dst, n, st);
}

// Device state in and out of a handle with one launch: what bounds it at the
// sizes of a step is the launches, of which a copy, a conversion (through the
// staging buffer) and a snapshot for each array took up to five in and four
// out, with a wait between those.  State in, steps, state out: 100 mixed steps
// of 1000 bodies 384 to 341 us, 12 of 16384 743 to 699, 10 plain FP32 steps of
// 4096 94.6 to 88.5.
struct Rec4 {
    double v[4];
};
__device__ __forceinline__ Rec4 rec_load(const float* p, size_t i)
{
    const float4 a = ((const float4*)p)[i];
    return {{a.x, a.y, a.z, a.w}};
}
__device__ __forceinline__ Rec4 rec_load(const double* p, size_t i)
{
    const double2 a = ((const double2*)p)[2 * i], b = ((const double2*)p)[2 * i + 1];
    return {{a.x, a.y, b.x, b.y}};
}
__device__ __forceinline__ void rec_store(float* p, size_t i, const Rec4& r)
{
    ((float4*)p)[i] = make_float4((float)r.v[0], (float)r.v[1], (float)r.v[2], (float)r.v[3]);
}
__device__ __forceinline__ void rec_store(double* p, size_t i, const Rec4& r)
{
    ((double2*)p)[2 * i] = make_double2(r.v[0], r.v[1]);
    ((double2*)p)[2 * i + 1] = make_double2(r.v[2], r.v[3]);
}

// Block row 0: positions (and their FP32 snapshot), 1: velocities.
template <typename From, typename To>
__global__ void state_copy_kernel(const From* __restrict__ pos, const From* __restrict__ vel, To* __restrict__ p,
                                  To* __restrict__ v, float* __restrict__ snap, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    if (blockIdx.y == 1) {
        rec_store(v, i, rec_load(vel, i));
        return;
    }
    const Rec4 r = rec_load(pos, i);
    rec_store(p, i, r);
    if (snap)
        rec_store(snap, i, r);
}

hipError_t launch_state_copy(const void* pos, const void* vel, bool from_f32, void* p, void* v, bool to_f32,
                             float4* snap, int n, hipStream_t st)
{
    const dim3 grid((n + 255) / 256, vel ? 2 : 1), block(256);
#define STATE_COPY(F, T)                                                                                            \
    hipLaunchKernelGGL((state_copy_kernel<F, T>), grid, block, 0, st, (const F*)pos, (const F*)vel, (T*)p, (T*)v, \
                       (float*)snap, n)
    if (from_f32 && to_f32)
        STATE_COPY(float, float);
    else if (from_f32)
        STATE_COPY(float, double);
    else if (to_f32)
        STATE_COPY(double, float);
    else
        STATE_COPY(double, double);
#undef STATE_COPY
    return hipGetLastError();
}

// ---- energy / momentum ---------------------------------------------------------
// Pass 1: one thread per body i computes phi_i = sum_{j != i} m_j / sqrt(r^2+eps2)
// (FP64, compensated chunks), kinetic_i and momentum_i; the workgroup reduces
// its 256 bodies with wavefront shuffles and LDS and writes one partial of 5
// values.  Pass 2: one workgroup adds the partials in a fixed order, so the
// result is deterministic.

__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1)
        v += __shfl_xor(v, off, 64);
    return v;
}

__global__ __launch_bounds__(256) void energy_pass1(const double4* __restrict__ pos,
                                                    const double4* __restrict__ vel, int n,
                                                    double eps2, double* __restrict__ part)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    const int il = i < n ? i : n - 1;
    const double4 p = pos[il];
    double phi = 0.0, c = 0.0;
    for (int jc = 0; jc < n; jc += kChunk) {
        const int je = jc + kChunk < n ? jc + kChunk : n;
        double a = 0.0;
        int j = jc;
        // four sources per trip, one wave-uniform choice between the short
        // forms of the correctly rounded sqrt and division (ref_inv.h; the
        // same bits inside their ranges) and the generic ones
        for (; j + 4 <= je; j += 4) {
            double d2[4], m[4], t[4];
            bool ok = true;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const double4 q = pos[j + k];
                double rx = q.x - p.x, ry = q.y - p.y, rz = q.z - p.z;
                d2[k] = rx * rx + ry * ry + rz * rz + eps2;
                m[k] = q.w;
                ok = ok && d2[k] >= kRefInv64Min && d2[k] <= kRefInv64Max && m[k] >= kRefDiv64NumMin &&
                     m[k] <= kRefDiv64NumMax;
            }
            if (__ballot(!ok) == 0) {
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    t[k] = ref_div64(m[k], ref_sqrt64(d2[k]));
            } else {
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    t[k] = m[k] / __builtin_sqrt(d2[k]);
            }
#pragma unroll
            for (int k = 0; k < 4; ++k)
                a += (j + k == il) ? 0.0 : t[k];
        }
        for (; j < je; ++j) {
            const double4 q = pos[j];
            double rx = q.x - p.x, ry = q.y - p.y, rz = q.z - p.z;
            double d2 = rx * rx + ry * ry + rz * rz + eps2;
            double t = q.w / __builtin_sqrt(d2);
            a += (j == il) ? 0.0 : t;
        }
        double y = a - c;
        double s = phi + y;
        c = (s - phi) - y;
        phi = s;
    }
    double v[5] = {0, 0, 0, 0, 0};
    if (i < n) {
        const double4 u = vel[i];
        v[0] = 0.5 * p.w * (u.x * u.x + u.y * u.y + u.z * u.z);
        v[1] = -0.5 * p.w * (phi - c);
        v[2] = p.w * u.x;
        v[3] = p.w * u.y;
        v[4] = p.w * u.z;
    }
    __shared__ double red[4][5];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        double w = wave_sum(v[k]);
        if (lane == 0)
            red[wave][k] = w;
    }
    __syncthreads();
    if (threadIdx.x < 5) {
        int k = threadIdx.x;
        part[5 * (size_t)blockIdx.x + k] = ((red[0][k] + red[1][k]) + red[2][k]) + red[3][k];
    }
}

__global__ __launch_bounds__(64) void energy_pass2(const double* __restrict__ part, int nparts,
                                                   double* __restrict__ out5)
{
    const int lane = threadIdx.x;
    for (int k = 0; k < 5; ++k) {
        double s = 0.0, c = 0.0;
        for (int b = lane; b < nparts; b += 64) {
            double y = part[5 * (size_t)b + k] - c;
            double t = s + y;
            c = (t - s) - y;
            s = t;
        }
        double w = wave_sum(s - c);
        if (lane == 0)
            out5[k] = w;
    }
}

// `out5` must hold 5 + 5 * ceil(n/256) doubles: the partials live after the result.
hipError_t launch_energy(const double4* pos, const double4* vel, int n, double eps2,
                         double* out5, hipStream_t st)
{
    const int blocks = (n + 255) / 256;
    double* part = out5 + 5;
    hipLaunchKernelGGL(energy_pass1, dim3(blocks), dim3(256), 0, st, pos, vel, n, eps2, part);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess)
        return e;
    hipLaunchKernelGGL(energy_pass2, dim3(1), dim3(64), 0, st, part, blocks, out5);
    return hipGetLastError();
}

}  // namespace utcnb

// probe_invdist_group.hip -- exhaustive device check of ref_inv_dist_y and
// ref_inv_dist_group (ref_inv.h).
//
// For every float d2 from 2^-96 to FLT_MAX and +inf: where y = v_rsq_f32(d2)
// has a non-zero significand, ref_inv_dist_y(d2, y) must equal
// (float)(1.0 / (double)sqrtf(d2)), as the compiler builds it with IEEE sqrt
// and division, bit for bit (the others are counted: the group function sends
// them elsewhere); and ref_inv_dist_group must equal it for groups of 8 and of
// 4 that mix values a fixed distance apart, NaN among them.
// Test infrastructure (run by tests/test_gpu_ref_split.py).
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>

#include "ref_inv.h"

#define CHK(x)                                                                                     \
    do {                                                                                           \
        hipError_t e_ = (x);                                                                       \
        if (e_ != hipSuccess) {                                                                    \
            std::printf("HIP error %s at line %d\n", hipGetErrorString(e_), __LINE__);             \
            return 1;                                                                              \
        }                                                                                          \
    } while (0)

struct Result {
    unsigned long long checked, bad, flagged, group_checked, group_bad;
    unsigned int first;
};

__device__ __attribute__((noinline)) float reference_inv(float d2) { return (float)(1.0 / (double)sqrtf(d2)); }

__device__ bool same(float a, float b) { return __float_as_uint(a) == __float_as_uint(b) || (a != a && b != b); }

__global__ void check_single(uint32_t lo, uint32_t hi, Result* r)
{
    unsigned long long n = 0, bad = 0, flagged = 0;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t u = (uint64_t)lo + blockIdx.x * blockDim.x + threadIdx.x; u <= (uint64_t)hi; u += stride) {
        const float x = __uint_as_float((uint32_t)u), y = __builtin_amdgcn_rsqf(x);
        ++n;
        if ((__float_as_uint(y) << 9) == 0) {
            ++flagged;
        } else if (!same(utcnb::ref_inv_dist_y(x, y), reference_inv(x))) {
            ++bad;
            r->first = (uint32_t)u;
        }
    }
    atomicAdd(&r->checked, n);
    atomicAdd(&r->bad, bad);
    atomicAdd(&r->flagged, flagged);
}

// Every value once: value u is member (u - lo) / step of the group that starts
// at lo + (u - lo) % step; members past hi are NaN.
template <int G>
__global__ void check_group(uint32_t lo, uint32_t hi, uint32_t step, Result* r)
{
    unsigned long long n = 0, bad = 0;
    const uint32_t stride = gridDim.x * blockDim.x;
    const uint32_t rounds = (step + stride - 1) / stride;  // every thread of the wave in every round
    for (uint32_t k = 0; k < rounds; ++k) {
        const uint64_t base = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x + (uint64_t)k * stride;
        float x[G], inv[G];
        for (int q = 0; q < G; ++q) {
            const uint64_t u = lo + base + (uint64_t)q * step;
            x[q] = base < step && u <= hi ? __uint_as_float((uint32_t)u) : __uint_as_float(0x7fc00000u);
        }
        utcnb::ref_inv_dist_group<G>(x, inv);
        for (int q = 0; q < G; ++q) {
            ++n;
            if (!same(inv[q], reference_inv(x[q])))
                ++bad;
        }
    }
    atomicAdd(&r->group_checked, n);
    atomicAdd(&r->group_bad, bad);
}

int main()
{
    Result* r;
    CHK(hipMalloc(&r, sizeof(Result)));
    CHK(hipMemset(r, 0, sizeof(Result)));
    const uint32_t lo = 0x0f800000u, hi = 0x7f800000u;  // 2^-96 .. +inf
    hipLaunchKernelGGL(check_single, dim3(4096), dim3(256), 0, 0, lo, hi, r);
    CHK(hipDeviceSynchronize());
    hipLaunchKernelGGL((check_group<8>), dim3(4096), dim3(256), 0, 0, lo, hi, (hi - lo) / 8 + 1, r);
    CHK(hipDeviceSynchronize());
    hipLaunchKernelGGL((check_group<4>), dim3(4096), dim3(256), 0, 0, lo, hi, (hi - lo) / 4 + 1, r);
    CHK(hipDeviceSynchronize());
    Result h;
    CHK(hipMemcpy(&h, r, sizeof(h), hipMemcpyDeviceToHost));
    CHK(hipFree(r));
    std::printf("checked %llu mismatches %llu flagged %llu group_checked %llu group_mismatches %llu first %08x\n", h.checked,
                h.bad, h.flagged, h.group_checked, h.group_bad, h.first);
    return h.bad || h.group_bad || h.checked != (uint64_t)hi - lo + 1 ? 2 : 0;
}

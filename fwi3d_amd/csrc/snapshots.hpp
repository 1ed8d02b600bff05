// Snapshot-store kernels: the forward wavefield every `sub` steps, kept in HBM for the
// imaging condition of the adjoint run (the role of zfpWrapper::set/get in the
// reference, src/include/zfpWrapper.hpp:78-116). FP32 slots are plain copies; 16-bit
// slots hold BF16 / FP16 codes of u / s with the per-snapshot scale of SnapView.
#pragma once
#include "common.hpp"

namespace fwi3d {

// Workgroups of the snapshot kernels: 4 of 256 threads per CU, each thread reads 16 bytes at
// a time.
inline unsigned snap_blocks(size_t n) { return (unsigned)std::min<size_t>(1024, (n / 4 + 255) / 256 + 1); }

// max|u| over n values into *maxbits (float bits; the word starts at zero). One atomic per
// workgroup, and none when the word already holds as much: with one per wave, 8192 on one
// word, they were the kernel's time: 99 us for 131 x 141 x 153 x 3 values, 12 us now.
__global__ __launch_bounds__(256) void snap_maxabs(const float* __restrict__ u, unsigned* __restrict__ maxbits,
                                                   long long n) {
    __shared__ float wm[4];
    float m = 0.f;
    const long long n4 = n >> 2;
    const float4* __restrict__ u4 = (const float4*)u;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += (long long)gridDim.x * blockDim.x) {
        const float4 v = u4[i];
        m = fmaxf(m, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
    }
    for (long long i = 4 * n4 + (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        m = fmaxf(m, fabsf(u[i]));
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
    if ((threadIdx.x & 63) == 0) wm[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        m = fmaxf(fmaxf(wm[0], wm[1]), fmaxf(wm[2], wm[3]));
        const unsigned b = __float_as_uint(m);
        if (b > __hip_atomic_load(maxbits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(maxbits, b);
    }
}

// 16-bit codes of u / s, s = max|u| / 2^15 (round to nearest even); u and dst are 16-byte
// aligned.
template <int FMT>
__device__ __forceinline__ unsigned short snap_code(float v) {
    return FMT == SNAP_BF16 ? bf16_rne(v) : __half_as_ushort(__float2half_rn(v));
}
template <int FMT>
__global__ __launch_bounds__(256) void snap_store(const float* __restrict__ u, void* __restrict__ dst,
                                                  const unsigned* __restrict__ maxbits, long long n) {
    const float m = __uint_as_float(*maxbits);
    const float inv = m > 0.f ? kSnapTop / m : 0.f;
    unsigned short* __restrict__ d = (unsigned short*)dst;
    const long long n4 = n >> 2;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += (long long)gridDim.x * blockDim.x) {
        const float4 v = ((const float4*)u)[i];
        ((ushort4*)d)[i] = make_ushort4(snap_code<FMT>(v.x * inv), snap_code<FMT>(v.y * inv), snap_code<FMT>(v.z * inv),
                                        snap_code<FMT>(v.w * inv));
    }
    for (long long i = 4 * n4 + (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        d[i] = snap_code<FMT>(u[i] * inv);
}

}  // namespace fwi3d

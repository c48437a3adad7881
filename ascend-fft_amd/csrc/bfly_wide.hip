// bfly_wide.hip -- C2C of 8192, 16384 and 32768 points, one transform per
// workgroup of n/32 threads (bfly_wide.hpp): one HBM read and one HBM write
// per element.
//
// HBM-bound in the aggregate, but a transform's load, passes and store follow
// each other inside its workgroup, and few workgroups share a CU (four at
// 8192, two at 16384, one at 32768), so the time depends on how well the
// workgroups' phases interleave.  Two things were measured to matter:
//   * 32 points per thread and one-component exchanges halve the LDS of a
//     transform: twice the workgroups per CU at 8192 and 16384 against the
//     16-point streaming kernels, and 32768 points fit a CU at all (two
//     kernels and two round trips before); three passes, two exchanges.
//   * The first workgroups start staggered (kStagger).
// Measured, the kernels AUTO ran before -> this one: 8192 x 2048 54.4 -> 49.6
// us, x 512 15.4 -> 14.3; 16384 x 1000 59.4 -> 56.3, x 512 31.2 -> 25.0, x 256
// 18.9 -> 17.6; 32768 x 256 51.3 -> 32.0 (4.2 TB/s), x 512 86.8 -> 62.5.
#include <hip/hip_runtime.h>

#include "bfly_hip.h"
#include "bfly_kernels.hpp"
#include "bfly_wide.hpp"

using namespace bfly_dev;

namespace {

// The plan of one length; T1: entries of the second pass's table (r R0 + k).
template <int N>
struct WidePlan {
    static constexpr int R0 = N == 32768 ? 32 : 16, R1 = N == 8192 ? 16 : 32, R2 = 32;
    static_assert(R0 * R1 * R2 == N, "three passes");
    static constexpr int T1 = R0 * R1;
};

// Staggered start.  All resident workgroups begin a launch together, load at
// the same time, then leave the memory idle while all of them compute.
// Instead workgroup b < kResident waits ((b >> SHIFT) & MASK) * STEP * 128
// clocks first, so that later ones load while earlier ones compute; the
// memory is busy either way, only the order changes.  The ramp is about the
// time of one round's loads (32768: 32 steps of 0.2 us).  32768 x 256 39.3 ->
// 32.0 us, x 512 75.5 -> 62.5 (steps twice as long), 16384 x 256 21.5 -> 17.6,
// x 512 28.9 -> 25.0, 8192 x 1024 24.6 -> 23.4, x 2048 50.8 -> 49.6.  Kernels
// with four or more smaller workgroups per CU and a prefetch gained nothing.
template <int N>
struct Stagger {
    static constexpr uint32_t SHIFT = N == 32768 ? 3 : 5, MASK = N == 32768 ? 31 : 7;
    static constexpr uint32_t kResident = 256 * (32768 / N);
};
template <int N>
uint32_t stagger_step(uint32_t batch) {
    return N == 32768 ? (batch <= 256 ? 4 : 7) : N == 16384 ? 8 : 2;
}

template <int N, int DIR>
__global__ __launch_bounds__(N / kWide) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_c2c_wide(
    const float2* __restrict__ in, float2* __restrict__ out, const float2* __restrict__ wN, float scale,
    uint64_t idist, uint64_t odist, uint32_t step) {
    using W = WidePlan<N>;
    constexpr int T = N / kWide;
    __shared__ float lds[lds_len(N)];
    __shared__ float2 t1[W::T1];
    __shared__ Wide64 tab[kWideTab<N>];
    if (blockIdx.x < Stagger<N>::kResident)
        for (uint32_t i = ((blockIdx.x >> Stagger<N>::SHIFT) & Stagger<N>::MASK) * step; i > 0; i--)
            __builtin_amdgcn_s_sleep(2);
    int t = threadIdx.x;
    const float2* src = in + (uint64_t)blockIdx.x * idist;
    float2 v[kWide];
#pragma unroll
    for (int m = 0; m < kWide / W::R0; m++)
#pragma unroll
        for (int r = 0; r < W::R0; r++) v[m * W::R0 + r] = ld_stream(&src[t + m * T + r * (N / W::R0)]);
    for (int i = t; i < W::T1; i += T) t1[i] = wN[(i / W::R0) * (i % W::R0) * (N / W::T1)];
    wide_table<N>(tab, t);
    // (the first exchange's barriers order the tables before their first read)
    stockham_wide<N, T, DIR, W::R0, 1, W::R0, W::R1, W::R2>(v, lds, tab, t1, t);
    if (scale != 1.0f) {  // uniform: the normalised entry point only
#pragma unroll
        for (int i = 0; i < kWide; i++) v[i] = make_float2(v[i].x * scale, v[i].y * scale);
    }
    float2* dst = out + (uint64_t)blockIdx.x * odist;
#pragma unroll
    for (int r = 0; r < W::R2; r++) st_stream(&dst[t + r * T], v[r]);
}

template <int N>
hipError_t launch_wide_rows(const float2* in, float2* out, const float2* wN, uint32_t batch, int sign, float scale,
                            uint64_t idist, uint64_t odist, hipStream_t s) {
    const uint32_t step = stagger_step<N>(batch);
    if (sign < 0)
        hipLaunchKernelGGL((k_c2c_wide<N, -1>), dim3(batch), dim3(N / kWide), 0, s, in, out, wN, scale, idist, odist,
                           step);
    else
        hipLaunchKernelGGL((k_c2c_wide<N, 1>), dim3(batch), dim3(N / kWide), 0, s, in, out, wN, scale, idist, odist,
                           step);
    return hipGetLastError();
}

}  // namespace

namespace bfly_kern {

hipError_t c2c_wide(const float2* in, float2* out, const float2* wN, uint32_t n, uint32_t batch, int sign,
                    float scale, uint64_t idist, uint64_t odist, hipStream_t s) {
    switch (n) {
        case 8192: return launch_wide_rows<8192>(in, out, wN, batch, sign, scale, idist, odist, s);
        case 16384: return launch_wide_rows<16384>(in, out, wN, batch, sign, scale, idist, odist, s);
        case 32768: return launch_wide_rows<32768>(in, out, wN, batch, sign, scale, idist, odist, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace bfly_kern

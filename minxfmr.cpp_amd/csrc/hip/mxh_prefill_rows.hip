// mxh_prefill_rows.hip — activation rows as input of the exact-weight prefill
// GEMM (mxh_gemm_codes.hip): a' = a 2^e (e per row, so max |a'| lies in
// [128, 256)) split into fp16 hi + lo (about 22 significant bits), with the
// sums of every 32-element sub-block of those values split the same way (they
// carry the min terms of Q4_K / Q5_K weights), optionally after the
// reference's rmsnorm or as silu(gate) * up.
//
// Four consecutive elements are stored in the order 0 2 1 3: the
// order in which the GEMM's code pairs leave its masks.
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include "mxh_device.h"
#include "mxh_internal.h"

namespace mxh {

namespace {

__device__ __forceinline__ uint16_t f16_bits(float v) { return __half_as_ushort(__float2half_rn(v)); }

// fp16 hi + lo of v (lo = v - hi rounded again) as hi | lo << 16
__device__ __forceinline__ uint32_t split_f16(float v) {
    const __half h = __float2half_rn(v);
    return (uint32_t)__half_as_ushort(h) | ((uint32_t)f16_bits(v - __half2float(h)) << 16);
}

// power-of-two scale 2^e that brings the row maximum into [128, 256)
__device__ __forceinline__ int row_exponent(float maxv) {
    if (!(maxv > 0.f) || maxv > 3.0e38f) return 0;
    int ex;
    (void)frexpf(maxv, &ex);  // maxv in [2^(ex-1), 2^ex)
    const int e = 8 - ex;
    return e < -100 ? -100 : (e > 100 ? 100 : e);
}

// block-wide max of non-negative floats (256 threads)
__device__ __forceinline__ float block_max_256(float v, float* red) {
    v = wave_max_all(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    const float r = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    __syncthreads();
    return r;
}

// Writes row values v (sub-block sb of 32, thread-owned) as a' = v 2^e split
// into fp16 hi / lo, and the split sum of each sub-block's hi + lo.
__device__ __forceinline__ void emit_subblock(const float* v, float scale, uint16_t* ah, uint16_t* al, uint16_t* sh,
                                              uint16_t* sl) {
    float s = 0.f;
    uint32_t ph[16], pl[16];
#pragma unroll
    for (int i = 0; i < 32; i += 2) {
        // stored pairs of a group of four: (0, 2) then (1, 3)
        const int e = (i & ~3) + ((i >> 1) & 1);
        const uint32_t p0 = split_f16(v[e] * scale), p1 = split_f16(v[e + 2] * scale);
        s += (__half2float(__ushort_as_half((uint16_t)p0)) + __half2float(__ushort_as_half((uint16_t)(p0 >> 16)))) +
             (__half2float(__ushort_as_half((uint16_t)p1)) + __half2float(__ushort_as_half((uint16_t)(p1 >> 16))));
        ph[i / 2] = (p0 & 0xffffu) | (p1 << 16);
        pl[i / 2] = (p0 >> 16) | (p1 & 0xffff0000u);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        reinterpret_cast<uint4*>(ah)[q] = make_uint4(ph[4 * q], ph[4 * q + 1], ph[4 * q + 2], ph[4 * q + 3]);
        reinterpret_cast<uint4*>(al)[q] = make_uint4(pl[4 * q], pl[4 * q + 1], pl[4 * q + 2], pl[4 * q + 3]);
    }
    const uint32_t ps = split_f16(s);
    *sh = (uint16_t)ps;
    *sl = (uint16_t)(ps >> 16);
}

// Rows of x (optionally the reference rmsnorm x / sqrt(mean(x^2) + eps) * w,
// rmsnorm.cpp:5-26, sum of squares in double, the same float products as
// rows_to_bf16) as GEMM input of gemm_q_f16.  One workgroup per row; k a
// multiple of 32 and at most 2 * 256 * 32.
constexpr int kRowSub = 2;  // sub-blocks per thread
__global__ __launch_bounds__(256) void rows_to_f16_kernel(const float* __restrict__ x, int ldx,
                                                          const float* __restrict__ nw, float eps, int k,
                                                          uint16_t* __restrict__ a_hi, uint16_t* __restrict__ a_lo,
                                                          int lda, uint16_t* __restrict__ s_hi,
                                                          uint16_t* __restrict__ s_lo, int lds,
                                                          float* __restrict__ rscale) {
    __shared__ double red[4];
    __shared__ float redf[4];
    const int row = blockIdx.x, nsb = k / 32;
    const float* xr = x + (size_t)row * ldx;
    float v[kRowSub][32];
    double ss = 0.0;
    float mx = 0.f;
#pragma unroll
    for (int u = 0; u < kRowSub; ++u) {
        const int sb = threadIdx.x + 256 * u;
#pragma unroll
        for (int i = 0; i < 32; ++i) v[u][i] = 0.f;
        if (sb < nsb) {
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const float4 f = reinterpret_cast<const float4*>(xr + 32 * sb)[q];
                v[u][4 * q] = f.x;
                v[u][4 * q + 1] = f.y;
                v[u][4 * q + 2] = f.z;
                v[u][4 * q + 3] = f.w;
            }
        }
#pragma unroll
        for (int i = 0; i < 32; ++i) ss += (double)v[u][i] * v[u][i];
    }
    float inv = 1.f;
    if (nw) {
        ss = wave_sum_d_lane63(ss);
        if ((threadIdx.x & 63) == 63) red[threadIdx.x >> 6] = ss;
        __syncthreads();
        inv = (float)(1.0 / sqrt(((red[0] + red[1]) + (red[2] + red[3])) / (double)k + (double)eps));
    }
#pragma unroll
    for (int u = 0; u < kRowSub; ++u) {
        const int sb = threadIdx.x + 256 * u;
        if (nw && sb < nsb) {
#pragma unroll
            for (int i = 0; i < 32; ++i) v[u][i] = v[u][i] * inv * nw[32 * sb + i];
        }
#pragma unroll
        for (int i = 0; i < 32; ++i) mx = fmaxf(mx, fabsf(v[u][i]));
    }
    const int e = row_exponent(block_max_256(mx, redf));
    const float scale = ldexpf(1.f, e);
    if (threadIdx.x == 0) rscale[row] = ldexpf(1.f, -e);
#pragma unroll
    for (int u = 0; u < kRowSub; ++u) {
        const int sb = threadIdx.x + 256 * u;
        if (sb < nsb)
            emit_subblock(v[u], scale, a_hi + (size_t)row * lda + 32 * sb, a_lo + (size_t)row * lda + 32 * sb,
                          s_hi + (size_t)row * lds + sb, s_lo + (size_t)row * lds + sb);
    }
}

// h = silu(gate) * up (transformer.cpp:183-185) as gemm_q_f16 input; gu
// rows are [gate | up], f a multiple of 32 and at most 2 * 256 * 32.
__global__ __launch_bounds__(256) void silu_mul_f16_kernel(const float* __restrict__ gu, int f,
                                                           uint16_t* __restrict__ h_hi, uint16_t* __restrict__ h_lo,
                                                           uint16_t* __restrict__ s_hi, uint16_t* __restrict__ s_lo,
                                                           float* __restrict__ rscale) {
    __shared__ float redf[4];
    const int row = blockIdx.x, nsb = f / 32, lds = nsb;
    const float* g = gu + (size_t)row * 2 * f;
    float v[kRowSub][32];
    float mx = 0.f;
#pragma unroll
    for (int u = 0; u < kRowSub; ++u) {
        const int sb = threadIdx.x + 256 * u;
#pragma unroll
        for (int i = 0; i < 32; ++i) v[u][i] = 0.f;
        if (sb < nsb) {
            // the sub-block's 32 gate and 32 up values as 16-byte loads
            const float4* gp = reinterpret_cast<const float4*>(g + 32 * sb);
            const float4* up = reinterpret_cast<const float4*>(g + f + 32 * sb);
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const float4 a = gp[q], b = up[q];
                const float ga[4] = {a.x, a.y, a.z, a.w}, ub[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
                for (int j = 0; j < 4; ++j) v[u][4 * q + j] = ga[j] / (1.0f + expf(-ga[j])) * ub[j];
            }
        }
#pragma unroll
        for (int i = 0; i < 32; ++i) mx = fmaxf(mx, fabsf(v[u][i]));
    }
    const int e = row_exponent(block_max_256(mx, redf));
    const float scale = ldexpf(1.f, e);
    if (threadIdx.x == 0) rscale[row] = ldexpf(1.f, -e);
#pragma unroll
    for (int u = 0; u < kRowSub; ++u) {
        const int sb = threadIdx.x + 256 * u;
        if (sb < nsb)
            emit_subblock(v[u], scale, h_hi + (size_t)row * f + 32 * sb, h_lo + (size_t)row * f + 32 * sb,
                          s_hi + (size_t)row * lds + sb, s_lo + (size_t)row * lds + sb);
    }
}

}  // namespace

int rows_to_f16_launch(const float* x, int ldx, const float* nw, float eps, int k, uint16_t* a_hi, uint16_t* a_lo,
                       int lda, uint16_t* s_hi, uint16_t* s_lo, int lds, float* rscale, int m, hipStream_t st) {
    if (m <= 0 || k % 32 || k > kRowSub * 256 * 32 || lda < k || lds < k / 32) return MXH_ERR_ARG;
    hipLaunchKernelGGL(rows_to_f16_kernel, dim3(m), dim3(256), 0, st, x, ldx, nw, eps, k, a_hi, a_lo, lda, s_hi, s_lo,
                       lds, rscale);
    return MXH_OK;
}

int silu_mul_f16_launch(const float* gu, int f, uint16_t* h_hi, uint16_t* h_lo, uint16_t* s_hi, uint16_t* s_lo,
                        float* rscale, int m, hipStream_t st) {
    if (m <= 0 || f % 32 || f > kRowSub * 256 * 32) return MXH_ERR_ARG;
    hipLaunchKernelGGL(silu_mul_f16_kernel, dim3(m), dim3(256), 0, st, gu, f, h_hi, h_lo, s_hi, s_lo, rscale);
    return MXH_OK;
}

}  // namespace mxh

// mxh_dequant.hip — GGUF block -> fp32 decode on the device, bit-exact with
// the reference CPU decoders (src/tensor/tensor.cpp:405-457) and with its
// load-time F16 / Q6_K conversions (third_party/gguf/gguf_reader.cpp:759-785,
// :905-1008; products and differences as in mxh_quant.h).
//
// Bound: HBM, nearly all of it the stores (4096 x 14336 Q6_K: 48 MB in, 235 MB
// out).  Rows of whole blocks are contiguous, so the matrix is one run of
// blocks and a thread writes four consecutive outputs: a wave's store is 1 KiB
// in one piece, and its codes are one dword a lane from at most 256 elements'
// blocks (the lanes that share a dword, a scale or a header hit the cache).
// One thread a run of 32 elements (scattered stores, byte loads) took 94 us
// there, this 52.
#include <hip/hip_runtime.h>

#include "mxh_device.h"
#include "mxh_internal.h"
#include "mxh_quant.h"

namespace mxh {
namespace {

// loads and stores at any byte address (the entry point takes any w) and any
// float address
struct __attribute__((packed, aligned(1))) U16 { uint16_t v; };
struct __attribute__((packed, aligned(1))) U32 { uint32_t v; };
typedef uint32_t u32x2u __attribute__((ext_vector_type(2), aligned(1)));
typedef uint32_t u32x4u __attribute__((ext_vector_type(4), aligned(1)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

__device__ __forceinline__ uint32_t ld16(const uint8_t* p) { return reinterpret_cast<const U16*>(p)->v; }
__device__ __forceinline__ uint32_t ld32(const uint8_t* p) { return reinterpret_cast<const U32*>(p)->v; }
__device__ __forceinline__ float byte_f(uint32_t v, int i) { return (float)((v >> (8 * i)) & 0xffu); }
__device__ __forceinline__ float sbyte_f(uint32_t v, int i) { return (float)(int)(int8_t)(v >> (8 * i)); }

// the bytes elements 4 u .. 4 u + 3 of the run of blocks at w come from, and
// their values
template <int TYPE>
struct Quad {
    uint32_t q, h, s;
    u32x4u hd;
    __device__ __forceinline__ void load(const uint8_t* __restrict__ w, int64_t u) {
        if constexpr (TYPE == MXH_Q4_K || TYPE == MXH_Q5_K) {
            const int l = (int)(u & 63), j = l >> 3, i = 4 * (l & 7);
            const uint8_t* blk = w + (u >> 6) * (TYPE == MXH_Q4_K ? 144 : 176);
            hd = *reinterpret_cast<const u32x4u*>(blk);
            q = ld32(blk + (TYPE == MXH_Q4_K ? 16 : 48) + 32 * (j >> 1) + i);
            if constexpr (TYPE == MXH_Q5_K) h = ld32(blk + 16 + i);
        } else if constexpr (TYPE == MXH_Q6_K) {
            // element 128 hh + 32 g + i of the block
            const int l = (int)(u & 63), hh = l >> 5, g = (l >> 3) & 3, i = 4 * (l & 7);
            const uint8_t* blk = w + (u >> 6) * 210;
            q = ld32(blk + 64 * hh + 32 * (g & 1) + i);
            h = ld32(blk + 128 + 32 * hh + i);
            s = ld16(blk + 208) | (uint32_t)blk[192 + 8 * hh + 2 * g + (i >> 4)] << 16;
        } else if constexpr (TYPE == MXH_Q8_0) {
            const uint8_t* blk = w + (u >> 3) * 34;
            q = ld32(blk + 2 + 4 * (u & 7));
            s = ld16(blk);
        } else if constexpr (TYPE == MXH_Q5_0) {
            const uint8_t* blk = w + (u >> 3) * 22;
            q = ld32(blk + 6 + 4 * (u & 3));
            h = ld32(blk + 2);
            s = ld16(blk);
        } else if constexpr (TYPE == MXH_F16) {
            const u32x2u v = *reinterpret_cast<const u32x2u*>(w + 8 * u);
            q = v.x, h = v.y;
        } else {
            hd = *reinterpret_cast<const u32x4u*>(w + 16 * u);
        }
    }
    __device__ __forceinline__ f32x4u value(int64_t u, int form) const {
        f32x4u y;
        if constexpr (TYPE == MXH_Q4_K || TYPE == MXH_Q5_K) {
            const int j = (int)(u & 63) >> 3;
            uint32_t sc, mn;
            k4_scale_min(hd.y, hd.z, hd.w, j, form, sc, mn);
            const float ds = half_bits_to_float(hd.x & 0xffffu) * (float)sc;
            const float ms = half_bits_to_float(hd.x >> 16) * (float)mn;
            uint32_t c = (q >> (4 * (j & 1))) & 0x0f0f0f0fu;
            if constexpr (TYPE == MXH_Q5_K) c |= ((h >> j) & 0x01010101u) << 4;
#pragma unroll
            for (int e = 0; e < 4; ++e) y[e] = ds * byte_f(c, e) - ms;
        } else if constexpr (TYPE == MXH_Q6_K) {
            const int g = (int)(u >> 3) & 3;
            const uint32_t c = ((q >> (4 * (g >> 1))) & 0x0f0f0f0fu) | (((h >> (2 * g)) & 0x03030303u) << 4);
            const float ds = half_bits_to_float(s & 0xffffu) * (float)(int)(int8_t)(s >> 16);
#pragma unroll
            for (int e = 0; e < 4; ++e) y[e] = ds * (float)((int)((c >> (8 * e)) & 0xffu) - 32);
        } else if constexpr (TYPE == MXH_Q8_0) {
            const float d = half_bits_to_float(s);
#pragma unroll
            for (int e = 0; e < 4; ++e) y[e] = d * sbyte_f(q, e);
        } else if constexpr (TYPE == MXH_Q5_0) {
            const int i = 4 * (int)(u & 7);  // elements i .. i + 3; 16 on from the high nibbles
            const uint32_t c = (q >> (i >= 16 ? 4 : 0)) & 0x0f0f0f0fu;
            const float d = half_bits_to_float(s);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                y[e] = d * (float)((int)(((c >> (8 * e)) & 0xffu) | (((h >> (i + e)) & 1u) << 4)) - 16);
        } else if constexpr (TYPE == MXH_F16) {
            y[0] = half_bits_to_float(q & 0xffffu), y[1] = half_bits_to_float(q >> 16);
            y[2] = half_bits_to_float(h & 0xffffu), y[3] = half_bits_to_float(h >> 16);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) y[e] = __uint_as_float(hd[e]);
        }
        return y;
    }
};

constexpr int kThreads = 256, kAhead = 4;  // quads a thread has in flight

template <int TYPE>
__global__ __launch_bounds__(kThreads) void dequant_kernel(const uint8_t* __restrict__ w, float* __restrict__ out,
                                                           int64_t quads, int form) {
    for (int64_t u0 = (int64_t)blockIdx.x * (kThreads * kAhead) + threadIdx.x; u0 < quads;
         u0 += (int64_t)gridDim.x * (kThreads * kAhead)) {
        Quad<TYPE> b[kAhead];
#pragma unroll
        for (int a = 0; a < kAhead; ++a) {
            const int64_t u = u0 + a * kThreads;
            b[a].load(w, u < quads ? u : quads - 1);
        }
#pragma unroll
        for (int a = 0; a < kAhead; ++a) {
            const int64_t u = u0 + a * kThreads;
            if (u < quads) *reinterpret_cast<f32x4u*>(out + 4 * u) = b[a].value(u, form);
        }
    }
}

template <int TYPE>
void launch(const void* w, float* out, int64_t rows, int64_t cols, int form, hipStream_t st) {
    const int64_t quads = rows * (cols / 4), wgs = (quads + kThreads * kAhead - 1) / (kThreads * kAhead);
    const unsigned grid = (unsigned)(wgs < (1 << 22) ? wgs : 1 << 22);
    hipLaunchKernelGGL(dequant_kernel<TYPE>, dim3(grid), dim3(kThreads), 0, st, (const uint8_t*)w, out, quads, form);
}

}  // namespace

int dequant_launch(int type, const void* w, float* out, int64_t rows, int64_t cols, int form, hipStream_t st) {
    if (rows <= 0 || cols <= 0 || cols % 32 || row_bytes(type, cols) == 0) return MXH_ERR_ARG;
    switch (type) {
    case MXH_Q4_K: launch<MXH_Q4_K>(w, out, rows, cols, form, st); break;
    case MXH_Q5_K: launch<MXH_Q5_K>(w, out, rows, cols, form, st); break;
    case MXH_Q8_0: launch<MXH_Q8_0>(w, out, rows, cols, form, st); break;
    case MXH_Q5_0: launch<MXH_Q5_0>(w, out, rows, cols, form, st); break;
    case MXH_Q6_K: launch<MXH_Q6_K>(w, out, rows, cols, form, st); break;
    case MXH_F16: launch<MXH_F16>(w, out, rows, cols, form, st); break;
    case MXH_F32: launch<MXH_F32>(w, out, rows, cols, form, st); break;
    default: return MXH_ERR_UNSUPPORTED;
    }
    return MXH_OK;
}

}  // namespace mxh

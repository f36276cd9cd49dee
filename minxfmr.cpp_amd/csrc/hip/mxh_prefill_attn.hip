// mxh_prefill_attn.hip — causal attention of a chunk of prompt tokens on the
// fp16 matrix cores, in flash form (running reference and sum per query, no
// score matrix in memory).
//
// Reference op: the attention of transformer.cpp:529-629 for each prompt
// token (scores q.k / sqrt(hd) over cache positions 0 .. pos, softmax
// softmax.cpp:4-18, weighted sum of V rows), with the chunk's own K/V rows
// already appended to the fp16 cache by qkv_prep_rows_kernel.
//
// Workgroup (g, y, z) serves kv head g and 64 query rows: the `group` q heads
// of g for T = 64 / group consecutive tokens (row r = token r / group, head
// r % group), over split z of the keys.  Keys stream through LDS in stages of
// 64, double-buffered.  Wave w of four takes query rows 32 (w & 1) .. +32 and
// key half w >> 1 of every stage; the two waves of a query set see disjoint
// keys and merge their (reference, sum, V sum) at the end, the splits of a
// tile in a second kernel.  Per 32-key block a wave computes
//
//   S^T = K Q^T      v_mfma_f32_32x32x16_f16; q is pre-scaled by
//                    log2(e) / sqrt(hd) and split into fp16 hi + lo (about
//                    22 significant bits); K is exact (the cache is fp16)
//   O^T += V^T P^T   P = 64 2^(S - ref) split into fp16 hi + lo; V exact
//
// ref is the row's largest score when it was last set: it moves (and the sums
// are rescaled, all by one rounded factor) only where a score exceeds it by
// more than 8, which is rare.  The factor 64 keeps the low halves of small
// probabilities out of the fp16 subnormals, and P stays at most 2^14.  It is
// multiplied, not added to the exponent: 6 + (S - ref) would be rounded at the
// magnitude of 6 (rms error of near-equal probabilities 1.3e-7, 7.4e-8 so).
//
// Lane l owns query l % 32 in both products (accumulator register i of lane l
// is row 8 (i / 4) + 4 (l / 32) + i % 4, column l % 32), so the softmax
// statistics are per lane; lanes l and l ^ 32 hold the two halves of a
// block's keys for the same query.  The K rows enter the first product in
// the order pi (bits 2 and 3 of the row index swapped), which puts keys
// 16 s + 8 (l / 32) .. +8 in registers 8 s .. 8 s + 7 of lane l: the B
// operand of k step s of the second product, with no exchange between lanes.
//
// LDS per stage: K as [64 keys][hd] with the 16-byte pieces of a row rotated
// by an XOR of the key (conflict-free first-product reads), and V transposed
// as [hd][64 + 8 keys] (a lane's 8 keys contiguous; the 144-byte row stride
// spreads 16 rows over all banks; no bank conflicts measured).  The next
// stage's global loads are in flight during the current stage's products.
//
// Bound: a block's 32 MFMAs (1,024 cycles at head dim 128) and its softmax
// (165 vector instructions, about 850 cycles) follow each other in a wave, and
// the two waves of a SIMD keep in step, so their times add up (counters at 512
// queries at 7680: matrix cores busy 48%, vector ALU 45%).  So the vector work
// was cut: the reference that seldom moves, one-instruction splits, loads
// without masks.  228 -> 156 us there; the first product one block ahead needs
// more registers than there are (spills, 258 us), wave priorities change
// nothing.  Few queries at long positions were a few workgroups' serial walk
// over the keys: they split them (see the launch).
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include "mxh_device.h"
#include "mxh_internal.h"
#include "mxh_plan.h"

namespace mxh {

namespace {

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kPaRows = 64;        // query rows per workgroup
constexpr float kPaScale = 64.f, kPaSlack = 8.f;  // P at most scale 2^slack

constexpr int kPaKeys = 64;        // keys per stage
constexpr int kPaThreads = 256;
constexpr int kPaVst = kPaKeys + 8;  // transposed V row stride (halves)

__host__ __device__ constexpr int pa_stage_halves(int hd) { return kPaKeys * hd + hd * kPaVst; }
// floats a wave leaves for the merge: V sums [hd][32], references, sums
__host__ __device__ constexpr int pa_merge_floats(int hd) { return hd * 32 + 64; }
__host__ __device__ constexpr size_t pa_lds_bytes(int hd) {
    const size_t st = (size_t)2 * pa_stage_halves(hd) * 2, mg = (size_t)4 * pa_merge_floats(hd) * 4;
    return st > mg ? st : mg;
}

// row m of a 32-key block -> key (bits 2 and 3 swapped)
__device__ __forceinline__ int pa_pi(int m) { return (m & ~12) | ((m & 4) << 1) | ((m & 8) >> 1); }

template <int HD>
__device__ __forceinline__ int pa_swz(int key) {
    constexpr int NCH = HD / 8, RS = HD == 128 ? 0 : HD == 64 ? 1 : 2;  // rows per 256 bytes = 1 << RS
    return (key >> RS) & (NCH - 1);
}

// the larger / the sum of a value in lanes l and l ^ 32, in both
__device__ __forceinline__ float pa_pair_max(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// p - h[HALF] in one instruction (written as C++ it is a conversion and a
// subtraction; exact)
template <int HALF>
__device__ __forceinline__ float pa_rest(float p, f16x2 h) {
    float d;
    if constexpr (HALF) asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(d) : "v"(h), "v"(p));
    else asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(d) : "v"(h), "v"(p));
    return d;
}

// a and b as fp16 hi + lo, both rounded to nearest (one instruction for a
// pair): cut off, a probability's halves left the V sums 7e-8 to 9e-8 low
// against lrun.  hi is made opaque: where a is a product the compiler would
// round it to fp16 in one step for lo and in two for hi, and where the two
// differ (one in some thousand q values) lo repairs an error that hi does not
// have (rms error of 200 queries at 0, 32/8 heads of 128: 4.1e-6).
__device__ __forceinline__ void pa_split(float a, float b, f16x2& hi, f16x2& lo) {
    hi = __builtin_convertvector((f32x2{a, b}), f16x2);
    asm("" : "+v"(hi));
    lo = __builtin_convertvector((f32x2{pa_rest<0>(a, hi), pa_rest<1>(b, hi)}), f16x2);
}

// One split's part of one row: V sums part[p][row][hd] and (reference, sum)
// ml[p][row], p = (tile nkv + g) splits + z
template <int HD>
__global__ __launch_bounds__(kPaThreads, 2) void attention_rows_mfma_kernel(
    const float* __restrict__ q, const __half* __restrict__ kc, const __half* __restrict__ vc,
    float* __restrict__ att, float* __restrict__ part, float2* __restrict__ ml, int p0, int m, int nh, int nkv,
    float qscale, int split_stages) {
    constexpr int NCH = HD / 8, KS = HD / 16, DB = HD / 32;
    constexpr int NKL = kPaKeys * NCH / kPaThreads;  // K pieces per thread per stage
    constexpr int NVB = kPaKeys / 4 * NCH;           // 4-key x 8-dim V blocks per stage
    static_assert(NKL * kPaThreads == kPaKeys * NCH && NVB <= kPaThreads, "");
    extern __shared__ __align__(16) _Float16 pa_smem[];

    const int g = blockIdx.x, group = nh / nkv, T = kPaRows / group;
    const int tile = gridDim.y - 1 - blockIdx.y;  // the tiles with the most keys start first
    const int t0 = tile * T;
    const int kvd = nkv * HD, qd = nh * HD;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int qg = wave & 1, kh = wave >> 1, n = lane & 31, h = lane >> 5;

    const int tmax = min(t0 + T, m) - 1;
    const int kend = p0 + tmax + 1;             // keys [0, kend) for the tile
    const int lim_min = p0 + t0 + 1;            // smallest per-row limit
    const int st0 = blockIdx.z * split_stages;
    const int nst = min((kend + kPaKeys - 1) / kPaKeys, st0 + split_stages);
    const size_t prt = ((size_t)tile * nkv + g) * gridDim.z + blockIdx.z;
    if (st0 >= nst) {  // no keys of this tile in the split
        if (tid < kPaRows) ml[prt * kPaRows + tid] = make_float2(-INFINITY, 0.f);
        return;
    }

    // this lane's query row
    const int r = 32 * qg + n, tl = r / group, hh = r % group, tok = t0 + tl;
    const bool valid = r < T * group && tok < m;
    const int lim = valid ? p0 + tok + 1 : lim_min;

    f16x8 qh[KS], ql[KS];
    {
        const float* qp = q + (size_t)tok * qd + (size_t)(g * group + hh) * HD;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            float v[8];
            if (valid) {
                const float4 a = *reinterpret_cast<const float4*>(qp + 16 * ks + 8 * h);
                const float4 b = *reinterpret_cast<const float4*>(qp + 16 * ks + 8 * h + 4);
                v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = 0.f;
            }
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                f16x2 hi, lo;
                pa_split(v[e] * qscale, v[e + 1] * qscale, hi, lo);
                qh[ks][e] = hi[0], qh[ks][e + 1] = hi[1], ql[ks][e] = lo[0], ql[ks][e + 1] = lo[1];
            }
        }
    }

    // stage loads: K pieces (key, 16-byte chunk) and V blocks (4 keys x 8
    // dims); keys past the last repeat it (their scores are masked)
    u32x4 kraw[NKL], vraw[4];
    const uint32_t row_b = 2u * (uint32_t)kvd;
    const int kk = tid / NCH, kcb = 16 * (tid % NCH);
    const int vk = 4 * (tid & 15), vcol = tid >> 4;
    const auto load = [&](int st) __attribute__((always_inline)) {
        const int last = kend - 1 - st * kPaKeys;  // (uniform)
        const size_t at = ((size_t)st * kPaKeys * kvd + (size_t)g * HD) * 2;
        const uint8_t *ks = reinterpret_cast<const uint8_t*>(kc) + at, *vs = reinterpret_cast<const uint8_t*>(vc) + at;
#pragma unroll
        for (int u = 0; u < NKL; ++u)
            kraw[u] = *reinterpret_cast<const u32x4*>(ks + (uint32_t)min(kk + kPaThreads / NCH * u, last) * row_b + kcb);
        if (NVB == kPaThreads || tid < NVB) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                vraw[i] = *reinterpret_cast<const u32x4*>(vs + (uint32_t)min(vk + i, last) * row_b + 16 * vcol);
        }
    };
    const auto store = [&](int buf) __attribute__((always_inline)) {
        _Float16* Ks = pa_smem + buf * pa_stage_halves(HD);
        _Float16* Vt = Ks + kPaKeys * HD;
#pragma unroll
        for (int u = 0; u < NKL; ++u) {
            const int key = kk + kPaThreads / NCH * u;
            *reinterpret_cast<u32x4*>(Ks + key * HD + 8 * (tid % NCH ^ pa_swz<HD>(key))) = kraw[u];
        }
        if (NVB == kPaThreads || tid < NVB) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const uint32_t sel = e & 1 ? 0x07060302u : 0x05040100u;  // the high or the low halves of two words
                *reinterpret_cast<uint2*>(Vt + (8 * vcol + e) * kPaVst + vk) =
                    make_uint2(__builtin_amdgcn_perm(vraw[1][e >> 1], vraw[0][e >> 1], sel),
                               __builtin_amdgcn_perm(vraw[3][e >> 1], vraw[2][e >> 1], sel));
            }
        }
    };

    load(st0);
    store(st0 & 1);
    if (st0 + 1 < nst) load(st0 + 1);
    __syncthreads();

    float mref = -INFINITY, lrun = 0.f;
    f32x16 o[DB];
#pragma unroll
    for (int d = 0; d < DB; ++d)
#pragma unroll
        for (int v = 0; v < 16; ++v) o[d][v] = 0.f;
    const int krow = 32 * kh + pa_pi(n);

    for (int st = st0; st < nst; ++st) {
        const _Float16* Ks = pa_smem + (st & 1) * pa_stage_halves(HD);
        const _Float16* Vt = Ks + kPaKeys * HD;
        const int kb = st * kPaKeys + 32 * kh;  // first key of this wave's block
        if (kb < kend) {
            f32x16 s;
#pragma unroll
            for (int v = 0; v < 16; ++v) s[v] = 0.f;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                const f16x8 a =
                    *reinterpret_cast<const f16x8*>(Ks + krow * HD + 8 * ((2 * ks + h) ^ pa_swz<HD>(krow)));
                s = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, qh[ks], s, 0, 0, 0);
                s = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, ql[ks], s, 0, 0, 0);
            }
            if (kb + 31 >= lim_min) {
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    if (kb + 16 * (v >> 3) + 8 * h + (v & 7) >= lim) s[v] = -INFINITY;
            }
            float mx = s[0];
#pragma unroll
            for (int v = 1; v < 16; ++v) mx = fmaxf(mx, s[v]);
            mx = pa_pair_max(mx);
            if (__any(mx > mref + kPaSlack)) {  // also the first block with an unmasked key
                const float mnew = fmaxf(mref, mx);
                // (every key masked so far: the sums are zero)
                const float alpha = mref == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mref - mnew);
                mref = mnew;
                lrun *= alpha;
#pragma unroll
                for (int d = 0; d < DB; ++d)
#pragma unroll
                    for (int v = 0; v < 16; ++v) o[d][v] *= alpha;
            }
            const float ref0 = mref == -INFINITY ? 0.f : mref;
            float p[16], ps[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                p[v] = kPaScale * __builtin_amdgcn_exp2f(s[v] - ref0);
                ps[v & 3] += p[v];
            }
            lrun += (ps[0] + ps[1]) + (ps[2] + ps[3]);
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                f16x8 bh, bl;
#pragma unroll
                for (int u = 0; u < 8; u += 2) {
                    f16x2 hi, lo;
                    pa_split(p[8 * t + u], p[8 * t + u + 1], hi, lo);
                    bh[u] = hi[0], bh[u + 1] = hi[1], bl[u] = lo[0], bl[u + 1] = lo[1];
                }
#pragma unroll
                for (int d = 0; d < DB; ++d) {
                    const f16x8 a =
                        *reinterpret_cast<const f16x8*>(Vt + (32 * d + n) * kPaVst + 32 * kh + 16 * t + 8 * h);
                    o[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, bh, o[d], 0, 0, 0);
                    o[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, bl, o[d], 0, 0, 0);
                }
            }
        }
        if (st + 1 < nst) store((st + 1) & 1);
        __syncthreads();
        if (st + 2 < nst) load(st + 2);
    }

    // merge the two key halves of each query set (stage buffers are free now)
    const float lsum = lrun + __shfl_xor(lrun, 32, 64);
    float* ms = reinterpret_cast<float*>(pa_smem);
    {
        float* mb = ms + wave * pa_merge_floats(HD);
#pragma unroll
        for (int d = 0; d < DB; ++d)
#pragma unroll
            for (int v = 0; v < 16; ++v) mb[(32 * d + 8 * (v >> 2) + 4 * h + (v & 3)) * 32 + n] = o[d][v];
        if (h == 0) {
            mb[HD * 32 + n] = mref;
            mb[HD * 32 + 32 + n] = lsum;
        }
    }
    __syncthreads();
    // thread: row 32 mq + mn, dims d0 .. d0 + ND
    constexpr int ND = HD / 4;
    const int mq = tid >> 7, mn = tid & 31, d0 = ((tid >> 5) & 3) * ND;
    const float* mb[2];
    float a[2], M = -INFINITY, L = 0.f;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        mb[i] = ms + (2 * i + mq) * pa_merge_floats(HD);
        M = fmaxf(M, mb[i][HD * 32 + mn]);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const float mi = mb[i][HD * 32 + mn];
        a[i] = mi == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mi - M);  // (no key of the row in that half)
        L += a[i] * mb[i][HD * 32 + 32 + mn];
    }
    const int row = 32 * mq + mn, mtok = t0 + row / group;
    float* op;
    float inv = 1.f;
    if (gridDim.z > 1) {
        op = part + (prt * kPaRows + row) * HD;
        if (d0 == 0) ml[prt * kPaRows + row] = make_float2(M, L);
    } else {
        if (row >= T * group || mtok >= m) return;
        op = att + (size_t)mtok * qd + (size_t)(g * group + row % group) * HD;
        inv = 1.0f / L;
    }
#pragma unroll
    for (int d = 0; d < ND; d += 4) {
        float w[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int at = (d0 + d + e) * 32 + mn;
            w[e] = (a[0] * mb[0][at] + a[1] * mb[1][at]) * inv;
        }
        *reinterpret_cast<float4*>(op + d0 + d) = make_float4(w[0], w[1], w[2], w[3]);
    }
}

// att from the splits' parts; a thread takes four dims of one row
template <int HD>
__global__ __launch_bounds__(256) void attention_rows_merge_kernel(const float* __restrict__ part,
                                                                   const float2* __restrict__ ml,
                                                                   float* __restrict__ att, int m, int nh, int nkv,
                                                                   int splits, int rows) {
    const int u = blockIdx.x * 256 + threadIdx.x, d = 4 * (u % (HD / 4)), wr = u / (HD / 4);  // row of all tiles
    if (wr >= rows) return;
    const int group = nh / nkv, T = kPaRows / group, row = wr % kPaRows, wg = wr / kPaRows;
    const int g = wg % nkv, tok = wg / nkv * T + row / group;
    if (row >= T * group || tok >= m) return;
    const size_t p = (size_t)wg * splits;
    float M = -INFINITY, L = 0.f;
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
    constexpr int kAhead = 8;  // splits whose loads are in flight together
    for (int z0 = 0; z0 < splits; z0 += kAhead) {
        float2 t[kAhead];
        float4 v[kAhead];
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            const size_t at = (p + min(z0 + i, splits - 1)) * kPaRows + row;
            t[i] = ml[at];
            v[i] = *reinterpret_cast<const float4*>(part + at * HD + d);
        }
        float m1 = M;
#pragma unroll
        for (int i = 0; i < kAhead; ++i) m1 = fmaxf(m1, t[i].x);
        const float a0 = M == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(M - m1);  // (split 0 holds key 0: m1 is finite)
        M = m1;
        L *= a0, s.x *= a0, s.y *= a0, s.z *= a0, s.w *= a0;
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            if (z0 + i >= splits || t[i].x == -INFINITY) continue;  // no key of the row in that split
            const float a = __builtin_amdgcn_exp2f(t[i].x - M);
            L += a * t[i].y;
            s.x += a * v[i].x, s.y += a * v[i].y, s.z += a * v[i].z, s.w += a * v[i].w;
        }
    }
    const float inv = 1.0f / L;
    *reinterpret_cast<float4*>(att + (size_t)tok * nh * HD + (size_t)(g * group + row % group) * HD + d) =
        make_float4(s.x * inv, s.y * inv, s.z * inv, s.w * inv);
}

template <int HD>
int attention_rows_mfma_launch_hd(const float* q, const __half* kc, const __half* vc, float* att, int p0, int m,
                                  int nh, int nkv, float qscale, float* part, size_t part_bytes, hipStream_t st) {
    static bool attr_set = false;  // above 64 KiB of LDS needs the opt-in, once per kernel
    if (!attr_set) {
        if (hipFuncSetAttribute((const void*)attention_rows_mfma_kernel<HD>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)pa_lds_bytes(HD)) != hipSuccess)
            return MXH_ERR_HIP;
        attr_set = true;
    }
    const int T = kPaRows / (nh / nkv), tiles = (m + T - 1) / T;
    const int64_t wgs = (int64_t)nkv * tiles;
    const AttnPlan plan = attention_plan(HD, wgs, (int)(((int64_t)p0 + m + kPaKeys - 1) / kPaKeys),
                                         (size_t)kPaRows * (HD + 2) * 4, device_cus(), part ? part_bytes : 0);
    const int splits = plan.splits, per = plan.stages;
    // (used with splits > 1 only)
    float2* ml = part ? reinterpret_cast<float2*>(part + (size_t)wgs * splits * kPaRows * HD) : nullptr;
    hipLaunchKernelGGL(attention_rows_mfma_kernel<HD>, dim3((unsigned)nkv, (unsigned)tiles, (unsigned)splits),
                       dim3(kPaThreads), pa_lds_bytes(HD), st, q, kc, vc, att, part, ml, p0, m, nh, nkv, qscale, per);
    if (splits > 1) {
        const int rows = (int)wgs * kPaRows;
        hipLaunchKernelGGL(attention_rows_merge_kernel<HD>, dim3((unsigned)((rows * (HD / 4) + 255) / 256)), dim3(256),
                           0, st, part, ml, att, m, nh, nkv, splits, rows);
    }
    return MXH_OK;
}

}  // namespace

int attention_rows_mfma_launch(const float* q, const __half* kc, const __half* vc, float* att, int p0, int m, int nh,
                               int nkv, int hd, float scale, float* part, size_t part_bytes, hipStream_t st) {
    if (m <= 0 || p0 < 0 || !attention_supported(nh, nkv, hd)) return MXH_ERR_ARG;
    const float qscale = scale * 1.4426950408889634f;  // scores in base-2 units
    switch (hd) {
    case 32: return attention_rows_mfma_launch_hd<32>(q, kc, vc, att, p0, m, nh, nkv, qscale, part, part_bytes, st);
    case 64: return attention_rows_mfma_launch_hd<64>(q, kc, vc, att, p0, m, nh, nkv, qscale, part, part_bytes, st);
    default: return attention_rows_mfma_launch_hd<128>(q, kc, vc, att, p0, m, nh, nkv, qscale, part, part_bytes, st);
    }
}

}  // namespace mxh

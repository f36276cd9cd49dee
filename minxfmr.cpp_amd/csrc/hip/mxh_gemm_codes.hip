// mxh_gemm_codes.hip — the prefill GEMM over quantized rows on the fp16
// matrix cores, pipelined through LDS, every weight exact.
//
// out[m][n] = sum_k a[m][k] w[n][k].  The weights enter the matrix cores as
// integer codes that fp16 holds exactly, the block scales meet fp32 partial
// sums (reference op: backend_matmul_rhs_transposed with m > 1,
// src/backend/backend_runtime.cpp:302-319; decoders tensor.cpp:395-457 and
// gguf_reader.cpp:905-1008):
//
//   Q4_K, Q5_K  w = d sc_j q - dmin m_j: codes sc_j q (< 2048), d per
//               256-element block; the min terms are a second contraction
//               over the activations' sub-block sums, eight per block.
//   Q8_0, Q5_0  w = d q: codes q (Q5_0: q - 16), d per 32-element block.
//   Q6_K        w = d sc_j (q - 32): sc_j (q - 32) needs 13 bits, so it is a
//               pair of codes, the fp16 rounding Wh and the exact rest Wl;
//               d per 256-element block.  Wl . a_lo, below 2^-23 of the
//               product, is not formed.
//
// Activations come as a 2^e (e per row) split into fp16 hi + lo (about 22
// bits, rows_to_f16), each four consecutive elements stored in the order
// 0 2 1 3: the order in which masking a dword of codes with 0x000f000f (and
// the same dword shifted by a byte) leaves pairs of fp16.
//
// Shape of the kernel.  8 waves, one workgroup per CU: WM along the
// activation rows x WN = 8 / WM along the weight rows, each wave 32 MI x
// 32 NJ outputs of v_mfma_f32_32x32x16_f16.  A K step is 64 elements.  The
// activations of a step and the raw weight bytes of a granule (two or four
// steps) go straight into LDS (global_load_lds_dwordx4), one barrier per step;
// every wave decodes the weight rows it multiplies itself, from LDS.  The
// granule is there for the memory pipe: a load whose lanes read 16 bytes of 64
// different rows takes about 60 ns of a CU on a full chip, a quarter of that
// when four lanes share 64 consecutive bytes (codes loaded a step at a time:
// 2241 against 2156 ns per 128 x 256 step, 907 against 675 per 32 x 256).
//
// What bounds it.  Per 128 x 256 x 64 step a SIMD has 2048 cycles of matrix
// work (two products) and about 130 VALU instructions per wave (1040 cycles):
// a wave's load addresses are scalar (a base in SGPRs plus a fixed lane
// offset), block headers are read once per 256 elements, a code pair costs one
// and-or and one packed fma, the min terms are formed in the registers of the
// lane that multiplies them, and the partial sums restart with a zero operand
// instead of being cleared.  (Decoding each code alone, with addresses and
// headers per step, cost about 330 per wave.)
//
// Measured (one MI355X, this kernel against a 128-row-tile kernel for Q4_K
// and an unpipelined one for the other types): Q4_K 512 x 24576 x 4096
// 283 -> 238 us, 512 x 4096 x 12288 at 104 us (498 TFLOP/s, 996 issued; a bf16
// library product of 8192^3 reaches 1200), Q5_K 129 x 4096 x 14336
// 665 -> 72 us, Q8_0 31 x 6144 x 1024 33 -> 16 us with the conversion of the
// rows.
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "mxh_device.h"
#include "mxh_gemm_f16.h"
#include "mxh_internal.h"

namespace mxh {

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 512;

// keeps the loads of a region ahead of its arithmetic in the instruction order
#define MXH_CODES_FENCE() __builtin_amdgcn_sched_barrier(0)

// 16 bytes per lane from global memory into LDS (lane i writes lds + 16 i):
// scalar base + lane offset, or a full lane address.  Inline assembly so that
// the compiler does not wait for every such load before the next LDS read (it
// cannot tell the stages apart); wait_vm waits for them.  The compiler does
// not see a memory instruction here, so the wait states between a VALU write
// of the base's SGPRs (5) or a write of M0 (1) and the load are in the asm.
__device__ __forceinline__ void g2l_s(uint64_t base, uint32_t off, uint32_t lds) {
    asm volatile("s_nop 4\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "{m0}"(lds) : "memory");
}
__device__ __forceinline__ void g2l_v(const void* addr, uint32_t lds) {
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(addr), "{m0}"(lds) : "memory");
}
// 4 bytes per lane (lane i writes lds + 4 i)
__device__ __forceinline__ void g2l4_s(uint64_t base, uint32_t off, uint32_t lds) {
    asm volatile("s_nop 4\n\tglobal_load_lds_dword %0, %1" ::"v"(off), "s"(base), "{m0}"(lds) : "memory");
}
// a uniform address, held in SGPRs
__device__ __forceinline__ uint64_t scalar_addr(const void* p) {
    const uint64_t v = (uint64_t)p;
    // (the builtin returns int: back to unsigned before widening)
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
    return ((uint64_t)hi << 32) | lo;
}

template <int N>
__device__ __forceinline__ void wait_vm() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    // vmcnt in bits 3:0 and 15:14; expcnt and lgkmcnt left at their maxima
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// LDS operations of this wave complete, then the workgroup barrier, with no
// wait for the global loads in flight
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

__device__ __forceinline__ f16x2 as_h2(uint32_t v) { return __builtin_bit_cast(f16x2, v); }
__device__ __forceinline__ uint32_t as_u(f16x2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ f16x2 splat(_Float16 v) { return f16x2{v, v}; }
__device__ __forceinline__ float half_lo(uint32_t v) { return (float)as_h2(v)[0]; }
__device__ __forceinline__ float half_hi(uint32_t v) { return (float)as_h2(v)[1]; }

constexpr uint32_t kMagic = 0x64006400u;  // fp16 1024: its low mantissa bits count units

// (v & mask) | magic in one instruction: at most one of the constants can be
// a scalar operand, so the compiler splits it in two when it sees both
__device__ __forceinline__ uint32_t code_pair(uint32_t v, uint32_t mask, uint32_t magic) {
    uint32_t r;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(v), "s"(mask), "v"(magic));
    return r;
}

// v << s for s >= 0, v >> -s otherwise
template <int S>
__device__ __forceinline__ uint32_t shl(uint32_t v) {
    if constexpr (S >= 0) return v << S;
    else return v >> -S;
}

__device__ __forceinline__ f16x8 pack8(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    return __builtin_bit_cast(f16x8, u32x4{a, b, c, d});
}

// ---- weight formats --------------------------------------------------------
// The codes of a row arrive in granules of kGR steps (64 elements each): kNT
// runs of kNC 16-byte pieces that lie side by side in the row, so that a load
// instruction reads 16 kNC consecutive bytes per row.  Piece p of step s of a
// granule is piece chunk(s, p) of run type(p).  kH 16-byte header pieces per
// row and 256-element block.  q_off / h_off: the runs' and headers' byte
// offsets in a row of nblk 256-element blocks; they are the same for every row
// and 32-bit, so they are scalar arithmetic (the tiled orders are those of
// mxh_types.h).  kQL: dwords of codes a lane reads per weight row and step;
// slice_chunk: the activation chunk (aoff) of slice sl of half-step h; kPair: a
// half-step is a whole 32-element block with its own d.
template <int F>
struct Fmt;

// blocks in tile j of tiles of T blocks
template <int T>
__device__ __forceinline__ uint32_t tile_blocks(uint32_t j, uint32_t nblk) {
    const uint32_t left = nblk - T * j;
    return left < T ? left : T;
}

struct FmtK {  // a 64-element group: low then high nibbles of 16 code bytes per lane half
    static constexpr bool kMin = true, kSplitW = false, kRuns = false, kPair = false;
    static constexpr int kQL = 4, kGR = 4;
    static __host__ __device__ constexpr int slice_chunk(int half, int sl) { return half + 2 * sl; }
};
struct FmtKRow : FmtK {  // a block's 128 code bytes side by side
    static constexpr int kNT = 1, kNC = 8;
    static __device__ __forceinline__ int type(int) { return 0; }
    static __device__ __forceinline__ int chunk(int s, int p) { return 2 * s + p; }
};

template <>
struct Fmt<GF_Q4K> : FmtKRow {
    static constexpr int kType = MXH_Q4_K, kH = 1;
    static __device__ __forceinline__ uint32_t q_off(uint32_t b, uint32_t, uint32_t) { return b * 144 + 16; }
    static __device__ __forceinline__ uint32_t h_off(uint32_t b, uint32_t, uint32_t) { return b * 144; }
};
template <>
struct Fmt<GF_Q4KT> : FmtK {
    static constexpr int kType = MXH_Q4_K, kH = 1, kNT = 2, kNC = 4;
    static __device__ __forceinline__ int type(int p) { return p; }
    static __device__ __forceinline__ int chunk(int s, int) { return s; }
    static __device__ __forceinline__ uint32_t q_off(uint32_t b, uint32_t t, uint32_t nblk) {
        const uint32_t j = b >> 4, nb = tile_blocks<16>(j, nblk);
        return j * 2304 + 16 * (nb + 4 * (b & 15) + 4 * nb * t);
    }
    static __device__ __forceinline__ uint32_t h_off(uint32_t b, uint32_t, uint32_t) {
        return (b >> 4) * 2304 + 16 * (b & 15);
    }
};
template <>
struct Fmt<GF_Q5K> : FmtKRow {
    static constexpr int kType = MXH_Q5_K, kH = 3;
    static __device__ __forceinline__ uint32_t q_off(uint32_t b, uint32_t, uint32_t) { return b * 176 + 48; }
    static __device__ __forceinline__ uint32_t h_off(uint32_t b, uint32_t p, uint32_t) { return b * 176 + 16 * p; }
};
template <>
struct Fmt<GF_Q5KT> : FmtKRow {
    static constexpr int kType = MXH_Q5_K, kH = 3;
    static __device__ __forceinline__ uint32_t q_off(uint32_t b, uint32_t, uint32_t nblk) {
        const uint32_t j = b >> 3;
        return j * 1408 + 16 * (3 * tile_blocks<8>(j, nblk) + 8 * (b & 7));
    }
    static __device__ __forceinline__ uint32_t h_off(uint32_t b, uint32_t p, uint32_t nblk) {
        const uint32_t j = b >> 3, l = b & 7;
        return j * 1408 + (p == 0 ? 16 * l : 16 * tile_blocks<8>(j, nblk) + 32 * l + 16 * (p - 1));
    }
};

// a step is two 32-element blocks, pieces (first, last 16 codes) of each; a
// granule is four of them; the header is the eight fp16 d of 256 elements
template <>
struct Fmt<GF_Q80T> {
    static constexpr int kType = MXH_Q8_0, kH = 1, kQL = 8, kGR = 2, kNT = 2, kNC = 4;
    static constexpr bool kMin = false, kSplitW = false, kRuns = false, kPair = true;
    static __host__ __device__ constexpr int slice_chunk(int half, int sl) { return 2 * half + sl; }
    static __device__ __forceinline__ int type(int p) { return p & 1; }
    static __device__ __forceinline__ int chunk(int s, int p) { return 2 * s + (p >> 1); }
    static __device__ __forceinline__ uint32_t q_off(uint32_t gr, uint32_t t, uint32_t nblk) {
        const uint32_t j = gr >> 4;
        return j * 2176 + 16 * (4 * (gr & 15) + t * tile_blocks<64>(j, 8 * nblk));
    }
    static __device__ __forceinline__ uint32_t h_off(uint32_t b, uint32_t, uint32_t nblk) {
        const uint32_t j = b >> 3;
        return j * 2176 + 32 * tile_blocks<64>(j, 8 * nblk) + 16 * (b & 7);
    }
};

// Q8_0 and Q5_0 rows in GGUF order: eight blocks are 272 (Q8_0) or 176 (Q5_0) bytes, so rows
// and every eighth block are 16-byte aligned.  A granule of four blocks comes
// as the 16-byte pieces that hold it, d and all; an odd one starts 8 bytes
// into its first piece.  Read in place since regrouping them into the tiled
// order first cost a read and a write of the weights: Q8_0 2 x 30000 x 14336
// 725 us so, 149 in place; 200 x 24576 x 4096 279 and 142 (tiled rows 127).
template <int BLOCK>
struct FmtBlock32 {
    static constexpr int kH = 0, kGR = 2, kNT = 1, kNC = (4 * BLOCK + 15) / 16, kBlock = BLOCK;
    static constexpr bool kMin = false, kSplitW = false, kRuns = false, kPair = true;
    static __host__ __device__ constexpr int slice_chunk(int half, int sl) { return 2 * half + sl; }
    static __device__ __forceinline__ int type(int) { return 0; }
    static __device__ __forceinline__ int chunk(int, int p) { return p; }
    static __device__ __forceinline__ uint32_t q_off(uint32_t gr, uint32_t, uint32_t) {
        return (gr >> 1) * (8 * BLOCK) + (gr & 1) * (4 * BLOCK - 8);
    }
    // byte of block `half` of step g of its 256 elements, in its granule's pieces
    static __host__ __device__ constexpr int block_at(int g, int half) {
        return 8 * (g >> 1) + BLOCK * (2 * (g & 1) + half);
    }
};
template <>
struct Fmt<GF_Q80> : FmtBlock32<34> {
    static constexpr int kType = MXH_Q8_0, kQL = 10;
};
template <>
struct Fmt<GF_Q50> : FmtBlock32<22> {
    static constexpr int kType = MXH_Q5_0, kQL = 12;
};

// a step is a 64-element chunk of the tiled layout: four runs of 16 elements
// (kRuns: 32 apart), so the activations are staged in that order
template <>
struct Fmt<GF_Q6KT> {
    static constexpr int kType = MXH_Q6_K, kH = 1, kQL = 6, kGR = 2, kNT = 3, kNC = 2;
    static constexpr bool kMin = false, kSplitW = true, kRuns = true, kPair = false;
    static __host__ __device__ constexpr int slice_chunk(int half, int sl) { return 2 * half + sl; }
    static __device__ __forceinline__ int type(int p) { return p; }
    static __device__ __forceinline__ int chunk(int s, int) { return s; }
    static __device__ __forceinline__ uint32_t q_off(uint32_t gr, uint32_t t, uint32_t nblk) {
        const uint32_t j = gr >> 5;
        return j * 3360 + 16 * (4 * tile_blocks<16>(j, nblk) * t + 2 * (gr & 31));
    }
    static __device__ __forceinline__ uint32_t h_off(uint32_t b, uint32_t, uint32_t nblk) {
        const uint32_t j = b >> 4;
        return j * 3360 + 192 * tile_blocks<16>(j, nblk) + 16 * (b & 15);
    }
    // the dword holding d of blocks b & ~1 and b | 1 (rows hold a multiple of eight blocks)
    static __device__ __forceinline__ uint32_t d_off(uint32_t b, uint32_t nblk) {
        const uint32_t j = b >> 4;
        return j * 3360 + 208 * tile_blocks<16>(j, nblk) + 2 * (b & 14);
    }
};

// ---- geometry ----------------------------------------------------------------
// Activations are staged per step, NST slots; codes per granule and headers
// (with the sub-block sums) per block, two slots each.  Slots are refilled at
// the end of a step: the activations of step t + NST at the end of step t,
// the next granule at the end of its predecessor's first step.
template <int F, int WM, int MI, int NJ, int NST>
struct Geo {
    using FM = Fmt<F>;
    static constexpr int WN = 8 / WM, BM = 32 * MI * WM, BN = 32 * NJ * WN;
    static constexpr int kA = BM * 256;                   // activation bytes of a stage (hi, lo)
    static constexpr int kAL = BM / 32;                   // direct loads per wave: activations of a stage,
    static constexpr int kWN = FM::kNT * FM::kNC * BN;    // (pieces of a granule)
    static constexpr int kWL = (kWN + 511) / 512;         // codes of a granule,
    static constexpr int kHN = FM::kH * BN + (FM::kMin ? 2 * BM : 0);
    static constexpr int kHL = (kHN + 511) / 512;         // headers and sub-block sums of a block,
    static constexpr int kDL = FM::kSplitW ? 1 : 0;       // 4-byte loads of d (Q6_K)
    static constexpr int kW = kWN * 16, kHdr = kHN * 16 + kDL * 2048;
    static constexpr size_t kLds = (size_t)NST * kA + 2 * (size_t)kW + 2 * (size_t)kHdr;
    // codes before or after the activations of the same refill: before where
    // the wait for the activations that follow must cover them
    static constexpr bool kWFirst = FM::kGR == 2 || NST > 2;
    static_assert(NST >= 2 && NST <= (FM::kGR == 2 ? 2 : 4), "a granule arrives before its first step");
    static_assert(kLds <= 160 * 1024, "LDS of a CU");
    static_assert(kHN % 64 == 0 && BN % 64 == 0 && BM % 32 == 0, "a wave's pieces are of one kind");
    // direct loads of codes and headers issued at the end of step s (s mod 4 counts)
    static constexpr int wloads(int s) {
        return s % FM::kGR == 0 ? kWL + ((s + FM::kGR) % 4 == 0 ? kHL + kDL : 0) : 0;
    }
    // loads issued after the activations of step t + 1 and in flight when they
    // are awaited at the end of step t
    static constexpr int ahead(int t) {
        int n = kWFirst ? 0 : wloads(t + 1 - NST + 4);
        for (int s = t + 2 - NST; s <= t - 1; ++s) n += kAL + wloads(s + 4);
        return n;
    }
};

// XOR of the 16-byte chunk index of activation row `row` (conflict-free
// operand reads: 8 consecutive rows take 8 different chunk slots)
__device__ __forceinline__ int a_swz(int row) { return (row & 7) ^ ((row >> 3) & 1); }

// XOR of the piece index of weight row `row` in a run of NC pieces (rows of
// nine or six pieces spread over the banks as they are)
template <int NC>
__device__ __forceinline__ int w_swz(int row) {
    if constexpr (NC & (NC - 1)) return 0;
    else return (row / (16 / NC)) & (NC - 1);
}

template <int F, int WM, int MI, int NJ, int NST>
__global__ __launch_bounds__(kThreads) void gemm_codes_kernel(CodesArgs a) {
    using G = Geo<F, WM, MI, NJ, NST>;
    using FM = Fmt<F>;
    constexpr int BM = G::BM, BN = G::BN, WN = G::WN;
    extern __shared__ __align__(16) uint8_t smem[];
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
    const uint8_t* codes = smem + (size_t)NST * G::kA;
    const uint8_t* hdrs = codes + 2 * (size_t)G::kW;

    // work item: split z, weight tile x, activation tile y, y fastest, dealt so
    // that XCD q (workgroup ids q, q + 8, ...) takes a contiguous range: the
    // activation tiles of one weight tile run on one XCD, whose L2 reads its
    // bytes once
    const int tn = (a.n + BN - 1) / BN, tm = (a.m + BM - 1) / BM;
    const int total = tn * tm * a.splits, per = (int)gridDim.x / 8;
    const int wi = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
    if (wi >= total) return;
    const int ty = wi % tm, tx = (wi / tm) % tn, tz = wi / (tm * tn);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wr = wave / WN, wc = wave % WN;
    const int m0 = ty * BM, n0 = tx * BN;
    const int nblk = a.row_blocks;
    const int b0 = tz * a.blocks, nb = min(a.blocks, a.k / 256 - b0);  // this split's 256-element blocks
    const int steps = 4 * nb;
    const size_t rb = row_bytes(FM::kType, 256 * nblk);
    const int lr = lane & 31, hh = lane >> 5;
    const uint32_t hmask = 0u - (uint32_t)hh;

    // ---- load roles (fixed lane offsets; the step moves the scalar base) ----
    uint32_t voff_a[G::kAL];
#pragma unroll
    for (int u = 0; u < G::kAL; ++u) {
        const int slot = (wave * G::kAL + u) * 64 + lane, p = slot % (BM * 8), row = p >> 3;
        const int c = (p & 7) ^ a_swz(row);
        const int e = FM::kRuns ? 32 * (c >> 1) + 8 * (c & 1) : 8 * c;
        voff_a[u] = (uint32_t)(min(m0 + row, a.m - 1) - m0) * (uint32_t)a.lda * 2u + 2u * (uint32_t)e;
    }
    const uint8_t* wrow0 = a.w + (size_t)n0 * rb;
    const uint64_t wbase = scalar_addr(wrow0);
    // piece slot (type, row, c) holds the row's piece c ^ w_swz(row) of the run:
    // a fixed piece of 16 consecutive rows takes 16 different bank groups
    uint32_t voff_w[G::kWL];
    int wtype[G::kWL], wslot[G::kWL];
#pragma unroll
    for (int u = 0; u < G::kWL; ++u) {
        const int s = (u * 512 + wave * 64) % G::kWN;  // padding waves repeat real pieces (same bytes, same place)
        wslot[u] = s;
        wtype[u] = s / (BN * FM::kNC);
        const int i = s % (BN * FM::kNC) + lane, row = i / FM::kNC;
        const int c = (i % FM::kNC) ^ w_swz<FM::kNC>(row);
        voff_w[u] = (uint32_t)(min(n0 + row, a.n - 1) - n0) * (uint32_t)rb + 16u * (uint32_t)c;
    }
    const uint32_t voff_d =
        (uint32_t)(min(n0 + (wave * 64) % BN + lane, a.n - 1) - n0) * (uint32_t)rb;  // (waves past BN / 64 repeat rows)
    // headers, then sub-block sums (hi rows, lo rows)
    constexpr int kHA = G::kHL ? G::kHL : 1;
    const uint8_t* hptr[kHA];
    int hpiece[kHA], hslot[kHA];
    uint32_t is_sum[kHA];
#pragma unroll
    for (int u = 0; u < G::kHL; ++u) {
        const int s = (u * 512 + wave * 64) % (G::kHN ? G::kHN : 1);
        hslot[u] = s;
        is_sum[u] = s >= FM::kH * BN;
        hpiece[u] = is_sum[u] ? 0 : s / BN;
        if (!is_sum[u]) {
            hptr[u] = wrow0 + (size_t)(min(n0 + s % BN + lane, a.n - 1) - n0) * rb;
        } else {
            const int i = s - FM::kH * BN + lane, row = i % BM;
            hptr[u] = reinterpret_cast<const uint8_t*>((i >= BM ? a.s_lo : a.s_hi) + (size_t)min(m0 + row, a.m - 1) * a.lds);
        }
    }
    uint64_t abase[G::kAL];  // load u of the wave reads hi or lo rows
#pragma unroll
    for (int u = 0; u < G::kAL; ++u)
        abase[u] = scalar_addr(((wave * G::kAL + u) / (BM / 8) ? a.a_lo : a.a_hi) + (size_t)m0 * a.lda);
    // (past the end the last step's, granule's or block's bytes again, never read)
    auto issue_a = [&](int st, int slot) __attribute__((always_inline)) {
        const int c = 4 * b0 + min(st, steps - 1);
        const int e = FM::kRuns ? 256 * (c >> 2) + 128 * ((c >> 1) & 1) + 16 * (c & 1) : 64 * c;
#pragma unroll
        for (int u = 0; u < G::kAL; ++u)
            g2l_s(abase[u] + 2 * (uint32_t)e, voff_a[u], lds0 + (uint32_t)slot * G::kA + (wave * G::kAL + u) * 1024);
    };
    // the granule that starts at step st, with its block's headers if the block does
    auto issue_w = [&](int st, bool head) __attribute__((always_inline)) {
        const int c = 4 * b0 + min(st, steps - FM::kGR);
        const uint32_t gr = (uint32_t)c / FM::kGR, b = (uint32_t)c >> 2;
        if (head) {
            const uint32_t hb = lds0 + NST * G::kA + 2 * G::kW + (uint32_t)((st >> 2) & 1) * G::kHdr;
#pragma unroll
            for (int u = 0; u < G::kHL; ++u) {
                if constexpr (FM::kH > 0) {
                    uint32_t off = FM::h_off(b, hpiece[u], nblk);
                    // (arithmetic, not a branch: the step stays one block of code)
                    if constexpr (FM::kMin) off += (16u * b - off) * is_sum[u];
                    g2l_v(hptr[u] + off, hb + hslot[u] * 16);
                }
            }
            if constexpr (G::kDL) g2l4_s(wbase + FM::d_off(b, nblk), voff_d, hb + G::kHN * 16 + wave * 256);
        }
        const uint32_t wb = lds0 + NST * G::kA + (uint32_t)((st / FM::kGR) & 1) * G::kW;
#pragma unroll
        for (int u = 0; u < G::kWL; ++u) g2l_s(wbase + FM::q_off(gr, wtype[u], nblk), voff_w[u], wb + wslot[u] * 16);
    };

    f32x16 acc[MI][NJ], P[MI][NJ];
    const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = zero;

    // operand reads: this lane's activation row of block i is 32 MI wr + 32 i + lr,
    // chunk c at offset aoff[c'] (the XOR is the same for every i)
    int aoff[4];
    const int arow = 32 * MI * wr + lr;
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) {
        const int c = FM::kRuns ? 2 * jj + hh : (jj & 1) + 2 * hh + 4 * (jj >> 1);
        aoff[jj] = arow * 128 + 16 * (c ^ a_swz(arow));
    }
    int col[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) col[j] = 32 * NJ * wc + 32 * j + lr;

    // The step is software-pipelined in four regions of one 16-element product
    // slice each: while a slice multiplies, the next slice's activations are
    // read from LDS and the next half-step's codes are decoded.  A stage's slot
    // is refilled as soon as every wave has read its last operands (before
    // the step's last slice), so NST - 1 stages are always in flight: with
    // one fewer (refilled in the middle of the next step) a step could not be
    // shorter than a stage's load latency, 1.1 - 1.6 us on a full chip.
    f16x8 A[2][2 * MI];           // activation operands (hi, lo per row block): this slice, the next
    uint32_t q[NJ][FM::kQL];      // raw codes of the step
    f16x8 W[2][2][NJ];            // decoded codes: half-step, slice
    f16x8 V[FM::kSplitW ? 2 : 1][2][NJ];  // Q6_K: their rests
    uint4 hd[NJ], qh[NJ];
    float dcol[NJ], d2[2][NJ];
    (void)qh;
    (void)V;
    (void)d2;
    auto read_a = [&](const uint8_t* stg, int half, int sl, int buf) __attribute__((always_inline)) {
        const int off = aoff[FM::slice_chunk(half, sl)];
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            A[buf][2 * i] = *reinterpret_cast<const f16x8*>(stg + off + 4096 * i);
            A[buf][2 * i + 1] = *reinterpret_cast<const f16x8*>(stg + BM * 128 + off + 4096 * i);
        }
    };
    auto read_head = [&](int t) __attribute__((always_inline)) {
        if constexpr (FM::kH == 0) return;
        const uint8_t* hb = hdrs + (size_t)((t >> 2) & 1) * G::kHdr;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            hd[j] = *reinterpret_cast<const uint4*>(hb + col[j] * 16);
            if constexpr (FM::kH == 3) qh[j] = *reinterpret_cast<const uint4*>(hb + ((1 + hh) * BN + col[j]) * 16);
        }
    };
    // d of the block whose header was read
    auto block_d = [&](int t) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            if constexpr (FM::kMin) dcol[j] = half_lo(hd[j].x);
            if constexpr (F == GF_Q6KT) {
                const uint8_t* hb = hdrs + (size_t)((t >> 2) & 1) * G::kHdr;
                const uint32_t v = *reinterpret_cast<const uint32_t*>(hb + G::kHN * 16 + col[j] * 4);
                dcol[j] = ((b0 + (t >> 2)) & 1) ? half_hi(v) : half_lo(v);
            }
        }
    };
    // the raw codes of step t (st: t modulo the granule)
    auto read_q = [&](int t, auto sc) __attribute__((always_inline)) {
        constexpr int g = decltype(sc)::value, st = g % FM::kGR;
        const uint8_t* wq = codes + (size_t)((t / FM::kGR) & 1) * G::kW;
        auto piece = [&](int j, int p) {
            return wq + (FM::type(p) * (BN * FM::kNC) + col[j] * FM::kNC + (FM::chunk(st, p) ^ w_swz<FM::kNC>(col[j]))) * 16;
        };
        // dword i of the words at a 4-byte aligned place of the row's pieces
        auto word = [&](int j, int at, int i) {
            return *reinterpret_cast<const uint32_t*>(wq + col[j] * (16 * FM::kNC) + at + 4 * i);
        };
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            if constexpr (F == GF_Q80) {
                // the lane's 16 codes of each block, and its d; the first
                // block's codes start in the middle of a dword
                const int b0q = FM::block_at(g, 0) + 16 * hh, b1q = FM::block_at(g, 1) + 2 + 16 * hh;
                uint32_t w[5];
#pragma unroll
                for (int i = 0; i < 5; ++i) w[i] = word(j, b0q, i);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    q[j][i] = __builtin_amdgcn_alignbyte(w[i + 1], w[i], 2);
                    q[j][4 + i] = word(j, b1q, i);
                }
                q[j][8] = word(j, FM::block_at(g, 0), 0);            // d in its low half
                q[j][9] = word(j, FM::block_at(g, 1) - 2, 0) >> 16;
            } else if constexpr (F == GF_Q50) {
                // per block four dwords of nibbles, the high bits, d
                uint32_t w[6];
#pragma unroll
                for (int i = 0; i < 6; ++i) w[i] = word(j, FM::block_at(g, 0), i);
#pragma unroll
                for (int i = 0; i < 4; ++i) q[j][i] = __builtin_amdgcn_alignbyte(w[i + 2], w[i + 1], 2);
                q[j][4] = __builtin_amdgcn_alignbyte(w[1], w[0], 2);
                q[j][5] = w[0];
#pragma unroll
                for (int i = 0; i < 5; ++i) q[j][6 + i] = word(j, FM::block_at(g, 1) + 2, (i + 1) % 5);
                q[j][11] = word(j, FM::block_at(g, 1) - 2, 0) >> 16;
            } else if constexpr (F == GF_Q6KT) {
#pragma unroll
                for (int p = 0; p < 3; ++p) {
                    const uint2 v = *reinterpret_cast<const uint2*>(piece(j, p) + 8 * hh);
                    q[j][2 * p] = v.x, q[j][2 * p + 1] = v.y;
                }
            } else {
#pragma unroll
                for (int p = 0; p < FM::kQL / 4; ++p) {
                    const uint4 v = *reinterpret_cast<const uint4*>(piece(j, 2 * p + hh));
                    q[j][4 * p] = v.x, q[j][4 * p + 1] = v.y, q[j][4 * p + 2] = v.z, q[j][4 * p + 3] = v.w;
                }
            }
        }
    };
    // codes of half-step `half` of a step g of its block into W[half] (V[half])
    auto decode = [&](auto gc, auto hc) __attribute__((always_inline)) {
        constexpr int g = decltype(gc)::value, half = decltype(hc)::value;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            if constexpr (FM::kMin) {
                uint32_t scp, mnp;
                k4_pair(hd[j].y, hd[j].z, hd[j].w, g, a.form, scp, mnp);
                // (1024 + sc) - 1024 for both sub-blocks, exact
                const f16x2 sc = as_h2(__builtin_amdgcn_perm(0x64u, scp, 0x04010400u)) - splat((_Float16)1024.f);
                const f16x2 sv0 = splat(sc[0]), sv1 = splat(sc[1]) * splat((_Float16)0.0625f);
                const f16x2 ov0 = sv0 * splat((_Float16)-1024.f), ov1 = sv1 * splat((_Float16)-1024.f);
                // dwords 2 half, 2 half + 1: eight low-nibble codes (sub-block
                // 2 g) and eight high-nibble codes (2 g + 1, as 16 q / 16)
                uint32_t l[4], h[4];
#pragma unroll
                for (int x = 0; x < 2; ++x) {
                    const uint32_t w0 = q[j][2 * half + x], w1 = w0 >> 8;
                    uint32_t l0 = code_pair(w0, 0x000f000fu, kMagic), l1 = code_pair(w1, 0x000f000fu, kMagic);
                    uint32_t h0 = code_pair(w0, 0x00f000f0u, kMagic), h1 = code_pair(w1, 0x00f000f0u, kMagic);
                    if constexpr (FM::kH == 3) {
                        const uint32_t b = half == 0 ? (x ? qh[j].y : qh[j].x) : (x ? qh[j].w : qh[j].z);
                        l0 = code_pair(shl<4 - 2 * g>(b), 0x00100010u, l0);
                        l1 = code_pair(shl<-4 - 2 * g>(b), 0x00100010u, l1);
                        h0 = code_pair(shl<7 - 2 * g>(b), 0x01000100u, h0);
                        h1 = code_pair(shl<-1 - 2 * g>(b), 0x01000100u, h1);
                    }
                    l[2 * x] = as_u(__builtin_elementwise_fma(as_h2(l0), sv0, ov0));
                    l[2 * x + 1] = as_u(__builtin_elementwise_fma(as_h2(l1), sv0, ov0));
                    h[2 * x] = as_u(__builtin_elementwise_fma(as_h2(h0), sv1, ov1));
                    h[2 * x + 1] = as_u(__builtin_elementwise_fma(as_h2(h1), sv1, ov1));
                }
                W[half][0][j] = pack8(l[0], l[1], l[2], l[3]);
                W[half][1][j] = pack8(h[0], h[1], h[2], h[3]);
            } else if constexpr (F == GF_Q50) {
                // this lane half's nibbles and high bits: elements 16 hh .. +15
                const uint32_t hb = q[j][6 * half + 4] >> (16 * hh);
                uint32_t o[8];
#pragma unroll
                for (int x = 0; x < 4; ++x) {
                    const uint32_t w0 = q[j][6 * half + x] >> (4 * hh);
                    // bit e of the four high bits to bits 4 + e and 18 + e
                    const uint32_t b = ((hb >> (4 * x)) & 15u) * 0x40010u;
                    const uint32_t c0 = code_pair(b, 0x00100010u, code_pair(w0, 0x000f000fu, kMagic));
                    const uint32_t c1 = code_pair(b >> 1, 0x00100010u, code_pair(w0 >> 8, 0x000f000fu, kMagic));
                    const f16x2 off = splat((_Float16)1040.f);
                    o[2 * x] = as_u(as_h2(c0) - off);
                    o[2 * x + 1] = as_u(as_h2(c1) - off);
                }
                W[half][0][j] = pack8(o[0], o[1], o[2], o[3]);
                W[half][1][j] = pack8(o[4], o[5], o[6], o[7]);
                d2[half][j] = half_lo(q[j][6 * half + 5]);
            } else if constexpr (F == GF_Q80T || F == GF_Q80) {
                uint32_t o[8];
#pragma unroll
                for (int x = 0; x < 4; ++x) {
                    const uint32_t u = q[j][4 * half + x] ^ 0x80808080u;  // code + 128
                    const f16x2 off = splat((_Float16)1152.f);
                    o[2 * x] = as_u(as_h2(__builtin_amdgcn_perm(0x64u, u, 0x04020400u)) - off);
                    o[2 * x + 1] = as_u(as_h2(__builtin_amdgcn_perm(0x64u, u, 0x04030401u)) - off);
                }
                W[half][0][j] = pack8(o[0], o[1], o[2], o[3]);
                W[half][1][j] = pack8(o[4], o[5], o[6], o[7]);
                if constexpr (F == GF_Q80) {
                    d2[half][j] = half_lo(q[j][8 + half]);
                } else {
                    const uint32_t dw = g == 0 ? hd[j].x : g == 1 ? hd[j].y : g == 2 ? hd[j].z : hd[j].w;
                    d2[half][j] = half ? half_hi(dw) : half_lo(dw);
                }
            } else {  // Q6_K: runs r = 2 half, 2 half + 1 (elements 32 r + 16 p + i of the block's half)
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    constexpr int sb = 8 * (g >> 1) + (g & 1) + 4 * half;
                    const uint32_t sw = sb + 2 * s < 4 ? hd[j].x : sb + 2 * s < 8 ? hd[j].y : sb + 2 * s < 12 ? hd[j].z : hd[j].w;
                    const f16x2 sc = splat((_Float16)(float)(int)(int8_t)((sw >> (8 * ((sb + 2 * s) & 3))) & 0xffu));
                    uint32_t oh[4], ol[4];
#pragma unroll
                    for (int x = 0; x < 2; ++x) {
                        const uint32_t w0 = q[j][2 * s + x], w1 = w0 >> 8;
                        const uint32_t b = q[j][4 + x] >> (2 * s);
                        f16x2 v0, v1;
                        if constexpr (half == 0) {
                            v0 = as_h2(code_pair(b << 4, 0x00300030u, code_pair(w0, 0x000f000fu, kMagic))) -
                                 splat((_Float16)1056.f);
                            v1 = as_h2(code_pair(b >> 4, 0x00300030u, code_pair(w1, 0x000f000fu, kMagic))) -
                                 splat((_Float16)1056.f);
                        } else {  // high nibbles in place: (1024 + 16 q) / 16 - 96 = q - 32
                            const f16x2 sx = splat((_Float16)0.0625f), of = splat((_Float16)-96.f);
                            v0 = __builtin_elementwise_fma(
                                as_h2(code_pair(b << 4, 0x03000300u, code_pair(w0, 0x00f000f0u, kMagic))), sx, of);
                            v1 = __builtin_elementwise_fma(
                                as_h2(code_pair(b >> 4, 0x03000300u, code_pair(w1, 0x00f000f0u, kMagic))), sx, of);
                        }
                        const f16x2 h0 = v0 * sc, h1 = v1 * sc;
                        oh[2 * x] = as_u(h0);
                        oh[2 * x + 1] = as_u(h1);
                        ol[2 * x] = as_u(__builtin_elementwise_fma(v0, sc, -h0));
                        ol[2 * x + 1] = as_u(__builtin_elementwise_fma(v1, sc, -h1));
                    }
                    W[half][s][j] = pack8(oh[0], oh[1], oh[2], oh[3]);
                    V[half][s][j] = pack8(ol[0], ol[1], ol[2], ol[3]);
                }
            }
        }
    };
    // one product slice over the operands in A[buf]
    auto multiply = [&](int half, int sl, int buf, bool first) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
                P[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[buf][2 * i + 1], W[half][sl][j], first ? zero : P[i][j], 0, 0, 0);
        if constexpr (FM::kSplitW) {
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j)
                    P[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[buf][2 * i], V[half][sl][j], P[i][j], 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
                P[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[buf][2 * i], W[half][sl][j], P[i][j], 0, 0, 0);
    };
    auto fold = [&](const float (&d)[NJ]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[i][j][e] = fmaf(d[j], P[i][j][e], acc[i][j][e]);
    };
    // min terms of the block's eight sub-blocks: lane half hh holds sub-blocks
    // 4 hh .. 4 hh + 3 of its rows, -dmin m and the sums both split into hi + lo
    auto min_terms = [&](int t) __attribute__((always_inline)) {
        const uint8_t* sb = hdrs + (size_t)((t >> 2) & 1) * G::kHdr + FM::kH * BN * 16;
        f16x4 sh[MI], sl[MI], bh[NJ], bl[NJ];
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            sh[i] = *reinterpret_cast<const f16x4*>(sb + (arow + 32 * i) * 16 + 8 * hh);
            sl[i] = *reinterpret_cast<const f16x4*>(sb + (BM + arow + 32 * i) * 16 + 8 * hh);
        }
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const uint32_t up = ((hd[j].w >> 4) & 0x0f0f0f0fu) | ((hd[j].z >> 2) & 0x30303030u);
            const uint32_t mn = (up & hmask) | (hd[j].z & 0x3f3f3f3fu & ~hmask);
            const float dmin = -half_hi(hd[j].x);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float v = dmin * (float)((mn >> (8 * e)) & 0xffu);
                bh[j][e] = (_Float16)v;
                bl[j][e] = (_Float16)(v - (float)bh[j][e]);
            }
        }
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x8f16(sl[i], bh[j], acc[i][j], 0, 0, 0);
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x8f16(sh[i], bl[j], acc[i][j], 0, 0, 0);
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x8f16(sh[i], bh[j], acc[i][j], 0, 0, 0);
            }
    };

    using C0 = std::integral_constant<int, 0>;
    using C1 = std::integral_constant<int, 1>;
    int slot = 0;
    auto step = [&](int t, auto gc) __attribute__((always_inline)) {
        constexpr int g = decltype(gc)::value;
        using GN = std::integral_constant<int, (g + 1) & 3>;
        const uint8_t* stg = smem + (size_t)slot * G::kA;
        const int nslot = slot == NST - 1 ? 0 : slot + 1;
        const uint8_t* nstg = smem + (size_t)nslot * G::kA;
        // a: slice (0, 0)
        read_a(stg, 0, 1, 1);
        MXH_CODES_FENCE();
        multiply(0, 0, 0, g == 0 || FM::kPair);
        if constexpr (FM::kMin && g == 1) min_terms(t);
        MXH_CODES_FENCE();
        // b: slice (0, 1)
        read_a(stg, 1, 0, 0);
        MXH_CODES_FENCE();
        multiply(0, 1, 1, false);
        decode(gc, C1{});
        if constexpr (FM::kPair) fold(d2[0]);
        MXH_CODES_FENCE();
        // c: slice (1, 0); the last reads of stage t
        read_a(stg, 1, 1, 1);
        MXH_CODES_FENCE();
        multiply(1, 0, 0, FM::kPair);
        MXH_CODES_FENCE();
        // d: slice (1, 1); every wave has read the step's activations and the
        // next step's are there: the slots are refilled and the next step's
        // first operands read
        wait_vm<G::ahead(g)>();
        lds_barrier();
        if constexpr (G::kWFirst && g % FM::kGR == 0) issue_w(t + FM::kGR, (g + FM::kGR) % 4 == 0);
        issue_a(t + NST, slot);
        if constexpr (!G::kWFirst && g % FM::kGR == 0) issue_w(t + FM::kGR, (g + FM::kGR) % 4 == 0);
        read_q(t + 1, GN{});
        if constexpr (g == 3) read_head(t + 1);
        read_a(nstg, 0, 0, 0);
        MXH_CODES_FENCE();
        multiply(1, 1, 1, false);
        if constexpr (FM::kPair) fold(d2[1]);
        decode(GN{}, C0{});
        if constexpr (!FM::kPair && g == 3) {
            fold(dcol);
            block_d(t + 1);
        }
        MXH_CODES_FENCE();
        slot = nslot;
    };

    issue_w(0, true);
#pragma unroll
    for (int st = 0; st < NST; ++st) issue_a(st, st);
    wait_vm<(NST - 1) * G::kAL>();
    lds_barrier();
    read_head(0);
    read_q(0, C0{});
    read_a(smem, 0, 0, 0);
    block_d(0);
    decode(C0{}, C0{});
    for (int t = 0; t < steps; t += 4) {
        step(t, std::integral_constant<int, 0>{});
        step(t + 1, std::integral_constant<int, 1>{});
        step(t + 2, std::integral_constant<int, 2>{});
        step(t + 3, std::integral_constant<int, 3>{});
    }
    wait_vm<0>();  // no load may still be writing LDS when the workgroup ends

    const bool partial = a.splits > 1;
    float* dst = partial ? a.part + (size_t)tz * a.m * a.n : a.out;
    const int ld = partial ? a.n : a.ldo;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int row = m0 + 32 * MI * wr + 32 * i + 8 * (e >> 2) + 4 * hh + (e & 3);
            if (row >= a.m) continue;
            const float rs = a.rscale[row];
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const int c = n0 + col[j];
                if (c >= a.n) continue;
                const size_t o = (size_t)row * ld + c;
                const float v = acc[i][j][e] * rs;
                dst[o] = !partial && a.res ? v + a.res[o] : v;
            }
        }
}

}  // namespace

template <int F, int WM, int MI, int NJ, int NST>
static int codes_launch(const CodesArgs& a, hipStream_t st) {
    using G = Geo<F, WM, MI, NJ, NST>;
    auto kern = gemm_codes_kernel<F, WM, MI, NJ, NST>;
    static bool attr_set = false;  // above 64 KiB of LDS needs the opt-in, once per kernel
    if (!attr_set) {
        if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)G::kLds) != hipSuccess)
            return MXH_ERR_HIP;
        attr_set = true;
    }
    const int items = (a.n + G::BN - 1) / G::BN * ((a.m + G::BM - 1) / G::BM) * a.splits;
    // a multiple of 8 workgroups (the kernel's XCD mapping)
    hipLaunchKernelGGL(kern, dim3((unsigned)((items + 7) / 8 * 8)), dim3(kThreads), G::kLds, st, a);
    return MXH_OK;
}

template <int F>
static int codes_tile(GemmTile t, const CodesArgs& a, hipStream_t st) {
    switch (t) {
    case GT_128x256:
        if constexpr (!Fmt<F>::kSplitW) return codes_launch<F, 2, 2, 2, 2>(a, st);
        else return MXH_ERR_UNSUPPORTED;  // (two code operands: out of registers)
    case GT_128x128: return codes_launch<F, 2, 2, 1, Fmt<F>::kGR == 2 ? 2 : 3>(a, st);
    case GT_64x256: return codes_launch<F, 1, 2, 1, Fmt<F>::kGR == 2 ? 2 : 4>(a, st);
    default: return codes_launch<F, 1, 1, 1, Fmt<F>::kGR == 2 ? 2 : 4>(a, st);
    }
}

int gemm_codes_launch(GemmFmt f, GemmTile t, const CodesArgs& a, hipStream_t st) {
    switch (f) {
    case GF_Q4K: return codes_tile<GF_Q4K>(t, a, st);
    case GF_Q4KT: return codes_tile<GF_Q4KT>(t, a, st);
    case GF_Q5K: return codes_tile<GF_Q5K>(t, a, st);
    case GF_Q5KT: return codes_tile<GF_Q5KT>(t, a, st);
    case GF_Q80: return codes_tile<GF_Q80>(t, a, st);
    case GF_Q80T: return codes_tile<GF_Q80T>(t, a, st);
    case GF_Q50: return codes_tile<GF_Q50>(t, a, st);
    case GF_Q6KT: return codes_tile<GF_Q6KT>(t, a, st);
    }
    return MXH_ERR_UNSUPPORTED;
}

// ---- dispatch ----------------------------------------------------------------

namespace {

__global__ void gemm_f16_reduce_kernel(const float* __restrict__ part, int splits, float* out, int ldo,
                                       const float* res, int m, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m * n) return;
    const int r = i / n, c = i % n;
    float v = 0.f;
    for (int s = 0; s < splits; ++s) v += part[(size_t)s * m * n + i];
    const size_t o = (size_t)r * ldo + c;
    out[o] = res ? v + res[o] : v;
}

// the same sums, four adjacent outputs per thread (n, ldo multiples of 4 and
// 16-byte aligned rows)
__global__ void gemm_f16_reduce4_kernel(const float4* __restrict__ part, int splits, float* out, int ldo,
                                        const float* res, int m, int n4) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m * n4) return;
    const int r = i / n4, c = i - r * n4;
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int s = 0; s < splits; ++s) {
        const float4 p = part[(size_t)s * m * n4 + i];
        v.x += p.x;
        v.y += p.y;
        v.z += p.z;
        v.w += p.w;
    }
    const size_t o = (size_t)r * ldo + 4 * (size_t)c;
    if (res) {
        const float4 q = *reinterpret_cast<const float4*>(res + o);
        v.x += q.x;
        v.y += q.y;
        v.z += q.z;
        v.w += q.w;
    }
    *reinterpret_cast<float4*>(out + o) = v;
}

void reduce_launch(const float* part, int splits, float* out, int ldo, const float* res, int m, int n,
                   hipStream_t st) {
    const bool vec = n % 4 == 0 && ldo % 4 == 0 && (uintptr_t)part % 16 == 0 && (uintptr_t)out % 16 == 0 &&
                     (uintptr_t)res % 16 == 0;
    if (vec)
        hipLaunchKernelGGL(gemm_f16_reduce4_kernel, dim3((m * (n / 4) + 255) / 256), dim3(256), 0, st,
                           reinterpret_cast<const float4*>(part), splits, out, ldo, res, m, n / 4);
    else
        hipLaunchKernelGGL(gemm_f16_reduce_kernel, dim3((m * n + 255) / 256), dim3(256), 0, st, part, splits, out,
                           ldo, res, m, n);
}

// Device workspace of the GEMMs, held by every GPU the library runs on from
// load until the process ends, so that no call allocates: partial tiles of
// split K (one array per Workspace), and a slab of rows regrouped for the
// kernel.
constexpr size_t kPartBytes = 64u << 20, kSlabBytes = 64u << 20;
static __device__ __align__(256) uint8_t g_partials[2][kPartBytes];
static __device__ __align__(256) uint8_t g_slab[kSlabBytes];
float* g_part_ptr[2] = {nullptr, nullptr};
uint8_t* g_slab_ptr = nullptr;

// Q6_K rows in GGUF order are only 2-aligned (210-byte blocks): regrouped into
// the tiled order, the block count rounded up to a multiple of eight (16-byte
// rows; the added blocks are never read).  Thread: one 64-element chunk.
// Bound by HBM: reads and writes each byte once.
__device__ __forceinline__ uint4 ld_u16x8(const uint8_t* p) {
    const uint16_t* h = reinterpret_cast<const uint16_t*>(p);
    return make_uint4(h[0] | ((uint32_t)h[1] << 16), h[2] | ((uint32_t)h[3] << 16), h[4] | ((uint32_t)h[5] << 16),
                      h[6] | ((uint32_t)h[7] << 16));
}

__global__ __launch_bounds__(256) void regroup_q6k_kernel(const uint8_t* __restrict__ w, uint8_t* __restrict__ o,
                                                          int rows, int k, int row_blocks) {
    const int units = k / 64;
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int row = (int)(t / units), c = (int)(t % units);
    if (row >= rows) return;
    const uint8_t* src = w + (size_t)row * row_bytes(MXH_Q6_K, k) + (size_t)(c >> 2) * 210;
    uint8_t* op = o + (size_t)row * row_bytes(MXH_Q6_K, 256 * (int64_t)row_blocks);
    const Q6KTileOffs f = q6k_tile_offsets(c, row_blocks);
    const int h = (c >> 1) & 1, p = c & 1;
    *reinterpret_cast<uint4*>(op + f.qa) = ld_u16x8(src + 64 * h + 16 * p);
    *reinterpret_cast<uint4*>(op + f.qb) = ld_u16x8(src + 64 * h + 32 + 16 * p);
    *reinterpret_cast<uint4*>(op + f.qh) = ld_u16x8(src + 128 + 32 * h + 16 * p);
    if ((c & 3) == 0) {
        *reinterpret_cast<uint4*>(op + f.sc) = ld_u16x8(src + 192);
        *reinterpret_cast<uint16_t*>(op + f.d) = *reinterpret_cast<const uint16_t*>(src + 208);
    }
}

bool al16(const void* p) { return ((uintptr_t)p & 15) == 0; }

}  // namespace

uint8_t* gemm_partials(size_t* bytes) {
    *bytes = kPartBytes;
    return reinterpret_cast<uint8_t*>(g_part_ptr[(int)Workspace::kStream]);
}

int gemm_workspace_init() {
    void *p = nullptr, *q = nullptr;
    if (int rc = check_hip(hipGetSymbolAddress(&p, HIP_SYMBOL(g_partials)), "hipGetSymbolAddress(partials)")) return rc;
    if (int rc = check_hip(hipGetSymbolAddress(&q, HIP_SYMBOL(g_slab)), "hipGetSymbolAddress(slab)")) return rc;
    for (int i = 0; i < 2; ++i) g_part_ptr[i] = reinterpret_cast<float*>(static_cast<uint8_t*>(p) + i * kPartBytes);
    g_slab_ptr = static_cast<uint8_t*>(q);
    return MXH_OK;
}

bool gemm_q_f16_supported(int type, int k) {
    if (k <= 0 || k % 256 || k > 16384) return false;
    switch (type) {
    case MXH_Q4_K: case MXH_Q4_K_TILED: case MXH_Q5_K: case MXH_Q5_K_TILED:
    case MXH_Q8_0: case MXH_Q8_0_TILED: case MXH_Q5_0: case MXH_Q6_K: return true;
    case MXH_Q6_K_TILED: return k % 2048 == 0;
    }
    return false;
}

int gemm_q_f16_run(int type, const uint16_t* a_hi, const uint16_t* a_lo, int lda, const uint16_t* s_hi,
                   const uint16_t* s_lo, int lds, const float* rscale, const void* w, float* out, int ldo,
                   const float* res, int m, int n, int k, int form, Workspace ws, hipStream_t st) {
    if (m <= 0 || n <= 0 || !gemm_q_f16_supported(type, k) || lda < k || lds < k / 32 || ldo < n) return MXH_ERR_ARG;
    float* part = g_part_ptr[(int)ws];
    // the direct loads are 16 bytes wide
    if (!al16(a_hi) || !al16(a_lo) || !al16(s_hi) || !al16(s_lo) || lda % 8 || lds % 8 || !part) return MXH_ERR_ARG;
    CodesArgs a{};
    a.a_hi = a_hi, a.a_lo = a_lo, a.s_hi = s_hi, a.s_lo = s_lo, a.rscale = rscale;
    a.out = out, a.res = res, a.part = part;
    a.lda = lda, a.lds = lds, a.ldo = ldo, a.m = m, a.n = n, a.k = k, a.form = form, a.row_blocks = k / 256;
    GemmFmt f;
    bool regroup = false;
    switch (type) {
    case MXH_Q4_K: f = GF_Q4K; break;
    case MXH_Q4_K_TILED: f = GF_Q4KT; break;
    case MXH_Q5_K: f = GF_Q5K; break;
    case MXH_Q5_K_TILED: f = GF_Q5KT; break;
    case MXH_Q8_0: f = GF_Q80; break;
    case MXH_Q8_0_TILED: f = GF_Q80T; break;
    case MXH_Q5_0: f = GF_Q50; break;
    case MXH_Q6_K_TILED: f = GF_Q6KT; break;
    default:  // Q6_K
        f = GF_Q6KT, regroup = true;
        a.row_blocks = (a.row_blocks + 7) / 8 * 8;
        break;
    }
    if (regroup ? ws != Workspace::kStream : !al16(w)) return MXH_ERR_ARG;  // (one slab)
    const size_t in_rb = row_bytes(type, k);
    const size_t rb = row_bytes(MXH_Q6_K, 256 * (int64_t)a.row_blocks);  // of a regrouped row
    // regrouped rows go through the slab in equal pieces, whole tiles of rows,
    // each under the plan for what it launches (2 x 30000 x 11008 under a plan
    // for all rows: seven launches of a seventh of the chip) - but under one for
    // all rows where the rows have a tiled order too, whose results are these
    const int slab_rows = regroup ? (int)(kSlabBytes / rb / 256 * 256) : n;
    const int pieces = (n - 1) / slab_rows + 1;
    const int step = pieces > 1 ? ((n - 1) / pieces + 256) / 256 * 256 : n;
    GemmPlan p = gemm_plan(f, m, n, k, device_cus(), kPartBytes);
    const bool per_piece = pieces > 1 && tiled_type(type, k) == type;
    for (int n0 = 0; n0 < n; n0 += step) {
        const int nn = std::min(step, n - n0);
        const uint8_t* src = static_cast<const uint8_t*>(w) + (size_t)n0 * in_rb;
        a.w = src;
        if (regroup) {
            const int64_t threads = (int64_t)nn * (k / 64);
            hipLaunchKernelGGL(regroup_q6k_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, st, src,
                               g_slab_ptr, nn, k, a.row_blocks);
            a.w = g_slab_ptr;
        }
        if (per_piece) p = gemm_plan(f, m, nn, k, device_cus(), kPartBytes);
        a.blocks = p.blocks, a.splits = p.splits;
        a.n = nn;
        a.out = out + n0;
        a.res = res ? res + n0 : nullptr;
        if (int rc = gemm_codes_launch(f, p.tile, a, st)) return rc;
        if (p.splits > 1) reduce_launch(a.part, p.splits, a.out, ldo, a.res, m, nn, st);
    }
    return MXH_OK;
}

}  // namespace mxh

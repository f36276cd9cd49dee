// mxh_sample.hip — top-k / temperature / top-p / min-p sampling on the device
// (reference: src/api/minxfmr.cpp:2091-2171, with a seeded draw).
//
// Keys: order-preserving bits of the logit above the complemented id, so ties
// go to the lower id, as the reference's partial_sort with `>` and an
// increasing initial order.  Pass 1, the whole chip: the largest logit of
// every group of 4 to 16 neighbouring ids (more above 196,608 ids).  Pass 2,
// one workgroup: the k-th largest group maximum T bounds the k-th largest key
// from below (k maxima reach it) and only groups whose maximum reaches it hold
// keys at or above it, so the logits of about k groups are read again, the
// hardly more than k keys at or above T are sorted, and the choice is made
// among the first k in double exactly as the reference makes it (exp of
// (l - max) / T, normalise, top-p cut and renormalise, min-p cut and
// renormalise).  Where more than kCandMax keys reach T (many equal logits, or
// large logits side by side), T is raised over the keys themselves first.
//
// Bound: the one workgroup's chain of barriers and LDS latencies, two launches
// and the wait for the id.  Selecting by sorting (64 lists sorted in LDS, then
// 4,096 keys by one workgroup) took 156 us for top_k 40 of 151,936 ids with
// the copies of its parameters and of the id; this 27.
//
// The uniform of draw d is splitmix64 at state seed + (d + 1) *
// 0x9E3779B97F4A7C15, the d-th value of the sequence that starts at `seed`.
#include <hip/hip_runtime.h>

#include "mxh_device.h"
#include "mxh_internal.h"

namespace mxh {

namespace {

constexpr int kCandMax = kSampleTopKMax;  // keys the workgroup sorts
constexpr int kThreads = 1024, kWaves = kThreads / 64;
constexpr int kGroupRegs = 12;  // group maxima a thread of pass 2 holds
constexpr int kGroupsMax = kThreads * kGroupRegs;

typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));  // 16 bytes at any float address

__device__ __forceinline__ uint32_t order_bits(float v) {
    const uint32_t u = __float_as_uint(v);
    if ((u & 0x7fffffffu) > 0x7f800000u) return 0u;  // NaN sorts last
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__device__ __forceinline__ uint64_t sort_key(float v, int idx) {
    return ((uint64_t)order_bits(v) << 32) | (uint32_t)(~(uint32_t)idx);
}

__device__ __forceinline__ int key_id(uint64_t k) { return (int)(~(uint32_t)(k & 0xffffffffu)); }

// ids per group: the fewest (a power of two, four at least) that leave at most
// kGroupsMax groups
int group_shift(int n) {
    int g = 2;
    while ((((int64_t)n + (1ll << g) - 1) >> g) > kGroupsMax) ++g;
    return g;
}
int group_count(int n) { return (int)(((int64_t)n + (1ll << group_shift(n)) - 1) >> group_shift(n)); }

// 1, 2 or 4 lanes per group (1 << lsh), four ids a load
__global__ __launch_bounds__(256) void group_max_kernel(const float* __restrict__ logits, int n, int gsh, int lsh,
                                                        int groups, uint32_t* __restrict__ gmax) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x, g = t >> lsh;
    uint32_t m = 0u;
    if (g < groups) {
        const int64_t end = (g + 1) << gsh;
        for (int64_t e = (g << gsh) + 4 * (t & ((1 << lsh) - 1)); e < end && e < n; e += 4 << lsh) {
            if (e + 4 <= n) {
                const f32x4u v = *reinterpret_cast<const f32x4u*>(logits + e);
#pragma unroll
                for (int i = 0; i < 4; ++i) m = max(m, order_bits(v[i]));
            } else {
                for (int64_t i = e; i < n; ++i) m = max(m, order_bits(logits[i]));
            }
        }
    }
    for (int off = 1; off < 1 << lsh; off <<= 1) m = max(m, (uint32_t)__shfl_xor((int)m, off, 64));
    if (g < groups && (t & ((1 << lsh) - 1)) == 0) gmax[g] = m;
}

__device__ __forceinline__ double draw_uniform(uint64_t seed, uint64_t d) {
    uint64_t z = seed + (d + 1) * 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    return (double)(z >> 11) * (1.0 / 9007199254740992.0);
}

// p[0] + p[1] + ... in that order: the loads of a stretch are issued together,
// only the additions form a chain
__device__ __forceinline__ double sum_in_order(const double* p, int m) {
    double s = 0.0;
#pragma unroll 16
    for (int i = 0; i < m; ++i) s += p[i];
    return s;
}

// First i with reached(p[0] + .. + p[i]) for non-negative p, m - 1 if none;
// *cum is that sum.  Whole stretches first (the sums only grow), then the one
// that holds it again.
template <class F>
__device__ __forceinline__ int first_reaching(const double* p, int m, F&& reached, double* cum) {
    double c = 0.0;
    int i = 0;
    for (; i + 16 <= m; i += 16) {
        double c1 = c;
#pragma unroll
        for (int j = 0; j < 16; ++j) c1 += p[i + j];
        if (reached(c1)) break;
        c = c1;
    }
    for (; i < m; ++i) {
        c += p[i];
        if (reached(c)) break;
    }
    *cum = c;
    return i < m ? i : m - 1;
}

// The choice among the k best ids in order (ids[0 .. k)), as the reference
// makes it (minxfmr.cpp:2104-2171), in double: exponentials and divisions by
// the whole workgroup, the sums by thread 0 in the reference's order.  The
// token goes to out[0] or, with tokens/pos, to tokens[*pos + 1] with the
// position advanced (the decode loop on the device); with prm the draw counter
// advances.  Called by every thread of the workgroup.
__device__ void choose(const float* __restrict__ logits, const int* ids, int k, double* pr, const SampleParams& sp,
                       SampleParams* prm, int* out, int* tokens, int* pos) {
    __shared__ double val;
    __shared__ int cut;
    const int tid = threadIdx.x;
    int pick = 0, m = k;  // pick: index into ids
    if (sp.temperature > 0.0) {
        double top_p = sp.top_p, min_p = sp.min_p;
        if (top_p <= 0.0 || top_p > 1.0) top_p = 1.0;
        if (min_p < 0.0) min_p = 0.0;
        if (min_p > 1.0) min_p = 1.0;
        const double mx = logits[ids[0]];
        for (int i = tid; i < k; i += kThreads) pr[i] = exp(((double)logits[ids[i]] - mx) / sp.temperature);
        __syncthreads();
        const auto divide = [&](double by) {  // pr[0 .. m) /= by
            for (int i = tid; i < m; i += kThreads) pr[i] /= by;
            __syncthreads();
        };
        if (tid == 0) val = sum_in_order(pr, m);
        __syncthreads();
        const double sum = val;
        if (sum > 0.0) {
            divide(sum);
            if (top_p < 1.0) {
                if (tid == 0) cut = first_reaching(pr, k, [&](double c) { return c >= top_p; }, &val) + 1;
                __syncthreads();
                m = cut;
                const double r = val;  // the sum of the kept, in the same order
                if (r > 0.0) divide(r);
            }
            if (min_p > 0.0 && m > 1) {
                const double thr = pr[0] * min_p;
                if (tid == 0) cut = m;
                __syncthreads();
                for (int i = 1 + tid; i < m; i += kThreads)
                    if (!(pr[i] >= thr)) {
                        atomicMin(&cut, i);
                        break;
                    }
                __syncthreads();
                m = cut;
                if (tid == 0) val = sum_in_order(pr, m);
                __syncthreads();
                const double r = val;
                if (r > 0.0) divide(r);
            }
            if (tid == 0) {
                const double u = draw_uniform(sp.seed, sp.draws) * sum_in_order(pr, m);
                double c;
                pick = first_reaching(pr, m, [&](double v) { return u < v; }, &c);
            }
        }
    }
    if (tid != 0) return;
    if (prm && sp.temperature > 0.0) prm->draws = sp.draws + 1;
    if (out) out[0] = ids[pick];
    if (tokens) {
        const int q = *pos;
        tokens[q + 1] = ids[pick];
        *pos = q + 1;
    }
}

// descending over the wave's lanes
__device__ __forceinline__ uint64_t sort64_desc(uint64_t v) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int k = 2; k <= 64; k <<= 1)
#pragma unroll
        for (int j = k >> 1; j > 0; j >>= 1) {
            const uint64_t o = (uint64_t)__shfl_xor((unsigned long long)v, j, 64);
            // the lower lane of a pair keeps the larger key in a descending run
            const bool larger = ((lane & k) == 0) == ((lane & j) == 0);
            v = (o > v) == larger ? o : v;
        }
    return v;
}

// keys of a descending run of 64 that are larger than v
__device__ __forceinline__ int run_larger(const uint64_t* run, uint64_t v) {
    int lo = 0;
#pragma unroll
    for (int step = 32; step > 0; step >>= 1)
        if (run[lo + step - 1] > v) lo += step;
    return lo + (run[lo] > v);
}

// prm: parameters in device memory, or null for `call`'s
__global__ __launch_bounds__(kThreads) void choose_topk_kernel(const float* __restrict__ logits, int n, int gsh,
                                                               int groups, const uint32_t* __restrict__ gmax,
                                                               SampleParams* prm, SampleParams call, int* out,
                                                               int* tokens, int* pos) {
    __shared__ __attribute__((aligned(16))) uint64_t s[kCandMax];  // keys, then the probabilities (doubles)
    __shared__ __attribute__((aligned(16))) uint16_t list[kGroupsMax];  // groups taken, then the ids in order
    __shared__ int part[2][4][kWaves];
    __shared__ int n_list, n_cand;
    __shared__ uint32_t bound;
    static_assert(sizeof(list) >= kCandMax * sizeof(int) && kGroupsMax <= 65536, "");
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const SampleParams sp = prm ? *prm : call;
    const int k = sp.top_k;

    uint32_t mx[kGroupRegs];
    uint32_t my_top = 0u;
#pragma unroll
    for (int r = 0; r < kGroupRegs; ++r) {
        const int g = tid + kThreads * r;
        mx[r] = g < groups ? gmax[g] : 0u;
        my_top = max(my_top, mx[r]);
    }
    if (tid == 0) n_list = 0, n_cand = 0, bound = 0u;
    // per-wave counts -> the workgroup's (part is double-buffered: one barrier a call)
    int turn = 0;
    const auto total3 = [&](int a, int b, int c, int (&t)[3]) {
        if (lane == 0) part[turn][0][wave] = a, part[turn][1][wave] = b, part[turn][2][wave] = c;
        __syncthreads();
        t[0] = t[1] = t[2] = 0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w)
            t[0] += part[turn][0][w], t[1] += part[turn][1][w], t[2] += part[turn][2][w];
        turn ^= 1;
    };

    // T: the k-th largest group maximum, from the top bit down, or a value
    // below it that few more maxima reach; 0 (every key) with fewer groups.
    // For k up to a quarter of the threads the largest maximum of each thread
    // stands for its groups (hardly more keys reach the k-th of those) and one
    // wave searches, without barriers: 2.4 us against 7.4.
    uint32_t T = 0u;
    if (k <= kThreads / 4) {
        uint32_t* tops = reinterpret_cast<uint32_t*>(s);
        tops[tid] = my_top;
        __syncthreads();
        if (wave == 0) {
            uint32_t v[kWaves];
#pragma unroll
            for (int w = 0; w < kWaves; ++w) v[w] = tops[lane + 64 * w];
            for (int bit = 31; bit >= 0; --bit) {
                const uint32_t c = T | (1u << bit);
                int t = 0;
#pragma unroll
                for (int w = 0; w < kWaves; ++w) t += __popcll(__ballot(v[w] >= c));
                if (t >= k) {
                    T = c;
                    if (t <= k + (k >> 3)) break;
                }
            }
            if (lane == 0) bound = T;
        }
        __syncthreads();
        T = bound;
    } else if (groups >= k) {
        for (int bit = 31; bit >= 0; --bit) {
            const uint32_t c = T | (1u << bit);
            int cnt = 0;
#pragma unroll
            for (int r = 0; r < kGroupRegs; ++r) cnt += __popcll(__ballot(mx[r] >= c));
            if (lane == 0) part[turn][0][wave] = cnt;
            __syncthreads();
            int t = 0;
#pragma unroll
            for (int w = 0; w < kWaves; ++w) t += part[turn][0][w];
            turn ^= 1;
            if (t >= k) {
                T = c;
                if (t <= k + (k >> 3)) break;
            }
        }
    }
    __syncthreads();

    // the groups whose maximum reaches T; one place a wave in the list
    {
        uint64_t in[kGroupRegs];
        int n_in = 0;
#pragma unroll
        for (int r = 0; r < kGroupRegs; ++r) {
            in[r] = __ballot(tid + kThreads * r < groups && mx[r] >= T);
            n_in += __popcll(in[r]);
        }
        if (n_in) {
            int base = 0;
            if (lane == 0) base = atomicAdd(&n_list, n_in);
            base = __builtin_amdgcn_readfirstlane(base);
#pragma unroll
            for (int r = 0; r < kGroupRegs; ++r) {
                if (in[r] >> lane & 1)
                    list[base + __popcll(in[r] & ((1ull << lane) - 1))] = (uint16_t)(tid + kThreads * r);
                base += __popcll(in[r]);
            }
        }
    }
    __syncthreads();

    // f(key, valid) over their ids, whole waves at a time
    const int64_t n_ids = (int64_t)n_list << gsh;
    const auto each = [&](auto&& f) {
        for (int64_t i = tid; i - lane < n_ids; i += kThreads) {
            const int64_t e = i < n_ids ? ((int64_t)list[i >> gsh] << gsh) + (i & ((1 << gsh) - 1)) : n;
            f(e < n ? sort_key(logits[e], (int)e) : 0ull);
        }
    };
    // the keys >= t to s (as many as fit); every real key is larger than zero
    const auto gather = [&](uint64_t t) {
        each([&](uint64_t key) {
            const bool in = key >= t && key != 0ull;
            const uint64_t mask = __ballot(in);
            if (!mask) return;
            int base = 0;
            if (lane == 0) base = atomicAdd(&n_cand, __popcll(mask));
            const int at = __builtin_amdgcn_readfirstlane(base) + __popcll(mask & ((1ull << lane) - 1));
            if (in && at < kCandMax) s[at] = key;
        });
        __syncthreads();
    };
    gather((uint64_t)T << 32);
    if (n_cand > kCandMax) {
        // The k-th largest key, or one below it that at most kCandMax reach:
        // two bits a pass.  It lies between T and the largest maximum, so the
        // value bits above their first difference are known; then the id's.
        if (tid == 0) bound = 0u;
        __syncthreads();
        atomicMax(&bound, my_top);
        __syncthreads();
        const uint32_t top = bound;
        int id_bits = 1;
        while (id_bits < 31 && (n >> id_bits)) ++id_bits;
        const uint32_t diff = T ^ top;
        const int vbits = diff ? 32 - __builtin_clz(diff) : 0;
        uint64_t t = (uint64_t)(vbits < 32 ? T >> vbits << vbits : 0u) << 32;
        int reach = n_cand;
        const auto narrow = [&](int bits, int low) {
            for (int hi = bits; hi > 0 && reach > kCandMax; hi -= 2) {
                const int sh = low + (hi > 1 ? hi - 2 : 0), steps = hi > 1 ? 3 : 1;
                const uint64_t c1 = t + (1ull << sh), c2 = t + (2ull << sh), c3 = t + (3ull << sh);
                int a = 0, b = 0, c = 0;
                each([&](uint64_t key) {
                    a += __popcll(__ballot(key >= c1));
                    b += __popcll(__ballot(key >= c2));
                    c += __popcll(__ballot(key >= c3));
                });
                int cnt[3];
                total3(a, b, c, cnt);
                for (int j = 0; j < steps; ++j)
                    if (cnt[j] >= k) t += 1ull << sh, reach = cnt[j];
            }
        };
        narrow(vbits, 32);
        if (reach > kCandMax) {
            t |= 0xffffffffull & (~0ull << id_bits);  // an id's complement has these bits set
            narrow(id_bits, 0);
        }
        __syncthreads();
        if (tid == 0) n_cand = 0;
        __syncthreads();
        gather(t);
    }

    // Sorted runs of 64, one a wave; a key's place is its place in its own run
    // plus the larger keys of every other run (keys are distinct).
    const int cand = n_cand, runs = (cand + 63) >> 6;
    int* ids = reinterpret_cast<int*>(list);
    constexpr int kRunRegs = kCandMax / kThreads;
    uint64_t key[kRunRegs];
#pragma unroll
    for (int r = 0; r < kRunRegs; ++r) {
        const int i = tid + kThreads * r;
        if (wave + kWaves * r < runs) {
            key[r] = sort64_desc(i < cand ? s[i] : 0ull);
            s[i] = key[r];
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kRunRegs; ++r) {
        const int run = wave + kWaves * r;
        if (run < runs) {
            int at = lane;
            for (int q = 0; q < runs; ++q)
                if (q != run) at += run_larger(s + 64 * q, key[r]);
            if (key[r] && at < k) ids[at] = key_id(key[r]);
        }
    }
    __syncthreads();
    choose(logits, ids, k, reinterpret_cast<double*>(s), sp, prm, out, tokens, pos);
}

}  // namespace

size_t sample_scratch_keys(int n) { return ((size_t)group_count(n) + 1) / 2; }

// Vocabularies taken: any for top_k above 64, else up to 4096 times 4096 /
// top_k (to the next power of two) ids, 8M at most.  The kernels have no such
// limit; it is what the entry point and the models have always refused.
int sample_launch(const float* logits, int n, SampleParams* prm, const SampleParams* call, int top_k, uint64_t* cand,
                  int* out, int* tokens, int* pos, hipStream_t st) {
    if (n <= 0 || top_k < 1 || top_k > kSampleTopKMax || top_k > n) return MXH_ERR_ARG;
    if (top_k <= 64) {
        int64_t lists = 4096;
        while (lists * top_k > 4096) lists >>= 1;
        if (n > 4096 * (lists < 2048 ? lists : 2048)) return MXH_ERR_UNSUPPORTED;
    }
    const int gsh = group_shift(n), lsh = gsh < 4 ? gsh - 2 : 2, groups = group_count(n);
    uint32_t* gmax = reinterpret_cast<uint32_t*>(cand);
    hipLaunchKernelGGL(group_max_kernel, dim3((unsigned)(((int64_t)(groups << lsh) + 255) / 256)), dim3(256), 0, st,
                       logits, n, gsh, lsh, groups, gmax);
    hipLaunchKernelGGL(choose_topk_kernel, dim3(1), dim3(kThreads), 0, st, logits, n, gsh, groups, gmax, prm,
                       call ? *call : SampleParams{}, out, tokens, pos);
    return MXH_OK;
}

// ---- logit edits before the choice (minxfmr.cpp:2047-2089) ---------------

namespace {

__device__ __forceinline__ bool edits_active(const EditParams* prm) {
    return prm->repeat_penalty != 1.0 || prm->frequency_penalty != 0.0 || prm->presence_penalty != 0.0;
}

// the penalty window: the last last_n ids of tokens[0 .. pos] (all when
// last_n < 0), as [*h0, *h1)
__device__ __forceinline__ void edit_window(const EditParams* prm, int pos, int* h0, int* h1) {
    const int len = pos + 1;
    int n = prm->last_n < 0 ? len : prm->last_n;
    if (n > len) n = len;
    *h0 = len - n;
    *h1 = len;
}

// suppressed ids to -inf; occurrences of each id in the window counted
__global__ void logit_count_kernel(float* __restrict__ logits, int n_vocab, const int* __restrict__ tokens,
                                   const int* __restrict__ pos_p, const EditParams* __restrict__ prm,
                                   const int* __restrict__ suppress, int* __restrict__ cnt) {
    const int tid = blockIdx.x * blockDim.x + threadIdx.x, nthr = gridDim.x * blockDim.x;
    for (int j = tid; j < prm->n_suppress; j += nthr) {
        const int id = suppress[j];
        if (id >= 0 && id < n_vocab) logits[id] = -INFINITY;
    }
    if (!edits_active(prm)) return;
    int h0, h1;
    edit_window(prm, *pos_p, &h0, &h1);
    for (int i = h0 + tid; i < h1; i += nthr) {
        const int t = tokens[i];
        if (t >= 0 && t < n_vocab) atomicAdd(cnt + t, 1);
    }
}

// each distinct id of the window (the one occurrence whose exchange returns
// its count) gets the reference's penalty, computed in double; the counts go
// back to zero for the next step
__global__ void logit_penalty_kernel(float* __restrict__ logits, int n_vocab, const int* __restrict__ tokens,
                                     const int* __restrict__ pos_p, const EditParams* __restrict__ prm,
                                     int* __restrict__ cnt) {
    if (!edits_active(prm)) return;
    const int tid = blockIdx.x * blockDim.x + threadIdx.x, nthr = gridDim.x * blockDim.x;
    int h0, h1;
    edit_window(prm, *pos_p, &h0, &h1);
    for (int i = h0 + tid; i < h1; i += nthr) {
        const int t = tokens[i];
        if (t < 0 || t >= n_vocab) continue;
        const int c = atomicExch(cnt + t, 0);
        if (c <= 0) continue;
        double l = (double)logits[t];
        if (prm->repeat_penalty != 1.0) l = l <= 0.0 ? l * prm->repeat_penalty : l / prm->repeat_penalty;
        l -= (double)c * prm->frequency_penalty + prm->presence_penalty;
        logits[t] = (float)l;
    }
}

}  // namespace

int logit_edits_launch(float* logits, int n_vocab, const int* tokens, const int* pos, const EditParams* prm,
                       const int* suppress, int* cnt, hipStream_t st) {
    if (n_vocab <= 0) return MXH_ERR_ARG;
    hipLaunchKernelGGL(logit_count_kernel, dim3(64), dim3(256), 0, st, logits, n_vocab, tokens, pos, prm, suppress,
                       cnt);
    hipLaunchKernelGGL(logit_penalty_kernel, dim3(64), dim3(256), 0, st, logits, n_vocab, tokens, pos, prm, cnt);
    return MXH_OK;
}

}  // namespace mxh

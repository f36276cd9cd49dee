// mxh_plan.h — how the prefill kernels share their work out over a device's
// CUs: estimates of the time from measured step times, the lowest taken.
// Plain C++.
#pragma once

#include <stddef.h>
#include <stdint.h>

namespace mxh {

// weight formats (GGUF block order, T: the tiled order of mxh_types.h)
enum GemmFmt { GF_Q4K, GF_Q4KT, GF_Q5K, GF_Q5KT, GF_Q80, GF_Q80T, GF_Q50, GF_Q6KT };

// tile shapes of the kernel (activation rows x weight rows)
enum GemmTile { GT_128x256, GT_128x128, GT_64x256, GT_32x256, GT_COUNT };

struct GemmPlan {
    GemmTile tile;
    int blocks, splits;
};

// The tile shape and split of K with the lowest estimate of
//   rounds of the device's CUs x (steps of a work item x time of a step + its start)
//   + the reduction of the partial tiles,
// the step's time lying between what it takes on a nearly idle chip and on a
// full one (ns, measured per format and tile at K = 4096 .. 14336, where the
// estimate is within 10% of the measured time of the shapes tried); 7.5 us is
// what a work item takes to start, fill its stages and store its outputs.  Q5_0
// was fitted from K = 1024 on, with that time per tile too (rms 5 to 9%).  A
// type's two orders, GGUF and tiled, share their costs: the split of K is part
// of the results, and these are the same bits through either.
inline GemmPlan gemm_plan(GemmFmt fmt, int m, int n, int k, int cus, size_t part_bytes) {
    struct Cost {
        float idle, full, item = 7500.f;
    };
    static const Cost cost[5][GT_COUNT] = {
        {{1420.f, 2130.f}, {830.f, 1160.f}, {800.f, 1110.f}, {490.f, 650.f}},       // Q4_K
        {{1680.f, 2280.f}, {980.f, 1270.f}, {950.f, 1220.f}, {650.f, 830.f}},       // Q5_K
        {{1720.f, 2300.f}, {980.f, 1180.f}, {950.f, 1200.f}, {600.f, 830.f}},       // Q8_0
        {{1e6f, 1e6f}, {1430.f, 1730.f}, {1560.f, 1830.f}, {1000.f, 1130.f}},       // Q6_K
        {{2460.f, 2470.f, 9100.f}, {1350.f, 1350.f, 5300.f}, {1250.f, 1280.f, 5500.f}, {1140.f, 780.f, 2000.f}}};  // Q5_0
    static const int bm[GT_COUNT] = {128, 128, 64, 32}, bn[GT_COUNT] = {256, 128, 256, 256};
    static const int cls_of[] = {0, 0, 1, 1, 2, 2, 4, 3};  // by GemmFmt
    const int cls = cls_of[fmt], nblk = k / 256;
    GemmPlan best{GT_128x256, nblk, 1};
    double best_cost = 1e30;
    for (int t = cls == 3 ? GT_128x128 : GT_128x256; t < GT_COUNT; ++t) {
        const int64_t tiles = (int64_t)((n + bn[t] - 1) / bn[t]) * ((m + bm[t] - 1) / bm[t]);
        for (int s = 1; s <= nblk && s <= 32; ++s) {
            const int blocks = (nblk + s - 1) / s;
            if ((nblk + blocks - 1) / blocks != s) continue;
            const double floats = (double)s * m * n;
            if (s > 1 && floats * 4 > (double)part_bytes) break;
            const Cost& c = cost[cls][t];
            const int64_t items = tiles * s, rounds = (items + cus - 1) / cus;
            const double load = items >= cus ? 1.0 : (double)items / cus;
            const double ns = rounds * (4.0 * blocks * (c.idle + load * (c.full - c.idle)) + c.item) +
                              (s > 1 ? 3000.0 + floats * 4 / 3000.0 : 0.0);
            if (ns < best_cost) {
                best_cost = ns;
                best = GemmPlan{(GemmTile)t, blocks, s};
            }
        }
    }
    return best;
}

// Splits of the keys among workgroups.  Measured: a stage takes kStage us
// alone (latencies) and at least kFull us of a CU's time for each workgroup on
// it, and kSlots workgroups fit a CU; a merge costs its launch (3.5 us), a
// little a split, and the parts' way through memory.  us without splits / with
// the splits chosen (m at p0, q heads / kv heads x head dim):
//   16 at 7680, 32/8 x 128   145 / 21      2 at 7000, 8/1 x 64     90 / 13
//   128 at 4000, 32/8 x 128   81 / 34      100 at 3000, 8/1 x 32   35 / 11
//   512 at 7680, 32/8 x 128  174 / 156     512 at 7680, 16/8 x 64 106 / 51
struct AttnPlan {
    int splits, stages;  // stages of 64 keys per split
};
// wgs: workgroups without splits; wg_bytes: a workgroup's part
inline AttnPlan attention_plan(int hd, int64_t wgs, int stages, size_t wg_bytes, int cus, size_t part_bytes) {
    constexpr int kSplitsMax = 32;
    const double kStart = 4.0, kStage = hd == 128 ? 1.45 : hd == 64 ? 0.85 : 0.7;
    const double kFull = hd == 128 ? 1.3 : hd == 64 ? 0.75 : 0.5;
    const int kSlots = hd == 128 ? 2 : hd == 64 ? 3 : 4;
    AttnPlan plan{1, stages};
    double best = 1e30;
    for (int s = 1; s <= kSplitsMax && s <= stages; ++s) {
        const size_t bytes = (size_t)wgs * s * wg_bytes;
        if (s > 1 && bytes > part_bytes) break;
        const int p = (stages + s - 1) / s;
        if ((stages + p - 1) / p != s) continue;  // the same stages in fewer splits
        const int64_t on_cu = (wgs * s + cus - 1) / cus, rounds = (on_cu + kSlots - 1) / kSlots;
        const double full = kFull * (double)on_cu, alone = kStage * (double)rounds;
        double us = kStart * (double)rounds + p * (full > alone ? full : alone);
        if (s > 1) us += 3.5 + 0.3 * s + (double)bytes / 5e6;
        if (us < best) best = us, plan = AttnPlan{s, p};
    }
    return plan;
}

}  // namespace mxh

// How a product of many rows is split over workgroups (gemm_rows.hip), and
// from which size on (host arithmetic, no device code); sanitize/plan_check.cpp
// checks the line against measured pairs on the CPU.
#pragma once

#include <algorithm>
#include <cstdint>

#include "common.h"

namespace qwh {
namespace plan {

constexpr uint32_t kRowsTile = 32;    // tokens, and weight rows, of one MFMA tile
constexpr uint32_t kRowsWaves = 4;    // wavefronts of a workgroup, a tile of rows each
constexpr uint32_t kDies = 8;

struct RowsPlan {
    int token_tiles = 1;  // per workgroup
    uint32_t slices = 1, slice_groups = 0;
    float us = 0.0f;      // estimated, without the activation pass
};

// One group step of a CU that holds `per_cu` workgroups (us), as sweeps of
// shapes from 896 x 896 to 12288 x 2048 at 64 to 1024 tokens measured it: a
// CU's first workgroup waits for its own loads and barriers, which more of
// them hide.
inline float rows_step_us(int token_tiles, uint32_t per_cu) {
    if (token_tiles == 2) return per_cu == 1 ? 0.76f : per_cu == 2 ? 1.13f : 0.53f * (float)per_cu;
    return per_cu == 1 ? 0.62f : per_cu == 2 ? 0.77f : 0.38f * (float)per_cu;
}

// Token tiles per workgroup and K slices by the least estimated time; a split
// writes its partial sums and reads them back, in a launch of its own unless
// the caller's next pass adds them (`folded`).
inline RowsPlan rows_plan(int cus, uint32_t tokens, uint32_t rows, uint32_t cols, uint32_t max_slices, bool folded) {
    const uint32_t groups = cols / 64, tiles = (tokens + kRowsTile - 1) / kRowsTile;
    const uint32_t row_blocks = (rows + kRowsWaves * kRowsTile - 1) / (kRowsWaves * kRowsTile);
    RowsPlan best;
    best.slice_groups = groups;
    for (int tt = 1; tt <= 2; ++tt)
        for (uint32_t want = 1; want <= max_slices; ++want) {
            RowsPlan p;
            p.token_tiles = tt;
            // Slices of whole weight chunks, none empty.
            p.slice_groups = ((groups + want - 1) / want + 3) & ~3u;
            p.slices = (groups + p.slice_groups - 1) / p.slice_groups;
            if (p.slices != want) continue;
            // The fullest die's share.
            const uint64_t units = ((uint64_t)row_blocks * p.slices + kDies - 1) / kDies;
            const uint64_t die_cus = std::max(1u, (uint32_t)cus / kDies);
            const uint32_t per_cu = (uint32_t)((units * ((tiles + tt - 1) / tt) + die_cus - 1) / die_cus);
            p.us = (float)std::min(p.slice_groups, groups) * rows_step_us(tt, per_cu);
            // (Even by the estimate, four and more slices that leave CUs two
            // workgroups lose to half as many: 2048 x 2048 q4 at 385 to 416
            // tokens 30.5 / 26.8, 4096 x 2048 at 192 25.0 / 23.4.)
            if (p.slices >= 4 && per_cu > 1 && !folded) p.us += 0.4f;
            if (p.slices > 1)
                p.us += (folded ? 0.5f : 3.0f) + (float)p.slices * (float)(tiles * kRowsTile) * (float)rows * 8.0f / 4.5e6f;
            if (best.us == 0.0f || p.us < best.us) best = p;
        }
    return best;
}

// The 16-token tiles (gemv_batch.hip) take less fixed time: their activation
// pass needs no whole row, and more and smaller workgroups fill the device.
// Both sides, f32 rows in and out, weights not yet cached (us, 16-token tiles
// against these): 2048 x 6144 at 128 tokens q4 26.1 / 23.6, q8 27.6 / 24.5;
// 6144 x 1024 at 256 20.7 / 17.9 and 22.6 / 20.3; 3584 x 896 at 512 23.0 /
// 18.3; 2048 x 2048 at 402 27.8 / 26.4 and 29.9 / 28.1; 12288 x 2048 at 402
// 91.9 / 59.1. They meet near 1.6e9 multiply-adds (8191 x 1024 q4 at 192 tokens
// 19.0 / 20.6, q8 23.8 / 23.3; 2048 x 6144 q5 at 144 30.7 / 32.1). Less than
// four row blocks, the last one often partly empty, gain only where the 16-token
// tiles have no good split, past 6144 values (100 x 6144 at 4000 tokens 60.9 /
// 69.7, 33 x 1088 at 44600 126 / 186, 300 x 4096 at 3000 57.8 / 61.0; 200 x 8128
// at 1000 83.5 / 36.4), or no form at all, q5 of an odd number of groups (33 x
// 1088 636 / 196).
inline bool rows_preferred(int format, uint32_t rows, uint32_t cols, uint32_t tokens) {
    const uint64_t work = (uint64_t)rows * cols * tokens;
    return tokens >= 128 && work >= 1600000000ull &&
           (rows >= 512 || cols > 6144 || (format == QWH_FORMAT_Q5 && cols / 64 % 2));
}

}  // namespace plan
}  // namespace qwh

// Where a few tokens' products run (host arithmetic, no device code): one
// launch of a per-token GEMV, which reads the matrix once per token, mostly
// from the caches, or the matrix-core form's two or three (activation digits,
// product, slice sum). gemv.hip asks it with the shapes its kernels have;
// sanitize/plan_check.cpp checks it against measured pairs on the CPU.
//
// Measured with the matrix not yet cached, as a model's layers find it (copies
// of 800 MB in turn; us, per-token GEMV / matrix cores): the launches saved
// are worth 5.8 us, and the GEMV's time grows with rows x K x tokens, by its
// kernel's layout:
//   q4            4096 x 1024 and 16 tokens 6.8 / 9.6, 12288 x 2048 and 4 10.4 /
//                 12.8; even at 105e6. Three slices a lane (K = 1536, 3072,
//                 6144) cost more: 2048 x 3072 even at 12 tokens, 2048 x 6144
//                 8.0 / 10.8 at 4 and 0.3 less at 6.
//   q5, q8        rows of a power of two from 256 to 4096, 3072 and 6144
//                 values: even at 50e6 (4096 x 1024 and 12 tokens, 4096 x 2048
//                 and 6), from 3072 on at 40e6 (1024 x 6144 and 7, 2048 x 3072
//                 and 6); with two tokens a third later (8191 x 3072 11.4 / 15.5).
//   q5, q8 else   a wavefront a row, whatever its length: K = 896 even at 17000
//                 rows x tokens, 2560 and 3584 at 9500, 5120 at 7900. (12288 x
//                 128 q5 and 12 tokens: 31 us slower than the matrix cores.)
//                 Where the matrix cores' form has one launch fewer (K of an odd
//                 number of groups, or short), half of that: 128 and 448 at
//                 9000. Two tokens gain up to 12288 rows of 512 values and more
//                 (12288 x 896 q8 9.7 / 13.0, 8191 x 2560 q5 13.1 / 14.7).
#pragma once

#include <cstdint>

#include "common.h"

namespace qwh {
namespace plan {

// The layout of the GEMV's rows: a lane takes `slices` 32-value slices, `lanes`
// of them a row.
struct RowLanes {
    uint32_t slices, lanes;
};

inline RowLanes row_lanes(uint32_t cols) {
    const uint32_t t = cols / 32;
    uint32_t lanes = 64;
    while (t % lanes) lanes /= 2;
    return {t / lanes, lanes};
}

// q5 / q8 rows without a kernel of their length: a wavefront a row.
inline bool wavefront_rows(int format, uint32_t cols) {
    const RowLanes r = row_lanes(cols);
    return format != QWH_FORMAT_Q4 &&
           !(r.slices == 1 ? r.lanes >= 8 : r.slices == 2 ? r.lanes == 64 : r.slices == 3 && r.lanes >= 32);
}

// A token's product on the per-token GEMV, in the weight values of the
// cheapest layout that take as long.
inline uint64_t token_gemv_work(int format, uint32_t rows, uint32_t cols) {
    const uint64_t values = (uint64_t)rows * cols;
    if (format == QWH_FORMAT_Q4)
        return cols > 3072 ? values * 105 / 64 : row_lanes(cols).slices == 3 ? values * 105 / 72 : values;
    if (!wavefront_rows(format, cols)) return cols > 2048 ? values * 5 / 4 : values;
    const uint64_t row = cols <= 2048 ? 3072 : 2400 + (uint64_t)cols * 4 / 5;
    return rows * row * (cols < 512 || cols / 64 % 2 ? 2 : 1);
}

// One product of `tokens` tokens.
inline bool token_gemv(int format, uint32_t rows, uint32_t cols, uint32_t tokens) {
    const bool q4 = format == QWH_FORMAT_Q4;
    if (tokens == 2 && cols >= 512 && rows <= 12288 && wavefront_rows(format, cols)) return true;
    const uint64_t most = q4 ? 105000000u : tokens == 2 ? 67200000u : 50400000u;
    return tokens >= 2 && tokens <= (q4 ? 16u : 12u) && token_gemv_work(format, rows, cols) * tokens <= most;
}

// A decoder layer's products, six launches against nine. Four steps (ms, this
// form / matrix cores): q4 0.6B at 3 and 8 sequences 3.51 / 5.18 and 4.59 /
// 5.67, 1.7B at 5 and 7 5.88 / 6.19 and 7.15 / 6.39; q8 0.6B at 8 5.58 / 5.83,
// 1.7B at 3 and 4 6.25 / 6.43 and 7.28 / 6.50; q5 1.7B at 3 and 4 5.81 / 6.39
// and 6.77 / 6.46. Each matrix counts by its own format. Two sequences, which
// gain as well (3.29 / 4.99), stay on the matrix cores: the prefill's tests hold
// a prompt's rows to the steps of a two-sequence decoder of the same products.
// (Other batches have no such twin.)
inline bool token_gemv_layer(const Matrix *const *matrices, uint32_t count, uint32_t tokens) {
    if (tokens < 3 || tokens > 8) return false;
    double share = 0.0;
    for (uint32_t i = 0; i < count; ++i) {
        const Matrix &m = *matrices[i];
        share += (double)token_gemv_work(m.format, m.rows, m.cols) * tokens / (m.format == QWH_FORMAT_Q4 ? 300e6 : 165e6);
    }
    return share <= 1.0;
}

}  // namespace plan
}  // namespace qwh

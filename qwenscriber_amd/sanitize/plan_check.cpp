// CPU check of the decode attention's scratch sizing (attention_plan.h),
// built with g++ only: for every shape and form the decoder step, the
// prefill and the attention entry points launch, the bytes they allocate
// (sized before the launch form is known) hold the records of the ranges
// the launch then writes. And of the products' rules (gemv_plan.h,
// rows_plan.h) against measured pairs. Exit status 0 when every case holds.
#include <cstdio>

#include "../csrc/attention_plan.h"
#include "../csrc/gemv_plan.h"
#include "../csrc/rows_plan.h"

using qwh::AttentionArgs;
namespace plan = qwh::plan;

namespace {

struct Heads {
    uint32_t heads, kv_heads, head_dim;
};

long cases = 0, failures = 0;

// `sized`: the bytes the caller allocated; the launch writes the records of
// the form it takes (decoder: q / k norms given).
void check(const char *who, int cus, const AttentionArgs &a, bool decoder, size_t sized) {
    uint32_t chunk = 0, splits = 0;
    plan::attention_shape(cus, a, decoder, chunk, splits);
    const size_t need = plan::record_bytes(a, splits);
    ++cases;
    // Every range starts below the capacity and the ranges cover it.
    const bool ranges_ok = splits >= 1 && (uint64_t)(splits - 1) * chunk < a.capacity &&
                           (uint64_t)splits * chunk >= a.capacity && chunk % (plan::kTile * plan::kWaves) == 0;
    if (need > sized || !ranges_ok) {
        ++failures;
        if (failures <= 20)
            std::printf("FAIL %s: cus %d heads %u/%u d %u batch %u capacity %u f32 %d decoder %d: "
                        "splits %u chunk %u need %zu sized %zu\n",
                        who, cus, a.heads, a.kv_heads, a.head_dim, a.batch, a.capacity, (int)a.f32_cache,
                        (int)decoder, splits, chunk, need, sized);
    }
}

// A few tokens' product as measured with cold weights (us, calls in a row):
// the per-token GEMV, and the matrix-core form.
struct Pair {
    int format;
    uint32_t rows, cols, tokens;
    float first, second;  // us: the form that the rule takes where it is faster, and the other
};

const Pair pairs[] = {
    {QWH_FORMAT_Q4, 4096, 1024, 16, 6.9f, 9.2f},
    {QWH_FORMAT_Q4, 12288, 2048, 4, 10.4f, 12.6f},
    {QWH_FORMAT_Q4, 8191, 1024, 8, 8.0f, 9.6f},
    {QWH_FORMAT_Q4, 2048, 3072, 8, 7.2f, 9.4f},
    {QWH_FORMAT_Q4, 2048, 3072, 16, 11.9f, 9.5f},
    {QWH_FORMAT_Q4, 8191, 3072, 4, 15.1f, 12.8f},
    {QWH_FORMAT_Q4, 2048, 6144, 4, 8.0f, 10.8f},
    {QWH_FORMAT_Q4, 1024, 6144, 16, 12.4f, 10.5f},
    {QWH_FORMAT_Q4, 256, 128, 2, 3.7f, 5.9f},
    {QWH_FORMAT_Q4, 4096, 1536, 16, 10.7f, 9.3f},
    {QWH_FORMAT_Q5, 4096, 1024, 8, 6.3f, 9.1f},
    {QWH_FORMAT_Q5, 8191, 1024, 12, 15.1f, 10.5f},
    {QWH_FORMAT_Q5, 1024, 3072, 8, 6.2f, 9.3f},
    {QWH_FORMAT_Q5, 2048, 6144, 2, 7.1f, 10.9f},
    {QWH_FORMAT_Q5, 2048, 6144, 6, 15.7f, 11.0f},
    {QWH_FORMAT_Q5, 12288, 128, 12, 38.2f, 6.8f},
    {QWH_FORMAT_Q5, 4096, 896, 2, 6.0f, 8.7f},
    {QWH_FORMAT_Q5, 4096, 896, 8, 15.4f, 8.9f},
    {QWH_FORMAT_Q5, 4096, 896, 12, 21.6f, 8.9f},
    {QWH_FORMAT_Q5, 2048, 3584, 12, 21.1f, 9.6f},
    {QWH_FORMAT_Q5, 8191, 3072, 2, 10.9f, 15.0f},
    {QWH_FORMAT_Q5, 12288, 2048, 2, 9.4f, 14.7f},
    {QWH_FORMAT_Q5, 1024, 896, 8, 5.7f, 9.8f},
    {QWH_FORMAT_Q8, 1024, 3072, 2, 4.4f, 9.4f},
    {QWH_FORMAT_Q8, 4096, 1024, 8, 6.6f, 9.1f},
    {QWH_FORMAT_Q8, 12288, 2048, 2, 11.0f, 14.4f},
    {QWH_FORMAT_Q8, 12288, 2048, 4, 19.4f, 14.7f},
    {QWH_FORMAT_Q8, 4096, 2048, 12, 16.7f, 9.9f},
    {QWH_FORMAT_Q8, 2048, 6144, 6, 16.9f, 11.4f},
    {QWH_FORMAT_Q8, 12288, 128, 12, 31.2f, 6.6f},
    {QWH_FORMAT_Q8, 4096, 896, 2, 5.7f, 8.9f},
    {QWH_FORMAT_Q8, 4096, 896, 12, 19.8f, 9.1f},
    {QWH_FORMAT_Q8, 2048, 448, 2, 3.9f, 6.1f},
    {QWH_FORMAT_Q8, 8191, 448, 8, 19.0f, 7.0f},
    {QWH_FORMAT_Q8, 1024, 2560, 4, 5.8f, 9.5f},
    {QWH_FORMAT_Q8, 4096, 3584, 8, 26.9f, 11.2f},
    {QWH_FORMAT_Q8, 1024, 5120, 4, 7.6f, 11.7f},
    {QWH_FORMAT_Q8, 2048, 5120, 8, 20.4f, 12.1f},
    {QWH_FORMAT_Q8, 8191, 6144, 2, 27.9f, 20.2f},
    {QWH_FORMAT_Q8, 8191, 512, 4, 4.8f, 9.4f},
    {QWH_FORMAT_Q8, 12288, 896, 2, 9.6f, 13.0f},
    {QWH_FORMAT_Q8, 8191, 1344, 2, 8.1f, 9.9f},
    {QWH_FORMAT_Q5, 8191, 2560, 2, 13.1f, 14.7f},
    {QWH_FORMAT_Q5, 12288, 128, 2, 10.1f, 6.5f},
};

// The rule takes the faster form of each pair, where they are apart.
void check_token_gemv() {
    for (const Pair &p : pairs) {
        const bool takes = plan::token_gemv(p.format, p.rows, p.cols, p.tokens);
        ++cases;
        if (takes == (p.first < p.second)) continue;
        ++failures;
        std::printf("FAIL few tokens: format %d %u x %u, %u tokens: per token %.1f us, matrix cores %.1f, rule %d\n", p.format,
                    p.rows, p.cols, p.tokens, p.first, p.second, (int)takes);
    }
    // A layer's matrices count by their own formats: 0.6B shapes, 8 sequences,
    // with q4 or q8 products; the 1.7B's at 3 and 5 with its down product in
    // the other format.
    auto layer = [](uint32_t hidden, uint32_t ffn, int format, int down, uint32_t tokens) {
        qwh::Matrix m[4];
        const uint32_t shapes[4][2] = {{4096, hidden}, {hidden, 2048}, {2 * ffn, hidden}, {hidden, ffn}};
        const qwh::Matrix *all[4];
        for (int i = 0; i < 4; ++i) {
            m[i].format = i == 3 ? down : format;
            m[i].rows = shapes[i][0], m[i].cols = shapes[i][1];
            all[i] = &m[i];
        }
        return plan::token_gemv_layer(all, 4, tokens);
    };
    const int q4 = QWH_FORMAT_Q4, q8 = QWH_FORMAT_Q8;
    const bool rule[] = {layer(1024, 3072, q4, q4, 8), layer(1024, 3072, q8, q8, 8), layer(2048, 6144, q4, q4, 5),
                         layer(2048, 6144, q8, q8, 3), !layer(2048, 6144, q4, q4, 6), !layer(2048, 6144, q8, q8, 4),
                         !layer(2048, 6144, q4, q8, 5), layer(2048, 6144, q4, q8, 4), !layer(2048, 6144, q8, q4, 4),
                         !layer(1024, 3072, q4, q4, 2), !layer(1024, 3072, q4, q4, 9)};
    for (const bool &holds : rule) {
        ++cases;
        if (!holds) ++failures, std::printf("FAIL layer rule %d\n", (int)(&holds - rule));
    }
}

// Many tokens' product: the 32-token tiles, and the 16-token ones.
const Pair many[] = {
    {QWH_FORMAT_Q4, 2048, 2048, 402, 26.4f, 27.8f},
    {QWH_FORMAT_Q8, 2048, 2048, 402, 28.1f, 29.9f},
    {QWH_FORMAT_Q4, 2048, 2048, 512, 27.7f, 30.7f},
    {QWH_FORMAT_Q8, 4096, 2048, 224, 26.9f, 30.0f},
    {QWH_FORMAT_Q4, 2048, 6144, 128, 23.7f, 26.1f},
    {QWH_FORMAT_Q5, 2048, 6144, 160, 32.4f, 33.1f},
    {QWH_FORMAT_Q8, 6144, 1024, 256, 20.2f, 22.6f},
    {QWH_FORMAT_Q4, 4096, 1024, 402, 20.1f, 22.6f},
    {QWH_FORMAT_Q5, 3584, 896, 512, 21.9f, 25.7f},
    {QWH_FORMAT_Q8, 896, 7680, 256, 29.6f, 30.7f},
    {QWH_FORMAT_Q4, 1024, 6144, 256, 25.1f, 27.1f},
    {QWH_FORMAT_Q8, 2048, 3072, 256, 25.3f, 27.4f},
    {QWH_FORMAT_Q5, 3000, 2560, 224, 27.2f, 30.9f},
    {QWH_FORMAT_Q8, 8191, 1024, 224, 22.9f, 27.7f},
    {QWH_FORMAT_Q4, 12288, 2048, 128, 27.2f, 36.0f},
    {QWH_FORMAT_Q4, 33, 1088, 44600, 186.2f, 126.9f},
    {QWH_FORMAT_Q5, 33, 1088, 44600, 196.2f, 636.5f},
    {QWH_FORMAT_Q8, 100, 6144, 4000, 71.7f, 65.3f},
    {QWH_FORMAT_Q4, 300, 4096, 3000, 61.0f, 57.8f},
    {QWH_FORMAT_Q8, 200, 8128, 1000, 38.6f, 85.0f},
    {QWH_FORMAT_Q4, 1600, 7808, 129, 28.0f, 57.6f},
    {QWH_FORMAT_Q8, 1480, 8256, 131, 35.7f, 44.2f},
};

void check_rows() {
    for (const Pair &p : many) {
        const bool takes = plan::rows_preferred(p.format, p.rows, p.cols, p.tokens);
        ++cases;
        if (takes == (p.first < p.second)) continue;
        ++failures;
        std::printf("FAIL many tokens: format %d %u x %u, %u tokens: 32-token tiles %.1f us, 16-token %.1f, rule %d\n", p.format,
                    p.rows, p.cols, p.tokens, p.first, p.second, (int)takes);
    }
}

}  // namespace

int main() {
    check_token_gemv();
    check_rows();
    // The Qwen3-ASR decoders (0.6B: 16 / 8 heads of 128; 1.7B the same
    // heads), the test suites' shapes, and every head layout the kernels
    // are built for.
    const Heads heads[] = {{16, 8, 128}, {4, 2, 128}, {5, 5, 64}, {8, 2, 64}, {16, 2, 128}, {16, 4, 64},
                           {2, 2, 256}, {4, 2, 256}, {8, 8, 128}, {64, 8, 128}};
    const int cus_list[] = {256, 304, 80, 1};
    const uint32_t capacities[] = {1, 2, 31, 64, 127, 128, 255, 256, 257, 600, 4096, 4352, 8192};
    for (const Heads &h : heads)
        for (int cus : cus_list)
            for (uint32_t capacity : capacities)
                for (uint32_t batch = 1; batch <= 300; batch += batch < 20 ? 1 : 37)
                    for (int f32 = 0; f32 < 2; ++f32) {
                        AttentionArgs a{};
                        a.heads = h.heads;
                        a.kv_heads = h.kv_heads;
                        a.head_dim = h.head_dim;
                        a.batch = batch;
                        a.capacity = capacity;
                        a.f32_cache = f32 != 0;
                        // The decoder sizes its scratch at create, before the
                        // norm pointers exist, and launches the decoder form.
                        const size_t at_create = plan::scratch_bytes(cus, a);
                        check("decoder step", cus, a, true, at_create);
                        // The attention entry points size and launch the
                        // plain form.
                        check("entry point", cus, a, false, at_create);
                        // The prefill sizes with its chunk's rows as the batch
                        // and the positions through the chunk as the capacity,
                        // norm pointers given, and launches the decoder form.
                        AttentionArgs p = a;
                        p.prefill = true;
                        check("prefill", cus, p, true, plan::scratch_bytes(cus, p));
                    }
    std::printf("plans: %ld cases, %ld failures\n", cases, failures);
    return failures ? 1 : 0;
}

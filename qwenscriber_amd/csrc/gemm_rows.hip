// Quantized matrices times many rows of f32 activations (kernels.zig:118-158
// linearQuantized with tokens = M: a prompt's positions, the audio tower's
// steps) on the f16 matrix cores.
//
// Each token's row is split once into two f16 terms of x * 2^s (s from the
// row's largest finite magnitude, so |x * 2^s| < 2^14): hi rounded to f16, lo
// the exact remainder rounded to f16. A value is kept to 2^-22 of itself or
// 2^-39 of what s was taken from, whichever is more. A row with a 64-value group
// more than 2^15 below its largest takes s from each group instead (an
// "uneven" row), so the split is at least as close as 23-bit integers per group
// (the small batch's digit planes) whatever the row holds: one s for a row with
// a value 1e8 times the others left them 1e-4 of themselves. The codes are
// small integers, exact in f16, and code * term products are exact in f32; the
// matrix core adds both terms' products of one group into one f32 partial,
// which takes the group's f16 scale in one FMA, in a workgroup with an uneven
// row times the token's 2^-s (2048 x 6144 q8 and 12288 x 2048 q4 at 402 tokens:
// 43.4 and 58.1 us, 47.0 and 68.2 with all rows uneven).
//
// Operands. One v_mfma_f32_32x32x16_f16 multiplies 32 tokens by 32 weight
// rows over 16 columns: lane l feeds token (or row) l % 32 and 8 columns, so
// a group is four steps s of two lane halves h: columns 32 h + 8 s .. + 7.
// Within those eight, the pair order is the one the format's decode gives for
// nothing: (i, i + 4) for nibbles, (2 i, 2 i + 1) for bytes; the activations
// are stored in that order.
//   activations  [32-token tile][group][step][hi, lo][lane][8] f16: a lane's
//                operand is one 16-byte word, a wavefront's 1 KiB in lane
//                order (whole-line loads, conflict-free LDS reads);
//   weights      lane l's half group row, 16 (q4), 16 + 4 (q5) or 32 (q8)
//                contiguous bytes, decoded in registers: every wavefront has
//                rows of its own, so no weight goes through LDS.
// With the tokens as the result's rows, a lane's 16 results of a tile belong
// to one weight row: one scale per lane and group.
//
// Where a SIMD has two and more wavefronts, near the shared issue of matrix cores
// and vector unit (two products per weight, and per group the decode and 16
// scale FMAs a tile): 12288 x 2048 q4 at 402 tokens keeps them busy 32 and 40 %
// of the cycles, 370 TFLOP/s, and at 2048 tokens reaches 440-475 (twice that in
// f16 products, of the 1.2 PFLOP/s an 8192^3 f16 matmul reaches on the same
// card). With one or two a SIMD it waits for its own loads and barriers: 4096 x
// 2048 18 and 19 %, 2048 x 2048 14 and 17 %. No LDS bank conflicts. Tiles of 64
// rows or 128 tokens a wavefront, or eight wavefronts, measured within 10 %.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.h"
#include "device.h"
#include "rows_plan.h"

namespace qwh {
namespace {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f16x __attribute__((ext_vector_type(16)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));

using plan::RowsPlan;
using plan::rows_plan;

constexpr int kTile = plan::kRowsTile;                 // tokens, and weight rows, of one MFMA tile
constexpr int kStepBytes = 2 * 64 * 16;                // hi and lo of one step
constexpr int kGroupPieces = 4 * kStepBytes / 16;      // 16-byte words of a (tile, group)

enum class Codes : int { Q4 = 0, Q5 = 1, Q8 = 2 };

constexpr int code_bytes(Codes c) { return c == Codes::Q4 ? 32 : c == Codes::Q5 ? 40 : 64; }
// Registers of a lane's half group row.
constexpr int code_words(Codes c) { return c == Codes::Q4 ? 4 : c == Codes::Q5 ? 5 : 8; }

__device__ __forceinline__ uint32_t sub2(uint32_t v, _Float16 bias) {
    const h2 b = {bias, bias};
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2, v) - b);
}

// The operand of step s from a lane's half group row w. An f16 with exponent
// bits 0x64 (0x54) holds 1024 + m (64 + m / 16) for a mantissa field m, so an
// AND-OR places two codes and one packed subtraction centres them, exactly.
template <Codes C>
__device__ __forceinline__ h8 decode(const uint32_t (&w)[code_words(C)], int s) {
    uint32_t r[4];
    if constexpr (C == Codes::Q4) {
        const uint32_t a = w[s], b = a >> 8;
        r[0] = sub2((a & 0x000f000fu) | 0x64006400u, (_Float16)1032.0f);
        r[1] = sub2((a & 0x00f000f0u) | 0x54005400u, (_Float16)72.0f);
        r[2] = sub2((b & 0x000f000fu) | 0x64006400u, (_Float16)1032.0f);
        r[3] = sub2((b & 0x00f000f0u) | 0x54005400u, (_Float16)72.0f);
    } else if constexpr (C == Codes::Q5) {
        // Byte s of the fifth bits holds the eight columns' in order: bit i
        // and bit i + 4 go to bits 4 and 20.
        const uint32_t f = (w[4] >> (8 * s)) & 0xffu, m = f | (f << 12);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            r[i] = sub2(((w[s] >> (4 * i)) & 0x000f000fu) | ((m << (4 - i)) & 0x00100010u) | 0x64006400u,
                        (_Float16)1040.0f);
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            r[i] = sub2(__builtin_amdgcn_perm(0x64646464u, w[2 * s + i / 2], i % 2 ? 0x04030402u : 0x04010400u),
                        (_Float16)1152.0f);
    }
    const u4 v = {r[0], r[1], r[2], r[3]};
    return __builtin_bit_cast(h8, v);
}

template <Codes C>
__device__ __forceinline__ void load_codes(const uint8_t *group_row, int h, uint32_t (&w)[code_words(C)]) {
    if constexpr (C == Codes::Q5) {
        __builtin_memcpy(w, group_row + 16 * h, 16);
        __builtin_memcpy(w + 4, group_row + 32 + 4 * h, 4);
    } else {
        constexpr int bytes = code_bytes(C) / 2;
        const u4 *p = reinterpret_cast<const u4 *>(group_row + bytes * h);
#pragma unroll
        for (int i = 0; i < bytes / 16; ++i) {
            const u4 v = p[i];
            w[4 * i] = v.x, w[4 * i + 1] = v.y, w[4 * i + 2] = v.z, w[4 * i + 3] = v.w;
        }
    }
}

// s_waitcnt operand: at most N vector memory operations and no LDS operation
// outstanding.
template <int N>
constexpr int kWait = (N & 15) | (7 << 4) | ((N >> 4) << 14);

template <int N, int I = 0, class F>
__device__ __forceinline__ void static_for(F f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<N, I + 1>(f);
    }
}

struct RowsArgs {
    const uint16_t *scales;
    const uint8_t *data;
    const uint8_t *halves;   // the split activations
    const float *factor;     // per token: 1, or 1 / rms with RMSNorm
    const float *scale;      // per token: 2^-s, or 0 of an uneven row
    const float *uneven;     // [32-token tile][group][token]: 2^-s of an uneven row's groups
    float *out;              // tokens x n, or tokens x n / 2 with pairs
    const float *residual;   // optional, tokens x n (may alias out): out = residual + W x; not with pairs
    float *part;             // non-null: [slice][token][n] partial sums instead of out
    uint32_t n, groups, tokens;
    uint32_t pairs;
    uint32_t row_blocks, token_blocks;
    uint32_t slices, slice_groups;
};

// silu(g) * u (math.zig:69-71).
__device__ __forceinline__ float silu_times(float g, float u) {
    return __fmul_rn(__fdiv_rn(g, __fadd_rn(1.0f, expf(-g))), u);
}

// A workgroup of W wavefronts covers 32 rows a wavefront and 32 * TT tokens over
// one K slice. Each group's activations (TT * 8
// KiB) are staged in LDS for all wavefronts, two buffers, one barrier a group;
// weights are loaded two groups (128 bytes of a row for q8) or four (q4) at a
// time, one such chunk ahead.
template <Codes C, int W, int TT>
__device__ __forceinline__ void rows_block(const RowsArgs &a, uint32_t row_block, uint32_t token_block,
                                           uint32_t slice) {
    constexpr int CG = C == Codes::Q4 ? 4 : 2;           // groups of a weight chunk
    constexpr int PIECES = TT * kGroupPieces;
    constexpr int PT = PIECES / (64 * W);                // 16-byte words per thread and group
    constexpr int CW = code_words(C);
    constexpr int WL = CG * (C == Codes::Q4 ? 1 : 2) + 1;  // loads of a weight chunk
    static_assert(PIECES % (64 * W) == 0, "whole words per thread");
    constexpr int D = 3;
    __shared__ u4 al[D][PIECES];
    __shared__ float inv[TT * kTile];
    __shared__ __attribute__((aligned(16))) float mult[W][64];  // a group's 2^-s by token, a copy for each wavefront
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int col = lane & 31, half = lane >> 5;
    const uint32_t tiles = (a.tokens + kTile - 1) / kTile;
    const uint32_t tile0 = token_block * TT;
    const uint32_t row0 = (row_block * W + wave) * kTile;
    const uint32_t g0 = slice * a.slice_groups;
    const uint32_t g1 = min(g0 + a.slice_groups, a.groups);
    const size_t row_bytes = (size_t)a.groups * code_bytes(C);

    // (Rows past the matrix read its last row; their results are dropped.)
    const uint32_t my_row = min(row0 + col, a.n - 1);
    const uint8_t *wp = a.data + my_row * row_bytes;
    const uint16_t *sp = a.scales + (size_t)my_row * a.groups;
    const u4 *ap[PT];  // this thread's words of group 0
#pragma unroll
    for (int m = 0; m < PT; ++m) {
        const int q = tid + 64 * W * m;
        const uint32_t tile = min(tile0 + q / kGroupPieces, tiles - 1);
        ap[m] = reinterpret_cast<const u4 *>(a.halves) + (size_t)tile * a.groups * kGroupPieces + q % kGroupPieces;
    }
    // This lane's token in the multipliers' order.
    const uint32_t my_token = min(tile0 * kTile + (TT == 2 ? lane : col), a.tokens - 1);
    const float my_scale = a.scale[my_token], my_factor = a.factor[my_token];

    f16x acc[TT];
#pragma unroll
    for (int t = 0; t < TT; ++t) acc[t] = f16x{};

    uint32_t rw[CG][CW];
    uint32_t rs[CG / 2];  // the chunk's scales, two to a word
    auto load_acts = [&](uint32_t g, int to) __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < PT; ++m)
            __builtin_amdgcn_global_load_lds(
                reinterpret_cast<const __attribute__((address_space(1))) uint32_t *>(
                    reinterpret_cast<uintptr_t>(ap[m] + (size_t)g * kGroupPieces)),
                reinterpret_cast<__attribute__((address_space(3))) uint32_t *>(
                    reinterpret_cast<uintptr_t>(&al[to][wave * 64 + 64 * W * m])), 16, 0, 0);
    };
    auto load_weights = [&](uint32_t g) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < CG; ++i) {
            const uint32_t gi = min(g + i, g1 - 1);
            load_codes<C>(wp + (size_t)gi * code_bytes(C), half, rw[i]);
        }
        // One load for the chunk's scales (one a group, from 32 rows' lines
        // each time, took 12 of 68 us). A last, shorter chunk reads the row's
        // last CG, shifted into place at their use.
        const uint32_t gs = min(g, a.groups - CG);
        __builtin_memcpy(rs, sp + gs, 2 * CG);
    };
    load_weights(g0);
    __builtin_amdgcn_sched_barrier(0);
    // (Before the copies to LDS: with one in flight the compiler waits for
    // everything.)
    const bool uneven = __builtin_amdgcn_ballot_w64(my_scale == 0.0f) != 0;  // the same in every wavefront
    if (tid < TT * kTile) inv[tid] = uneven ? my_factor : __fmul_rn(my_scale, my_factor);
    __builtin_amdgcn_sched_barrier(0);
    load_acts(g0, 0);
    load_acts(min(g0 + 1, g1 - 1), 1);
    __builtin_amdgcn_s_waitcnt(kWait<PT>);  // the first weights and words (the steps' counts assume a step before)
    __builtin_amdgcn_sched_barrier(0);
    int buf = 0;
    uint32_t cw[CG][CW];
    uint32_t cs[CG / 2];
    auto take_chunk = [&](uint32_t gc) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < CG; ++i)
#pragma unroll
            for (int k = 0; k < CW; ++k) cw[i][k] = rw[i][k];
#pragma unroll
        for (int i = 0; i < CG / 2; ++i) cs[i] = rs[i];
        if (gc + CG > a.groups) {
            uint64_t v = 0;
            __builtin_memcpy(&v, cs, 2 * CG);
            v >>= 16 * (gc + CG - a.groups);
            __builtin_memcpy(cs, &v, 2 * CG);
        }
    };
    // p = this buffer's group times the codes w.
    auto multiply = [&](const uint32_t (&w)[CW], f16x (&p)[TT]) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < TT; ++t) p[t] = f16x{};
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const h8 b = decode<C>(w, s);
#pragma unroll
            for (int t = 0; t < TT; ++t) {
                const u4 *word = &al[buf][t * kGroupPieces + s * 128 + lane];
                const h8 hi = __builtin_bit_cast(h8, word[0]), lo = __builtin_bit_cast(h8, word[64]);
                p[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(hi, b, p[t], 0, 0, 0);
                p[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(lo, b, p[t], 0, 0, 0);
            }
        }
    };
    // Group gc + i of the chunk taken at gc; `tail`: of the last, shorter chunk.
    auto step = [&](auto at, auto tail, uint32_t gc) __attribute__((always_inline)) {
        constexpr int i = decltype(at)::value;
        constexpr bool ahead = !decltype(tail)::value;
        const uint32_t g = gc + i;
        // This group's words have landed (what was issued after them, the
        // next group's and in some steps a chunk of weights, may still be on
        // its way: vector memory completes in order), in every wavefront
        // after the barrier; the buffer refilled now was last read before it.
        // No weights follow the last chunk (the compiler would drop loads that
        // nothing uses, and a count that expects them would not wait). In the
        // two-group chunks of q5 and q8 the codes taken at i == 0 are awaited
        // by the compiler's own wait, which with copies to LDS in flight is
        // for everything: once a chunk nothing travels. Counting PT there
        // keeps the next words in flight: 4096 x 2048 q8 at 402 tokens 34.9 ->
        // 31.2 us, where a CU has one workgroup, but 2048 x 6144 43.0 -> 44.1
        // and 896 x 7680 34.1 -> 35.7, where it has two.
        constexpr int after = PT + (ahead && (i == 1 || i == 2 || CG == 2) ? WL : 0);
        __builtin_amdgcn_s_waitcnt(kWait<after>);
        __builtin_amdgcn_s_barrier();
        load_acts(min(g + 2, g1 - 1), buf == 0 ? 2 : buf - 1);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (i == 0 && ahead) {
            // The next chunk's weights travel while this one multiplies.
            load_weights(min(gc + CG, g1 - 1));
            __builtin_amdgcn_sched_barrier(0);
        }
        f16x p[TT];
        multiply(cw[i], p);
        const float sv = dev::f16_bits_to_f32((uint16_t)(cs[i / 2] >> (16 * (i % 2))));
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
            for (int k = 0; k < 16; ++k) acc[t][k] = fmaf(p[t][k], sv, acc[t][k]);
        buf = buf == D - 1 ? 0 : buf + 1;
    };
    if (uneven) {
        // A group at a time, the next one's codes and multipliers loaded
        // meanwhile (8 to 17 % slower than the loop below).
        const float *mp = a.uneven + (size_t)(my_token / kTile) * a.groups * kTile + my_token % kTile;
        uint16_t next_s = sp[g0];
        float next_m = mp[(size_t)g0 * kTile];
        for (uint32_t g = g0; g < g1; ++g) {
            __builtin_amdgcn_s_waitcnt(kWait<0>);
            __builtin_amdgcn_s_barrier();
            load_acts(min(g + 2, g1 - 1), buf == 0 ? 2 : buf - 1);
            uint32_t w[CW];
#pragma unroll
            for (int k = 0; k < CW; ++k) w[k] = rw[0][k];
            const float sv = dev::f16_bits_to_f32(next_s);
            mult[wave][lane] = my_scale == 0.0f ? next_m : my_scale;
            const uint32_t gn = min(g + 1, g1 - 1);
            load_codes<C>(wp + (size_t)gn * code_bytes(C), half, rw[0]);
            next_s = sp[gn];
            next_m = mp[(size_t)gn * kTile];
            f16x p[TT];
            multiply(w, p);
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int t = 0; t < TT; ++t)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float *q = &mult[wave][t * kTile + 8 * j + 4 * half];
#pragma unroll
                    for (int k = 0; k < 4; ++k) acc[t][4 * j + k] = fmaf(p[t][4 * j + k], sv * q[k], acc[t][4 * j + k]);
                }
            buf = buf == D - 1 ? 0 : buf + 1;
        }
    } else {
        // (Whole chunks apart from the last: an exit inside the chunk would make
        // the compiler's own waits drain the loads in flight.)
        uint32_t gc = g0;
        for (; gc + CG <= g1; gc += CG) {
            take_chunk(gc);
            static_for<CG>([&](auto at) __attribute__((always_inline)) { step(at, std::false_type{}, gc); });
        }
        if (gc < g1) {
            take_chunk(gc);
            static_for<CG>([&](auto at) __attribute__((always_inline)) {
                if (gc + decltype(at)::value < g1) step(at, std::true_type{}, gc);
            });
        } else {
            // (The last chunk's step loaded weights that nothing multiplies: a
            // use, or a compiler that takes that step out of the loop may drop
            // them from under the waits that count them.)
#pragma unroll
            for (int i = 0; i < CG; ++i)
#pragma unroll
                for (int k = 0; k < CW; ++k) asm volatile("" ::"v"(rw[i][k]));
#pragma unroll
            for (int i = 0; i < CG / 2; ++i) asm volatile("" ::"v"(rs[i]));
        }
    }

    __builtin_amdgcn_s_waitcnt(kWait<0>);  // (the last words, copied past the end, before the LDS is given back)
    // Register k of lane l: token 8 (k / 4) + 4 (l / 32) + k % 4, row l % 32.
    // (The form of the output is chosen outside the loops, and only ragged
    // tiles test their bounds: per-element branches here cost more than a
    // group of the loop above.)
    const bool whole = (tile0 + TT) * kTile <= a.tokens && row0 + kTile <= a.n;
    auto each = [&](auto put) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
            for (int k = 0; k < 16; ++k) {
                const uint32_t tt = t * kTile + 8 * (k / 4) + 4 * half + k % 4;
                put(tile0 * kTile + tt, row0 + col, __fmul_rn(acc[t][k], inv[tt]));
            }
    };
    if (a.part) {
        float *part = a.part + (size_t)slice * a.tokens * a.n;
        if (whole)
            each([&](uint32_t tok, uint32_t row, float v) { part[(size_t)tok * a.n + row] = v; });
        else
            each([&](uint32_t tok, uint32_t row, float v) {
                if (tok < a.tokens && row < a.n) part[(size_t)tok * a.n + row] = v;
            });
    } else if (a.pairs) {
        // Rows 2 j and 2 j + 1 are gate and up: neighbouring lanes.
        each([&](uint32_t tok, uint32_t row, float v) {
            const float y = silu_times(v, dev::xor_lane<1>(v));
            if (tok < a.tokens && row < a.n && !(col & 1)) a.out[(size_t)tok * (a.n / 2) + (row >> 1)] = y;
        });
    } else if (whole && !a.residual) {
        each([&](uint32_t tok, uint32_t row, float v) { a.out[(size_t)tok * a.n + row] = v; });
    } else {
        each([&](uint32_t tok, uint32_t row, float v) {
            if (tok < a.tokens && row < a.n) {
                const float res = a.residual ? a.residual[(size_t)tok * a.n + row] : 0.0f;
                a.out[(size_t)tok * a.n + row] = res + v;
            }
        });
    }
}

// Workgroup id to (row block, K slice, token block): consecutive ids run on
// the eight dies in turn, so a die takes whole (row block, slice) units and
// walks their token blocks: a weight line is fetched into one die's L2, and
// with as many slices as dies a die reads one slice of the activations.
using plan::kDies;

template <Codes C, int W, int TT>
__global__ __launch_bounds__(64 * W, 2) void gemm_rows_kernel(const RowsArgs a) {
    const uint32_t die = blockIdx.x % kDies, at = blockIdx.x / kDies;
    const uint32_t unit = at / a.token_blocks * kDies + die;
    const uint32_t row_block = unit / a.slices;
    if (row_block >= a.row_blocks) return;
    rows_block<C, W, TT>(a, row_block, at % a.token_blocks, unit % a.slices);
}

// out = the slices' sum, in slice order.
__global__ __launch_bounds__(256) void rows_reduce_kernel(const float *part, uint32_t slices, size_t plane, float *out) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= plane) return;
    float w[kRowsMaxSlices];
#pragma unroll
    for (uint32_t s = 0; s < kRowsMaxSlices; ++s) w[s] = s < slices ? part[s * plane + i] : 0.0f;
    float v = w[0];
#pragma unroll
    for (uint32_t s = 1; s < kRowsMaxSlices; ++s)
        if (s < slices) v += w[s];
    out[i] = v;
}

// ---------------------------------------------------------------------------
// The split activations. One workgroup per token, thread i with values 8 i ..
// 8 i + 7 of each 8 * blockDim stretch, the whole row in registers (rows to
// kPrepPasses stretches; longer rows are read twice).
// ---------------------------------------------------------------------------
constexpr int kPrepPasses = 4;
constexpr uint32_t kPrepThreads = 256;
constexpr uint32_t kPrepWidest = 8 * kPrepThreads * kPrepPasses;

struct PrepRowsArgs {
    const float *x;            // tokens x k (not with Pairs)
    const float *weight;       // RmsNorm
    float eps;
    uint32_t k, tokens;
    // Partial sums [slices][tokens][part_n] of the product that made the
    // input (slices 0: none). RmsNorm: added to x, the sum also stored to
    // x_out (may be x); Pairs (part_n = 2 k): value j is silu(row 2 j) * row
    // 2 j + 1.
    const float *part;
    uint32_t slices, part_n;
    float *x_out;
    uint32_t bytes;            // pair order: 1 for byte codes, 0 for nibbles
    uint8_t *halves;
    float *factor, *scale, *uneven;
};

__device__ __forceinline__ void read8(const float *p, float (&v)[8]) {
    const float4 a = reinterpret_cast<const float4 *>(p)[0], b = reinterpret_cast<const float4 *>(p)[1];
    v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w;
    v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
}

// Adds (first: sets) the slices' values at p, in slice order, all loads first.
__device__ __forceinline__ void slices8(const float *p, uint32_t slices, size_t plane, float (&v)[8]) {
    float4 w[kRowsMaxSlices][2];
#pragma unroll
    for (uint32_t s = 0; s < kRowsMaxSlices; ++s)
        if (s < slices) {
            w[s][0] = reinterpret_cast<const float4 *>(p + s * plane)[0];
            w[s][1] = reinterpret_cast<const float4 *>(p + s * plane)[1];
        }
    auto put = [&](uint32_t s, auto op) {
        v[0] = op(v[0], w[s][0].x), v[1] = op(v[1], w[s][0].y), v[2] = op(v[2], w[s][0].z), v[3] = op(v[3], w[s][0].w);
        v[4] = op(v[4], w[s][1].x), v[5] = op(v[5], w[s][1].y), v[6] = op(v[6], w[s][1].z), v[7] = op(v[7], w[s][1].w);
    };
    put(0, [](float, float b) { return b; });
#pragma unroll
    for (uint32_t s = 1; s < kRowsMaxSlices; ++s)
        if (s < slices) put(s, [](float a, float b) { return __fadd_rn(a, b); });
}

template <RowsInput::Form F>
__device__ __forceinline__ void input8(const PrepRowsArgs &a, uint32_t t, uint32_t e, float (&v)[8]) {
    const size_t plane = (size_t)a.tokens * a.part_n;
    if constexpr (F == RowsInput::Pairs) {
        float f[2][8];
        slices8(a.part + (size_t)t * a.part_n + 2 * e, a.slices, plane, f[0]);
        slices8(a.part + (size_t)t * a.part_n + 2 * e + 8, a.slices, plane, f[1]);
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = silu_times(f[i / 4][2 * (i % 4)], f[i / 4][2 * (i % 4) + 1]);
        return;
    }
    read8(a.x + (size_t)t * a.k + e, v);
    if constexpr (F == RowsInput::RmsNorm) {
        if (a.slices) {
            float sum[8];
            slices8(a.part + (size_t)t * a.part_n + e, a.slices, plane, sum);
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = __fadd_rn(v[i], sum[i]);
        }
    }
}

// The largest finite magnitude of a group, eight values of it in each of eight
// neighbouring lanes.
__device__ __forceinline__ float largest8(const float (&v)[8]) {
    float m = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float x = fabsf(v[i]);
        m = x < __builtin_inff() ? fmaxf(m, x) : m;
    }
    m = fmaxf(m, dev::xor_lane<4>(m));
    m = fmaxf(m, dev::xor_lane<2>(m));
    return fmaxf(m, dev::xor_lane<1>(m));
}

// The spread that a row's groups share one s within: their largest magnitudes'
// exponents.
constexpr int kEvenSpread = 15;

// `largest`: of the group; `row`: its row's exponent; `even`: the row's spread
// is within kEvenSpread.
__device__ __forceinline__ void split8(const PrepRowsArgs &a, const float (&v)[8], uint32_t t, uint32_t e, float largest,
                                       int row, bool even) {
    const int ex = even ? row : dev::chunk_exponent(largest);
    const float up = __builtin_ldexpf(1.0f, 14 - ex);
    h8 hi, lo;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        // Element 2 j, 2 j + 1 of the operand: columns j, j + 4 for nibbles.
        const float x = (a.bytes ? v[i] : v[(i >> 1) + 4 * (i & 1)]) * up;
        hi[i] = (_Float16)x;
        const float rest = x - (float)hi[i];
        lo[i] = fabsf(rest) < __builtin_inff() ? (_Float16)rest : (_Float16)0.0f;  // (inf and NaN are hi's)
    }
    const uint32_t g = e >> 6, s = (e >> 3) & 3, h = (e >> 5) & 1;
    uint8_t *to = a.halves + ((((size_t)(t / kTile) * (a.k >> 6) + g) * 4 + s) * 2 * 64 + h * 32 + t % kTile) * 16;
    *reinterpret_cast<h8 *>(to) = hi;
    *reinterpret_cast<h8 *>(to + 64 * 16) = lo;
    if (!even && (e & 63) == 0)
        a.uneven[((size_t)(t / kTile) * (a.k >> 6) + g) * kTile + t % kTile] = __builtin_ldexpf(1.0f, ex - 14);
}

// Workgroup id to token: eight consecutive tokens, whose words share 128-byte
// lines, run on one die, so that its L2 joins their 16-byte stores (from
// different dies they reach memory one by one: 12.7 us for 402 rows of 7680
// values).
__device__ __forceinline__ uint32_t prep_token() {
    const uint32_t die = blockIdx.x % kDies, at = blockIdx.x / kDies;
    return (at / 8 * kDies + die) * 8 + at % 8;
}

uint32_t prep_grid(uint32_t tokens) { return (tokens + 8 * kDies - 1) / (8 * kDies) * (8 * kDies); }

struct RowSpread {
    int exponent;
    bool even;
};

// From each thread's largest and least group (groups of zeros are left out);
// lds: two words a wavefront.
__device__ __forceinline__ RowSpread row_spread(float most, float least, float2 *lds) {
    most = dev::wave_max(most);
    least = -dev::wave_max(-least);
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = make_float2(most, least);
    __syncthreads();
    for (uint32_t w = 0; w < blockDim.x >> 6; ++w) {
        most = fmaxf(most, lds[w].x);
        least = fminf(least, lds[w].y);
    }
    const int exponent = dev::chunk_exponent(most);
    return {exponent, exponent - dev::chunk_exponent(least) <= kEvenSpread || !(most > 0.0f)};
}

template <RowsInput::Form F>
__global__ __launch_bounds__(kPrepThreads) void prep_rows_kernel(const PrepRowsArgs a) {
    __shared__ float red[4];
    __shared__ float2 spread[4];
    const uint32_t t = prep_token();
    if (t >= a.tokens) return;
    const uint32_t stretch = 8 * blockDim.x;
    float v[kPrepPasses][8];
    float sum = 0.0f, factor = 1.0f;
#pragma unroll
    for (int p = 0; p < kPrepPasses; ++p) {
        const uint32_t e = p * stretch + 8 * threadIdx.x;
#pragma unroll
        for (int i = 0; i < 8; ++i) v[p][i] = 0.0f;
        if (p * stretch < a.k && e < a.k) {
            input8<F>(a, t, e, v[p]);
            if (F == RowsInput::RmsNorm && a.slices) {
                float *to = a.x_out + (size_t)t * a.k + e;
                reinterpret_cast<float4 *>(to)[0] = make_float4(v[p][0], v[p][1], v[p][2], v[p][3]);
                reinterpret_cast<float4 *>(to)[1] = make_float4(v[p][4], v[p][5], v[p][6], v[p][7]);
            }
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) sum += v[p][i] * v[p][i];
    }
    if constexpr (F == RowsInput::RmsNorm) {
        // math.zig:120-130; the factor joins the token's output multiplier.
        sum = dev::wave_sum(sum);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = sum;
        __syncthreads();
        sum = red[0];
        for (uint32_t w = 1; w < blockDim.x >> 6; ++w) sum += red[w];
        factor = __fdiv_rn(1.0f, __fsqrt_rn(__fadd_rn(__fdiv_rn(sum, (float)a.k), a.eps)));
    }
    float largest[kPrepPasses], most = 0.0f, least = __builtin_inff();
#pragma unroll
    for (int p = 0; p < kPrepPasses; ++p) {
        const uint32_t e = p * stretch + 8 * threadIdx.x;
        if (F == RowsInput::RmsNorm && e < a.k) {
            float w[8];
            read8(a.weight + e, w);
#pragma unroll
            for (int i = 0; i < 8; ++i) v[p][i] = __fmul_rn(v[p][i], w[i]);
        }
        largest[p] = largest8(v[p]);
        most = fmaxf(most, largest[p]);
        least = largest[p] > 0.0f ? fminf(least, largest[p]) : least;
    }
    const RowSpread row = row_spread(most, least, spread);
#pragma unroll
    for (int p = 0; p < kPrepPasses; ++p) {
        const uint32_t e = p * stretch + 8 * threadIdx.x;
        if (e < a.k) split8(a, v[p], t, e, largest[p], row.exponent, row.even);
    }
    if (threadIdx.x == 0) a.factor[t] = factor, a.scale[t] = row.even ? __builtin_ldexpf(1.0f, row.exponent - 14) : 0.0f;
}

// Rows of more than kPrepWidest f32 values: read once for the largest, once
// to split.
__global__ __launch_bounds__(kPrepThreads) void prep_rows_wide_kernel(const PrepRowsArgs a) {
    __shared__ float2 spread[4];
    const uint32_t t = prep_token();
    if (t >= a.tokens) return;
    float v[8], most = 0.0f, least = __builtin_inff();
    for (uint32_t e = 8 * threadIdx.x; e < a.k; e += 8 * kPrepThreads) {
        input8<RowsInput::F32>(a, t, e, v);
        const float m = largest8(v);
        most = fmaxf(most, m);
        least = m > 0.0f ? fminf(least, m) : least;
    }
    const RowSpread row = row_spread(most, least, spread);
    for (uint32_t e = 8 * threadIdx.x; e < a.k; e += 8 * kPrepThreads) {
        input8<RowsInput::F32>(a, t, e, v);
        split8(a, v, t, e, largest8(v), row.exponent, row.even);
    }
    if (threadIdx.x == 0) a.factor[t] = 1.0f, a.scale[t] = row.even ? __builtin_ldexpf(1.0f, row.exponent - 14) : 0.0f;
}

size_t halves_bytes(uint32_t tokens, uint32_t cols) {
    return (size_t)((tokens + kTile - 1) / kTile) * kTile * cols * 4;
}

size_t uneven_bytes(uint32_t tokens, uint32_t cols) {
    return (size_t)((tokens + kTile - 1) / kTile) * kTile * (cols / 64) * sizeof(float);
}

constexpr int kWaves = plan::kRowsWaves;

template <Codes C>
void launch_rows(hipStream_t s, const RowsPlan &plan, const RowsArgs &a) {
    const uint32_t grid = (a.row_blocks * plan.slices + kDies - 1) / kDies * kDies * a.token_blocks;
    if (plan.token_tiles == 2) gemm_rows_kernel<C, kWaves, 2><<<grid, 64 * kWaves, 0, s>>>(a);
    else gemm_rows_kernel<C, kWaves, 1><<<grid, 64 * kWaves, 0, s>>>(a);
}

}  // namespace

bool gemm_rows_supported(const Matrix &w) {
    // (Four groups: the scales' chunk load.)
    return (w.format == QWH_FORMAT_Q4 || w.format == QWH_FORMAT_Q5 || w.format == QWH_FORMAT_Q8) && w.cols % 64 == 0 &&
           w.cols >= 256 && w.rows != 0;
}

bool gemm_rows_preferred(const Matrix &w, uint32_t tokens) {
    return gemm_rows_supported(w) && plan::rows_preferred(w.format, w.rows, w.cols, tokens);
}

size_t rows_activation_bytes(uint32_t tokens, uint32_t cols) {
    return halves_bytes(tokens, cols) + uneven_bytes(tokens, cols) + 2 * (size_t)tokens * sizeof(float);
}

size_t rows_partial_bytes(int cus, uint32_t tokens, const Matrix &w) {
    const uint32_t slices = std::max(rows_plan(cus, tokens, w.rows, w.cols, kRowsMaxSlices, false).slices,
                                     rows_plan(cus, tokens, w.rows, w.cols, kRowsMaxSlices, true).slices);
    return slices > 1 ? (size_t)slices * tokens * w.rows * sizeof(float) : 0;
}

hipError_t launch_prep_rows(hipStream_t s, const RowsInput &in, int format, uint32_t tokens, uint32_t cols, void *acts) {
    if (tokens == 0 || cols == 0 || cols % 64) return hipErrorInvalidValue;
    PrepRowsArgs p{};
    p.x = in.x;
    p.weight = in.weight;
    p.eps = in.eps;
    p.k = cols;
    p.tokens = tokens;
    p.part = in.sums.part;
    p.slices = in.sums.slices;
    p.part_n = in.sums.rows;
    p.x_out = in.sums.x_out;
    p.bytes = format == QWH_FORMAT_Q8 ? 1u : 0u;
    p.halves = static_cast<uint8_t *>(acts);
    p.uneven = reinterpret_cast<float *>(p.halves + halves_bytes(tokens, cols));
    p.factor = reinterpret_cast<float *>(p.halves + halves_bytes(tokens, cols) + uneven_bytes(tokens, cols));
    p.scale = p.factor + tokens;
    if (p.slices > kRowsMaxSlices || (p.slices && !p.part)) return hipErrorInvalidValue;
    if (in.form == RowsInput::Pairs && (!p.slices || p.part_n != 2 * cols)) return hipErrorInvalidValue;
    if (in.form == RowsInput::RmsNorm && p.slices && (p.part_n != cols || !p.x_out)) return hipErrorInvalidValue;
    if (p.slices && in.form != RowsInput::Pairs && in.form != RowsInput::RmsNorm) return hipErrorInvalidValue;
    if (cols > kPrepWidest) {
        if (in.form != RowsInput::F32) return hipErrorInvalidValue;
        prep_rows_wide_kernel<<<prep_grid(tokens), kPrepThreads, 0, s>>>(p);
        return hipGetLastError();
    }
    const uint32_t threads = std::min(kPrepThreads, (cols / 8 + 63) / 64 * 64);
    switch (in.form) {
    case RowsInput::F32: prep_rows_kernel<RowsInput::F32><<<prep_grid(tokens), threads, 0, s>>>(p); break;
    case RowsInput::RmsNorm: prep_rows_kernel<RowsInput::RmsNorm><<<prep_grid(tokens), threads, 0, s>>>(p); break;
    case RowsInput::Pairs: prep_rows_kernel<RowsInput::Pairs><<<prep_grid(tokens), threads, 0, s>>>(p); break;
    }
    return hipGetLastError();
}

hipError_t launch_gemm_rows(hipStream_t s, int cus, const void *acts, const Matrix &w, uint32_t tokens,
                            const RowsOutput &out, uint32_t *slices_left) {
    if (slices_left) *slices_left = 0;
    if (tokens == 0 || !gemm_rows_supported(w)) return hipErrorInvalidValue;
    if (out.pairs && (w.rows % 2 || out.residual)) return hipErrorInvalidValue;
    // (Without a caller that adds them, only a plain product has its slices added.)
    const bool split = out.partials && (slices_left || !(out.pairs || out.residual));
    const RowsPlan plan = rows_plan(cus, tokens, w.rows, w.cols, split ? kRowsMaxSlices : 1, slices_left != nullptr);
    RowsArgs a{};
    a.scales = reinterpret_cast<const uint16_t *>(w.scales);
    a.data = w.data;
    a.halves = static_cast<const uint8_t *>(acts);
    a.uneven = reinterpret_cast<const float *>(a.halves + halves_bytes(tokens, w.cols));
    a.factor = reinterpret_cast<const float *>(a.halves + halves_bytes(tokens, w.cols) + uneven_bytes(tokens, w.cols));
    a.scale = a.factor + tokens;
    a.out = out.out;
    a.residual = out.residual;
    a.pairs = out.pairs ? 1u : 0u;
    a.n = w.rows;
    a.groups = w.cols / 64;
    a.tokens = tokens;
    a.row_blocks = (w.rows + kWaves * kTile - 1) / (kWaves * kTile);
    a.token_blocks = ((tokens + kTile - 1) / kTile + plan.token_tiles - 1) / plan.token_tiles;
    a.slices = plan.slices;
    a.slice_groups = plan.slice_groups;
    if (plan.slices > 1) a.part = out.partials;
    switch (w.format) {
    case QWH_FORMAT_Q4: launch_rows<Codes::Q4>(s, plan, a); break;
    case QWH_FORMAT_Q5: launch_rows<Codes::Q5>(s, plan, a); break;
    default: launch_rows<Codes::Q8>(s, plan, a); break;
    }
    if (plan.slices > 1 && slices_left) {
        *slices_left = plan.slices;
    } else if (plan.slices > 1) {
        const size_t plane = (size_t)tokens * w.rows;
        rows_reduce_kernel<<<(uint32_t)((plane + 255) / 256), 256, 0, s>>>(out.partials, plan.slices, plane, out.out);
    }
    return hipGetLastError();
}

}  // namespace qwh

// The audio tower's convolution front end: model.zig:509-644 convolveAndPack
// and projectConvStep, with kernels.zig:302-427 conv3x3Stride2Gelu.
//
// The log-mel spectrogram is cut into chunks of 2 * n_window frames (the last
// one zero filled); each chunk goes through three 3x3, stride-2, padding-1
// convolutions with bias and GELU ([out][in][3][3] f16 weights, channel-major
// planes, as the checkpoint stores them); every valid time step of the third
// stage is flattened channel-major over the remaining frequency bins and
// projected by conv_out; the sinusoidal position of the step within its chunk
// (model.zig:751-763) is added.
//
// Convolution kernel: a workgroup computes 64 output channels over an 8 x 8
// tile of output positions of one image. The input channels go through LDS in
// stages of 8: the 17 x 17 input patch the tile reads (zero outside the
// plane, which is the padding) and the stage's weights as f32, laid out
// [channel][tap][output channel] so a thread reads its four output channels'
// weights with one 16-byte LDS load. A thread accumulates 4 output channels x
// 4 positions in f32 FMAs (the reference sums each input channel's nine taps
// before adding them to the output; the order here differs, within f32
// rounding), then adds the bias and applies GELU (the reference's erf fit).
#include <algorithm>

#include "common.h"
#include "device.h"

namespace qwh {
namespace {

constexpr int kOcTile = 64;    // output channels per workgroup
constexpr int kTile = 8;       // output rows and columns per workgroup
constexpr int kPatch = 2 * kTile + 1;
constexpr int kCi = 8;         // input channels per LDS stage

struct ConvArgs {
    float *out;                // [batch][out_ch][oh][ow]
    const float *in;           // [batch][in_ch][h][w]
    const uint16_t *weights;   // [out_ch][in_ch][9] f16 bits
    const float *bias;         // [out_ch]
    uint32_t out_ch, in_ch, h, w, oh, ow, tiles_w;
};

__global__ __launch_bounds__(256) void conv3x3s2_gelu_kernel(const ConvArgs a) {
    __shared__ float patch[kCi][kPatch * kPatch];
    __shared__ float4 wts[kCi][9][kOcTile / 4];
    const int t = threadIdx.x;
    const uint32_t oc0 = blockIdx.x * kOcTile;
    const uint32_t tile_r = blockIdx.y / a.tiles_w, tile_c = blockIdx.y % a.tiles_w;
    const uint32_t b = blockIdx.z;
    const int ocg = t >> 4;             // four output channels oc0 + 4 ocg ..
    const int pg = t & 15;              // four positions: tile row pg / 2, columns 4 (pg % 2) ..
    const int pr = pg >> 1, pc = (pg & 1) * 4;
    const int in_r0 = (int)(tile_r * kTile) * 2 - 1, in_c0 = (int)(tile_c * kTile) * 2 - 1;
    const float *in = a.in + (size_t)b * a.in_ch * a.h * a.w;
    float acc[4][4] = {};
    for (uint32_t ci0 = 0; ci0 < a.in_ch; ci0 += kCi) {
        __syncthreads();  // the previous stage's reads are done
        for (int i = t; i < kCi * kPatch * kPatch; i += 256) {
            const int c = i / (kPatch * kPatch), rem = i % (kPatch * kPatch);
            const int r = in_r0 + rem / kPatch, col = in_c0 + rem % kPatch;
            float v = 0.0f;
            if (ci0 + c < a.in_ch && r >= 0 && r < (int)a.h && col >= 0 && col < (int)a.w)
                v = in[((size_t)(ci0 + c) * a.h + r) * a.w + col];
            patch[c][rem] = v;
        }
        for (int i = t; i < kCi * 9 * kOcTile; i += 256) {
            const int oc = i % kOcTile, tap = (i / kOcTile) % 9, c = i / (kOcTile * 9);
            float v = 0.0f;
            if (ci0 + c < a.in_ch && oc0 + oc < a.out_ch)
                v = dev::f16_bits_to_f32(a.weights[((size_t)(oc0 + oc) * a.in_ch + ci0 + c) * 9 + tap]);
            reinterpret_cast<float *>(&wts[c][tap][0])[oc] = v;
        }
        __syncthreads();
        const int stage = a.in_ch - ci0 < (uint32_t)kCi ? (int)(a.in_ch - ci0) : kCi;
        for (int c = 0; c < stage; ++c) {
#pragma unroll
            for (int tap = 0; tap < 9; ++tap) {
                const int kh = tap / 3, kw = tap % 3;
                const float4 wv = wts[c][tap][ocg];
                const float *row = &patch[c][(2 * pr + kh) * kPatch + 2 * pc + kw];
                const float x[4] = {row[0], row[2], row[4], row[6]};
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    acc[0][j] = fmaf(wv.x, x[j], acc[0][j]);
                    acc[1][j] = fmaf(wv.y, x[j], acc[1][j]);
                    acc[2][j] = fmaf(wv.z, x[j], acc[2][j]);
                    acc[3][j] = fmaf(wv.w, x[j], acc[3][j]);
                }
            }
        }
    }
    const uint32_t orow = tile_r * kTile + pr;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint32_t oc = oc0 + 4 * ocg + k;
        if (oc >= a.out_ch || orow >= a.oh) continue;
        const float bias = a.bias[oc];
        float *dst = a.out + (((size_t)b * a.out_ch + oc) * a.oh + orow) * a.ow;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t ocol = tile_c * kTile + pc + j;
            if (ocol < a.ow) dst[ocol] = dev::gelu(bias + acc[k][j]);
        }
    }
}

// ---- Matrix-core form (input channels a multiple of 16) ----
//
// The convolution as an implicit GEMM on v_mfma_f32_32x32x16_f16: rows are
// output channels, columns are output positions (row-major over the output
// plane), and the reduction runs over (tap, input channel) in stages of 16
// input channels, one 16-deep MFMA step per tap. A weight is f16 as it is. An
// activation is two f16 terms of x * s: hi its f16 rounding, lo 2^11 times the
// exact remainder rounded to f16, with s a power of two for the image from a
// bound on its largest magnitude, |x * s| < 2^15. So a value keeps 22
// significant bits down to 2^-29 of the bound, and nothing above 2^-51 of it is
// lost, whatever the other images hold; the products are exact and summed in
// f32 by the matrix core, each term's in accumulators of its own. (Two bf16
// terms of both operands, without a scale, took four products a tap and kept
// 2^-17.)
//
// The terms are stored once by whoever makes the activations (the "halves"
// layout): [image][stage][plane][row][parity][slot] 16-byte words of 8
// channels, plane = 2 * term + channel half, rows and columns padded by one
// zero on each side and the padded columns split by parity. A tap of stride 2
// reads one parity, so the 32 positions of an operand are consecutive words:
// the patch is copied to LDS as it is, and read without tests for the border.
//
// Workgroup: 256 output channels (four wavefronts of 64) x 64 positions (or 32,
// where the grid is small: launch_mfma, which may also split the stages over
// workgroups); a wavefront's 64 x 64 tile takes eight products from four LDS
// words and two weight words a lane. A stage's patch (at most 2 * ceil(63 / ow) + 3 rows) is
// copied by global-to-LDS loads one stage ahead, and a tap's weights, stored
// in operand order, are loaded a whole stage before their use. Bound by its
// waits and by the last, partly empty wave of workgroups: the matrix cores are
// busy 42 % of conv2's cycles, the LDS 21 % (half of that bank conflicts), its
// wavefronts wait 70 % of theirs. 30 s of audio, 480 channels, under the tracer:
// conv2 (64 x 50 planes) 706 -> 264 us, conv3 204 -> 86 us.
typedef _Float16 ch8 __attribute__((ext_vector_type(8)));
typedef _Float16 ch4 __attribute__((ext_vector_type(4)));
typedef float cf32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t cu4 __attribute__((ext_vector_type(4)));

constexpr int kMfOc = 256;       // output channels per workgroup, 64 per wavefront
constexpr int kMfPos = 64;       // output positions per workgroup at most (one or two 32-column MFMA tiles)
constexpr int kMfIc = 16;        // input channels per stage
constexpr int kMfRounds = 9;     // patch words per thread at most
constexpr uint32_t kConvMaxSlices = 6;

// A tensor in the halves layout: padded planes of (h + 2) rows x 2 parities x
// slots words.
struct HalvesPlane {
    uint32_t slots, words;       // of a row and parity; of a plane
};

__host__ __device__ inline HalvesPlane halves_plane(uint32_t h, uint32_t w) {
    const uint32_t slots = (w + 3) / 2;
    return {slots, (h + 2) * 2 * slots};
}

struct ConvMfmaArgs {
    const uint8_t *in;           // halves
    const uint8_t *wprep;        // [stage][tap][oc / 32][lane][8] f16
    const float *bias;
    const float *scales;         // per image, scale_stride apart: input [1]: 2^-e; halves output [2]: its 2^e
    float *out;                  // [batch][out_ch][oh * ow] f32, or null
    uint8_t *halves;             // the output in the halves layout, or null
    uint32_t out_ch, oc_tiles, stages, h, w, oh, ow, positions;
    uint32_t patch_rows, pos_tiles, units, oc_blocks;
    uint32_t slices, slice_stages, scale_stride;
    float *part;                 // slices > 1: [slice][batch][out_ch][positions] sums, for conv_finish_kernel
    uint32_t batch;
};

// The two terms of v * s, the second times 2^11.
constexpr float kLoUp = 2048.0f, kLoDown = 1.0f / 2048.0f;
__device__ __forceinline__ void split_half(float v, float s, _Float16 &hi, _Float16 &lo) {
    const float x = v * s;
    hi = (_Float16)x;
    const float rest = (x - (float)hi) * kLoUp;
    lo = fabsf(rest) < __builtin_inff() ? (_Float16)rest : (_Float16)0.0f;  // (inf and NaN are hi's)
}

// s_waitcnt operand: at most N vector memory operations and no LDS operation
// outstanding.
template <int N>
constexpr int kConvWait = (N & 15) | (7 << 4) | ((N >> 4) << 14);
// The same for vector memory alone.
template <int N>
constexpr int kConvLoads = kConvWait<N> | (15 << 8);

// NT: 32-position tiles; R: rounds of 256 patch words. (Three workgroups a CU
// where their LDS allows it: one register more would leave two.)
template <int NT, int R, bool HALVES>
__global__ __launch_bounds__(256, NT == 1 && R <= 6 ? 3 : 2) void conv3x3s2_gelu_mfma_kernel(const ConvMfmaArgs a) {
    __shared__ cu4 patch[2][R * 256];
    const int t = threadIdx.x;
    const int lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int half = lane >> 5;
    // Consecutive workgroups run on the eight dies in turn: a position tile's
    // channel blocks stay on one die, next to each other.
    const uint32_t die = blockIdx.x & 7, at = blockIdx.x >> 3;
    const uint32_t inner = a.oc_blocks * a.slices;
    const uint32_t unit = at / inner * 8 + die;
    if (unit >= a.units) return;
    const uint32_t b = unit / a.pos_tiles, p0 = unit % a.pos_tiles * (32 * NT);
    const uint32_t slice = at % inner / a.oc_blocks, oc_block = at % a.oc_blocks;
    const uint32_t first_stage = slice * a.slice_stages, last_stage = min(first_stage + a.slice_stages, a.stages) - 1;
    const uint32_t oc0 = oc_block * kMfOc + wave * 64;
    const HalvesPlane in_plane = halves_plane(a.h, a.w);
    const uint32_t slots = in_plane.slots;
    const uint32_t patch_plane = a.patch_rows * 2 * slots;  // words of a patch plane
    const uint32_t r_first = p0 / a.ow;

    if (HALVES && p0 == 0 && slice == 0) {
        // The output planes' zero border (this workgroup's channels, once per
        // image): the first and last row, and in the others what is left and
        // right of the columns.
        const HalvesPlane o = halves_plane(a.oh, a.ow);
        const uint32_t first = oc_block * (kMfOc / kMfIc);
        const uint32_t count = min((uint32_t)(kMfOc / kMfIc), a.out_ch / kMfIc - first) * 4;
        cu4 *to = reinterpret_cast<cu4 *>(a.halves) + ((size_t)b * (a.out_ch / kMfIc) + first) * 4 * o.words;
        for (uint32_t i = t; i < o.words; i += 256) {
            const uint32_t row = i / (2 * o.slots), rest = i % (2 * o.slots);
            const uint32_t col = 2 * (rest % o.slots) + rest / o.slots;
            if (row >= 1 && row <= a.oh && col >= 1 && col <= a.ow) continue;
            for (uint32_t p = 0; p < count; ++p) to[(size_t)p * o.words + i] = cu4{0, 0, 0, 0};
        }
    }

    // Patch words t, t + 256, ...: their source within a stage (the last word
    // again past the patch, the last row again past the plane: both unused).
    uint32_t from[R];
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const uint32_t u = min((uint32_t)(t + 256 * k), 4 * patch_plane - 1);
        const uint32_t plane = u / patch_plane, rem = u % patch_plane;
        const uint32_t row = min(2 * r_first + rem / (2 * slots), a.h + 1);
        from[k] = plane * in_plane.words + row * 2 * slots + rem % (2 * slots);
    }
    const cu4 *image = reinterpret_cast<const cu4 *>(a.in) + (size_t)b * a.stages * 4 * in_plane.words;
    auto copy_patch = [&](uint32_t stage, int buf) __attribute__((always_inline)) {
        const cu4 *src = image + (size_t)stage * 4 * in_plane.words;
#pragma unroll
        for (int k = 0; k < R; ++k)
            __builtin_amdgcn_global_load_lds(
                reinterpret_cast<const __attribute__((address_space(1))) uint32_t *>(
                    reinterpret_cast<uintptr_t>(src + from[k])),
                reinterpret_cast<__attribute__((address_space(3))) uint32_t *>(
                    reinterpret_cast<uintptr_t>(&patch[buf][wave * 64 + 256 * k])), 16, 0, 0);
    };
    // B operand: this lane's position (column lane % 32) and channel half.
    uint32_t cell[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const uint32_t p = min(p0 + 32 * j + (lane & 31), a.positions - 1);  // (past the plane: never stored)
        cell[j] = half * patch_plane + 2 * (p / a.ow - r_first) * 2 * slots + p % a.ow;
    }
    // A operand: weights of oc0 + 32 i + lane % 32, channels 8 half .. + 7.
    // (A wavefront past the channels multiplies the last ones' and stores
    // nothing: a branch around its products would make the compiler wait for
    // every load in flight at each stage.)
    const cu4 *weights = reinterpret_cast<const cu4 *>(a.wprep) + (size_t)min(oc0 / 32, a.oc_tiles - 2) * 64 + lane;
    const size_t tap_words = (size_t)a.oc_tiles * 64;
    ch8 wa[9][2];
    auto load_tap = [&](uint32_t stage, int tap) __attribute__((always_inline)) {
        const cu4 *src = weights + ((size_t)stage * 9 + tap) * tap_words;
        wa[tap][0] = __builtin_bit_cast(ch8, src[0]);
        wa[tap][1] = __builtin_bit_cast(ch8, src[64]);
        __builtin_amdgcn_sched_barrier(0);  // (else it sinks to the stage's end)
    };
    cf32x16 acc[2][NT] = {}, acc_lo[2][NT] = {};
    copy_patch(first_stage, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int tap = 0; tap < 9; ++tap) load_tap(first_stage, tap);
    int buf = 0;
    for (uint32_t s = first_stage; s <= last_stage; ++s, buf ^= 1) {
        const uint32_t next = min(s + 1, last_stage);
        // This stage's patch has landed (the 18 weight words a lane loaded
        // after it may still travel), in every wavefront after the barrier;
        // the other buffer was last read before it.
        __builtin_amdgcn_s_waitcnt(kConvWait<18>);
        __builtin_amdgcn_s_barrier();
        copy_patch(next, buf ^ 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int tap = 0; tap < 9; ++tap) {
            // This tap's weights: the 16 words of the other taps and R of the
            // patch were loaded since, and loads complete in order. (Left to
            // itself the compiler waits for everything once a copy to LDS is
            // in flight.)
            __builtin_amdgcn_s_waitcnt(kConvLoads<16 + R>);
            const uint32_t step = (2 * (tap / 3) + (tap % 3 & 1)) * slots + (tap % 3 >> 1);
#pragma unroll
            for (int term = 0; term < 2; ++term) {
                ch8 x[NT];
#pragma unroll
                for (int j = 0; j < NT; ++j)
                    x[j] = __builtin_bit_cast(ch8, patch[buf][cell[j] + term * 2 * patch_plane + step]);
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < NT; ++j) {
                        cf32x16 &to = term ? acc_lo[i][j] : acc[i][j];
                        to = __builtin_amdgcn_mfma_f32_32x32x16_f16(wa[tap][i], x[j], to, 0, 0, 0);
                    }
            }
            load_tap(next, tap);
        }
    }
    __builtin_amdgcn_s_waitcnt(kConvWait<0>);  // (the last copy, unused, before the LDS is given back)
    // (The last stage loaded weights that nothing multiplies: a use, or a
    // compiler that takes that stage out of the loop may drop them from under
    // the waits that count them.)
#pragma unroll
    for (int tap = 0; tap < 9; ++tap)
#pragma unroll
        for (int i = 0; i < 2; ++i) asm volatile("" ::"v"(__builtin_bit_cast(cu4, wa[tap][i])));
    if (oc0 >= a.out_ch) return;
    // (Computed again: no register of the loop's, at its limit, holds them.)
    const int out_lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)), out_half = out_lane >> 5;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = fmaf(acc_lo[i][j][r], kLoDown, acc[i][j][r]);
    // Value r of a lane: output channel 8 (r / 4) + 4 half + r % 4 of the
    // tile's 32, position column lane % 32.
    if (a.part) {
        float *part = a.part + ((size_t)slice * a.batch + b) * a.out_ch * a.positions;
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const uint32_t pos = p0 + 32 * j + (out_lane & 31);
            if (pos >= a.positions) continue;
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const uint32_t oc = oc0 + 32 * i + 8 * (r / 4) + 4 * out_half + r % 4;
                    if (oc < a.out_ch) part[(size_t)oc * a.positions + pos] = acc[i][j][r];
                }
        }
        return;
    }
    const float *scales = a.scales + (size_t)b * a.scale_stride;
    const float inverse = scales[1];
    const float up = HALVES ? scales[2] : 0.0f;
    const HalvesPlane o = halves_plane(a.oh, a.ow);
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const uint32_t pos = p0 + 32 * j + (out_lane & 31);
        if (pos >= a.positions) continue;
        const uint32_t row = pos / a.ow + 1, col = pos % a.ow + 1;
        const uint32_t word = (row * 2 + (col & 1)) * o.slots + (col >> 1);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t oc = oc0 + 32 * i + 8 * q + 4 * out_half;
                if (oc >= a.out_ch) continue;
                float y[4];
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    y[k] = dev::gelu(a.bias[min(oc + k, a.out_ch - 1)] + acc[i][j][4 * q + k] * inverse);
                if constexpr (HALVES) {
                    ch4 hi, lo;
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        _Float16 p, l;
                        split_half(y[k], up, p, l);
                        hi[k] = p, lo[k] = l;
                    }
                    // (Channels oc .. oc + 3 are half of a word of eight.)
                    uint8_t *to = a.halves + ((((size_t)b * (a.out_ch / kMfIc) + oc / kMfIc) * 4 + (q & 1)) * o.words +
                                              word) * 16 + 8 * out_half;
                    *reinterpret_cast<ch4 *>(to) = hi;
                    *reinterpret_cast<ch4 *>(to + (size_t)2 * o.words * 16) = lo;
                } else {
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        if (oc + k < a.out_ch) a.out[((size_t)b * a.out_ch + oc + k) * a.positions + pos] = y[k];
                }
            }
    }
}

// The slices' sums in slice order, scaled, with bias and GELU: a thread takes
// eight channels of a position (one word of the halves layout).
template <bool HALVES>
__global__ __launch_bounds__(256) void conv_finish_kernel(const ConvMfmaArgs a) {
    const uint32_t words = (a.out_ch + 7) / 8;
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (uint64_t)a.batch * words * a.positions) return;
    const uint32_t pos = (uint32_t)(i % a.positions);
    const uint32_t oc = (uint32_t)(i / a.positions % words) * 8, b = (uint32_t)(i / a.positions / words);
    const size_t plane = (size_t)a.batch * a.out_ch * a.positions;
    float v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const float *p = a.part + ((size_t)b * a.out_ch + min(oc + k, a.out_ch - 1)) * a.positions + pos;
        float w[kConvMaxSlices];
#pragma unroll
        for (uint32_t s = 0; s < kConvMaxSlices; ++s) w[s] = s < a.slices ? p[s * plane] : 0.0f;
        v[k] = w[0];
#pragma unroll
        for (uint32_t s = 1; s < kConvMaxSlices; ++s)
            if (s < a.slices) v[k] += w[s];
    }
    const float *scales = a.scales + (size_t)b * a.scale_stride;
    const float inverse = scales[1];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = dev::gelu(a.bias[min(oc + k, a.out_ch - 1)] + v[k] * inverse);
    if constexpr (HALVES) {
        // (out_ch is a multiple of 16.)
        const HalvesPlane o = halves_plane(a.oh, a.ow);
        const uint32_t row = pos / a.ow + 1, col = pos % a.ow + 1;
        const uint32_t word = (row * 2 + (col & 1)) * o.slots + (col >> 1);
        const float up = scales[2];
        ch8 hi, lo;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            _Float16 p, l;
            split_half(v[k], up, p, l);
            hi[k] = p, lo[k] = l;
        }
        ch8 *to = reinterpret_cast<ch8 *>(a.halves) +
                  (((size_t)b * (a.out_ch / kMfIc) + oc / kMfIc) * 4 + (oc >> 3 & 1)) * o.words + word;
        to[0] = hi;
        to[(size_t)2 * o.words] = lo;
    } else {
#pragma unroll
        for (int k = 0; k < 8; ++k)
            if (oc + k < a.out_ch) a.out[((size_t)b * a.out_ch + oc + k) * a.positions + pos] = v[k];
    }
}

// What a call prepares: each convolution's weights in operand order with the
// sum of magnitudes per output channel (a workgroup per channel; channels
// past out_ch are zero), and the partial maxima of |x| over finite values of
// each image of an input (the workgroups after them, `partials` to an image, four
// rows to a wavefront).
struct ConvWeightsJob {
    const uint16_t *weights;     // [out_ch][in_ch][9] f16 bits
    uint8_t *wprep;
    float *norms;                // [oc_pad]
    uint32_t out_ch, oc_pad, in_ch;
};

struct ConvPrepArgs {
    ConvWeightsJob job[2];
    // Row r of image b: x + b * image_stride + r * row_stride, at most
    // row_values values: what is left of `limit` after b * image_used + r *
    // row_used of it.
    const float *x;
    uint64_t image_stride, row_stride, limit, image_used, row_used;
    uint32_t rows, row_values;
    float *partial;              // [image][partials]
    uint32_t partials;
};

constexpr int kPrepIc = 512;

__global__ __launch_bounds__(256) void conv_prep_kernel(const ConvPrepArgs a) {
    __shared__ uint16_t rows[kPrepIc * 9];
    __shared__ float red[4];
    uint32_t block = blockIdx.x;
    float v = 0.0f;
    float *to;
    const bool maxima = block >= a.job[0].oc_pad + a.job[1].oc_pad;
    if (maxima) {
        block -= a.job[0].oc_pad + a.job[1].oc_pad;
        const uint64_t image = block / a.partials;
        // (Four rows' loads at a time; past the last row, that row again, and
        // past a row's end its last value.)
        for (uint32_t r = (block % a.partials * 4 + (threadIdx.x >> 6)) * 4; r < a.rows; r += a.partials * 16) {
            const float *row[4];
            uint32_t last[4], longest = 0;
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) {
                const uint64_t at = min(r + k, a.rows - 1);
                row[k] = a.x + image * a.image_stride + at * a.row_stride;
                last[k] = (uint32_t)min((uint64_t)a.row_values, a.limit - image * a.image_used - at * a.row_used) - 1;
                longest = max(longest, last[k]);
            }
            for (uint32_t i = threadIdx.x & 63; i <= longest; i += 64) {
                float m[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) m[k] = fabsf(row[k][min(i, last[k])]);
#pragma unroll
                for (int k = 0; k < 4; ++k) v = m[k] < __builtin_inff() ? fmaxf(v, m[k]) : v;
            }
        }
        v = dev::wave_max(v);
        to = a.partial + block;
    } else {
        const uint32_t n = block >= a.job[0].oc_pad ? 1 : 0;
        const ConvWeightsJob &j = a.job[n];
        // Eight consecutive channels, whose words share 128-byte lines, on one
        // die (block ids run on the eight dies in turn), so that its L2 joins
        // their stores.
        const uint32_t id = block - (n ? a.job[0].oc_pad : 0);
        const uint32_t oc = (id / 64 * 8 + id % 8) * 8 + id / 8 % 8;
        const uint16_t *row = j.weights + (size_t)min(oc, j.out_ch - 1) * j.in_ch * 9;
        // A channel's weights through LDS, kPrepIc input channels at a time;
        // items (stage, channel half, tap) are eight channels' of a tap.
        for (uint32_t ic = 0; ic < j.in_ch; ic += kPrepIc) {
            const uint32_t n = min((uint32_t)kPrepIc, j.in_ch - ic) * 9;
            uint16_t r[kPrepIc * 9 / 256];  // (all loads first; past the row, its last value again)
#pragma unroll
            for (int k = 0; k < kPrepIc * 9 / 256; ++k) r[k] = row[ic * 9 + min(threadIdx.x + 256u * k, n - 1)];
            __syncthreads();
#pragma unroll
            for (int k = 0; k < kPrepIc * 9 / 256; ++k)
                if (threadIdx.x + 256u * k < n) rows[threadIdx.x + 256u * k] = r[k];
            __syncthreads();
            for (uint32_t i = threadIdx.x; i < n / 8; i += 256) {
                const uint32_t tap = i % 9, h = i / 9 % 2, stage = ic / kMfIc + i / 18;
                ch8 w;
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const uint16_t bits = rows[((i / 18) * kMfIc + 8 * h + k) * 9 + tap];
                    w[k] = oc < j.out_ch ? __builtin_bit_cast(_Float16, bits) : (_Float16)0.0f;
                    v += fabsf((float)w[k]);
                }
                *reinterpret_cast<ch8 *>(j.wprep + ((((size_t)stage * 9 + tap) * (j.oc_pad / 32) + oc / 32) * 64 +
                                                    h * 32 + oc % 32) * 16) = w;
            }
        }
        v = dev::wave_sum(v);
        to = j.norms + oc;
    }
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0)
        *to = maxima ? fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3])) : (red[0] + red[1]) + (red[2] + red[3]);
}

// An image's scales {2^e, 2^-e} for magnitudes to m, with room for the bound's
// own rounding.
__device__ __forceinline__ float2 scale_of(float m) {
    const int e = dev::chunk_exponent(fminf(m * 1.01f, 3.4e38f));
    return make_float2(__builtin_ldexpf(1.0f, 15 - e), __builtin_ldexpf(1.0f, e - 15));
}

// The scales of the tower's intermediate tensors from bounds on their
// magnitudes, one workgroup a chunk: the first, of conv1's result, from the
// partial maxima of the chunk through conv1's weight sums, the second from the
// first's bound through conv2's: |gelu(y)| <= |y| <= |bias| + sum |w| * bound.
// (A bound a thousand times the largest value still keeps it to 2^-41.)
struct ConvScaleArgs {
    const float *partial;
    uint32_t partials;
    const uint16_t *conv1;       // [channels][9] f16 bits
    const float *bias1, *norms2, *bias2;
    uint32_t channels;
    float *scales;               // per chunk, {s, 1 / s} of the first, then of the second
};

__device__ __forceinline__ float block_max_256(float v, float *red) {
    v = dev::wave_max(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

__global__ __launch_bounds__(256) void conv_scale_kernel(const ConvScaleArgs a) {
    __shared__ float red[4];
    float v = 0.0f;
    for (uint32_t i = threadIdx.x; i < a.partials; i += 256) v = fmaxf(v, a.partial[(size_t)blockIdx.x * a.partials + i]);
    float bound = block_max_256(v, red);
    v = 0.0f;
    for (uint32_t c = threadIdx.x; c < a.channels; c += 256) {
        float sum = 0.0f;
        for (int k = 0; k < 9; ++k) sum += fabsf(dev::f16_bits_to_f32(a.conv1[(size_t)c * 9 + k]));
        v = fmaxf(v, fabsf(a.bias1[c]) + sum * bound);
    }
    bound = block_max_256(v, red);
    v = 0.0f;
    for (uint32_t c = threadIdx.x; c < a.channels; c += 256) v = fmaxf(v, fabsf(a.bias2[c]) + a.norms2[c] * bound);
    const float next = block_max_256(v, red);
    if (threadIdx.x == 0) {
        const float2 first = scale_of(bound), second = scale_of(next);
        reinterpret_cast<float4 *>(a.scales)[blockIdx.x] = make_float4(first.x, first.y, second.x, second.y);
    }
}

// f32 [image][channel][h][w] to the halves layout, border included: a thread
// per word pair (both terms), channels in groups of eight. Each workgroup takes
// its image's scale from the (at most 256) partial maxima; an image's first
// one stores it.
__global__ __launch_bounds__(256) void to_halves_kernel(const float *in, uint32_t channels, uint32_t h, uint32_t w,
                                                        const float *partial, uint32_t partials, float *scales,
                                                        uint8_t *out) {
    __shared__ float red[4];
    const HalvesPlane p = halves_plane(h, w);
    const float2 scale = scale_of(block_max_256(
        threadIdx.x < partials ? partial[(size_t)blockIdx.z * partials + threadIdx.x] : 0.0f, red));
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) reinterpret_cast<float2 *>(scales)[blockIdx.z] = scale;
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= p.words) return;
    const uint32_t c0 = blockIdx.y * 8, b = blockIdx.z;
    const uint32_t row = i / (2 * p.slots), rest = i % (2 * p.slots);
    const uint32_t col = 2 * (rest % p.slots) + rest / p.slots;
    const bool inside = row >= 1 && row <= h && col >= 1 && col <= w;
    const float up = scale.x;
    const float *src = in + (((size_t)b * channels + c0) * h + (inside ? row - 1 : 0)) * w + (inside ? col - 1 : 0);
    ch8 hi, lo;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        _Float16 x, y;
        split_half(inside ? src[(size_t)k * h * w] : 0.0f, up, x, y);
        hi[k] = x, lo[k] = y;
    }
    uint8_t *to = out + ((((size_t)b * (channels / kMfIc) + c0 / kMfIc) * 4 + (c0 / 8 & 1)) * p.words + i) * 16;
    *reinterpret_cast<ch8 *>(to) = hi;
    *reinterpret_cast<ch8 *>(to + (size_t)2 * p.words * 16) = lo;
}

// conv1 of the tower (one input channel) from the log-mel [bins][frames]
// straight to the halves layout: image b is the chunk_frames frames from
// chunk first + b (zero past the clip, model.zig:557-563). A thread takes one
// word position of the padded output plane and 16 channels: its nine samples
// are read once, each output is bias + the taps in the reference's order, then
// GELU and the two terms; border words are zero.
struct Conv1HalvesArgs {
    const float *mel;
    const uint16_t *weights;
    const float *bias, *scales;  // (four scales an image)
    uint8_t *out;
    uint32_t bins, frames, chunk_frames, first, channels, oh, ow;
};

__global__ __launch_bounds__(256) void conv1_halves_kernel(const Conv1HalvesArgs a) {
    __shared__ float wts[kMfIc][9];
    __shared__ float bs[kMfIc];
    const uint32_t c0 = blockIdx.y * kMfIc, b = blockIdx.z;
    if (threadIdx.x < kMfIc * 9)
        wts[threadIdx.x / 9][threadIdx.x % 9] = dev::f16_bits_to_f32(a.weights[(size_t)c0 * 9 + threadIdx.x]);
    if (threadIdx.x < kMfIc) bs[threadIdx.x] = a.bias[c0 + threadIdx.x];
    __syncthreads();
    const HalvesPlane p = halves_plane(a.oh, a.ow);
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= p.words) return;
    const uint32_t prow = i / (2 * p.slots), rest = i % (2 * p.slots);
    const uint32_t pcol = 2 * (rest % p.slots) + rest / p.slots;
    cu4 *to = reinterpret_cast<cu4 *>(a.out) + ((size_t)b * (a.channels / kMfIc) + blockIdx.y) * 4 * p.words + i;
    if (prow < 1 || prow > a.oh || pcol < 1 || pcol > a.ow) {
#pragma unroll
        for (int k = 0; k < 4; ++k) to[(size_t)k * p.words] = cu4{0, 0, 0, 0};
        return;
    }
    const uint64_t frame0 = (uint64_t)(a.first + b) * a.chunk_frames;
    float x[9];
    bool ok[9];
#pragma unroll
    for (int tap = 0; tap < 9; ++tap) {
        const int r = (int)(prow - 1) * 2 + tap / 3 - 1, c = (int)(pcol - 1) * 2 + tap % 3 - 1;
        ok[tap] = r >= 0 && r < (int)a.bins && c >= 0 && c < (int)a.chunk_frames;
        x[tap] = ok[tap] && frame0 + c < a.frames ? a.mel[(size_t)r * a.frames + frame0 + c] : 0.0f;
    }
    const float up = a.scales[4 * (size_t)b];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        ch8 hi, lo;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            float acc = 0.0f;
#pragma unroll
            for (int tap = 0; tap < 9; ++tap)
                if (ok[tap]) acc = fmaf(wts[8 * h + k][tap], x[tap], acc);
            _Float16 u, l;
            split_half(dev::gelu(bs[8 * h + k] + acc), up, u, l);
            hi[k] = u, lo[k] = l;
        }
        to[(size_t)h * p.words] = __builtin_bit_cast(cu4, hi);
        to[(size_t)(2 + h) * p.words] = __builtin_bit_cast(cu4, lo);
    }
}

// One input channel (conv1 of the tower, on the log-mel): each thread takes
// one output position of one image and a range of output channels; its nine
// input samples are read once, each output is bias + the taps in the
// reference's order (rows, then columns; taps outside the plane skipped),
// then GELU. Stores are coalesced over positions.
constexpr uint32_t kC1Oc = 64;   // output channels per workgroup column
__global__ __launch_bounds__(256) void conv1_gelu_kernel(const ConvArgs a) {
    __shared__ float wts[kC1Oc][9];
    __shared__ float bs[kC1Oc];
    const uint32_t t = threadIdx.x;
    const uint32_t oc0 = blockIdx.y * kC1Oc;
    const uint32_t b = blockIdx.z;
    const uint32_t positions = a.oh * a.ow;
    const uint32_t p = blockIdx.x * 256 + t;
    for (uint32_t i = t; i < kC1Oc * 9; i += 256) {
        const uint32_t oc = oc0 + i / 9;
        wts[i / 9][i % 9] = oc < a.out_ch ? dev::f16_bits_to_f32(a.weights[(size_t)oc * 9 + i % 9]) : 0.0f;
    }
    if (t < kC1Oc) bs[t] = oc0 + t < a.out_ch ? a.bias[oc0 + t] : 0.0f;
    __syncthreads();
    if (p >= positions) return;
    const uint32_t orow = p / a.ow, ocol = p % a.ow;
    const float *in = a.in + (size_t)b * a.h * a.w;
    float x[9];
    bool ok[9];
#pragma unroll
    for (int tap = 0; tap < 9; ++tap) {
        const int r = (int)orow * 2 + tap / 3 - 1, c = (int)ocol * 2 + tap % 3 - 1;
        ok[tap] = r >= 0 && r < (int)a.h && c >= 0 && c < (int)a.w;
        x[tap] = ok[tap] ? in[(size_t)r * a.w + c] : 0.0f;
    }
    const uint32_t end = a.out_ch - oc0 < kC1Oc ? a.out_ch - oc0 : kC1Oc;
    float *out = a.out + ((size_t)b * a.out_ch + oc0) * positions + p;
    for (uint32_t k = 0; k < end; ++k) {
        float acc = 0.0f;
#pragma unroll
        for (int tap = 0; tap < 9; ++tap)
            if (ok[tap]) acc = fmaf(wts[k][tap], x[tap], acc);
        out[(size_t)k * positions] = dev::gelu(bs[k] + acc);
    }
}

// Chunks [first, first + count) of the log-mel [bins][frames] into
// [count][bins][chunk_frames], frames past the clip zero (model.zig:557-563).
__global__ void gather_chunks_kernel(const float *mel, uint32_t bins, uint32_t frames, uint32_t chunk_frames,
                                     uint32_t first, uint32_t count, float *out) {
    const uint64_t n = (uint64_t)count * bins * chunk_frames;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t t = (uint32_t)(i % chunk_frames);
        const uint32_t bin = (uint32_t)((i / chunk_frames) % bins);
        const uint32_t c = (uint32_t)(i / ((uint64_t)chunk_frames * bins));
        const uint64_t frame = (uint64_t)(first + c) * chunk_frames + t;
        out[i] = frame < frames ? mel[(uint64_t)bin * frames + frame] : 0.0f;
    }
}

// projectConvStep's flatten (model.zig:615-631). Every chunk but the clip's
// last is whole, so row r of a run of chunks is step r % steps_per_chunk of
// chunk r / steps_per_chunk; its features are channel-major over the
// frequency bins: flat[r][c * bins + f] = conv3[chunk][c][f][step].
__global__ void pack_steps_kernel(const float *conv3, uint32_t channels, uint32_t bins, uint32_t steps_per_chunk,
                                  uint32_t rows, float *flat) {
    const uint32_t features = channels * bins;
    const uint64_t n = (uint64_t)rows * features;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t r = (uint32_t)(i / features), k = (uint32_t)(i % features);
        const uint32_t c = k / bins, f = k % bins;
        const uint32_t chunk = r / steps_per_chunk, step = r % steps_per_chunk;
        flat[i] = conv3[(((uint64_t)chunk * channels + c) * bins + f) * steps_per_chunk + step];
    }
}

// addSinusoidalPosition (model.zig:751-763) from a table of f32 values the
// host computed in f64: encoder row first + r is step (first + r) %
// steps_per_chunk of its chunk.
__global__ void add_positions_kernel(float *rows, const float *table, uint32_t first, uint32_t count, uint32_t width,
                                     uint32_t steps_per_chunk) {
    const uint64_t n = (uint64_t)count * width;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t r = (uint32_t)(i / width), k = (uint32_t)(i % width);
        rows[i] += table[(uint64_t)((first + r) % steps_per_chunk) * width + k];
    }
}

unsigned blocks_for(uint64_t n) {
    const uint64_t b = (n + 255) / 256;
    return (unsigned)(b < 65535 ? (b ? b : 1) : 65535);
}

}  // namespace

hipError_t launch_conv3x3s2_gelu(hipStream_t s, float *out, const float *in, const uint16_t *weights, const float *bias,
                                 uint32_t batch, uint32_t out_ch, uint32_t in_ch, uint32_t h, uint32_t w) {
    ConvArgs a{};
    a.out = out, a.in = in, a.weights = weights, a.bias = bias;
    a.out_ch = out_ch, a.in_ch = in_ch, a.h = h, a.w = w;
    a.oh = (h - 1) / 2 + 1, a.ow = (w - 1) / 2 + 1;
    a.tiles_w = (a.ow + kTile - 1) / kTile;
    const uint32_t tiles_h = (a.oh + kTile - 1) / kTile;
    if (in_ch == 1) {
        const dim3 grid1((a.oh * a.ow + 255) / 256, (out_ch + kC1Oc - 1) / kC1Oc, batch);
        conv1_gelu_kernel<<<grid1, 256, 0, s>>>(a);
        return hipGetLastError();
    }
    const dim3 grid((out_ch + kOcTile - 1) / kOcTile, tiles_h * a.tiles_w, batch);
    conv3x3s2_gelu_kernel<<<grid, 256, 0, s>>>(a);
    return hipGetLastError();
}

namespace {

// Patch rows for `positions` positions starting anywhere in a row of `ow`.
uint32_t mfma_patch_rows(uint32_t ow, uint32_t positions = kMfPos) { return 2 * ((positions - 1 + ow - 1) / ow) + 3; }

uint32_t mfma_oc_pad(uint32_t out_ch) { return (out_ch + 63) / 64 * 64; }

// Workgroups that look for an image's largest magnitude: four rows a wavefront,
// more of them where the images alone fill the device; at most 256 to an image.
uint32_t maxima_blocks(uint32_t images, uint32_t rows) {
    return std::min({(rows + 15) / 16, std::max(1u, 2048 / images), 256u});
}
// An image that lies in one piece is read in rows of this many values.
constexpr uint32_t kMaximaRow = 256;
uint32_t maxima_rows(uint32_t channels, uint32_t h, uint32_t w) {
    return (uint32_t)(((uint64_t)channels * h * w + kMaximaRow - 1) / kMaximaRow);
}

// Workspace pieces of a prepared convolution: operand-order weights, channel
// sums, partial maxima and scales, 256-byte aligned.
size_t piece(size_t bytes) { return (bytes + 255) & ~(size_t)255; }
size_t wprep_bytes(uint32_t out_ch, uint32_t in_ch) { return piece((size_t)mfma_oc_pad(out_ch) * in_ch * 9 * 2); }
size_t norms_bytes(uint32_t out_ch) { return piece((size_t)mfma_oc_pad(out_ch) * sizeof(float)); }
// (At least images * maxima_blocks, and no less for more images: a caller sizes for
// its largest run.)
size_t maxima_bytes(uint32_t images, uint32_t rows) {
    return piece(std::min<size_t>((size_t)images * std::min((rows + 15) / 16, 256u), std::max(images, 2048u)) * sizeof(float));
}
size_t scale_bytes(uint32_t images) { return piece((size_t)images * 4 * sizeof(float)); }

size_t halves_image_bytes(uint32_t channels, uint32_t h, uint32_t w) {
    return (size_t)channels / kMfIc * 4 * halves_plane(h, w).words * 16;
}

template <int NT, bool HALVES>
hipError_t launch_mfma_tiles(hipStream_t s, ConvMfmaArgs a, uint32_t slices) {
    const HalvesPlane p = halves_plane(a.h, a.w);
    a.patch_rows = std::min(mfma_patch_rows(a.ow, 32 * NT), a.h + 2);
    a.pos_tiles = (a.positions + 32 * NT - 1) / (32 * NT);
    a.units = a.batch * a.pos_tiles;
    a.oc_blocks = (a.out_ch + kMfOc - 1) / kMfOc;
    a.slice_stages = (a.stages + slices - 1) / slices;
    a.slices = (a.stages + a.slice_stages - 1) / a.slice_stages;
    if (a.slices == 1) a.part = nullptr;
    const uint32_t grid = (a.units + 7) / 8 * 8 * a.oc_blocks * a.slices;
    const uint32_t rounds = (a.patch_rows * 2 * p.slots * 4 + 255) / 256;
    if (rounds <= 2) conv3x3s2_gelu_mfma_kernel<NT, 2, HALVES><<<grid, 256, 0, s>>>(a);
    else if (rounds <= 4) conv3x3s2_gelu_mfma_kernel<NT, 4, HALVES><<<grid, 256, 0, s>>>(a);
    else if (rounds <= 6) conv3x3s2_gelu_mfma_kernel<NT, 6, HALVES><<<grid, 256, 0, s>>>(a);
    else if (rounds <= 8) conv3x3s2_gelu_mfma_kernel<NT, 8, HALVES><<<grid, 256, 0, s>>>(a);
    else if (rounds <= kMfRounds) conv3x3s2_gelu_mfma_kernel<NT, kMfRounds, HALVES><<<grid, 256, 0, s>>>(a);
    else return hipErrorInvalidValue;
    if (a.slices > 1) {
        const uint64_t n = (uint64_t)a.batch * ((a.out_ch + 7) / 8) * a.positions;
        conv_finish_kernel<HALVES><<<(uint32_t)((n + 255) / 256), 256, 0, s>>>(a);
    }
    return hipGetLastError();
}

// 32-position workgroups where 64-position ones leave compute units idle or
// unevenly filled: a compute unit's share took about 42 us a workgroup of 32
// positions and 63 of 64 (30 stages; 30 s of audio conv3 89 / 82 us, conv2 253
// / 252; 4 s conv2 54 / 78, conv3 40 / 66; 11 s conv2 122 / 131).
//
// A few chunks leave most compute units idle even so, behind a chain of all
// the stages: the stages are then split over workgroups, as many as fill the
// device once, and a second pass adds the slices (us, one launch / split in
// `cus / workgroups`: conv2 44 / 28 of one chunk and 45 / 33 of two, conv3 36 /
// 15, 36 / 17, of four 36 / 19 and of eight 36 / 25; a second slice of a
// device more than half full gained nothing).
template <bool HALVES>
hipError_t launch_mfma(hipStream_t s, int cus, ConvMfmaArgs a, uint32_t batch, float *part) {
    a.batch = batch;
    a.part = part;
    auto groups = [&](uint32_t positions) {
        return (uint64_t)batch * ((a.positions + positions - 1) / positions) * ((a.out_ch + kMfOc - 1) / kMfOc);
    };
    auto share = [&](uint32_t positions) { return (groups(positions) + (uint32_t)cus - 1) / (uint32_t)cus; };
    if (2 * share(32) > 3 * share(64)) return launch_mfma_tiles<2, HALVES>(s, a, 1);
    const uint64_t fill = std::min<uint64_t>((uint32_t)cus / groups(32), a.stages / 5);
    return launch_mfma_tiles<1, HALVES>(s, a, (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(kConvMaxSlices, fill)));
}

// The slices' sums: a split launch has at most `cus` workgroups of 32
// positions by kMfOc channels.
size_t conv_part_bytes(int cus) { return (size_t)cus * 32 * kMfOc * sizeof(float); }

ConvMfmaArgs mfma_args(const void *in, const void *wprep, const float *bias, const float *scales, uint32_t scale_stride,
                       uint32_t out_ch, uint32_t in_ch, uint32_t h, uint32_t w) {
    ConvMfmaArgs a{};
    a.in = static_cast<const uint8_t *>(in);
    a.wprep = static_cast<const uint8_t *>(wprep);
    a.bias = bias;
    a.scales = scales;
    a.scale_stride = scale_stride;
    a.out_ch = out_ch;
    a.oc_tiles = mfma_oc_pad(out_ch) / 32;
    a.stages = in_ch / kMfIc;
    a.h = h, a.w = w;
    a.oh = (h - 1) / 2 + 1, a.ow = (w - 1) / 2 + 1;
    a.positions = a.oh * a.ow;
    return a;
}

}  // namespace

bool conv_mfma_supported(uint32_t in_ch, uint32_t h, uint32_t w) {
    if (in_ch == 0 || in_ch % kMfIc || h == 0 || w == 0) return false;
    const uint32_t ow = (w - 1) / 2 + 1;
    // Four planes of patch words, kMfRounds of 256, in each of two LDS buffers.
    return (uint64_t)mfma_patch_rows(ow) * 2 * ((w + 3) / 2) * 4 <= 256u * kMfRounds;
}

// One convolution over f32 planes: images of at most this many bytes of
// activation terms at a time (at least one).
constexpr size_t kConvGroupBytes = (size_t)256 << 20;

uint32_t conv_mfma_group(uint32_t batch, uint32_t in_ch, uint32_t h, uint32_t w) {
    const size_t image = halves_image_bytes(in_ch, h, w);
    return (uint32_t)std::min<size_t>(batch, std::max<size_t>(1, kConvGroupBytes / image));
}

size_t conv_mfma_bytes(int cus, uint32_t batch, uint32_t out_ch, uint32_t in_ch, uint32_t h, uint32_t w) {
    return wprep_bytes(out_ch, in_ch) + norms_bytes(out_ch) + maxima_bytes(batch, maxima_rows(in_ch, h, w)) + scale_bytes(batch) +
           conv_part_bytes(cus) +
           conv_mfma_group(batch, in_ch, h, w) * halves_image_bytes(in_ch, h, w);
}

hipError_t launch_conv3x3s2_gelu_mfma(hipStream_t s, int cus, float *out, const float *in, const uint16_t *weights,
                                      const float *bias, uint32_t batch, uint32_t out_ch, uint32_t in_ch, uint32_t h,
                                      uint32_t w, void *scratch) {
    if (!conv_mfma_supported(in_ch, h, w) || batch == 0 || batch > 65535) return hipErrorInvalidValue;
    uint8_t *at = static_cast<uint8_t *>(scratch);
    uint8_t *wprep = at;
    float *norms = reinterpret_cast<float *>(at += wprep_bytes(out_ch, in_ch));
    float *partial = reinterpret_cast<float *>(at += norms_bytes(out_ch));
    float *scales = reinterpret_cast<float *>(at += maxima_bytes(batch, maxima_rows(in_ch, h, w)));
    float *part = reinterpret_cast<float *>(at += scale_bytes(batch));
    uint8_t *halves = at + conv_part_bytes(cus);
    ConvPrepArgs p{};
    p.job[0] = {weights, wprep, norms, out_ch, mfma_oc_pad(out_ch), in_ch};
    p.x = in;
    p.rows = maxima_rows(in_ch, h, w);
    p.row_values = kMaximaRow;
    p.row_stride = p.row_used = kMaximaRow;
    p.image_stride = p.limit = (uint64_t)in_ch * h * w;
    p.partial = partial;
    p.partials = maxima_blocks(batch, p.rows);
    conv_prep_kernel<<<p.job[0].oc_pad + batch * p.partials, 256, 0, s>>>(p);
    ConvMfmaArgs a = mfma_args(halves, wprep, bias, scales, 2, out_ch, in_ch, h, w);
    const uint32_t group = conv_mfma_group(batch, in_ch, h, w);
    for (uint32_t b = 0; b < batch; b += group) {
        const uint32_t n = std::min(group, batch - b);
        to_halves_kernel<<<dim3((halves_plane(h, w).words + 255) / 256, in_ch / 8, n), 256, 0, s>>>(
            in + (size_t)b * in_ch * h * w, in_ch, h, w, partial + (size_t)b * p.partials, p.partials,
            scales + 2 * (size_t)b, halves);
        a.scales = scales + 2 * (size_t)b;
        a.out = out + (size_t)b * out_ch * a.positions;
        const hipError_t e = launch_mfma<false>(s, cus, a, n, part);
        if (e != hipSuccess) return e;
    }
    return hipGetLastError();
}

// The tower's three convolutions with conv2 and conv3 in this form.
namespace {

struct TowerPieces {
    size_t wprep2, wprep3, norms2, norms3, partial, scales, part, halves1, halves2, total;
};

TowerPieces tower_pieces(int cus, const ConvTower &c) {
    const uint32_t h1 = (c.bins - 1) / 2 + 1, w1 = (c.chunk_frames - 1) / 2 + 1;
    const uint32_t h2 = (h1 - 1) / 2 + 1, w2 = (w1 - 1) / 2 + 1;
    TowerPieces p{};
    size_t at = 0;
    auto take = [&](size_t bytes) {
        const size_t here = at;
        at += bytes;
        return here;
    };
    p.wprep2 = take(wprep_bytes(c.channels, c.channels));
    p.wprep3 = take(wprep_bytes(c.channels, c.channels));
    p.norms2 = take(norms_bytes(c.channels));
    p.norms3 = take(norms_bytes(c.channels));
    p.partial = take(maxima_bytes(c.chunks, c.bins));
    p.scales = take(scale_bytes(c.chunks));
    p.part = take(conv_part_bytes(cus));
    p.halves1 = take(piece(c.group * halves_image_bytes(c.channels, h1, w1)));
    p.halves2 = take(piece(c.group * halves_image_bytes(c.channels, h2, w2)));
    p.total = at;
    return p;
}

}  // namespace

bool conv_tower_supported(const ConvTower &c) {
    const uint32_t h1 = (c.bins - 1) / 2 + 1, w1 = (c.chunk_frames - 1) / 2 + 1;
    const uint32_t h2 = (h1 - 1) / 2 + 1, w2 = (w1 - 1) / 2 + 1;
    return conv_mfma_supported(c.channels, h1, w1) && conv_mfma_supported(c.channels, h2, w2);
}

size_t conv_tower_bytes(int cus, const ConvTower &c) { return tower_pieces(cus, c).total; }

hipError_t launch_conv_tower_prep(hipStream_t s, int cus, const ConvTower &c, const float *mel, uint32_t frames, void *scratch) {
    uint8_t *base = static_cast<uint8_t *>(scratch);
    const TowerPieces at = tower_pieces(cus, c);
    const uint32_t pad = mfma_oc_pad(c.channels);
    ConvPrepArgs p{};
    p.job[0] = {c.weights[1], base + at.wprep2, reinterpret_cast<float *>(base + at.norms2), c.channels, pad, c.channels};
    p.job[1] = {c.weights[2], base + at.wprep3, reinterpret_cast<float *>(base + at.norms3), c.channels, pad, c.channels};
    p.x = mel;
    p.rows = c.bins;
    p.row_values = c.chunk_frames;
    p.image_stride = p.image_used = c.chunk_frames;
    p.row_stride = p.limit = frames;
    p.partial = reinterpret_cast<float *>(base + at.partial);
    p.partials = maxima_blocks(c.chunks, c.bins);
    conv_prep_kernel<<<2 * pad + c.chunks * p.partials, 256, 0, s>>>(p);
    ConvScaleArgs q{};
    q.partial = p.partial;
    q.partials = p.partials;
    q.conv1 = c.weights[0];
    q.bias1 = c.bias[0];
    q.norms2 = p.job[0].norms;
    q.bias2 = c.bias[1];
    q.channels = c.channels;
    q.scales = reinterpret_cast<float *>(base + at.scales);
    conv_scale_kernel<<<c.chunks, 256, 0, s>>>(q);
    return hipGetLastError();
}

hipError_t launch_conv_tower(hipStream_t s, int cus, const ConvTower &c, const float *mel, uint32_t frames, uint32_t first,
                             uint32_t count, float *out, void *scratch) {
    uint8_t *base = static_cast<uint8_t *>(scratch);
    const TowerPieces at = tower_pieces(cus, c);
    const float *scales = reinterpret_cast<const float *>(base + at.scales) + 4 * (size_t)first;
    const uint32_t h1 = (c.bins - 1) / 2 + 1, w1 = (c.chunk_frames - 1) / 2 + 1;
    Conv1HalvesArgs k{};
    k.mel = mel;
    k.weights = c.weights[0];
    k.bias = c.bias[0];
    k.scales = scales;
    k.out = base + at.halves1;
    k.bins = c.bins, k.frames = frames, k.chunk_frames = c.chunk_frames, k.first = first, k.channels = c.channels;
    k.oh = h1, k.ow = w1;
    conv1_halves_kernel<<<dim3((halves_plane(h1, w1).words + 255) / 256, c.channels / kMfIc, count), 256, 0, s>>>(k);
    ConvMfmaArgs a = mfma_args(base + at.halves1, base + at.wprep2, c.bias[1], scales, 4, c.channels, c.channels, h1, w1);
    a.halves = base + at.halves2;
    const hipError_t e = launch_mfma<true>(s, cus, a, count, reinterpret_cast<float *>(base + at.part));
    if (e != hipSuccess) return e;
    ConvMfmaArgs a3 = mfma_args(base + at.halves2, base + at.wprep3, c.bias[2], scales + 2, 4, c.channels, c.channels, a.oh,
                                a.ow);
    a3.out = out;
    return launch_mfma<false>(s, cus, a3, count, reinterpret_cast<float *>(base + at.part));
}

hipError_t launch_gather_chunks(hipStream_t s, const float *mel, uint32_t bins, uint32_t frames, uint32_t chunk_frames,
                                uint32_t first, uint32_t count, float *out) {
    gather_chunks_kernel<<<blocks_for((uint64_t)count * bins * chunk_frames), 256, 0, s>>>(mel, bins, frames, chunk_frames,
                                                                                          first, count, out);
    return hipGetLastError();
}

hipError_t launch_pack_steps(hipStream_t s, const float *conv3, uint32_t channels, uint32_t bins, uint32_t steps_per_chunk,
                             uint32_t rows, float *flat) {
    pack_steps_kernel<<<blocks_for((uint64_t)rows * channels * bins), 256, 0, s>>>(conv3, channels, bins,
                                                                                  steps_per_chunk, rows, flat);
    return hipGetLastError();
}

hipError_t launch_add_positions(hipStream_t s, float *rows, const float *table, uint32_t first, uint32_t count,
                                uint32_t width, uint32_t steps_per_chunk) {
    add_positions_kernel<<<blocks_for((uint64_t)count * width), 256, 0, s>>>(rows, table, first, count, width,
                                                                            steps_per_chunk);
    return hipGetLastError();
}

}  // namespace qwh

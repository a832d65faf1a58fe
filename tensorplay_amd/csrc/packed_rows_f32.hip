// Packed weights against float32 activations without LDS for those.  First, up to eight rows in blocks of FOUR (int4 layout and n-bit rows, as packed_rows_kernel.h, whose
// blocks of 16 rows multiply padding where the rows do not fill them: one row costs what sixteen do).
//
// What bounds it: about evenly the float32 matrix instructions (some 16 clocks each) and the dequantization (2.3 to 4 vector instructions a
// code), which follow each other: a round of 128 k and 32 channels per wavefront takes 1.5 us with one block of rows, 2.4 with two.
// v_mfma_f32_4x4x1 multiplies sixteen independent blocks of 4 x 4 by one k.  Four of them are 16 channels, four of those groups four tiles of
// 32 k: lane (i, q) dequantizes the 32 codes of channel i in tile q, as the blocks of 16 rows do, and the activations, first operand, come to
// the four blocks of a group from one of them (cbsz 2).  Hence
//   * lane (row, b, q) loads eight k of its row, 32 q + 8 b .. + 7: register v, block abid hold k = 32 q + 8 abid + v, so nothing is staged in
//     LDS, and 128 k of four rows are two 16-byte loads a lane;
//   * a wavefront is 32 channels and R blocks of four rows; a workgroup's eight wavefronts are CW x 32 channels times 8 / CW steps of 128 k at a
//     time, and slices of K (summed by packed_rows_finish_kernel) fill the chip where the channels do not;
//   * sums go over 16 k and those over the wavefront's share (a quarter of its tiles each of the four q); the four q meet by two swaps between lanes,
//     which leave row q in lane group q, the wavefronts meet in LDS by halves;
//   * a last step that is partial repeats the last tile with scale, zero and activations cleared: zeros that meet finite numbers only.
// Measured (us, this kernel / what ran before, in a graph): int4, one row of 4096 x 4096 9.2 / 14.3, 8192 x 8192 15.5 / 29.5; two rows of 2048 x 2048
// 5.9 / 8.5; seven of 8192 x 8192 22 / 30; n-bit rows, 4 rows of 11008 -> 4096 with 8 bits 20 / 28, 2 rows of 5120 -> 13824 with 1 bit 21.5 / 37.5, 7 rows of
// 8192 x 8192 with 4 bits 26 / 35.  A lane per channel (64 channels a wavefront, one k for all blocks) reads a quarter of the activations
// but a line per lane: int4 the same times, two rows of 4096 -> 11008 14.6, n-bit rows half as fast again (4 rows, 2 bits, 4864 -> 9728 28.7, here
// 20.7; 6 rows, 8 bits 50, here 33.5).
#include "packed_rows_bits.h"

namespace tpq {
namespace {

typedef uint32_t quads_pair __attribute__((ext_vector_type(2)));

// per register of four: the sum over the four lane groups of 16, register e in lane group e
__device__ __forceinline__ float over_groups(float4_t v) {
    auto swap16 = [](float a, float b) __attribute__((always_inline)) {  // rows 0, 2 of a beside rows 0, 2 of b, and rows 1, 3
        const quads_pair t = __builtin_bit_cast(quads_pair, __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b), false, false));
        return __builtin_bit_cast(float, static_cast<uint32_t>(t.x)) + __builtin_bit_cast(float, static_cast<uint32_t>(t.y));
    };
    const float e = swap16(v[0], v[1]), f = swap16(v[2], v[3]);
    const quads_pair t = __builtin_bit_cast(quads_pair, __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, e), __builtin_bit_cast(uint32_t, f), false, false));
    return __builtin_bit_cast(float, static_cast<uint32_t>(t.x)) + __builtin_bit_cast(float, static_cast<uint32_t>(t.y));
}

template <class Source, int R>
__global__ __launch_bounds__(8 * kWave) void packed_quads_kernel(const PackedRowsArgs a, int cw_shift) {
    using P = RowsParams<TPQ_DTYPE_F32, Source::kTypedParams>;
    constexpr int kDepth = 3, kChains = R == 1 ? 2 : 1, NB = 2;
    __shared__ float sums[8][R][NB][kWave];
    const int lane = threadIdx.x & (kWave - 1), q = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kw_shift = 3 - cw_shift, k_wave = wave & ((1 << kw_shift) - 1);
    const int n0 = ((blockIdx.x << cw_shift) + (wave >> kw_shift)) * (16 * NB), m0 = blockIdx.y * (4 * R);
    const int tiles = a.K / 32, steps = (tiles + 3) / 4, begin = blockIdx.z * a.steps_per_slice;
    const int end = steps < begin + a.steps_per_slice ? steps : begin + a.steps_per_slice;
    const int count = end - begin > k_wave ? ((end - begin - k_wave - 1) >> kw_shift) + 1 : 0;  // steps of this wavefront

    uint32_t w_off[NB], p_off[NB];
    const uint32_t group_bytes = static_cast<uint32_t>(a.N) * 8u;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        const int n = n0 + 16 * nb + (lane & 15);
        w_off[nb] = Source::lane_offset(a, n, 0);
        p_off[nb] = static_cast<uint32_t>(n < a.N ? n : a.N - 1) * 8u;
    }
    const char* x_row[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int row = m0 + 4 * r + (lane & 3);
        x_row[r] = static_cast<const char*>(a.x) + (static_cast<size_t>(row < a.M ? row : a.M - 1) * a.K + 8 * ((lane >> 2) & 3)) * 4;  // rows past M: the last one again, dropped
    }

    struct Step {
        typename Source::Words w[NB];
        typename P::raw_t p[NB];
        pr_word4 x[R][2];
        bool live;
    };
    auto load = [&](int j, Step& d) __attribute__((always_inline)) {
        const int step = begin + k_wave + ((j < count ? j : count - 1) << kw_shift);  // past the last: that one again
        int tile = 4 * step + q;
        d.live = tile < tiles;
        tile = d.live ? tile : tiles - 1;
        const uint32_t group = static_cast<uint32_t>((static_cast<float>(tile) + 0.5f) * a.inv_tiles_per_group);  // exact: tile < 2^20
        auto from = (TPQ_GLOBAL char*)a.w;
        auto params = (TPQ_GLOBAL char*)a.sz;
        asm volatile("" : "+s"(from), "+s"(params));  // the loads stay here (see pinned_global)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            const pr_word2 t = *(TPQ_GLOBAL pr_word2*)(params + (group * group_bytes + p_off[nb]));
            d.p[nb].x = t.x; d.p[nb].y = t.y;
            Source::load(from, w_off[nb] + static_cast<uint32_t>(tile) * static_cast<uint32_t>(Source::kStepBytes / 4), d.w[nb]);
        }
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int h = 0; h < 2; ++h) d.x[r][h] = *((TPQ_GLOBAL pr_word4*)pinned_global(x_row[r] + static_cast<size_t>(tile) * 128) + h);
    };

    float4_t acc[NB][R];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int r = 0; r < R; ++r) acc[nb][r] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
    uint32_t magic[2] = {Source::kMagic0, Source::kMagic1};
    asm volatile("" : "+v"(magic[0]), "+v"(magic[1]));  // registers: one v_and_or_b32 per pair of codes
    auto multiply = [&](Step& d, int j) __attribute__((always_inline)) {
        float scale[NB], zero[NB];
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) { scale[nb] = P::scale(d.p[nb]); zero[nb] = P::zero(d.p[nb]); }
        if (4 * (begin + k_wave + (j << kw_shift)) + 4 > tiles) {
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) { scale[nb] = d.live ? scale[nb] : 0.0f; zero[nb] = d.live ? zero[nb] : 0.0f; }
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int h = 0; h < 2; ++h) d.x[r][h] = d.live ? d.x[r][h] : pr_word4{0u, 0u, 0u, 0u};
        }
        float4_t piece[kChains][NB][R];
        // a chain is 16 k; with one block of rows both halves of the tile are under way (a product waits for the one before it)
        pr_static_for<0, 16>([&](auto pair_c) __attribute__((always_inline)) {
            constexpr int kPair = decltype(pair_c)::value;
            constexpr int kAt = kChains == 2 ? (kPair >> 1) + 8 * (kPair & 1) : kPair, kChain = kChains == 2 ? kPair & 1 : 0;
            constexpr bool kFirst = kChains == 2 ? kPair < 2 : (kPair & 7) == 0, kLast = kChains == 2 ? kPair >= 14 : (kPair & 7) == 7;
            float w[NB][2];
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                const half2_t h = __builtin_bit_cast(half2_t, Source::pair(d.w[nb], kAt, magic)) -
                                  half2_t{static_cast<_Float16>(Source::offset(kAt, 0)), static_cast<_Float16>(Source::offset(kAt, 1))};
                if constexpr (Source::kTypedParams) {
                    w[nb][0] = __builtin_fmaf(static_cast<float>(h.x), scale[nb], zero[nb]);
                    w[nb][1] = __builtin_fmaf(static_cast<float>(h.y), scale[nb], zero[nb]);
                } else {
                    w[nb][0] = less_zero<0>(h, zero[nb]) * scale[nb];
                    w[nb][1] = less_zero<1>(h, zero[nb]) * scale[nb];
                }
            }
            pr_static_for<0, 2>([&](auto v_c) __attribute__((always_inline)) {
                constexpr int kV = decltype(v_c)::value, kIn = (2 * kAt + kV) & 7, kBlock = (2 * kAt) >> 3;
#pragma unroll
                for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        const uint32_t bits = d.x[r][kIn >> 2][kIn & 3];
                        piece[kChain][nb][r] = __builtin_amdgcn_mfma_f32_4x4x1f32(__builtin_bit_cast(float, bits), w[nb][kV],
                                                                                 kFirst && kV == 0 ? float4_t{0.0f, 0.0f, 0.0f, 0.0f} : piece[kChain][nb][r], 2, kBlock, 0);
                    }
            });
            if constexpr (kLast) {
#pragma unroll
                for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                    for (int r = 0; r < R; ++r)
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[nb][r][e] += piece[kChain][nb][r][e];
            }
        });
    };

    if (count > 0) {
        Step ring[kDepth];
        pr_static_for<0, kDepth>([&](auto d) __attribute__((always_inline)) { load(decltype(d)::value, ring[decltype(d)::value]); });
        int j = 0;
        for (; j + kDepth < count; j += kDepth)
            pr_static_for<0, kDepth>([&](auto d) __attribute__((always_inline)) {
                multiply(ring[decltype(d)::value], j + decltype(d)::value);
                load(j + kDepth + decltype(d)::value, ring[decltype(d)::value]);
                __builtin_amdgcn_sched_barrier(0);
            });
        pr_static_for<0, kDepth>([&](auto d) __attribute__((always_inline)) {
            if (j + decltype(d)::value < count) multiply(ring[decltype(d)::value], j + decltype(d)::value);
        });
    }

#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) sums[wave][r][nb][lane] = over_groups(acc[nb][r]);
    __syncthreads();
    // an output per thread: one of the channel positions, its blocks of 16 channels and of four rows
    for (int t = wave; t < (R * NB << cw_shift); t += 8) {
        const int c = t / (R * NB), r = t % (R * NB) / NB, nb = t % NB;
        const int m = m0 + 4 * r + q, n = ((blockIdx.x << cw_shift) + c) * (16 * NB) + 16 * nb + (lane & 15);
        if (m >= a.M || n >= a.N) continue;
        const float(*from)[R][NB][kWave] = sums + (c << kw_shift);
        float s;
        if (cw_shift == 0)
            s = ((from[0][r][nb][lane] + from[1][r][nb][lane]) + (from[2][r][nb][lane] + from[3][r][nb][lane])) +
                ((from[4][r][nb][lane] + from[5][r][nb][lane]) + (from[6][r][nb][lane] + from[7][r][nb][lane]));
        else
            s = (from[0][r][nb][lane] + from[1][r][nb][lane]) + (from[2][r][nb][lane] + from[3][r][nb][lane]);
        const size_t at = static_cast<size_t>(m) * a.N + n;
        if (a.partial != nullptr) {
            a.partial[static_cast<size_t>(blockIdx.z) * a.M * a.N + at] = s;
            continue;
        }
        if (a.bias != nullptr) s += a.bias[n];
        if (a.after != nullptr) s += static_cast<const float*>(a.after)[n];
        static_cast<float*>(a.y)[at] = s;
    }
}

// ---- more rows: a lane per channel ----------------------------------------------------------------------------
// From nine rows on, where that is the faster way (packed_rows_f32_plan).  What bounds it: the matrix instructions, 32 clocks for 16 rows x 64 channels x one k
// (v_mfma_f32_16x16x1, four blocks of 16 channels), and the dequantization behind them.  What the kernel with its activations in LDS spends beside those, barriers between
// its rounds and wavefronts that only fetch, is not here: a wavefront takes tiles of 32 k for itself, MB blocks of 16 rows and, QB, one of four rows (v_mfma_f32_4x4x1 with
// the channels of a lane side by side), so that 19 rows cost 20 and not 32.
//   * lane n is channel n: its 32 codes of a tile, dequantized, are the second operand as they are, its (scale, zero) one load.  n-bit rows are read a line per lane: with so
//     many rows to multiply that is still the smaller part;
//   * activations, first operand, reach all four blocks from one (cbsz 2): lane (row, b) loads eight k of its row, 8 b .. + 7, register v, block abid hold k = 8 abid + v;
//     of the block of four (cbsz 4), lane (row, b) holds k = 2 b, + 1;
//   * sums go over 16 k, those over a group of three or four tiles, the groups over the wavefront's share: in one chain over 2944 k the error against float64 is 1.14 times that of
//     the staged kernel, whose steps of 128 k are summed first.  Three blocks of rows and more have no registers for both: the groups' sum lies in LDS, each lane's own words
//     (read, added to and written once in four tiles; slices of up to 48 tiles, where one chain is as precise by the variances of the roundings - (1 / 256 - 1 / 1024) K <= 4.5 -
//     go without).  The eight wavefronts' sums meet in LDS by halves, up to two blocks 16 rows at a time.
// Measured (us, before / with this, in a graph): int4 19 rows 4096 x 4096 17.4 / 13.4, 35 rows 26.5 / 19.2, 17 rows 11008 -> 4096 35.5 / 25.6; 8 bits, 36 rows 4096 x 4096 30 / 24.8.
typedef float float16_t __attribute__((ext_vector_type(16)));
constexpr int kLanesGroupBlocks = 2, kLanesOneChain = 48;  // blocks of 16 rows whose groups are summed in registers; tiles of a slice without groups in LDS
constexpr int kLanesPitch = kWave + 4;  // of a row of sums in LDS: the four rows that a wavefront stores at once lie 16 banks apart

constexpr int lanes_words(int mb, int qb) { return mb <= kLanesGroupBlocks ? 16 : 16 * mb + 4 * qb; }  // of LDS a lane of each wavefront

// one block of rows, up to 4 bits: two workgroups on a compute unit, three tiles in flight each
template <class Source, int MB, int QB>
constexpr bool lanes_in_pairs() { return MB == 1 && QB == 0 && sizeof(typename Source::Words) <= 16; }

template <class Source, int MB, int QB>
__global__ __launch_bounds__(8 * kWave, (lanes_in_pairs<Source, MB, QB>() ? 4 : 2)) void packed_lanes_kernel(const PackedRowsArgs a) {
    using P = RowsParams<TPQ_DTYPE_F32, Source::kTypedParams>;
    constexpr int kDepth = lanes_in_pairs<Source, MB, QB>() ? 3 : MB == 1 ? 4 : MB == 2 ? 3 : 2, kChains = MB == 1 ? 2 : 1;
    constexpr bool kGroups = MB <= kLanesGroupBlocks;
    extern __shared__ float lanes_sums[];  // [8][lanes_words(MB, QB)][kLanesPitch]
    auto sums = reinterpret_cast<float(*)[lanes_words(MB, QB)][kLanesPitch]>(lanes_sums);
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = blockIdx.x * kWave + lane, m0 = blockIdx.y * (16 * MB + 4 * QB);
    const int tiles = a.K / 32, begin = blockIdx.z * a.steps_per_slice;  // (steps_per_slice: tiles)
    const int end = tiles < begin + a.steps_per_slice ? tiles : begin + a.steps_per_slice;
    const int count = end - begin > wave ? (end - begin - wave + 7) / 8 : 0;  // tiles of this wavefront

    const uint32_t w_off = Source::lane_offset(a, n, 0);
    const uint32_t p_off = static_cast<uint32_t>(n < a.N ? n : a.N - 1) * 8u, group_bytes = static_cast<uint32_t>(a.N) * 8u;
    const char* x_row[MB];
#pragma unroll
    for (int b = 0; b < MB; ++b) {
        const int row = m0 + 16 * b + (lane & 15);
        x_row[b] = static_cast<const char*>(a.x) + (static_cast<size_t>(row < a.M ? row : a.M - 1) * a.K + 8 * (lane >> 4)) * 4;  // rows past M: the last one again, dropped
    }
    const int quad_row = m0 + 16 * MB + (lane & 3);
    const char* const x_quad = static_cast<const char*>(a.x) + (static_cast<size_t>(quad_row < a.M ? quad_row : a.M - 1) * a.K + 2 * (lane >> 2)) * 4;
    struct Tile {
        typename Source::Words w;
        typename P::raw_t p;
        pr_word4 x[MB][2];
        pr_word2 x_quad;
    };
    auto load = [&](int j, Tile& d) __attribute__((always_inline)) {
        const int tile = begin + wave + 8 * (j < count ? j : count - 1);  // past the last: that one again
        const uint32_t group = static_cast<uint32_t>((static_cast<float>(tile) + 0.5f) * a.inv_tiles_per_group);  // exact: tile < 2^20
        auto from = (TPQ_GLOBAL char*)a.w + static_cast<size_t>(tile) * (Source::kStepBytes / 4);
        auto params = (TPQ_GLOBAL char*)a.sz;
        asm volatile("" : "+s"(from), "+s"(params));  // the loads stay here (see pinned_global)
        const pr_word2 t = *(TPQ_GLOBAL pr_word2*)(params + (group * group_bytes + p_off));
        d.p.x = t.x; d.p.y = t.y;
        Source::load(from, w_off, d.w);
#pragma unroll
        for (int b = 0; b < MB; ++b)
#pragma unroll
            for (int h = 0; h < 2; ++h) d.x[b][h] = *((TPQ_GLOBAL pr_word4*)pinned_global(x_row[b] + static_cast<size_t>(tile) * 128) + h);
        if constexpr (QB) d.x_quad = *(TPQ_GLOBAL pr_word2*)pinned_global(x_quad + static_cast<size_t>(tile) * 128);
    };

    float16_t acc[MB] = {}, group_sum[kGroups ? MB : 1] = {};
    float4_t acc_quad = {}, group_quad = {};
    auto flush = [&]() __attribute__((always_inline)) {
        if constexpr (kGroups) {
#pragma unroll
            for (int b = 0; b < MB; ++b) {
                acc[b] += group_sum[b];
                group_sum[b] = float16_t{};
            }
            if constexpr (QB) {
                acc_quad += group_quad;
                group_quad = float4_t{};
            }
        }
    };
    // kGroups: nothing; else the lane's words of LDS := the same (first) or += acc, and acc := 0
    auto to_lds = [&](bool first) __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < MB; ++b)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                float& at = sums[wave][16 * b + e][lane];
                at = first ? acc[b][e] : at + acc[b][e];
                acc[b][e] = 0.0f;
            }
        if constexpr (QB) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float& at = sums[wave][16 * MB + e][lane];
                at = first ? acc_quad[e] : at + acc_quad[e];
                acc_quad[e] = 0.0f;
            }
        }
    };
    bool first_group = true;
    const bool in_groups = end - begin > kLanesOneChain;
    uint32_t magic[2] = {Source::kMagic0, Source::kMagic1};
    asm volatile("" : "+v"(magic[0]), "+v"(magic[1]));
    auto multiply = [&](const Tile& d) __attribute__((always_inline)) {
        const float scale = P::scale(d.p), zero = P::zero(d.p);
        float16_t piece[kChains][MB];
        float4_t piece_quad[kChains];
        pr_static_for<0, 16>([&](auto pair_c) __attribute__((always_inline)) {
            constexpr int kPair = decltype(pair_c)::value;
            constexpr int kAt = kChains == 2 ? (kPair >> 1) + 8 * (kPair & 1) : kPair, kChain = kChains == 2 ? kPair & 1 : 0;
            constexpr bool kFirst = kChains == 2 ? kPair < 2 : (kPair & 7) == 0, kLast = kChains == 2 ? kPair >= 14 : (kPair & 7) == 7;
            const half2_t h = __builtin_bit_cast(half2_t, Source::pair(d.w, kAt, magic)) -
                              half2_t{static_cast<_Float16>(Source::offset(kAt, 0)), static_cast<_Float16>(Source::offset(kAt, 1))};
            float w[2];
            if constexpr (Source::kTypedParams) {
                w[0] = __builtin_fmaf(static_cast<float>(h.x), scale, zero);
                w[1] = __builtin_fmaf(static_cast<float>(h.y), scale, zero);
            } else {
                w[0] = less_zero<0>(h, zero) * scale;
                w[1] = less_zero<1>(h, zero) * scale;
            }
            pr_static_for<0, 2>([&](auto v_c) __attribute__((always_inline)) {
                constexpr int kV = decltype(v_c)::value, kIn = (2 * kAt + kV) & 7, kBlock = (2 * kAt) >> 3;
#pragma unroll
                for (int b = 0; b < MB; ++b) {
                    const uint32_t bits = d.x[b][kIn >> 2][kIn & 3];
                    piece[kChain][b] = __builtin_amdgcn_mfma_f32_16x16x1f32(__builtin_bit_cast(float, bits), w[kV], kFirst && kV == 0 ? float16_t{} : piece[kChain][b], 2, kBlock, 0);
                }
                if constexpr (QB) {
                    const uint32_t bits = kV ? d.x_quad.y : d.x_quad.x;
                    piece_quad[kChain] = __builtin_amdgcn_mfma_f32_4x4x1f32(__builtin_bit_cast(float, bits), w[kV], kFirst && kV == 0 ? float4_t{} : piece_quad[kChain], 4, kAt, 0);
                }
            });
            if constexpr (kLast) {
#pragma unroll
                for (int b = 0; b < MB; ++b)
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        if constexpr (kGroups) group_sum[b][e] += piece[kChain][b][e];
                        else acc[b][e] += piece[kChain][b][e];
                    }
                if constexpr (QB) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        if constexpr (kGroups) group_quad[e] += piece_quad[kChain][e];
                        else acc_quad[e] += piece_quad[kChain][e];
                    }
                }
            }
        });
    };

    if (count > 0) {
        Tile ring[kDepth];
        pr_static_for<0, kDepth>([&](auto d) __attribute__((always_inline)) { load(decltype(d)::value, ring[decltype(d)::value]); });
        int j = 0;
        for (; j + kDepth < count; j += kDepth) {
            pr_static_for<0, kDepth>([&](auto d) __attribute__((always_inline)) {
                multiply(ring[decltype(d)::value]);
                load(j + kDepth + decltype(d)::value, ring[decltype(d)::value]);
                if constexpr (decltype(d)::value == kDepth - 1) flush();
                __builtin_amdgcn_sched_barrier(0);
            });
            if constexpr (!kGroups) {
                static_assert(kDepth == 2, "a group of four tiles is two turns of the ring");
                if (in_groups && (j & 2)) {
                    to_lds(first_group);
                    first_group = false;
                }
            }
        }
        pr_static_for<0, kDepth>([&](auto d) __attribute__((always_inline)) {
            if (j + decltype(d)::value < count) multiply(ring[decltype(d)::value]);
        });
        flush();
    }

    if constexpr (!kGroups) {
        to_lds(first_group);
        __syncthreads();
    }
    auto store = [&](int row, int at_lane, int m) __attribute__((always_inline)) {  // row: of words in LDS
        if (m >= a.M || n >= a.N) return;
        float part[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) part[k] = sums[k][row][at_lane];
        float s = ((part[0] + part[1]) + (part[2] + part[3])) + ((part[4] + part[5]) + (part[6] + part[7]));
        const size_t at = static_cast<size_t>(m) * a.N + n;
        if (a.partial != nullptr) {
            a.partial[static_cast<size_t>(blockIdx.z) * a.M * a.N + at] = s;
            return;
        }
        if (a.bias != nullptr) s += a.bias[n];
        if (a.after != nullptr) s += static_cast<const float*>(a.after)[n];
        static_cast<float*>(a.y)[at] = s;
    };
    if constexpr (kGroups) {
#pragma unroll
        for (int b = 0; b < MB; ++b) {
            if (b > 0) __syncthreads();
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int e = 0; e < 4; ++e) sums[wave][4 * (lane >> 4) + e][16 * c + (lane & 15)] = acc[b][4 * c + e];
            __syncthreads();
#pragma unroll
            for (int h = 0; h < 2; ++h) store(wave + 8 * h, lane, m0 + 16 * b + wave + 8 * h);
        }
        if constexpr (QB) {
            __syncthreads();
#pragma unroll
            for (int e = 0; e < 4; ++e) sums[wave][e][lane] = acc_quad[e];
            __syncthreads();
            if (wave < 4) store(wave, lane, m0 + 16 * MB + wave);
        }
    } else {  // as the products left them: row 4 q + e of a block, channel 16 c + i in word 4 c + e of lane (i, q)
#pragma unroll
        for (int h = 0; h < 2 * MB; ++h) {
            const int row = wave + 8 * h, in_block = row & 15;
            store((row & ~15) + 4 * (lane >> 4) + (in_block & 3), (in_block >> 2) * 16 + (lane & 15), m0 + row);
        }
        if constexpr (QB) {
            if (wave < 4) store(16 * MB + wave, lane, m0 + 16 * MB + wave);
        }
    }
}

template <class Source, int MB, int QB>
int launch_packed_lanes(const PackedRowsArgs& a, const dim3& grid, hipStream_t s) {
    constexpr size_t smem = static_cast<size_t>(8) * lanes_words(MB, QB) * kLanesPitch * sizeof(float);
    static_assert(smem <= 160 * 1024, "LDS of one compute unit");
    auto kernel = packed_lanes_kernel<Source, MB, QB>;
    static std::atomic<uint64_t> configured{0};
    if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(kernel), smem, configured, "packed rows (float32)")) return rc;
    kernel<<<grid, 8 * kWave, smem, s>>>(a);
    return TPQ_OK;
}

template <class Source>
int launch_packed_f32(PackedRowsArgs a, int quads, int cw, int slices, hipStream_t s) {
    const int channels = cw == 0 ? kWave : 32 * cw;
    const dim3 grid(static_cast<unsigned>((a.N + channels - 1) / channels), static_cast<unsigned>((a.M + 4 * quads - 1) / (4 * quads)), static_cast<unsigned>(slices));
    if (cw > 0) {
        if (quads == 1)
            packed_quads_kernel<Source, 1><<<grid, 8 * kWave, 0, s>>>(a, cw >> 1);
        else
            packed_quads_kernel<Source, 2><<<grid, 8 * kWave, 0, s>>>(a, cw >> 1);
    } else {
        int rc;
        switch (quads) {
            case 4: rc = launch_packed_lanes<Source, 1, 0>(a, grid, s); break;
            case 5: rc = launch_packed_lanes<Source, 1, 1>(a, grid, s); break;
            case 8: rc = launch_packed_lanes<Source, 2, 0>(a, grid, s); break;
            case 9: rc = launch_packed_lanes<Source, 2, 1>(a, grid, s); break;
            case 12: rc = launch_packed_lanes<Source, 3, 0>(a, grid, s); break;
            case 13: rc = launch_packed_lanes<Source, 3, 1>(a, grid, s); break;
            default: rc = launch_packed_lanes<Source, 4, 0>(a, grid, s); break;
        }
        if (rc) return rc;
    }
    if (int rc = check_launch("packed rows (float32)")) return rc;
    if (a.partial == nullptr) return TPQ_OK;
    const int64_t quarters = static_cast<int64_t>(a.M) * a.N / 4;
    packed_rows_finish_kernel<TPQ_DTYPE_F32><<<static_cast<unsigned>((quarters + 255) / 256), 256, 0, s>>>(
        a.partial, slices, quarters, a.bias, static_cast<const float*>(a.after), a.N / 4, static_cast<float*>(a.y));
    return check_launch("packed rows (sum of the slices)");
}

}  // namespace

int packed_rows_f32(const PackedRowsBits& c, int quads, int cw, int slices, int steps_per_slice) {
    PackedRowsArgs a{};
    a.x = c.x; a.w = c.packed; a.sz = c.sz; a.bias = c.bias; a.after = c.after; a.y = c.out; a.partial = slices > 1 ? static_cast<float*>(c.workspace) : nullptr;
    a.M = static_cast<int>(c.M); a.N = static_cast<int>(c.N); a.K = static_cast<int>(c.K);
    a.tiles_per_group = static_cast<int>(c.group / 32);
    a.inv_tiles_per_group = 1.0f / static_cast<float>(a.tiles_per_group);
    a.steps_per_slice = steps_per_slice;
    switch (c.bits) {
        case 0: return launch_packed_f32<SourceInt4>(a, quads, cw, slices, c.stream);
        case 1: return c.lsb_first ? launch_packed_f32<SourceBits<1, true>>(a, quads, cw, slices, c.stream) : launch_packed_f32<SourceBits<1, false>>(a, quads, cw, slices, c.stream);
        case 2: return launch_packed_f32<SourceBits<2, false>>(a, quads, cw, slices, c.stream);
        case 4: return launch_packed_f32<SourceBits<4, false>>(a, quads, cw, slices, c.stream);
        default: return launch_packed_f32<SourceBits<8, false>>(a, quads, cw, slices, c.stream);
    }
}

}  // namespace tpq

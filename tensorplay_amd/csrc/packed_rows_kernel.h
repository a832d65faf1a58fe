// Weight-only product of a block of activation rows (a prompt, a decode batch: 9 .. a few hundred rows) with a packed
// weight, float16 / bfloat16 / float32, groups of any multiple of 32, K % 32 == 0:
//   y[m][n] = sum_k x[m][k] w[n][k],  w dequantized in registers, once per 16 MB rows, on its way into the matrix cores.
// The weight comes from one of two sources: the int4 device layout (tiles of 8 channels x 32 k) or rows of n-bit codes.
//
// What bounds it: with few rows the stream of the weight and the latency of its first bytes; from about 48 rows on what a
// compute unit does per step of 128 k and 32 channels, of which four things cost about the same (clocks per round of the loop
// at 64 rows, two multiplying wavefronts per SIMD): the activations through its vector memory path (64 KB at 21.6 clocks per
// KB, 1400), the fragment reads from LDS (1024 + 512 for writing them), the dequantization (1280) and the products (1024).
// Taken out one at a time they all shorten the loop, none by much (4096 x 4096 at 256 rows, bfloat16: 17.0 us, without
// activations 13.3, without dequantization 16.5, without products 15.4, loads of weights and barriers alone 8.9).  Hence
//   * a workgroup owns 64 channels (128 where that still fills the chip: half the activation bytes per product; 32 with few rows, which then
//     need no slices) and a slice of K (a few slices of K fill the chip where N / 64 workgroups do not; their fp32 sums meet in a second kernel,
//     added in slice order, float32 four at a time by halves);
//   * up to 64 rows, with 128 channels up to 128 (whose two rounds of activations fill 128 KB of LDS): a taller tile dequantizes
//     its channels once for more rows, and 203 rows of 4096 -> 11008 are 172 tiles of 112 rows in one round of workgroups instead of 344 of 64
//     in two (2 bits 48.5 -> 32, int4 41 -> 28 us; int4 at 256 rows 43 -> 34, at 384 66 -> 53);
//   * its eight multiplying wavefronts are CW channel positions x KW steps of 128 k: a round of the loop covers KW steps, whose
//     activations two more wavefronts fetch by direct global -> LDS loads (whole lines, one copy per workgroup, the
//     swizzle of the fragment reads applied on the global side) into a ring of two to three rounds while the rounds before are multiplied:
//     with two, a round's loads were all waited for before the next ones were asked for (us, two rounds / as many as fit: 85 rows of
//     2240 -> 2560 in groups of 64 16.2 / 12.4, 150 and 256 rows of 4096 x 4096 14.4 / 12.7 and 15.6 / 14.0, 240 rows of 4096 -> 11008 34.5 / 31.9, 48
//     rows of 11008 -> 4096 15.7 / 15.4; tiles of one and two blocks of rows keep two: nothing gained).  A direct
//     load blocks the wavefront that issues it until the memory path accepts it, and vector loads return in order, so in a
//     multiplying wavefront it would stand in front of the products and tie the weights' prefetch to the activations';
//   * packed weights and parameters are loaded two rounds ahead, into registers (four rounds: the same times, 40 registers
//     more, and the tall tiles spill);
//   * a lane (i, q) dequantizes the 32 codes of channel i at k = 128 s + 32 q: codes are brought under an fp16 exponent in place
//     and one v_fma_mix per code applies scale and zero point in fp32, rounded once to the operand type (float16: the mix
//     instruction's own rounding; bfloat16: v_cvt_pk_bf16_f32; float32: no rounding).  They are the A operand of
//     v_mfma_f32_16x16x32_{f16,bf16} (float32: v_mfma_f32_16x16x4_f32), the activations as they lie in memory the B operand;
//   * where the kernels for fewer rows keep the weight in float32 (scales applied to sums), a 16-bit weight is not rounded here
//     either: SPLIT, the rounding's remainder goes through the matrix cores as a second operand.  The groups of 32 lie across a
//     lane group's k range, so scales cannot be applied to sums instead;
//   * a sum that comes out NaN there (SPLIT, or a last step that is partial) is formed again term by term, by the lane that stores
//     it: an infinite activation meets the weight's remainder, which is zero or of the other sign, an infinite weight meets the zeros
//     behind K, and a weight beyond the 16-bit range becomes two infinities of opposite signs; the sum itself is infinite or finite.
//     Finite results pay one comparison;
//   * with float32 activations sums are formed over 16 k, these added up over a step and the steps over the slice (16-bit operands
//     keep one chain, their products' own roundings are larger): in one chain over the slice
//     the roundings of the long sum weigh twice as much as all others together (error against float64 with 8 bits, 4096 x 4096 at
//     19 rows: one chain 3.3e-7, so 1.3e-7; the one-row kernels 1.9e-7);
//   * the KW partial sums of a tile meet in LDS at the end.
// Measured (us, weights from HBM, this kernel / what ran before): int4, bfloat16, 11008 -> 4096 in groups of 64: 24 / 48 / 128 / 256
// rows 12.4 / 22.8, 14.8 / 39, 24 / 43, 36 / 71; 4096 x 4096 in groups of 128: 33 rows (SPLIT) 10.8 / 12.5, 64 / 256 rows 11.2 / 20, 15.8 / 34;
// 4768 -> 13544 in groups of 32 (K % 128 != 0): 3 / 33 rows (SPLIT) 19.4 / 92, 31 / 868.  float32 4096 x 4096: 64 rows 26.7 /
// 47 (bound by its MFMAs, 32 clocks for 16 x 16 x 4; most shapes of fewer rows: packed_rows_f32.hip).  2 bits: 4096 -> 11008 at 203 rows 32 /
// 67, (SPLIT) at 40 rows 20 / 31; 4096 x 4096 in groups of 32 (SPLIT): 1 / 16 / 80 rows 10.1 / 25, 10.4 / 46, 17.6 / 175.
// Rows >= M repeat row M - 1, steps of k behind the end of the slice are loaded (from the last step) and not multiplied, the
// chunks of a last partial step behind K are cleared in LDS.
#pragma once

#include <atomic>
#include <type_traits>

#include "int4_lane.h"

namespace tpq {
namespace {

typedef __attribute__((address_space(3))) void* pr_lds_ptr;
typedef uint32_t pr_word4 __attribute__((ext_vector_type(4)));
typedef _Float16 pr_half8 __attribute__((ext_vector_type(8)));
typedef __bf16 pr_bf8 __attribute__((ext_vector_type(8)));

constexpr int pr_vmcnt(int n) { return (n & 0xF) | ((n >> 4) << 14) | (0x7 << 4) | (0xF << 8); }  // s_waitcnt immediate, vmcnt only

// a workgroup's eight multiplying wavefronts: CW (1, 2 or 4) positions of two blocks of 16 channels x 8 / CW steps of k,
constexpr int kRowsNB = 2;
// and two more that only request activations
constexpr int kRowsProducers = 2, kRowsThreads = (8 + kRowsProducers) * kWave;
constexpr int kRowsAhead = 2;  // rounds of packed weights in registers

#define TPQ_GLOBAL const __attribute__((address_space(1)))
typedef uint32_t pr_word2 __attribute__((ext_vector_type(2)));

struct PackedRowsArgs {
    const void* x;         // [M][K]
    const void* w;         // packed
    const void* sz;        // int4: [K / group][N][2] of the activation type; n-bit: the same in float32
    const float* bias;     // added in fp32 before the rounding (n-bit modules), or null
    const void* after;     // of the activation type, added to the rounded product, which is rounded again (int4 modules), or null
    void* y;               // [M][N]
    float* partial;        // [slices][M][N], or null: y
    int M, N, K, tiles_per_group, steps_per_slice;
    float inv_tiles_per_group;
};

// code - zero, rounded once (one instruction instead of a conversion and a subtraction)
template <int HALF>
__device__ __forceinline__ float less_zero(half2_t codes, float zero) {
    float out;
    if constexpr (HALF == 0)
        asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel_hi:[1,0,0]" : "=v"(out) : "v"(codes), "v"(zero));
    else
        asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(out) : "v"(codes), "v"(zero));
    return out;
}

// ---- the two weight sources ------------------------------------------------------------------------------
// codes(): the lane's 32 codes as 16 pairs under fp16 exponents, pair p = codes 2 p, 2 p + 1 in k order
// offset(p, half): what the exponent adds to the code (and to its bias) in that half

// int4 device layout, [N / 8][K / 32] tiles of 8 rows x 16 bytes: word r of a row holds k = 2 r + 8 j, + 1 in nibbles j, 4 + j
struct SourceInt4 {
    static constexpr int kLoads = 1, kStepBytes = 512;  // (bytes from a step to the next)
    static constexpr bool kTypedParams = true;          // (scale, zero) in the activation type; value = (code - 8) scale + zero
    struct Words { uint4 v[1]; };
    // byte offset of the lane's codes in step 0, and how far the last step's lie behind K (a partial last step)
    static __device__ __forceinline__ uint32_t lane_offset(const PackedRowsArgs& a, int n, int q) {
        const int tiles = a.N / 8, tile = n >> 3;
        return static_cast<uint32_t>(tile < tiles ? tile : tiles - 1) * static_cast<uint32_t>(a.K / 32) * 128u + static_cast<uint32_t>(q * 128 + (n & 7) * 16);
    }
    static __device__ __forceinline__ uint32_t edge_back(int tiles_behind) { return static_cast<uint32_t>(tiles_behind) * 128u; }
    static __device__ __forceinline__ void load(TPQ_GLOBAL char* step_base, uint32_t off, Words& d) {
        const pr_word4 t = __builtin_nontemporal_load((TPQ_GLOBAL pr_word4*)(step_base + off));
        d.v[0] = make_uint4(t.x, t.y, t.z, t.w);
    }
    static constexpr float offset(int p, int) { return ((p >> 2) & 1) ? 72.0f : 1032.0f; }  // exponent + 8
    static __device__ __forceinline__ uint32_t pair(const Words& d, int p, const uint32_t (&magic)[2]) {
        const int j = p >> 2, r = p & 3;  // k = 8 j + 2 r, + 1
        const uint32_t w = r == 0 ? d.v[0].x : r == 1 ? d.v[0].y : r == 2 ? d.v[0].z : d.v[0].w;
        const uint32_t t = j & 2 ? w >> 8 : w;
        return (j & 1) ? (t & 0x00F000F0u) | magic[1] : (t & 0x000F000Fu) | magic[0];
    }
    static constexpr uint32_t kMagic0 = 0x64006400u, kMagic1 = 0x54005400u;
    // one code less its bias, for the rare sums that are formed again
    static __device__ __forceinline__ float code(const PackedRowsArgs& a, int n, int k) {
        const size_t tile = static_cast<size_t>(n >> 3) * (a.K / 32) + (k >> 5);
        const uint32_t w = static_cast<const uint32_t*>(a.w)[tile * 32 + (n & 7) * 4 + ((k >> 1) & 3)];
        return static_cast<float>(static_cast<int>((w >> (4 * ((k >> 3) & 3) + 16 * (k & 1))) & 15u) - 8);
    }
};

// rows of n-bit codes, 8 / BITS per byte (one for 5 .. 8 bits), the first in the most significant bits or (LSB) the least
template <int BITS, bool LSB>
struct SourceBits {
    static constexpr int kPerByte = 8 / BITS, kBytes = 32 / kPerByte;  // bytes of a lane's 32 codes: 4, 8, 16 or 32
    static constexpr int kLoads = kBytes == 32 ? 2 : 1, kStepBytes = 4 * kBytes;
    static constexpr bool kTypedParams = false;  // float32 (scale, zero); value = (code - zero) scale
    static constexpr uint32_t kField = (1u << BITS) - 1u;
    struct Words { uint32_t v[kBytes / 4]; };
    static __device__ __forceinline__ uint32_t lane_offset(const PackedRowsArgs& a, int n, int q) {
        return static_cast<uint32_t>(n < a.N ? n : a.N - 1) * static_cast<uint32_t>(a.K / kPerByte) + static_cast<uint32_t>(q * kBytes);
    }
    static __device__ __forceinline__ uint32_t edge_back(int tiles_behind) { return static_cast<uint32_t>(tiles_behind * kBytes); }
    static __device__ __forceinline__ void load(TPQ_GLOBAL char* step_base, uint32_t off, Words& d) {
        TPQ_GLOBAL char* const p = step_base + off;
        if constexpr (kBytes == 4) {
            d.v[0] = __builtin_nontemporal_load((TPQ_GLOBAL uint32_t*)p);
        } else if constexpr (kBytes == 8) {
            const pr_word2 t = __builtin_nontemporal_load((TPQ_GLOBAL pr_word2*)p);
            d.v[0] = t.x; d.v[1] = t.y;
        } else {
#pragma unroll
            for (int e = 0; e < kBytes / 16; ++e) {
                const pr_word4 t = __builtin_nontemporal_load((TPQ_GLOBAL pr_word4*)p + e);
                d.v[4 * e] = t.x; d.v[4 * e + 1] = t.y; d.v[4 * e + 2] = t.z; d.v[4 * e + 3] = t.w;
            }
        }
    }
    static constexpr int pos(int c) { return LSB ? (c % kPerByte) * BITS : 8 - (c % kPerByte + 1) * BITS; }  // bit position of code c in its byte
    static constexpr uint32_t exponent(int p) { return static_cast<uint32_t>(25 - p) << 10; }               // fp16 bits of 2^(10 - p)
    // 8-bit codes are signed (the reference's unpack ends in int8): byte ^ 0x80 = value + 128
    static constexpr float offset(int p, int half) { return static_cast<float>(1 << (10 - pos(2 * p + half))) + (BITS == 8 ? 128.0f : 0.0f); }
    static __device__ __forceinline__ uint32_t pair(const Words& d, int p, const uint32_t (&)[2]) {
        const int lo = 2 * p, hi = 2 * p + 1, byte_lo = lo / kPerByte, byte_hi = hi / kPerByte;
        uint32_t w = d.v[byte_lo >> 2];
        if constexpr (BITS == 8) w ^= 0x80808080u;
        const uint32_t both = __builtin_amdgcn_perm(0u, w, 0x0C000C00u | (byte_lo & 3) | ((byte_hi & 3) << 16));
        return (both & ((kField << pos(lo)) | (kField << (pos(hi) + 16)))) | (exponent(pos(lo)) | (exponent(pos(hi)) << 16));
    }
    static constexpr uint32_t kMagic0 = 0, kMagic1 = 0;
    static constexpr float kMostCode = BITS == 8 ? 128.0f : static_cast<float>((1 << BITS) - 1);
    static __device__ __forceinline__ float code(const PackedRowsArgs& a, int n, int k) {
        const uint32_t byte = static_cast<const uint8_t*>(a.w)[static_cast<size_t>(n) * (a.K / kPerByte) + k / kPerByte];
        if constexpr (BITS == 8) return static_cast<float>(static_cast<int>(byte ^ 0x80u) - 128);
        else return static_cast<float>((byte >> (LSB ? (k % kPerByte) * BITS : 8 - (k % kPerByte + 1) * BITS)) & kField);
    }
};

template <int FIRST, int LAST, class F>
__device__ __forceinline__ void pr_static_for(F&& f) {
    if constexpr (FIRST < LAST) {
        f(std::integral_constant<int, FIRST>{});
        pr_static_for<FIRST + 1, LAST>(f);
    }
}

// step(0), step(1), .. for all but the last of `left` rounds, last() for that one, as nested straight-line code
template <int R, int MOST, class F, class G>
__device__ __forceinline__ void pr_last_rounds(int left, F&& step, G&& last) {
    if constexpr (R + 1 < MOST) {
        if (R + 1 < left) {
            step(std::integral_constant<int, R>{});
            pr_last_rounds<R + 1, MOST>(left, step, last);
            return;
        }
    }
    last(std::integral_constant<int, R>{});
}

// ---- operand types -----------------------------------------------------------------------------------
template <int DT>
struct RowsArith {  // 16-bit
    static constexpr int kElem = 2, kChunks = 16;  // 16-byte chunks of a row and step
    // four words = the eight dequantized weights of a 16-byte chunk
    static __device__ __forceinline__ uint32_t pack(float lo, float hi) {
        typedef float f2_t __attribute__((ext_vector_type(2)));
        const f2_t v = {lo, hi};
        if constexpr (DT == TPQ_DTYPE_BF16) {
            typedef __bf16 bf2_t __attribute__((ext_vector_type(2)));
            return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf2_t));
        } else {
            return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, half2_t));
        }
    }
    static __device__ __forceinline__ float4_t mfma(const pr_word4& a, const pr_word4& b, float4_t c) {
        if constexpr (DT == TPQ_DTYPE_BF16) return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(pr_bf8, a), __builtin_bit_cast(pr_bf8, b), c, 0, 0, 0);
        else return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(pr_half8, a), __builtin_bit_cast(pr_half8, b), c, 0, 0, 0);
    }
};
template <>
struct RowsArith<TPQ_DTYPE_F32> {
    static constexpr int kElem = 4, kChunks = 32;
};

// (scale, zero) of one channel and group
template <int DT, bool TYPED>
struct RowsParams {
    using raw_t = typename std::conditional<TYPED && DT != TPQ_DTYPE_F32, uint32_t, uint2>::type;
    static __device__ __forceinline__ float scale(raw_t p) {
        if constexpr (TYPED && DT != TPQ_DTYPE_F32) return Elem<DT>::load(static_cast<uint16_t>(p & 0xFFFFu));
        else return __builtin_bit_cast(float, p.x);
    }
    static __device__ __forceinline__ float zero(raw_t p) {
        if constexpr (TYPED && DT != TPQ_DTYPE_F32) return Elem<DT>::load(static_cast<uint16_t>(p >> 16));
        else return __builtin_bit_cast(float, p.y);
    }
};

// four sums of the channels n .. n + 3 rounded (+ after[n ..], rounded again)
template <int DT>
__device__ __forceinline__ void store_rows_result(const float4_t& s, typename Elem<DT>::storage* y, const typename Elem<DT>::storage* after, int n) {
    typename Elem<DT>::storage o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = Elem<DT>::store(s[e]);
    if (after != nullptr) {
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = Elem<DT>::store(Elem<DT>::load(o[e]) + Elem<DT>::load(after[n + e]));
    }
    if constexpr (DT == TPQ_DTYPE_F32) *reinterpret_cast<float4_t*>(y) = float4_t{o[0], o[1], o[2], o[3]};
    else *reinterpret_cast<uint2*>(y) = make_uint2(o[0] | (static_cast<uint32_t>(o[1]) << 16), o[2] | (static_cast<uint32_t>(o[3]) << 16));
}

// One row's sum over k in [k0, k1) term by term, the weight as the kernel's dequantization defines it (SPLIT: not rounded); ends at
// the first NaN.
template <int DT, class Source, bool SPLIT>
__device__ float one_sum(const PackedRowsArgs& a, int m, int n, int k0, int k1) {
    using P = RowsParams<DT, Source::kTypedParams>;
    const auto* const x = static_cast<const typename Elem<DT>::storage*>(a.x) + static_cast<size_t>(m) * a.K;
    float sum = 0.0f;
    for (int k = k0; k < k1 && sum == sum; ++k) {
        const auto params = static_cast<const typename P::raw_t*>(a.sz)[static_cast<size_t>((k >> 5) / a.tiles_per_group) * a.N + n];
        const float code = Source::code(a, n, k), scale = P::scale(params), zero = P::zero(params);
        float w = Source::kTypedParams ? __builtin_fmaf(code, scale, zero) : (code - zero) * scale;
        if constexpr (!SPLIT) w = Elem<DT>::load(Elem<DT>::store(w));
        sum = __builtin_fmaf(Elem<DT>::load(x[k]), w, sum);
    }
    return sum;
}

// Slots of one step of activations each in a workgroup's ring: two rounds of the small ones, up to three of those from 12 KB on, as far as a
// compute unit's LDS holds them
constexpr int rows_ring_slots(int slot_bytes, int kw) {
    const int most = 160 * 1024 / slot_bytes, wanted = slot_bytes >= 12 * 1024 ? 3 * kw : 2 * kw;
    return most < wanted ? most : wanted;
}

template <int DT, class Source, int MB, int CW, bool EDGE, bool SPLIT>
__global__ __launch_bounds__(kRowsThreads) void packed_rows_kernel(const PackedRowsArgs a) {
    using A = RowsArith<DT>;
    using P = RowsParams<DT, Source::kTypedParams>;
    using storage = typename Elem<DT>::storage;
    constexpr int KW = 8 / CW, NB = kRowsNB, kRows = 16 * MB, kStepBytes = A::kChunks * 16;
    constexpr int kLoadsPerStep = kRows * kStepBytes / 1024, kMine = kLoadsPerStep / kRowsProducers;  // 1 KB loads of a step, a requesting wavefront's
    constexpr int kRowsPerLoad = 64 / A::kChunks, kSlot = kLoadsPerStep * 1024, kSlots = rows_ring_slots(kSlot, KW);
    static_assert(!SPLIT || DT != TPQ_DTYPE_F32, "float32 weights are not rounded");
    static_assert(kLoadsPerStep % kRowsProducers == 0 && kSlots >= 2 * KW, "every wavefront loads the same number of pieces");
    extern __shared__ uint4 pr_lds[];  // [kSlots][kRows][kStepBytes], later the partial sums [CW][NB][MB][KW][64 lanes]
    char* const lds = reinterpret_cast<char*>(pr_lds);

    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int cw = wave % CW, kk = wave / CW;
    const int i = lane & 15, q = lane >> 4;
    const int m0 = blockIdx.y * kRows;
    const int steps_all = (a.K + 127) / 128, s_begin = blockIdx.z * a.steps_per_slice;
    const int s_end = steps_all < s_begin + a.steps_per_slice ? steps_all : s_begin + a.steps_per_slice;
    const int rounds = (s_end - s_begin + KW - 1) / KW;
    const int edge_chunks = EDGE ? (a.K % 128) * A::kElem / 16 : A::kChunks;  // 16-byte chunks of a row in the last step of K
    auto step_of = [&](int round, int k) __attribute__((always_inline)) {     // clamped: a step behind the slice repeats its last one
        const int s = s_begin + round * KW + k;
        return s < s_end ? s : s_end - 1;
    };

    // LDS traffic only: the loads of weights stay in flight
    auto lds_barrier = []() __attribute__((always_inline)) { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    // ---- the requesting wavefronts: pieces of 1 KB, kRowsPerLoad rows of a step each; step t of the slice in slot t % kSlots, one barrier
    // per round.  One round is asked for at first (more would stand in front of the first weights: 232 rows of 6656 -> 576, two rounds of
    // the loop, 13.3 -> 13.7 us), and from the first barrier on what the ring holds, so that loads are under way while a round is waited for.
    if (wave >= 8) {
        const uint32_t row_bytes = static_cast<uint32_t>(a.K) * A::kElem;
        const char* const x_base = static_cast<const char*>(a.x) + static_cast<size_t>(m0) * row_bytes;
        const uint32_t ring_addr = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((pr_lds_ptr)pr_lds));
        const int first = (wave - 8) * kMine;
        uint32_t x_off[kMine];  // byte offset of the lane's chunk in step 0
        auto chunk_of = [&](int j) __attribute__((always_inline)) { return (lane % A::kChunks) ^ (((first + j) * kRowsPerLoad + lane / A::kChunks) & 15); };
#pragma unroll
        for (int j = 0; j < kMine; ++j) {
            const int row = (first + j) * kRowsPerLoad + lane / A::kChunks;
            x_off[j] = static_cast<uint32_t>(m0 + row < a.M ? row : a.M - 1 - m0) * row_bytes + static_cast<uint32_t>(chunk_of(j)) * 16;
        }
        const int total = rounds * KW;
        int asked = 0, fill = 0;  // steps asked for; the slot of the next one
        auto ask_up_to = [&](int limit) __attribute__((always_inline)) {
            for (limit = limit < total ? limit : total; asked < limit; ++asked) {
                const int step = step_of(0, asked);
                const char* const from = x_base + static_cast<size_t>(step) * kStepBytes;
#pragma unroll
                for (int j = 0; j < kMine; ++j) {
                    uint32_t off = x_off[j];
                    if constexpr (EDGE) {  // the last chunk of the row in place of the ones behind it
                        const int behind = chunk_of(j) - ((step == steps_all - 1 ? edge_chunks : A::kChunks) - 1);
                        off -= static_cast<uint32_t>(behind > 0 ? behind : 0) * 16;
                    }
                    const uint32_t to = ring_addr + fill * kSlot + (first + j) * 1024;
                    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(to), "v"(off), "s"(from) : "memory", "m0");
                }
                fill = fill + 1 == kSlots ? 0 : fill + 1;
            }
        };
        // all but the loads of the last `steps` steps have landed
        auto wait_but = [&](int steps) __attribute__((always_inline)) {
            bool done = false;
            pr_static_for<0, kSlots - KW + 1>([&](auto e) __attribute__((always_inline)) {
                constexpr int N = kSlots - KW - decltype(e)::value, kCount = N * kMine < 63 ? N * kMine : 63;  // (the counter ends at 63: a wait for more)
                if (!done && steps >= N) {
                    __builtin_amdgcn_s_waitcnt(pr_vmcnt(kCount));
                    done = true;
                }
            });
        };
        ask_up_to(KW);
        for (int round = 0; round < rounds; ++round) {
            wait_but(asked - (round + 1) * KW);
            if constexpr (EDGE) {  // zeros over what was fetched in place of chunks behind K
#pragma unroll
                for (int k = 0; k < KW; ++k) {
                    if (step_of(round, k) == steps_all - 1) {
                        char* const slot = lds + static_cast<uint32_t>(round * KW + k) % static_cast<uint32_t>(kSlots) * kSlot;
#pragma unroll
                        for (int j = 0; j < kMine; ++j)
                            if (chunk_of(j) >= edge_chunks) *reinterpret_cast<uint4*>(slot + (first + j) * 1024 + lane * 16) = make_uint4(0, 0, 0, 0);
                    }
                }
            }
            lds_barrier();  // round `round` is there, and everybody is done with the round before it
            ask_up_to(kSlots + round * KW);
        }
        __syncthreads();  // the products of the last round are done
        __syncthreads();  // the sums are in LDS
        return;
    }

    // ---- weights
    struct Loaded {
        typename Source::Words w[NB];
        typename P::raw_t p[NB];
    };
    uint32_t w_off[NB], p_off[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const int n = blockIdx.x * (16 * NB * CW) + (cw * NB + b) * 16 + i;
        w_off[b] = Source::lane_offset(a, n, q);
        p_off[b] = static_cast<uint32_t>(n < a.N ? n : a.N - 1) * static_cast<uint32_t>(sizeof(typename P::raw_t));
    }
    const int last_tile = a.K / 32 - 1;
    const uint32_t group_bytes = static_cast<uint32_t>(a.N) * static_cast<uint32_t>(sizeof(typename P::raw_t));
    auto load_w = [&](int round, Loaded& d) __attribute__((always_inline)) {
        const int step = step_of(round, kk);
        int tile = 4 * step + q;
        uint32_t back = 0;
        if constexpr (EDGE) {
            const int behind = tile - last_tile;
            tile = behind > 0 ? last_tile : tile;
            back = Source::edge_back(behind > 0 ? behind : 0);
        }
        // exact: tile < 2^20
        const uint32_t group = static_cast<uint32_t>((static_cast<float>(tile) + 0.5f) * a.inv_tiles_per_group);
        const uint32_t group_off = group * group_bytes;
        auto from = (TPQ_GLOBAL char*)a.w + static_cast<size_t>(step) * Source::kStepBytes;
        auto params = (TPQ_GLOBAL char*)a.sz;
        asm volatile("" : "+s"(from), "+s"(params));  // the loads stay here (see pinned_global)
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            Source::load(from, w_off[b] - back, d.w[b]);
            if constexpr (sizeof(typename P::raw_t) == 4) {
                d.p[b] = *(TPQ_GLOBAL uint32_t*)(params + (group_off + p_off[b]));
            } else {
                const pr_word2 t = *(TPQ_GLOBAL pr_word2*)(params + (group_off + p_off[b]));
                d.p[b].x = t.x; d.p[b].y = t.y;
            }
        }
    };
    uint32_t magic[2];  // in VGPRs behind opaque moves: v_and_or_b32 takes one literal only
    asm volatile("v_mov_b32 %0, %1" : "=v"(magic[0]) : "s"(Source::kMagic0));
    asm volatile("v_mov_b32 %0, %1" : "=v"(magic[1]) : "s"(Source::kMagic1));
    // float16 and n-bit rows, whose scales are float32: remainders of small weights would lie on the grid of float16's subnormals, large
    // weights beyond its range.  NORMALIZE multiplies a channel's scales by a power of two (exact) that brings the bound of its
    // first group to 64 .. 128, and the float32 sums by its inverse.  A group may then be 2^9 times as large as the first, or
    // 2^14 times smaller and still be held to 2^-18.  At most 2^16, for a first group that is nearly zero and says nothing about
    // the others: below weights of 1e-7 the grid shows (at 1e-8 3e-5 of a weight).  (int4: scale and zero point are float16, so every weight and remainder is a whole multiple of 2^-24 already.)
    constexpr bool NORMALIZE = SPLIT && DT == TPQ_DTYPE_F16 && !Source::kTypedParams;
    int power[NB] = {};
    // pair p of a block's codes, dequantized
    auto weight_pair = [&](const Loaded& d, int b, int p, float scale, float zero, float& lo, float& hi) __attribute__((always_inline)) {
        half2_t h = __builtin_bit_cast(half2_t, Source::pair(d.w[b], p, magic));
        if constexpr (DT == TPQ_DTYPE_F32 || SPLIT) {  // the offset leaves exactly, in fp16
            h = h - half2_t{static_cast<_Float16>(Source::offset(p, 0)), static_cast<_Float16>(Source::offset(p, 1))};
            if constexpr (Source::kTypedParams) {
                lo = __builtin_fmaf(static_cast<float>(h.x), scale, zero);
                hi = __builtin_fmaf(static_cast<float>(h.y), scale, zero);
            } else {  // zero points are whole numbers as a rule: one rounding
                lo = less_zero<0>(h, zero) * scale;
                hi = less_zero<1>(h, zero) * scale;
            }
        } else {  // the offset folded into the constant: an error of 2^-24 x 1032 scale at most, below the operand type's rounding
            const float z_lo = Source::kTypedParams ? zero - Source::offset(p, 0) * scale : -(zero + Source::offset(p, 0)) * scale;
            const float z_hi = Source::kTypedParams ? zero - Source::offset(p, 1) * scale : -(zero + Source::offset(p, 1)) * scale;
            lo = __builtin_fmaf(static_cast<float>(h.x), scale, z_lo);
            hi = __builtin_fmaf(static_cast<float>(h.y), scale, z_hi);
        }
    };
    // Dequantized weights that go with one 16-byte chunk of the lane's activations, of two chunks in turn: four words (eight
    // 16-bit values, four floats) per block
    constexpr int kChunkPairs = DT == TPQ_DTYPE_F32 ? 2 : 4;
    uint32_t wq[2][NB][4];
    uint32_t wr[SPLIT ? 2 : 1][NB][4];  // SPLIT: what their rounding left
    // pairs [first, last) of the NB kChunkPairs pairs of chunk u
    auto dequantize = [&](const Loaded& d, auto u_c, auto first, auto last) __attribute__((always_inline)) {
        constexpr int U = decltype(u_c)::value;
#pragma unroll
        for (int e = decltype(first)::value; e < decltype(last)::value; ++e) {
            const int b = e % NB, p = e / NB;
            float lo, hi;
            const float scale = NORMALIZE ? __builtin_amdgcn_ldexpf(P::scale(d.p[b]), power[b]) : P::scale(d.p[b]);
            weight_pair(d, b, U * kChunkPairs + p, scale, P::zero(d.p[b]), lo, hi);
            if constexpr (DT == TPQ_DTYPE_F32) {
                wq[U & 1][b][2 * p] = __builtin_bit_cast(uint32_t, lo);
                wq[U & 1][b][2 * p + 1] = __builtin_bit_cast(uint32_t, hi);
            } else {
                const uint32_t rounded = A::pack(lo, hi);
                wq[U & 1][b][p] = rounded;
                if constexpr (SPLIT)
                    wr[U & 1][b][p] = A::pack(lo - Elem<DT>::load(static_cast<uint16_t>(rounded & 0xFFFFu)), hi - Elem<DT>::load(static_cast<uint16_t>(rounded >> 16)));
            }
        }
    };
    // the values exist from here on (moved down to their use, the codes would have to live on beside the ones loaded next)
    auto settle = [&](auto u_c) __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                uint32_t& v = wq[decltype(u_c)::value & 1][b][e];
                asm volatile("" : "+v"(v));
                if constexpr (SPLIT) {
                    uint32_t& rest = wr[decltype(u_c)::value & 1][b][e];
                    asm volatile("" : "+v"(rest));
                }
            }
    };

    float4_t acc[NB][MB];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int r = 0; r < MB; ++r) acc[b][r] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};

    // A step's products in pieces: piece c = u MB + r is chunk u of the lane's activations for row block r
    constexpr int kU = A::kChunks / 4, kPieces = kU * MB, kFragments = kPieces < 3 ? kPieces : 3;
    const char* const frag_base = lds + i * kStepBytes;
    int slot = kk;  // of this wavefront's step in the current round
    pr_word4 frag[kFragments];
    auto read_piece = [&](const char* from, auto c) __attribute__((always_inline)) {
        constexpr int C = decltype(c)::value;
        if constexpr (C < kPieces)
            frag[C % kFragments] = *reinterpret_cast<const pr_word4*>(from + (C % MB) * (16 * kStepBytes) + ((kU * q + C / MB) ^ i) * 16);
    };
    // float32: a piece's own sum, added to its step's while the next piece multiplies
    float4_t piece[DT == TPQ_DTYPE_F32 ? 2 : 1][NB], step_sum[NB][DT == TPQ_DTYPE_F32 ? MB : 1];
    auto add_piece = [&](auto c) __attribute__((always_inline)) {
        if constexpr (DT == TPQ_DTYPE_F32) {
            constexpr int C = decltype(c)::value, U = C / MB, r = C % MB;
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float more = piece[C & 1][b][e];
                    if constexpr (U == 0) step_sum[b][r][e] = more;
                    else if constexpr (U + 1 < kU) step_sum[b][r][e] += more;
                    else acc[b][r][e] += step_sum[b][r][e] + more;
                }
        }
    };
    auto multiply_piece = [&](auto c) __attribute__((always_inline)) {
        constexpr int C = decltype(c)::value, U = C / MB, r = C % MB;
        if constexpr (DT == TPQ_DTYPE_F32) {
            const float4_t f = __builtin_bit_cast(float4_t, frag[C % kFragments]);
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int b = 0; b < NB; ++b)
                    piece[C & 1][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(__builtin_bit_cast(float, wq[U & 1][b][t]), f[t],
                                                                           t == 0 ? float4_t{0.0f, 0.0f, 0.0f, 0.0f} : piece[C & 1][b], 0, 0, 0);
            if constexpr (C > 0) add_piece(std::integral_constant<int, C - 1>{});
            if constexpr (C == kPieces - 1) add_piece(c);
        } else {
            if constexpr (SPLIT) {
#pragma unroll
                for (int b = 0; b < NB; ++b)
                    acc[b][r] = A::mfma(pr_word4{wr[U & 1][b][0], wr[U & 1][b][1], wr[U & 1][b][2], wr[U & 1][b][3]}, frag[C % kFragments], acc[b][r]);
            }
#pragma unroll
            for (int b = 0; b < NB; ++b)
                acc[b][r] = A::mfma(pr_word4{wq[U & 1][b][0], wq[U & 1][b][1], wq[U & 1][b][2], wq[U & 1][b][3]}, frag[C % kFragments], acc[b][r]);
        }
    };
    // The products of one step (weights d, in ring slot SLOT) and, dealt over their pieces, the dequantization of the following
    // chunk's weights: the matrix cores and the vector ALU are separate pipes, and both multiplying wavefronts of a SIMD are in
    // the same phase.  The order of the pieces is fixed: left to itself the compiler dequantizes first and multiplies
    // afterwards.  The last chunk prepares the first one of the next step (next; NEXT), and the ring slot is asked for again
    // as soon as its last codes are used.
    constexpr int kShare = NB * kChunkPairs;
    auto products = [&](Loaded& d, const Loaded& next, int load_round, auto has_next, auto load_c) __attribute__((always_inline)) {
        constexpr bool NEXT = decltype(has_next)::value, LOAD = decltype(load_c)::value;
        const char* const from = frag_base + slot * kSlot;
        slot = slot + KW >= kSlots ? slot + KW - kSlots : slot + KW;
        pr_static_for<0, kFragments - 1>([&](auto c) __attribute__((always_inline)) { read_piece(from, c); });
        pr_static_for<0, kPieces>([&](auto c) __attribute__((always_inline)) {
            constexpr int C = decltype(c)::value, U = C / MB, r = C % MB;
            constexpr std::integral_constant<int, r * kShare / MB> first{};
            constexpr std::integral_constant<int, (r + 1) * kShare / MB> last{};
            constexpr std::integral_constant<int, (U + 1) % kU> following{};
            read_piece(from, std::integral_constant<int, C + kFragments - 1>{});
            multiply_piece(c);
            if constexpr (U + 1 < kU) dequantize(d, following, first, last);
            else if constexpr (NEXT) dequantize(next, following, first, last);
            if constexpr (r == MB - 1 && (U + 1 < kU || NEXT)) settle(following);
            if constexpr (LOAD && r == MB - 1 && U + 2 == kU) load_w(load_round, d);
            __builtin_amdgcn_sched_barrier(0);
        });
    };

    Loaded ring[kRowsAhead];
    auto phase = [&](int round, auto slot_c, auto load_c) __attribute__((always_inline)) {  // a round that is not the last; slot_c = round % kRowsAhead
        constexpr int SLOT = decltype(slot_c)::value;
        products(ring[SLOT], ring[(SLOT + 1) % kRowsAhead], round + kRowsAhead, std::true_type{}, load_c);
        lds_barrier();
    };
    pr_static_for<0, kRowsAhead>([&](auto r) __attribute__((always_inline)) { load_w(decltype(r)::value, ring[decltype(r)::value]); });
    if constexpr (NORMALIZE) {
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            float most = (Source::kMostCode + fabsf(P::zero(ring[0].p[b]))) * fabsf(P::scale(ring[0].p[b]));
            most = fmaxf(most, __shfl_xor(most, 16));  // the four lanes of a channel: up to four groups of 32
            most = fmaxf(most, __shfl_xor(most, 32));
            const int up = 7 - __builtin_amdgcn_frexp_expf(most);
            power[b] = up < 16 ? up : 16;
        }
    }
    dequantize(ring[0], std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{}, std::integral_constant<int, kShare>{});
    settle(std::integral_constant<int, 0>{});
    lds_barrier();
    int round = 0;
    for (; round + kRowsAhead < rounds; round += kRowsAhead)
        pr_static_for<0, kRowsAhead>([&](auto r) __attribute__((always_inline)) { phase(round + decltype(r)::value, r, std::true_type{}); });
    // 1 .. kRowsAhead rounds left, their weights all asked for; in the last one a wavefront whose step lies behind the slice multiplies nothing
    pr_last_rounds<0, kRowsAhead>(rounds - round, [&](auto r) __attribute__((always_inline)) { phase(round + decltype(r)::value, r, std::false_type{}); },
                                  [&](auto r) __attribute__((always_inline)) {
                                      constexpr int SLOT = decltype(r)::value;
                                      if (s_begin + (round + SLOT) * KW + kk < s_end) products(ring[SLOT], ring[SLOT], 0, std::false_type{}, std::false_type{});
                                  });
    __syncthreads();

    // ---- the KW sums of a tile meet in LDS; wavefront t finishes tiles t, t + 8, ...
    float4_t* const sums = reinterpret_cast<float4_t*>(lds);
    if constexpr (NORMALIZE) {
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int down = -__shfl(power[b], 4 * q + e);  // element e: channel 4 q + e
#pragma unroll
                for (int r = 0; r < MB; ++r) acc[b][r][e] = __builtin_amdgcn_ldexpf(acc[b][r][e], down);
            }
    }
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int r = 0; r < MB; ++r) sums[(((cw * NB + b) * MB + r) * KW + kk) * kWave + lane] = acc[b][r];
    __syncthreads();
    for (int t = wave; t < CW * NB * MB; t += 8) {
        float4_t s = sums[(t * KW) * kWave + lane];
        auto add = [](const float4_t& a, const float4_t& b) { return float4_t{a[0] + b[0], a[1] + b[1], a[2] + b[2], a[3] + b[3]}; };
        if constexpr (KW == 8) {  // by halves: eight in a row are 8 % more error in float32 than the four of two slices had
            float4_t part[KW];
#pragma unroll
            for (int k = 0; k < KW; ++k) part[k] = sums[(t * KW + k) * kWave + lane];
            s = add(add(add(part[0], part[1]), add(part[2], part[3])), add(add(part[4], part[5]), add(part[6], part[7])));
        } else {
#pragma unroll
            for (int k = 1; k < KW; ++k) s = add(s, sums[(t * KW + k) * kWave + lane]);
        }
        const int block = t / MB, r = t % MB;
        const int m = m0 + 16 * r + i, n = blockIdx.x * (16 * NB * CW) + block * 16 + 4 * q;
        if (m >= a.M || n >= a.N) continue;  // N % 4 == 0: all four channels exist
        if constexpr (SPLIT || EDGE) {
            const int k0 = s_begin * 128, k1 = s_end * 128 < a.K ? s_end * 128 : a.K;
            const float all = (s[0] + s[1]) + (s[2] + s[3]);
            if (all != all) {  // one copy of the loop: four of them cost every call 0.2 us
#pragma unroll 1
                for (int e = 0; e < 4; ++e) {
                    float v = e == 0 ? s[0] : e == 1 ? s[1] : e == 2 ? s[2] : s[3];
                    if (v != v) v = one_sum<DT, Source, SPLIT>(a, m, n + e, k0, k1);
                    s = float4_t{e == 0 ? v : s[0], e == 1 ? v : s[1], e == 2 ? v : s[2], e == 3 ? v : s[3]};
                }
            }
        }
        const size_t at = static_cast<size_t>(m) * a.N + n;
        if (a.partial != nullptr) {
            *reinterpret_cast<float4_t*>(a.partial + static_cast<size_t>(blockIdx.z) * a.M * a.N + at) = s;
            continue;
        }
        if (a.bias != nullptr) {
#pragma unroll
            for (int e = 0; e < 4; ++e) s[e] += a.bias[n + e];
        }
        store_rows_result<DT>(s, static_cast<storage*>(a.y) + at, static_cast<const storage*>(a.after), n);
    }
}

// y = round(sum over the slices, in a fixed order (+ bias)); a thread takes four consecutive elements (N % 4 == 0)
template <int DT>
__global__ __launch_bounds__(256) void packed_rows_finish_kernel(const float* __restrict__ partial, int slices, int64_t quads, const float* __restrict__ bias,
                                                                 const typename Elem<DT>::storage* __restrict__ after, int quads_per_row,
                                                                 typename Elem<DT>::storage* __restrict__ y) {
    const int64_t e = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (e >= quads) return;
    // four slices requested together; a batch past the last slice asks for the last one again and leaves it out of the sum
    float4_t sum = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int z0 = 0; z0 < slices; z0 += 4) {
        float4_t more[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) more[j] = reinterpret_cast<const float4_t*>(partial)[static_cast<int64_t>(z0 + j < slices ? z0 + j : slices - 1) * quads + e];
        if constexpr (DT == TPQ_DTYPE_F32) {  // four by halves: in one chain, eleven slices' roundings show (40 rows of 11008 -> 1024 1.23e-7 of the result for 1.19e-7)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const float m1 = z0 + 1 < slices ? more[1][v] : 0.0f, m2 = z0 + 2 < slices ? more[2][v] : 0.0f, m3 = z0 + 3 < slices ? more[3][v] : 0.0f;
                sum[v] += (more[0][v] + m1) + (m2 + m3);
            }
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (z0 + j < slices) sum = float4_t{sum[0] + more[j][0], sum[1] + more[j][1], sum[2] + more[j][2], sum[3] + more[j][3]};
        }
    }
    const int n = bias != nullptr || after != nullptr ? static_cast<int>(static_cast<uint32_t>(e) % static_cast<uint32_t>(quads_per_row)) * 4 : 0;
    if (bias != nullptr) {
#pragma unroll
        for (int j = 0; j < 4; ++j) sum[j] += bias[n + j];
    }
    store_rows_result<DT>(sum, y + e * 4, after, n);
}

// ---- launch ------------------------------------------------------------------------------------------
struct PackedRowsPlan {
    int mb;        // blocks of 16 rows per workgroup: 1 .. 4, with 128 channels 3 .. 8 (float32: 1, 2)
    int cw;        // channel positions: 2 (64 channels per workgroup), 4 (128; 16-bit, three blocks of rows and more, K % 128 == 0) or 1 (32; up to
                   // 32 rows, float32 16)
    int slices, steps_per_slice;  // (steps of 128 k)
    int quads;     // float32, kernels without LDS for the activations: a quarter of the rows per workgroup (of 32 cw channels; cw 0: a lane per channel,
                   // steps_per_slice in tiles of 32 k); 0: the kernel above
    bool split;    // the weights' remainders multiplied too (64 channels per workgroup)
};

// (a 64-bit division takes several times as long as a 32-bit one)
inline int64_t ceil_div(int64_t a, int64_t b) {
    const int64_t up = a + b - 1;
    return up <= 0x7FFFFFFF ? static_cast<uint32_t>(up) / static_cast<uint32_t>(b) : up / b;
}

// (16-bit) weights rounded once: int4, n-bit, 8-bit; not rounded: int4, n-bit
enum RowsWeights { kRowsRounded, kRowsRoundedBits, kRowsRoundedBytes, kRowsUnrounded, kRowsUnroundedBits };

constexpr int64_t kRowsAnyRoom = int64_t{1} << 60;  // floats of a workspace that holds the slices of any plan

// ---- float32 ---------------------------------------------------------------------------------------------
// Three kernels, one of which a call runs, by estimates (us).
// Fitted to the device times of all plans of 85 shapes (k 1024 .. 8192, channels 512 .. 11008) at 25 row counts up to 64, in groups of 32, 64 and
// 128; the plan that they take is 2 % (8 bits 4 %) above the best on average, with one cost for all widths it was 4 (9, up to 124).  What a round of the loop costs depends on the width of the codes: int4 (one instruction from pair to floats), 1, 2 and 4 bits (an instruction more a
// code), 8 bits (twice the bytes, and with a lane per channel a line per lane and tile).  A workgroup that a compute unit gets after its first (a turn) costs its rounds
// again, and what does not hide behind the one before it.  (10.4 and 98.5: int4 takes no staged tile of 16 rows, and 1 to 4 bits none in turns; the others were never slower.)
struct RowsF32Cost {
    double quads, quads_turn, quads_round[2], quads_slices, quads_bytes;                // blocks of four rows: one, two of them
    double narrow, narrow_turn, narrow_round;                                        // activations staged, 32 channels per workgroup
    double staged, staged_round[2], staged_turn[2], staged_slices, staged_bytes;        // 64 channels; one block of 16 rows, two
    double lanes, lanes_round, lanes_block, lanes_four, lanes_turn, lanes_short, lanes_slices, lanes_bytes;  // a lane per channel: a round, a block of 16, one of four
};
constexpr RowsF32Cost kRowsF32Costs[3] = {
    {2.0, 1.0, {1.6, 2.4}, 2.0, 2.0, 3.9, 0.0, 2.25, 3.5, {10.4, 4.3}, {0.2, 0.9}, 1.3, 1.6, 3.3, 0.2, 0.9, 0.5, 0.0, 0.3, 1.8, 1.45},        // int4
    {1.0, 1.2, {1.9, 2.4}, 1.0, 3.0, 3.8, 0.45, 2.85, 2.7, {2.45, 5.05}, {98.5, 4.7}, 3.0, 0.55, 4.25, 0.3, 1.0, 0.5, 1.7, 0.3, 1.85, 1.4},  // 1, 2, 4 bits
    {1.8, 2.5, {1.4, 2.0}, 1.3, 0.4, 4.6, 0.4, 2.65, 3.4, {2.45, 4.8}, {3.55, 5.15}, 2.65, 0.95, 4.15, 1.3, 0.8, 0.0, 2.4, 0.0, 2.55, 0.95},  // 8 bits
};

// The best plan so far.  A call is replayed in a graph as well as made eagerly, where the host needs 7.2 us for one launch and 10.8 for two and an
// allocation: the sum of both times decides (us, eager and in a graph: nine rows, int4 2048 -> 2048 one slice 9.5, 9.5, eight slices 10.8, 7.2; 1280 -> 768 8.0, 8.0 and
// 10.8, 6.5).
struct RowsF32Choice {
    PackedRowsPlan plan{};
    double best = 1e30;
    void offer(double us, int quads, int mb, int cw, int64_t slices, int64_t steps_per_slice) {
        const double host = slices > 1 ? 10.8 : 7.2, both = us + (us > host ? us : host);
        if (both >= best) return;
        best = both;
        plan = PackedRowsPlan{mb, cw, static_cast<int>(slices), static_cast<int>(steps_per_slice), quads, false};
    }
};

// every number of slices that `units` can be cut into: (slices, units of one, us of their sums written and read at 4 TB/s)
template <class F>
inline void rows_slices(int64_t units, int64_t M, int64_t N, int64_t room_floats, F&& each) {
    for (int64_t z = 1; z <= 16 && z <= units; ++z) {
        if (z > 1 && z * M * N > room_floats) break;
        const int64_t per = ceil_div(units, z);
        if (ceil_div(units, per) == z) each(z, per, z > 1 ? static_cast<double>(z * M * N) * 8.0 / 4e6 : 0.0);
    }
}

// Up to eight rows: blocks of four.  Against the blocks of 16 (us, those / these, eager): four rows, 2 bits 4864 -> 9728 34.8 / 20.8; int4
// 1408 -> 1152 7.7 / 7.6 (in a graph 7.8 / 5.2), 4096 x 4096 11.8 / 9.3; two rows of 4096 -> 11008 28.2 / 15; one row, 2 bits, 5248 -> 3104 15.9 / 11.4; eight rows,
// 4 bits, 4096 -> 11008 30.5 / 26.4, 2048 x 2048 10.9 / 9.5, int4 4096 x 4096 12.1 / 11.3; six rows, 8 bits, 4864 -> 10880 37.9 / 33.5.  From three
// blocks on the two kinds cost the same (12 rows of 11008 -> 4096 24.4 / 24.4, 16 rows of 4096 x 4096 12.3 / 14.1): a product of sixteen 4 x 4
// blocks takes half the clocks of one of 16 x 16.
constexpr int64_t kQuadRows = 8;

// From nine rows on: activations staged in LDS, or a lane per channel: 16 to 64 rows a workgroup, and where one to four rows are left over by blocks of 16, those as a
// block of four.  Slices so short that a wavefront's four tiles in flight are not filled, on workgroups that take turns, are the worst of both kinds (10 rows 3968 -> 4864
// with 1 bit in 16 slices 25, in three 17; 16 rows 5632 -> 8480 with 8 bits in eleven 65, three 40): the estimates of turns keep calls away from them, and a round is the least.
// Staged / a lane per channel, us in a graph: int4 19 rows 4096 x 4096 17.8 / 13.6, 35 rows 26.2 / 19.3, 80 rows 42.9 / 35.4, 17 rows 11008 -> 4096 35.2 / 25.8; 36 rows
// with 8 bits 29.8 / 24.7; but 64 rows 2048 -> 8192 23.9 / 27.6, 50 rows 2048 x 2048 with 1 bit 12.4 / 13.6, 14 rows 8064 -> 1536 with 8 bits 15.6 / 17.5, 20 rows
// 2560 -> 8192 with 8 bits 25 / 31.
inline PackedRowsPlan packed_rows_f32_plan(int64_t M, int64_t N, int64_t K, int64_t room_floats, int bits) {
    const RowsF32Cost& cost = kRowsF32Costs[bits == 0 ? 0 : bits == 8 ? 2 : 1];
    RowsF32Choice choice;
    auto turns_of = [](int64_t workgroups) { return static_cast<double>((workgroups + 255) >> 8); };  // 256 compute units
    const int64_t steps = (K + 127) / 128, tiles = K / 32, blocks = (M + 15) / 16, columns = (N + 63) / 64;
    if (M <= kQuadRows) {
        const int quads = static_cast<int>((M + 3) / 4);
        rows_slices(steps, M, N, room_floats, [&](int64_t z, int64_t per, double sums_us) {
            for (int shift = 0; shift < 2; ++shift) {
                const double turns = turns_of(((N + (32 << shift) - 1) >> (5 + shift)) * z), rounds = static_cast<double>((per + (8 >> shift) - 1) >> (3 - shift));
                choice.offer(cost.quads + turns * (cost.quads_turn + cost.quads_round[quads - 1] * rounds) + (z > 1 ? cost.quads_slices + cost.quads_bytes * sums_us : 0.0), quads, 0, 1 << shift, z, per);
            }
        });
        return choice.plan;
    }
    if (blocks == 1) {  // no slices is what the narrow tiles are for
        const double turns = turns_of((N + 31) / 32);
        choice.offer(cost.narrow + cost.narrow_turn * (turns - 1.0) + cost.narrow_round * turns * static_cast<double>((steps + 7) >> 3), 0, 1, 1, 1, steps);
    }
    const int64_t staged_tiles = ceil_div(blocks, 2);
    const int mb16 = static_cast<int>(ceil_div(blocks, staged_tiles));
    rows_slices(steps, M, N, room_floats, [&](int64_t z, int64_t per, double sums_us) {
        if (z > 1 && per < 4) return;  // less than a round of the loop
        const double turns = turns_of(columns * staged_tiles * z), rounds = static_cast<double>((per + 3) >> 2);
        choice.offer(cost.staged + turns * rounds * cost.staged_round[mb16 - 1] + (turns - 1.0) * cost.staged_turn[mb16 - 1] + (z > 1 ? cost.staged_slices + cost.staged_bytes * sums_us : 0.0), 0, mb16, 2, z, per);
    });
    const int64_t lanes_tiles = ceil_div(blocks, 4);
    const bool four = lanes_tiles == 1 && M > 16 && M % 16 >= 1 && M % 16 <= 4;
    const int sixteens = static_cast<int>(four ? blocks - 1 : ceil_div(blocks, lanes_tiles));
    const double round_us = cost.lanes_round + cost.lanes_block * sixteens + (four ? cost.lanes_four : 0.0);
    rows_slices(tiles, M, N, room_floats, [&](int64_t z, int64_t per, double sums_us) {
        const double turns = turns_of(columns * lanes_tiles * z), rounds = static_cast<double>((per + 7) >> 3);
        if (z > 1 && turns > 1.0 && per <= 8) return;
        choice.offer(cost.lanes + (sixteens > 3 ? 0.3 : 0.0) + turns * rounds * round_us + (turns - 1.0) * (cost.lanes_turn + cost.lanes_short * (rounds < 4.0 ? 4.0 - rounds : 0.0)) +
                         (z > 1 ? cost.lanes_slices + cost.lanes_bytes * sums_us : 0.0),
                     4 * sixteens + (four ? 1 : 0), 0, 0, z, per);
    });
    return choice.plan;
}

// ---- float16, bfloat16 ----------------------------------------------------------------------------------
// Tile height, channels per workgroup and slices of K by an estimate (us) fitted to a sweep of 1 .. 8 slices and both widths
// over six shapes and 16 .. 256 rows (128 channels and 5 .. 8 blocks of rows, on the same line: 1.36 and 1.49 us a round at 7 and 8; unrounded
// weights 1.29, 1.43, 1.66 and 1.86 us at 1 .. 4 blocks, n-bit rows 1.4 times that): 4 for the launch, the first loads and the epilogue, per
// round what the comment on the kernel says, per round of workgroups over the compute units, and for the second kernel 2.5 + the bytes of
// the slices' sums (written and read) at 4 TB/s.  Rounded n-bit weights by all plans of 50 shapes at 16 row counts: rounds of 8 bits are twice as long
// (us, with the costs of int4 / with their own: 8 bits 132 rows 2560 -> 1152 16.3 / 11.8, 129 rows 1920 -> 896 12.6 / 10.5; 2 bits 154 rows 5888 -> 6272
// 31 / 26), and the plans taken with 8 bits are 1.6 % above the best on average, 4.1 before.  Within 5 % of the sweep's best nearly everywhere (11008 -> 4096 at 128 rows 24.8, best 22.7).
// Few rows: 32 channels per workgroup, eight steps of k a round.  Half the rounds on twice the compute units, so a few thousand k
// need no slices, and where the card would be as fast with them the host saves a launch and an allocation (us, slices / this, eager and then
// in a graph: int4 in groups of 64, 28 rows 4096 x 4096 11.2 / 7.6, 8.4 / 7.6; 20 rows 2048 x 2048 10.9 / 7.0, 6.7 / 5.2; 32 rows 3072 -> 8192
// 8.7 / 7.4, 9.0 / 7.7; 2 bits in groups of 64, three rows 2944 -> 5832 15.4 / 9.9, 15.8 / 10.2).
// Unrounded int4 weights, whose few rows of an odd k come here: 3 for the second kernel (us, one slice / sliced, eager and then in a graph: two rows
// 3776 -> 616 9.0 / 11.6, 8.8 / 6.6; 31 rows 4800 -> 3584 14.1 / 11.8, 14.2 / 11.3; 46 rows 1824 -> 1688 11.2 / 11.4, 11.2 / 9.6; and where half a
// microsecond of the device would cost an eager call four: two rows 2272 -> 512 7.5 / 11.7, 7.2 / 6.5; 79 rows 1280 -> 1024 8.6 / 11.5, 8.5 / 8.2).
// A call plans twice (workspace, launch), so what the heights have in common, the
// divisions above all, is worked out once: 203 rows of 4096 -> 11008 0.12 us of host time instead of 0.83.
struct RowsCost {
    double round, block, wide_round, wide_block;  // a round of the loop and a block of 16 rows in it: up to 64 channels, 128
    double second, bytes;                         // slices: the second kernel; factor of what their sums, written and read, take at 4 TB/s
    int tall;                                     // from this many blocks on a workgroup costs 2 us more
};
constexpr RowsCost kRowsCosts[5] = {
    {0.5, 0.18, 0.45, 0.13, 2.5, 1.0, 9}, {0.55, 0.19, 0.55, 0.14, 2.3, 1.0, 7}, {1.3, 0.18, 1.08, 0.2, 1.6, 1.4, 6},
    {1.08, 0.19, 0.0, 0.0, 3.0, 1.0, 9}, {1.51, 0.27, 0.0, 0.0, 2.5, 1.0, 9},
};
inline PackedRowsPlan packed_rows_plan(int dtype, int64_t M, int64_t N, int64_t K, int64_t room_floats, RowsWeights weights = kRowsRounded, int bits = 0) {
    if (dtype == TPQ_DTYPE_F32) return packed_rows_f32_plan(M, N, K, room_floats, bits);
    PackedRowsPlan p;
    p.quads = 0;
    p.split = weights >= kRowsUnrounded;
    const RowsCost& cost = kRowsCosts[weights];
    const int64_t blocks = (M + 15) / 16, steps = (K + 127) / 128;
    int64_t best = 1;
    double best_us = 1e30;
    p.cw = 2;
    // the slices that K can be cut into, and the steps of each
    int cuts = 0;
    int64_t slices_of[16], steps_of[16];
    for (int64_t z = 1; z <= 16 && z <= steps; ++z) {
        if (z > 1 && z * M * N > room_floats) break;
        const int64_t per = ceil_div(steps, z);
        if (ceil_div(steps, per) != z) continue;
        slices_of[cuts] = z;
        steps_of[cuts++] = per;
    }
    for (int cw = blocks <= 2 ? 1 : 2; cw <= (K % 128 == 0 && !p.split ? 4 : 2); cw *= 2) {
        // 32 and 64 channels: tiles of equal height, as few as the tallest allows; 128 channels: any height that tiles of equal height can have
        const int kw_shift = cw == 1 ? 3 : cw == 2 ? 2 : 1, most = cw <= 2 ? 4 : 8;
        const int64_t fewest = ceil_div(blocks, most);
        const int tallest = static_cast<int>(ceil_div(blocks, fewest));
        for (int mb = tallest; mb >= (cw <= 2 ? tallest : 3); --mb) {
            const int64_t row_tiles = ceil_div(blocks, mb);
            if (ceil_div(blocks, row_tiles) != mb) continue;
            const int64_t tiles = ((N + 32 * cw - 1) / (32 * cw)) * row_tiles;
            const double round_us = (cw <= 2 ? cost.round + cost.block * mb : cost.wide_round + cost.wide_block * mb) + (cw == 1 ? 0.2 * mb : 0.0);
            const double fixed_us = cw == 1 ? 3.4 : mb >= cost.tall ? 6.0 : 4.0;
            for (int c = 0; c < cuts; ++c) {
                if (cw == 1 && c > 0) break;  // no slices is what they are for
                const int64_t z = slices_of[c], rounds = (steps_of[c] + (1 << kw_shift) - 1) >> kw_shift;
                const double waves = static_cast<double>((tiles * z + 255) >> 8);  // 256 compute units
                double us = waves * (fixed_us + round_us * static_cast<double>(rounds));
                if (z > 1) us += cost.second + cost.bytes * (static_cast<double>(z * M * N) * 8.0 / 4e6);
                if (us < best_us) { best_us = us; best = z; p.cw = cw; p.mb = mb; }
            }
        }
    }
    if (const char* e = tuning_env("TPQ_ROWS_SLICES")) best = std::atoi(e);
    if (const char* e = tuning_env("TPQ_ROWS_CW")) p.cw = std::atoi(e);
    p.steps_per_slice = static_cast<int>((steps + best - 1) / best);
    p.slices = static_cast<int>((steps + p.steps_per_slice - 1) / p.steps_per_slice);
    return p;
}

template <int DT, class Source, int MB, int CW, bool EDGE, bool SPLIT>
int launch_packed_rows_shape(const PackedRowsArgs& a, int slices, hipStream_t s) {
    constexpr int KW = 8 / CW, NB = kRowsNB;
    constexpr int kSlot = 16 * MB * RowsArith<DT>::kChunks * 16;
    constexpr size_t stage = static_cast<size_t>(rows_ring_slots(kSlot, KW)) * kSlot, sums = static_cast<size_t>(8) * NB * MB * 1024;
    constexpr size_t smem = stage > sums ? stage : sums;
    static_assert(smem <= 160 * 1024, "LDS of one compute unit");
    auto kernel = packed_rows_kernel<DT, Source, MB, CW, EDGE, SPLIT>;
    static std::atomic<uint64_t> configured{0};
    if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(kernel), smem, configured, "packed rows")) return rc;
    const dim3 grid(static_cast<unsigned>((a.N + 16 * NB * CW - 1) / (16 * NB * CW)), static_cast<unsigned>((a.M + 16 * MB - 1) / (16 * MB)), static_cast<unsigned>(slices));
    kernel<<<grid, kRowsThreads, smem, s>>>(a);
    return check_launch("packed rows");
}

template <int DT, class Source, int MB, int CW>
int launch_packed_rows_as(const PackedRowsArgs& a, const PackedRowsPlan& p, hipStream_t s) {
    if constexpr (CW <= 2) {
        if constexpr (DT != TPQ_DTYPE_F32) {
            if (p.split) return a.K % 128 != 0 ? launch_packed_rows_shape<DT, Source, MB, CW, true, true>(a, p.slices, s)
                                               : launch_packed_rows_shape<DT, Source, MB, CW, false, true>(a, p.slices, s);
        }
        if (a.K % 128 != 0) return launch_packed_rows_shape<DT, Source, MB, CW, true, false>(a, p.slices, s);
    }
    return launch_packed_rows_shape<DT, Source, MB, CW, false, false>(a, p.slices, s);
}

template <int DT, class Source>
int launch_packed_rows(PackedRowsArgs a, const PackedRowsPlan& p, hipStream_t s) {
    a.steps_per_slice = p.steps_per_slice;
    a.inv_tiles_per_group = 1.0f / static_cast<float>(a.tiles_per_group);
    if (p.slices == 1) a.partial = nullptr;
    int rc;
    const bool wide = p.cw == 4;
    if (p.mb == 1) rc = p.cw == 1 ? launch_packed_rows_as<DT, Source, 1, 1>(a, p, s) : launch_packed_rows_as<DT, Source, 1, 2>(a, p, s);
    else if (p.mb == 2) {
        if constexpr (DT == TPQ_DTYPE_F32) rc = launch_packed_rows_as<DT, Source, 2, 2>(a, p, s);
        else rc = p.cw == 1 ? launch_packed_rows_as<DT, Source, 2, 1>(a, p, s) : launch_packed_rows_as<DT, Source, 2, 2>(a, p, s);
    } else {
        if constexpr (DT == TPQ_DTYPE_F32) rc = fail(TPQ_ERR_RUNTIME, "packed rows: no such tile");
        else if (p.mb == 8) rc = launch_packed_rows_shape<DT, Source, 8, 4, false, false>(a, p.slices, s);
        else if (p.mb == 7) rc = launch_packed_rows_shape<DT, Source, 7, 4, false, false>(a, p.slices, s);
        else if (p.mb == 6) rc = launch_packed_rows_shape<DT, Source, 6, 4, false, false>(a, p.slices, s);
        else if (p.mb == 5) rc = launch_packed_rows_shape<DT, Source, 5, 4, false, false>(a, p.slices, s);
        else if (p.mb == 3) rc = wide ? launch_packed_rows_as<DT, Source, 3, 4>(a, p, s) : launch_packed_rows_as<DT, Source, 3, 2>(a, p, s);
        else rc = wide ? launch_packed_rows_as<DT, Source, 4, 4>(a, p, s) : launch_packed_rows_as<DT, Source, 4, 2>(a, p, s);
    }
    if (rc != TPQ_OK || a.partial == nullptr) return rc;
    const int64_t quads = static_cast<int64_t>(a.M) * a.N / 4;
    packed_rows_finish_kernel<DT><<<static_cast<unsigned>((quads + 255) / 256), 256, 0, s>>>(
        a.partial, p.slices, quads, a.bias, static_cast<const typename Elem<DT>::storage*>(a.after), a.N / 4, static_cast<typename Elem<DT>::storage*>(a.y));
    return check_launch("packed rows (sum of the slices)");
}

}  // namespace
}  // namespace tpq

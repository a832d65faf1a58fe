// The two gradients of a linear layer in float32, one launch (and one that adds slices, where there are any):
//   grad_x[M][K] = g[M][N] w[N][K]          grad_w[N][K] = g[M][N]^T x[M][K]
// the straight-through backward of the quantized training linears (reference tensorplay/ao/quantization/int8_dyn_act_int4_weight.py:
// 86-95, two plain float32 products).
//
// What bounds it: the matrix cores.  v_mfma_f32_16x16x4_f32 takes 32 clocks for 2048 flops, a sixteenth of what bfloat16 does, so every
// float32 value is taken apart into three bfloat16 parts on its way into LDS (8 + 8 + 8 bits: exact from 2^-110 on, x = h + m + l) and a
// product is the six part products down to 2^-18 of it (hh, hm, mh, mm, hl, lh; what is left out is below 2^-23 of it): six bfloat16
// instructions for the work of sixteen.  No scaling: the parts keep float32's exponent.  Two float16 parts would need three products
// instead of six, but a scale for each row and column, whose maxima are a pass of their own, and lose what lies 2^17 below a row's
// largest value.
//   * tile 128 x 128, 32 k a stage; 4 wavefronts of 64 x 64, v_mfma_f32_32x32x16_bf16: 12 fragments of 16 bytes from LDS for 24
//     instructions (384 of 768 clocks per 16 k); up to three workgroups a compute unit, so that one takes values apart (6.5 vector
//     instructions each, 832 clocks a stage) while another multiplies (1536 clocks a stage);
//   * the next stage's float32 values travel to registers while a stage is multiplied: half of the wavefronts fetch one operand,
//     half the other.  An operand whose k is its slow index (both of grad_w, the weight of grad_x) is read as quads of rows x 8 k
//     and transposed by the choice of registers;
//   * LDS: [part][chunk of 8 k][slot] of 16 bytes, a slot per row: fragment reads are 512 consecutive bytes, and so are the
//     writes, row 4 i + e of a transposed operand having the slot 32 e + i.  A wavefront's two column fragments then lie at
//     columns 4 i + 0, 1 (or 2, 3): a lane stores two neighbours;
//   * the k range is cut into slices where tiles are few, so that workgroups of both products are about equally long, up to all places for
//     one tile (262144 rows, 64 -> 64: 328 slices, 128 us, at most eight slices 1915, the library products 554; 16 rows, 64 -> 65536
//     32 / 454 / 97; 65536 rows, 128 -> 128 44 / 487 / 241; 32 rows, 512 -> 4096 15 / 36 / 37); their float32 sums, about a tile for each
//     place, meet in a second kernel, in slice order;
//   * where that is not float32's result a tile's slice is formed again with float32 instructions: a value below 2^-110 whose lowest
//     bits the parts lose (its l is a subnormal bfloat16; seen in the bits that l cuts off, half an instruction a value), a sum that is not
//     finite (an infinite value has h = inf and m = NaN, one next to 2^64 can have h x h = inf), and sums of up to three terms, whose
//     error is that of a term (against float64, one / two / three terms: six products 3.7e-8 / 3.7e-8 / 3.6e-8, float32 2.5e-8 / 3.1e-8 /
//     3.5e-8; from four on the six products have the smaller one).  512 rows, 2048 -> 4096 with such a value in every stage 166 us, with
//     a row of infinities, which only the end shows, 240 (the library products 131); the test for them costs the others 3 of 98.
// Measured (us, both gradients with the adding launch / float32 library products): 512 rows, 2048 -> 4096 101 / 131 (the matrix cores are
// busy for 55 % of it by the counters; the write-back of 32 MB at the end of the launch takes 7, the rest is stages in which the workgroups
// of a unit wait for each other's phases), 295 rows, 808 -> 3840 38 / 48, 128 rows, 2048 -> 2048 28 / 37, 72 rows, 1280 -> 712 15 / 37, 1024
// rows, 4096 -> 4096 360 / 468, 8 rows of the same 38 / 38.  Error against float64 at the first: 3.4e-7 (grad_x 3.5e-7), the products 4.0e-7
// (1.15e-6).  float32 values kept in LDS and taken apart by the wavefronts that multiply them (no barrier between the two, each value
// twice): 113 - 130.
// Rows behind the operand's end repeat its last ones and are not stored; k behind the end is cleared in both operands.
#include "tpq_common.h"

namespace tpq {
namespace {

typedef __bf16 fg_bf8 __attribute__((ext_vector_type(8)));
typedef float fg_f2 __attribute__((ext_vector_type(2)));
typedef float fg_f4 __attribute__((ext_vector_type(4)));
typedef float fg_f16 __attribute__((ext_vector_type(16)));

constexpr int kTile = 128, kStageK = 32, kThreads = 256, kParts = 3;
constexpr int kChunkBytes = kTile * 16 + 64;  // (64: the four chunks of a row read along k fall into different banks)
constexpr int kPartBytes = (kStageK / 8) * kChunkBytes, kOperandBytes = kParts * kPartBytes;

// c[m][n] = sum over k of a(m, k) b(n, k); b lies as [k][n], a as [m][k] (ALONG) or [k][m]
struct Product {
    const float *a, *b;
    float* c;        // [M][N], or [slices][M][N] in the workspace
    int M, N, K;
    int tiles_m, tiles_n, slices, stages_per_slice;
};

struct GradArgs {
    Product p[2];    // grad_x, grad_w
    int first;       // workgroups of p[0]
};

// the float32 values of one operand and stage that a thread carries: ALONG rows t / 4 + 32 j, k 8 (t % 4) .. + 7;
// else rows 4 (t % 32) .. + 3 at k 8 (t / 32) + j
template <bool ALONG>
__device__ __forceinline__ void fetch(const float* __restrict__ base, int rows, int row0, int K, int k0, int t, fg_f4 (&v)[8]) {
    if constexpr (ALONG) {
        const int k = k0 + 8 * (t & 3);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int row = row0 + (t >> 2) + 32 * j;
            const float* const p = base + static_cast<size_t>(row < rows ? row : rows - 1) * K;
#pragma unroll
            for (int h = 0; h < 2; ++h) v[2 * j + h] = *reinterpret_cast<const fg_f4*>(p + (k + 4 * h < K ? k + 4 * h : K - 4));
        }
    } else {
        const int row = row0 + 4 * (t & 31), k = k0 + 8 * (t >> 5);
        const float* const p = base + (row < rows ? row : rows - 4);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = *reinterpret_cast<const fg_f4*>(p + static_cast<size_t>(k + j < K ? k + j : K - 1) * rows);
    }
}

// zeros for k >= K
template <bool ALONG>
__device__ __forceinline__ void clear_behind(int K, int k0, int t, fg_f4 (&v)[8]) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int k = ALONG ? k0 + 8 * (t & 3) + 4 * (j & 1) : k0 + 8 * (t >> 5) + j;
        if (k >= K) v[j] = fg_f4{0.0f, 0.0f, 0.0f, 0.0f};
    }
}

// Eight values as three chunks of bfloat16 parts: h is the upper half of the value after half a unit was added (to nearest; beyond the
// largest bfloat16 it is infinite, m NaN and the sum is formed again), m the upper half of x - h, l what is left, 8 bits at most.  cut
// gathers what is left of l: nothing from 2^-110 on.
// v_cvt_pk_bf16_f32 and v_dot2_f32_bf16, half as many instructions, take 8 - 10 % longer.
__device__ __forceinline__ void store_parts(const float (&x)[8], char* lds, uint32_t& cut) {
    uint32_t h[4], m[4], l[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t upper[2], middle[2], lower[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const float v = x[2 * i + e];
            upper[e] = __builtin_bit_cast(uint32_t, v) + 0x8000u;
            const float r = v - __builtin_bit_cast(float, upper[e] & 0xFFFF0000u);
            middle[e] = __builtin_bit_cast(uint32_t, r);
            lower[e] = __builtin_bit_cast(uint32_t, r - __builtin_bit_cast(float, middle[e] & 0xFFFF0000u));
        }
        h[i] = __builtin_amdgcn_perm(upper[1], upper[0], 0x07060302u);
        m[i] = __builtin_amdgcn_perm(middle[1], middle[0], 0x07060302u);
        l[i] = __builtin_amdgcn_perm(lower[1], lower[0], 0x07060302u);
        cut |= lower[0] | lower[1];
        asm volatile("" : "+v"(cut));
    }
    *reinterpret_cast<uint4*>(lds) = make_uint4(h[0], h[1], h[2], h[3]);
    *reinterpret_cast<uint4*>(lds + kPartBytes) = make_uint4(m[0], m[1], m[2], m[3]);
    *reinterpret_cast<uint4*>(lds + 2 * kPartBytes) = make_uint4(l[0], l[1], l[2], l[3]);
}

template <bool ALONG>
__device__ __forceinline__ void put(const fg_f4 (&v)[8], char* lds, int t, uint32_t& cut) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float x[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = ALONG ? v[2 * e + (j >> 2)][j & 3] : v[j][e];
        const int chunk = ALONG ? t & 3 : t >> 5, slot = 32 * e + (ALONG ? t >> 2 : t & 31);
        store_parts(x, lds + chunk * kChunkBytes + slot * 16, cut);
    }
}

// the same values as they are: part p holds k 4 p .. 4 p + 3 of each chunk
template <bool ALONG>
__device__ __forceinline__ void put_whole(const fg_f4 (&v)[8], char* lds, int t) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            fg_f4 x;
#pragma unroll
            for (int j = 0; j < 4; ++j) x[j] = ALONG ? v[2 * e + p][j] : v[4 * p + j][e];
            const int chunk = ALONG ? t & 3 : t >> 5, slot = 32 * e + (ALONG ? t >> 2 : t & 31);
            *reinterpret_cast<fg_f4*>(lds + p * kPartBytes + chunk * kChunkBytes + slot * 16) = x;
        }
}

__device__ __forceinline__ fg_bf8 fragment(const char* lds) { return __builtin_bit_cast(fg_bf8, *reinterpret_cast<const uint4*>(lds)); }

// a workgroup's tile and its slice of k
struct Place {
    int m0, n0, begin, end, slice;
};

// Sums of a lane to memory.  Register e: slot 8 (e / 4) + 4 half + e % 4 of a fragment; row slot 32 f + s is row s of 32 rows (ALONG) or
// row 4 s + f, column slot 32 f + s column 4 s + f: the two column fragments are neighbours
template <bool ALONG>
__device__ __forceinline__ void write_sums(const Product& p, const Place& at, int wave, int lane, const fg_f16 (&acc)[2][2]) {
    const int i = lane & 31, half = lane >> 5, wm = wave >> 1, wn = wave & 1;
    const int n = at.n0 + 4 * i + 2 * wn;
    float* const c = p.c + static_cast<size_t>(at.slice) * p.M * p.N;
    if (n >= p.N) return;
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int in = 8 * (e >> 2) + 4 * half + (e & 3);
            const int m = at.m0 + (ALONG ? 32 * (2 * wm + f) + in : 4 * in + 2 * wm + f);
            if (m < p.M) *reinterpret_cast<fg_f2*>(c + static_cast<size_t>(m) * p.N + n) = fg_f2{acc[f][0][e], acc[f][1][e]};
        }
}

// A tile's slice again, with float32 instructions
template <bool ALONG>
__device__ __forceinline__ void whole_product(const Product& p, const Place& at, char* lds) {
    int thread = threadIdx.x;
    asm volatile("" : "+v"(thread));  // (or what the two forms have in common is kept in registers from the first to the second)
    const int t = thread & 127, lane = thread & 63, wave = thread >> 6, i = lane & 31, half = lane >> 5, wm = wave >> 1, wn = wave & 1;
    const bool first_operand = wave < 2;
    char* const lds_b = lds + kOperandBytes;
    fg_f16 acc[2][2];
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[f >> 1][f & 1][e] = 0.0f;
    for (int k0 = at.begin; k0 < at.end; k0 += kStageK) {
        fg_f4 v[8];
        if (first_operand) fetch<ALONG>(p.a, p.M, at.m0, p.K, k0, t, v);
        else fetch<false>(p.b, p.N, at.n0, p.K, k0, t, v);
        if (k0 + kStageK > p.K) {
            if (first_operand) clear_behind<ALONG>(p.K, k0, t, v);
            else clear_behind<false>(p.K, k0, t, v);
        }
        __syncthreads();
        if (first_operand) put_whole<ALONG>(v, lds, t);
        else put_whole<false>(v, lds_b, t);
        __syncthreads();
#pragma unroll 1
        for (int chunk = 0; chunk < kStageK / 8; ++chunk) {
            // a lane's half multiplies k 4 half .. + 3 of the chunk, in both operands
            const char* const la = lds + half * kPartBytes + chunk * kChunkBytes + (64 * wm + i) * 16;
            const char* const lb = lds_b + half * kPartBytes + chunk * kChunkBytes + (64 * wn + i) * 16;
            fg_f4 a[2], b[2];
#pragma unroll
            for (int f = 0; f < 2; ++f) {
                a[f] = *reinterpret_cast<const fg_f4*>(la + f * 32 * 16);
                b[f] = *reinterpret_cast<const fg_f4*>(lb + f * 32 * 16);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int f = 0; f < 4; ++f)
                    acc[f >> 1][f & 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[f >> 1][e], b[f & 1][e], acc[f >> 1][f & 1], 0, 0, 0);
        }
    }
    write_sums<ALONG>(p, at, wave, lane, acc);
}

template <bool ALONG>
__device__ __forceinline__ void product(const Product& p, int block, int blocks, char* lds, uint32_t* inexact) {
    // consecutive workgroups go round the eight dies: each die gets one run of neighbouring tiles, whose operands its L2 holds
    const int die = block & 7, each = blocks >> 3, more = blocks & 7;
    const int id = die * each + (die < more ? die : more) + (block >> 3);
    const int tiles = p.tiles_m * p.tiles_n, slice = id / tiles, tile = id - slice * tiles;
    // groups of eight tile rows, down each group's columns
    const int group = tile / (8 * p.tiles_n), in_group = tile - group * 8 * p.tiles_n;
    const int high = p.tiles_m - 8 * group < 8 ? p.tiles_m - 8 * group : 8;
    const int tile_n = in_group / high, tile_m = 8 * group + in_group - tile_n * high;
    const int m0 = tile_m * kTile, n0 = tile_n * kTile;
    const int begin = slice * p.stages_per_slice * kStageK;
    const int end = begin + p.stages_per_slice * kStageK < p.K ? begin + p.stages_per_slice * kStageK : p.K;
    const Place at{m0, n0, begin, end, slice};

    const int t = threadIdx.x & 127, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i = lane & 31, half = lane >> 5, wm = wave >> 1, wn = wave & 1;
    const bool first_operand = wave < 2;
    char* const lds_b = lds + kOperandBytes;
    fg_f4 v[8];
    const auto load = [&](int k0) {
        if (first_operand) fetch<ALONG>(p.a, p.M, m0, p.K, k0, t, v);
        else fetch<false>(p.b, p.N, n0, p.K, k0, t, v);
    };
    const auto store = [&](int k0) {
        if (k0 + kStageK > p.K) {
            if (first_operand) clear_behind<ALONG>(p.K, k0, t, v);
            else clear_behind<false>(p.K, k0, t, v);
        }
        uint32_t cut = 0;
        if (first_operand) put<ALONG>(v, lds, t, cut);
        else put<false>(v, lds_b, t, cut);
        return (cut & 0xFFFFu) != 0;
    };

    fg_f16 acc[2][2];
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[f >> 1][f & 1][e] = 0.0f;

    load(begin);
    if (threadIdx.x == 0) *inexact = p.K < 4;
    const bool first_cut = store(begin);
    __syncthreads();
    if (first_cut) *inexact = 1;
    uint32_t stop = 0;  // what *inexact was between the two barriers before a stage, the same for all of the workgroup
    for (int k0 = begin; k0 < end; k0 += kStageK) {
        const bool more_stages = k0 + kStageK < end;
        if (more_stages) load(k0 + kStageK);
#pragma unroll
        for (int s = 0; s < kStageK / 16; ++s) {
            const char* const la = lds + (2 * s + half) * kChunkBytes + (64 * wm + i) * 16;
            const char* const lb = lds_b + (2 * s + half) * kChunkBytes + (64 * wn + i) * 16;
            fg_bf8 a[kParts][2], b[kParts][2];
#pragma unroll
            for (int part = 0; part < kParts; ++part)
#pragma unroll
                for (int f = 0; f < 2; ++f) {
                    a[part][f] = fragment(la + part * kPartBytes + f * 32 * 16);
                    b[part][f] = fragment(lb + part * kPartBytes + f * 32 * 16);
                }
            constexpr int kA[6] = {2, 0, 1, 1, 0, 0}, kB[6] = {0, 2, 1, 0, 1, 0};  // small products first
#pragma unroll
            for (int e = 0; e < 6; ++e)
#pragma unroll
                for (int f = 0; f < 4; ++f)
                    acc[f >> 1][f & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[kA[e]][f >> 1], b[kB[e]][f & 1], acc[f >> 1][f & 1], 0, 0, 0);
        }
        stop = __builtin_amdgcn_readfirstlane(stop);
        if (stop || !more_stages) break;
        __syncthreads();
        if (store(k0 + kStageK)) *inexact = 1;
        __syncthreads();
        stop = *inexact;
    }

    // parts that do not add up to their value, or a sum that is not finite (its product with zero is NaN)
    float left[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int e = 0; e < 16; ++e)
#pragma unroll
        for (int f = 0; f < 4; ++f) left[f] = __builtin_fmaf(acc[f >> 1][f & 1][e], 0.0f, left[f]);
    const float any = (left[0] + left[1]) + (left[2] + left[3]);
    if (any != any) *inexact = 1;
    __syncthreads();
    const uint32_t again = *inexact;
    write_sums<ALONG>(p, at, wave, lane, acc);
    if (__builtin_amdgcn_readfirstlane(again)) whole_product<ALONG>(p, at, lds);
}

__global__ __launch_bounds__(kThreads, 3) void f32_grads_kernel(const GradArgs args) {
    __shared__ __attribute__((aligned(16))) char lds[2 * kOperandBytes];
    __shared__ uint32_t inexact;
    const int block = static_cast<int>(blockIdx.x);
    if (block < args.first) product<true>(args.p[0], block, args.first, lds, &inexact);
    else product<false>(args.p[1], block - args.first, static_cast<int>(gridDim.x) - args.first, lds, &inexact);
}

struct Finish {
    const fg_f4* partial;
    fg_f4* out;
    int64_t quads;
    int slices, parts, blocks;  // parts: neighbouring slices go to one of this many threads
};

// The slices' sums, added in slice order; blocks of both products in one launch.  Many slices of a small output, whose quads are too few
// threads for the chip, are shared out over parts of a workgroup, whose sums are then added in part order: 512 slices one after the other
// would be their requests' latency.  A larger output (more than 128 workgroups of quads) is the slower that way (256 rows, 1648 -> 2560, nine
// slices: 40 / 36 us).
__global__ __launch_bounds__(256) void f32_grads_finish_kernel(const Finish x, const Finish w) {
    __shared__ fg_f4 sums[256];
    const bool second = static_cast<int>(blockIdx.x) >= x.blocks;
    const Finish f = second ? w : x;
    const int each = 256 / f.parts, part = static_cast<int>(threadIdx.x) / each;
    const int64_t q = static_cast<int64_t>(static_cast<int>(blockIdx.x) - (second ? x.blocks : 0)) * each + static_cast<int>(threadIdx.x) % each;
    const int per = (f.slices + f.parts - 1) / f.parts, first = part * per, last = first + per < f.slices ? first + per : f.slices;
    fg_f4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
    if (q < f.quads && first < last) {
        sum = f.partial[first * f.quads + q];
        for (int s = first + 1; s < last; ++s) sum += f.partial[s * f.quads + q];
    }
    if (f.parts > 1) {
        sums[threadIdx.x] = sum;
        __syncthreads();
        for (int p = 1; p < f.parts && p * per < f.slices; ++p) sum += sums[(p * each + static_cast<int>(threadIdx.x)) & 255];
    }
    if (q < f.quads && part == 0) f.out[q] = sum;
}

constexpr int64_t kPlaces = 512;  // two workgroups on each of 256 compute units
constexpr int kLeastStages = 4;
constexpr int64_t kFewQuads = 128 * 256;

struct Plan {
    int64_t tiles_m, tiles_n, slices, stages;
};

Plan plan_of(int64_t M, int64_t N, int64_t K, int64_t stages_each) {
    Plan p{(M + kTile - 1) / kTile, (N + kTile - 1) / kTile, 1, 0};
    const int64_t stages = (K + kStageK - 1) / kStageK;
    int64_t slices = (stages + stages_each / 2) / stages_each;
    if (slices < 1) slices = 1;
    p.stages = (stages + slices - 1) / slices;
    p.slices = (stages + p.stages - 1) / p.stages;
    return p;
}

// Plans of grad_x and grad_w: about the stages that each place gets if all are shared out evenly.  Nine to sixteen slices of a product only
// where all workgroups find a place at once: the few that would not start when the others end, and then take as long (248 rows, 1536 ->
// 2944: 516 workgroups 47 us, 468 37; 180 rows, 1408 -> 3584 44 / 39).  With more slices they are short (55 rows, 1408 -> 3584: 616 workgroups,
// 28 slices, 22 us, 517 23), and where the tiles fill the places by themselves there is nothing to lose.
void plans(int64_t M, int64_t K, int64_t N, bool want_x, bool want_w, Plan (&plan)[2]) {
    const auto tiles = [](int64_t a, int64_t b) { return ((a + kTile - 1) / kTile) * ((b + kTile - 1) / kTile); };
    const int64_t tiles_x = want_x ? tiles(M, K) : 0, tiles_w = want_w ? tiles(N, K) : 0;
    const int64_t all = tiles_x * ((N + kStageK - 1) / kStageK) + tiles_w * ((M + kStageK - 1) / kStageK);
    int64_t each = (all + kPlaces - 1) / kPlaces;
    if (each < kLeastStages) each = kLeastStages;
    const auto settled = [](const Plan& p) { return p.slices <= 8 || p.slices > 16; };
    for (;; each += each / 8 + 1) {
        plan[0] = plan_of(M, K, N, each);
        plan[1] = plan_of(N, K, M, each);
        const int64_t x = tiles_x * plan[0].slices, w = tiles_w * plan[1].slices;
        if ((settled(plan[0]) && settled(plan[1])) || tiles_x + tiles_w >= kPlaces || x + w <= kPlaces) return;
    }
}

}  // namespace
}  // namespace tpq

using namespace tpq;

namespace tpq {
namespace {
inline bool grads_sizes_ok(int64_t M, int64_t K, int64_t N) {
    return M > 0 && K > 0 && N > 0 && K % 4 == 0 && N % 4 == 0 && M <= (1 << 24) && K <= (1 << 24) && N <= (1 << 24);
}
}  // namespace
}  // namespace tpq

// Up to three rows the tiles are padding but for those and grad_w is formed with float32 instructions too (us, this / library products:
// 4096 x 4096 at 1, 2, 4 rows 55 / 41, 54 / 41, 38 / 40; 8192 x 8192 207 / 137, 199 / 137, 145 / 139; 4096 -> 11008 126 / 109, 138 / 109,
// 94 / 110; small layers, where the calls are what counts, 2048 x 2048 21 / 40 at any of them).
TPQ_EXPORT int tpq_f32_linear_grads_takes(const float* grad, const float* x, const float* w, int64_t M, int64_t K, int64_t N) {
    return M >= 4 && grads_sizes_ok(M, K, N) && aligned(grad, 16) && aligned(x, 16) && aligned(w, 16);
}

TPQ_EXPORT size_t tpq_f32_linear_grads_workspace_bytes(int64_t M, int64_t K, int64_t N, int want_x, int want_w) {
    if (M <= 0 || K <= 0 || N <= 0) return 0;
    Plan plan[2];
    plans(M, K, N, want_x != 0, want_w != 0, plan);
    size_t bytes = 0;
    if (want_x && plan[0].slices > 1) bytes += static_cast<size_t>(plan[0].slices * M * K) * 4;
    if (want_w && plan[1].slices > 1) bytes += static_cast<size_t>(plan[1].slices * N * K) * 4;
    return bytes;
}

TPQ_EXPORT int tpq_f32_linear_grads(const float* grad, const float* x, const float* w, int64_t M, int64_t K, int64_t N, float* grad_x,
                                    float* grad_w, void* workspace, size_t workspace_bytes, void* stream) {
    TPQ_REQUIRE(M >= 0 && K >= 0 && N >= 0, TPQ_ERR_INVALID_VALUE, "tpq_f32_linear_grads: negative dimension");
    TPQ_REQUIRE(grads_sizes_ok(M, K, N), TPQ_ERR_UNSUPPORTED,
                "tpq_f32_linear_grads: sizes of 1 to 2^24, K and N multiples of 4");
    if (grad_x == nullptr && grad_w == nullptr) return TPQ_OK;
    TPQ_REQUIRE(grad && (grad_x == nullptr || w) && (grad_w == nullptr || x), TPQ_ERR_INVALID_VALUE, "tpq_f32_linear_grads: null pointer");
    TPQ_REQUIRE(aligned(grad, 16) && aligned(x, 16) && aligned(w, 16) && aligned(grad_x, 16) && aligned(grad_w, 16) && aligned(workspace, 16),
                TPQ_ERR_UNSUPPORTED, "tpq_f32_linear_grads: operands must be 16-byte aligned");
    TPQ_REQUIRE(workspace_bytes >= tpq_f32_linear_grads_workspace_bytes(M, K, N, grad_x != nullptr, grad_w != nullptr) &&
                    (workspace != nullptr || workspace_bytes == 0),
                TPQ_ERR_INVALID_VALUE, "tpq_f32_linear_grads: workspace too small");
    Plan plan[2];
    plans(M, K, N, grad_x != nullptr, grad_w != nullptr, plan);
    GradArgs args{};
    Finish finish[2] = {};
    int64_t blocks[2] = {0, 0};
    float* space = static_cast<float*>(workspace);
    const int m = static_cast<int>(M), k = static_cast<int>(K), n = static_cast<int>(N);
    args.p[0] = Product{grad, w, grad_x, m, k, n, 0, 0, 0, 0};
    args.p[1] = Product{grad, x, grad_w, n, k, m, 0, 0, 0, 0};
    for (int e = 0; e < 2; ++e) {
        Product& p = args.p[e];
        if (p.c == nullptr) continue;
        p.tiles_m = static_cast<int>(plan[e].tiles_m);
        p.tiles_n = static_cast<int>(plan[e].tiles_n);
        p.slices = static_cast<int>(plan[e].slices);
        p.stages_per_slice = static_cast<int>(plan[e].stages);
        blocks[e] = plan[e].tiles_m * plan[e].tiles_n * plan[e].slices;
        if (p.slices > 1) {
            const int64_t quads = static_cast<int64_t>(p.M) * p.N / 4;
            const int parts = p.slices > 8 && quads <= kFewQuads ? 16 : 1;
            finish[e] = Finish{reinterpret_cast<const fg_f4*>(space), reinterpret_cast<fg_f4*>(p.c), quads, p.slices, parts, static_cast<int>((quads * parts + 255) / 256)};
            p.c = space;
            space += p.slices * quads * 4;
        }
    }
    TPQ_REQUIRE(blocks[0] + blocks[1] < (1 << 24), TPQ_ERR_UNSUPPORTED, "tpq_f32_linear_grads: too many tiles");
    args.first = static_cast<int>(blocks[0]);
    hipStream_t s = static_cast<hipStream_t>(stream);
    f32_grads_kernel<<<dim3(static_cast<unsigned>(blocks[0] + blocks[1])), dim3(kThreads), 0, s>>>(args);
    if (int rc = check_launch("tpq_f32_linear_grads")) return rc;
    const int adding = finish[0].blocks + finish[1].blocks;
    if (adding == 0) return TPQ_OK;
    f32_grads_finish_kernel<<<dim3(adding), dim3(256), 0, s>>>(finish[0], finish[1]);
    return check_launch("tpq_f32_linear_grads (finish)");
}

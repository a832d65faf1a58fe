// Dynamically quantized linear of 1 .. 16 activation rows in ONE launch: the rows are quantized to int8 by every workgroup for itself
// and meet the weight (int8 rows, or packed 2-bit ternary codes) on the matrix cores; same bits as the row quantizer and the
// product behind it.
//
// What bounds it: at these sizes a launch.  The quantizer is 2.5 - 3 us for a few KB, its codes travel through memory, the product waits
// for it, and the host pays two launches and a buffer for the codes; the weight of such a layer streams in 1 - 4 us.  Hence
//   * a workgroup is 16 wavefronts and NB blocks of 16 channels, NB the smallest that leaves at most one workgroup per compute unit, so that
//     a compute unit quantizes the rows once;
//   * a wavefront takes segments of a row, 512 elements each (SEGS <= 4: at most 32768 elements, about 1 us of vector work a workgroup;
//     beyond, the quantizer's own launch is the cheaper one), and asks for its share of the weight before it looks at them: up to
//     W = 4 steps of it in registers, every load of the workgroup in flight at once;
//   * maxima and codes meet in LDS, rows 16 bytes apart from a multiple of the step so that the sixteen rows of an operand read lie in
//     different banks; barriers wait for LDS only;
//   * products as in int8_decode_kernel.h and ternary_decode_mfma.h: the weight as the A operand as it lies (ternary: expanded in
//     registers, the activations in the order of its fields), wavefront (b, ks) block b and the steps ks, ks + 16 / NB, ...; exact
//     int32 sums, so it does not matter which.
#include "int8_gemm_kernel.h"
#include "quantize_row.h"
#include "ternary_decode_mfma.h"

namespace tpq {
namespace {

constexpr int kFewWaves = 16, kFewRows = 16, kFewSegment = kWave * kVec, kFewSegments = 4 * kFewWaves, kFewMaxSteps = 4,
              kFewFullSteps = 2;  // int8 rows in four segments

struct FewRowsOut {
    void* out;           // [M][N]
    const float* cs;     // [N], or null: w_scale
    const float* bias;   // [N] or null
    float w_scale;
    int dtype;
};

// int8 rows [N][K], K % 16 == 0: lane (i, q) holds the 32 bytes of row i at 32 q of a step of 128 k
struct FewInt8 {
    static constexpr int kStep = 128, kLoads = 2;
    static __device__ __forceinline__ void load(const uint8_t* w, size_t n, int K, int step, int q, uint4 (&d)[kLoads]) {
        const uint8_t* const row = w + n * K;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int k = step * kStep + 32 * q + 16 * h;
            d[h] = nt_load(reinterpret_cast<const uint4*>(row + (k < K ? k : K - 16)));  // behind K: any codes, they meet zeros
        }
    }
    static __device__ __forceinline__ void multiply(const uint4 (&d)[kLoads], const char* x_row, int step, int q, v4i (&acc)[2]) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
            acc[h] = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(v4i, d[h]), *reinterpret_cast<const v4i*>(x_row + step * kStep + 32 * q + 16 * h), acc[h], 0, 0, 0);
    }
};

// packed ternary rows [N][K / 4], K % 64 == 0: lane (i, q) holds the 64 codes of row i at 64 q of a step of 256 k
struct FewTernary {
    static constexpr int kStep = 256, kLoads = 1;
    static __device__ __forceinline__ void load(const uint8_t* w, size_t n, int K, int step, int q, uint4 (&d)[kLoads]) {
        const int k = step * kStep + 64 * q;
        d[0] = nt_load(reinterpret_cast<const uint4*>(w + n * (static_cast<size_t>(K) >> 2) + ((k < K ? k : K - 64) >> 2)));
    }
    static __device__ __forceinline__ void multiply(const uint4 (&d)[kLoads], const char* x_row, int step, int q, v4i (&acc)[2]) {
        const uint32_t words[4] = {d[0].x, d[0].y, d[0].z, d[0].w};
#pragma unroll
        for (int p = 0; p < 4; ++p)
            acc[p & 1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ternary_fields_to_i8(words[p]),
                                                               transpose_4x4_bytes(*reinterpret_cast<const uint4*>(x_row + step * kStep + 64 * q + 16 * p)), acc[p & 1], 0, 0, 0);
    }
};

__host__ __device__ constexpr int few_pitch(int K, int step) { return (K + step - 1) / step * step + 16; }

// grid: ceil(N / (16 << nb_shift)); block: 1024; LDS: M few_pitch(K) bytes.  M <= 16, K % 16 == 0 (FewTernary: 64), M segs_per_row <= 16 SEGS,
// ceil(K / kStep) << nb_shift <= 16 W, segs_per_row = ceil(K / 512) <= 16
template <class Source, int XDT, int SEGS, int W>
__global__ __launch_bounds__(kFewWaves * kWave) void few_rows_kernel(const typename Elem<XDT>::storage* __restrict__ x, const uint8_t* __restrict__ w, int M, int N, int K,
                                                                    int nb_shift, int segs_per_row, float inv_segs_per_row, float eps, FewRowsOut o) {
    extern __shared__ uint4 few_codes[];  // [M][pitch] bytes
    __shared__ float seg_most[kFewSegments], row_scales[kFewRows];
    __shared__ int red[kFewWaves][4][kWave];
    char* const codes = reinterpret_cast<char*>(few_codes);
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = lane & 15, q = lane >> 4;
    const int pitch = few_pitch(K, Source::kStep), steps = pitch / Source::kStep;  // (the 16 spare bytes are less than a step)
    const int segs = M * segs_per_row;
    const QParams quantizer{eps, 127.0f, -127, 127, 0, 1};  // constants: what other parameters would need is not compiled in
    auto row_of = [&](int seg) { return static_cast<int>((static_cast<float>(seg) + 0.5f) * inv_segs_per_row); };  // exact: seg < 64
    auto lds_barrier = []() __attribute__((always_inline)) { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    // ---- requests: this wavefront's pieces of the rows, then its share of the weight
    int row[SEGS], k0[SEGS];
    RawChunk<XDT> raw[SEGS];
#pragma unroll
    for (int j = 0; j < SEGS; ++j) {
        const int seg = wave + j * kFewWaves < segs ? wave + j * kFewWaves : segs - 1;  // past the last: that one again, nothing is kept of it
        row[j] = __builtin_amdgcn_readfirstlane(row_of(seg));
        k0[j] = (seg - row[j] * segs_per_row) * kFewSegment + lane * kVec;
        raw[j] = load_raw<XDT, false>(x + static_cast<size_t>(row[j]) * K + chunk_start(k0[j], K));
    }
    __builtin_amdgcn_sched_barrier(0);
    const int block = wave & ((1 << nb_shift) - 1), ks = wave >> nb_shift, ks_count = kFewWaves >> nb_shift;
    const int n0 = ((blockIdx.x << nb_shift) + block) * 16;
    uint4 wq[W][Source::kLoads];
#pragma unroll
    for (int j = 0; j < W; ++j) {
        const int step = ks + j * ks_count, n = n0 + i;
        Source::load(w, static_cast<size_t>(n < N ? n : N - 1), K, step < steps ? step : ks < steps ? ks : 0, q, wq[j]);  // past the end: the first one again; channels past N: a valid row, result dropped
    }
    // element v of a lane's sums: row i, channel n0 + 4 q + v; wavefront ks of a block finishes the elements ks, ks + ks_count, ..  What
    // it needs for them travels with the weight; no branch around a load: some readable word where there is none
    float col_scale[2], bias_n[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const int n = n0 + 4 * q + ((ks + e * ks_count) & 3), at = n < N ? n : N - 1;
        const float* const some = reinterpret_cast<const float*>(w);
        col_scale[e] = *pinned_global(o.cs ? o.cs + at : some);
        bias_n[e] = *pinned_global(o.bias ? o.bias + at : some);
    }
    __builtin_amdgcn_sched_barrier(0);

    // ---- maxima
    float v[SEGS][kVec];
#pragma unroll
    for (int j = 0; j < SEGS; ++j) {
        unpack_chunk<XDT>(raw[j], v[j]);
        float most = 0.0f;
#pragma unroll
        for (int e = 0; e < kVec; ++e) most = fmaxf(most, fabsf(v[j][e]));
        most = wave_max(most);
        if (lane == 0 && wave + j * kFewWaves < segs) seg_most[wave + j * kFewWaves] = most;
    }
    for (int t = threadIdx.x, spare = (pitch - 16 - K) / 16; t < M * spare; t += kFewWaves * kWave) {  // zeros behind K
        const int r = static_cast<int>(static_cast<uint32_t>(t) / static_cast<uint32_t>(spare));
        *reinterpret_cast<uint4*>(codes + r * pitch + K + (t - r * spare) * 16) = make_uint4(0, 0, 0, 0);
    }
    lds_barrier();
    // ---- codes: sixteen lanes find the parameters of a segment's row (at most 16 segments), the wavefront's segments side by side
    static_assert(SEGS <= 4, "a group of sixteen lanes per segment");
    const int my = q < SEGS ? q : 0, my_seg = wave + my * kFewWaves < segs ? wave + my * kFewWaves : segs - 1;
    const int my_row = row_of(my_seg);
    float row_most = seg_most[my_row * segs_per_row + (i < segs_per_row ? i : 0)];
    over_16_lanes(row_most, [](float a, float b) { return fmaxf(a, b); });
    const RowScale mine = scale_of_row(row_most, quantizer);
#pragma unroll
    for (int j = 0; j < SEGS; ++j) {
        if (wave + j * kFewWaves < segs) {
            RowScale r;
            r.scale = from_lane(mine.scale, 16 * j);
            r.inverse = from_lane(mine.inverse, 16 * j);
            r.shortcut = __builtin_amdgcn_readlane(mine.shortcut, 16 * j) != 0;
            r.lean = __builtin_amdgcn_readlane(mine.lean, 16 * j) != 0;
            uint32_t lo, hi;
            quantize_eight(v[j], r, quantizer, lo, hi);
            if (k0[j] < K) *reinterpret_cast<uint2*>(codes + row[j] * pitch + k0[j]) = make_uint2(lo, hi);  // K % 8 == 0: chunks do not overlap
            if (k0[j] == 0) row_scales[row[j]] = r.scale;
        }
    }
    lds_barrier();

    // ---- products
    const char* const x_row = codes + (i < M ? i : M - 1) * pitch;  // columns past M: results dropped
    v4i acc[2] = {};
#pragma unroll
    for (int j = 0; j < W; ++j)
        if (ks + j * ks_count < steps) Source::multiply(wq[j], x_row, ks + j * ks_count, q, acc);
#pragma unroll
    for (int e = 0; e < 4; ++e) red[wave][e][lane] = acc[0][e] + acc[1][e];
    lds_barrier();
    const float row_scale = row_scales[i < M ? i : M - 1];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const int element = ks + e * ks_count, n = n0 + 4 * q + element;
        if (element >= 4) break;
        int sum = 0;
        for (int s = 0; s < ks_count; ++s) sum += red[(s << nb_shift) + block][element][lane];
        if (i < M && n < N) {
            float f = __fmul_rn(__fmul_rn(static_cast<float>(sum), row_scale), o.cs ? col_scale[e] : o.w_scale);
            if (o.bias) f = __fadd_rn(f, bias_n[e]);
            const size_t idx = static_cast<size_t>(i) * N + n;
            if (o.dtype == TPQ_DTYPE_F32) static_cast<float*>(o.out)[idx] = f;
            else if (o.dtype == TPQ_DTYPE_F16) static_cast<uint16_t*>(o.out)[idx] = f32_to_f16_bits(f);
            else static_cast<uint16_t*>(o.out)[idx] = f32_to_bf16_bits(f);
        }
    }
}

struct FewRowsPlan {
    int nb_shift, steps_per_wave, segments;  // segments and steps of a wavefront; 0 segments: not for this kernel
};

// Where one launch is the shorter way.  Measured (us, two launches / one; a pass called eagerly, then the kernels alone in a graph), weights
// from HBM:
//   int8, up to two segments: 16 rows 1024 x 1024 float32 9.8 / 6.4, 6.2 / 5.6; 1024 -> 8192 9.7 / 6.4, 6.9 / 5.9; one row 4096 x 4096 9.4 / 6.4, 7.9 /
//     6.9; 4096 -> 8192 10.4 / 9.6, 10.9 / 11.1; 7424 -> 1536 9.4 / 8.5, 8.1 / 8.5; four rows 3072 -> 8192 11.7 / 8.9, 12.0 / 9.7
//   three or four segments, where the vector work is 1.3 us longer: only in well filled segments and with little weight to wait for: 16 rows
//     2048 -> 4096 9.4 / 7.9, 7.5 / 7.5; eight rows 4096 x 4096 9.5 / 9.3, 9.3 / 9.7; but seven rows 3328 -> 1280 10.4 / 8.4, 7.8 / 8.5 and three rows
//     7328 -> 3632 11.2 / 13.8, 11.7 / 14.4
//   beyond 2^25 weights the streams of the row and flight kernels are the better ones: one row 8192 x 8192 16.3 / 16.8, 16.7 / 18.5; ternary 4096 ->
//     11008 9.6 / 10.7 in a graph
//   ternary (two linears and a relu): two rows 1024 <-> 3712 24.9 / 15.7, 16.9 / 10.6; eight rows 2560 <-> 6912 24.9 / 19.3, 19.1 / 18.9; K that is no
//     multiple of 256, five rows 3712 <-> 3200 37 / 15.8, 36 / 15.2; 16 rows 2048 x 2048 24.5 / 17.4, 15.0 / 16.6; one row 4096 <-> 8192 25 / 15.6, 16 / 14.2
inline FewRowsPlan few_rows_plan(int64_t M, int64_t N, int64_t K, int step, int k_multiple) {
    const FewRowsPlan none{0, 0, 0};
    if (M < 1 || M > kFewRows || N < 1 || N > 16 * 8 * 256 || K < k_multiple || K % k_multiple || K > 16 * kFewSegment || N * K > (int64_t{1} << 25)) return none;
    const int64_t segs = M * ((K + kFewSegment - 1) / kFewSegment);
    if (segs > kFewSegments) return none;
    FewRowsPlan p{0, 0, segs <= kFewWaves ? 1 : segs <= 2 * kFewWaves ? 2 : 4};
    while (((N + 15) / 16 + (1 << p.nb_shift) - 1) >> p.nb_shift > 256) ++p.nb_shift;
    const int64_t shares = (((K + step - 1) / step << p.nb_shift) + kFewWaves - 1) / kFewWaves;
    if (shares > kFewMaxSteps) return none;
    if (step == FewInt8::kStep && p.segments == 4 && (shares > kFewFullSteps || M * K * 16 < segs * kFewSegment * 15)) return none;
    p.steps_per_wave = static_cast<int>(shares);
    return p;
}

// For whom a call that the kernel takes should go to it: 2 everybody, 1 who makes it eagerly (the host saves a launch and a buffer, the device is
// longer by the vector work of the rows in every workgroup, so the two launches are the shorter ones to replay), 0 nobody.  us, two launches / one, in a
// graph and eager:
//   four segments: int8 with two steps a wavefront, eight rows 3968 -> 1708 9.0 / 9.5, 10.7 / 9.7, 11 rows 2528 -> 2460 8.1 / 9.6, 9.4 / 9.8; with one, 16 rows 1984 -> 2272 8.1 /
//     8.7, 10.6 / 8.7, but up to 48 of the 64 filled, 12 rows 1936 -> 3832 8.4 / 8.1.  Ternary with K % 256 == 0, two linears: 16 rows 2048 x 2048 15.6 / 17.4, 25.9 / 17.5; other K,
//     whose product of codes is the slower one, 16 rows 1984 x 1984 22.4 / 17.8
//   int8 rows off 64 bytes, whose steps touch twice the lines: four steps a wavefront, one row 7392 -> 1348 10.2 / 11.6, 10.8 / 11.7, two rows 6160 -> 820 9.8 / 11.7, 10.6 /
//     11.8; three steps and two segments, three rows 4272 -> 924 9.2 / 10.5, 10.6 / 10.6 (one segment, 3 rows in four are shorter)
inline int few_rows_pays(const FewRowsPlan& p, int64_t M, int64_t K, int step) {
    if (!p.segments) return 0;
    if (step != FewInt8::kStep) return p.segments == 4 && K % step == 0 ? 1 : 2;
    const bool off_lines = K % 64 != 0;
    if (off_lines && p.steps_per_wave == 4) return 0;
    const bool full = p.segments == 4 && (p.steps_per_wave > 1 || M * ((K + kFewSegment - 1) / kFewSegment) > 48);
    return full || (off_lines && p.segments == 2 && p.steps_per_wave == 3) ? 1 : 2;
}

template <class Source, int XDT>
int launch_few_rows(const void* x, const uint8_t* w, int64_t M, int64_t N, int64_t K, const FewRowsPlan& p, float eps, const FewRowsOut& o, hipStream_t s) {
    const dim3 grid(static_cast<unsigned>(((N + 15) / 16 + (1 << p.nb_shift) - 1) >> p.nb_shift));
    const size_t smem = static_cast<size_t>(M) * few_pitch(static_cast<int>(K), Source::kStep);
    const int per_row = static_cast<int>((K + kFewSegment - 1) / kFewSegment);
    auto run = [&](auto segs, auto steps) {
        few_rows_kernel<Source, XDT, decltype(segs)::value, decltype(steps)::value><<<grid, kFewWaves * kWave, smem, s>>>(
            static_cast<const typename Elem<XDT>::storage*>(x), w, static_cast<int>(M), static_cast<int>(N), static_cast<int>(K), p.nb_shift,
            per_row, 1.0f / static_cast<float>(per_row), eps, o);
    };
    auto with_segments = [&](auto segs) {
        constexpr int kMost = Source::kStep == FewInt8::kStep && decltype(segs)::value == 4 ? kFewFullSteps : kFewMaxSteps;
        if (p.steps_per_wave == 1) run(segs, std::integral_constant<int, 1>{});
        else if (p.steps_per_wave == 2) run(segs, std::integral_constant<int, 2>{});
        else if constexpr (kMost > kFewFullSteps) {
            if (p.steps_per_wave == 3) run(segs, std::integral_constant<int, 3>{});
            else run(segs, std::integral_constant<int, 4>{});
        }
    };
    if (p.segments == 1) with_segments(std::integral_constant<int, 1>{});
    else if (p.segments == 2) with_segments(std::integral_constant<int, 2>{});
    else with_segments(std::integral_constant<int, 4>{});
    return check_launch("linear of a few rows, quantized in the product");
}

template <class Source>
int few_rows(const void* x, int x_dtype, const uint8_t* w, int64_t M, int64_t N, int64_t K, int k_multiple, float eps, const FewRowsOut& o, void* stream) {
    const FewRowsPlan p = few_rows_plan(M, N, K, Source::kStep, k_multiple);
    TPQ_REQUIRE(x && w && o.out, TPQ_ERR_INVALID_VALUE, "few rows linear: null pointer");
    TPQ_REQUIRE(p.segments && aligned(x, 16) && aligned(w, 16), TPQ_ERR_UNSUPPORTED, "few rows linear: a shape or an alignment that it does not take");
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (x_dtype == TPQ_DTYPE_F32) return launch_few_rows<Source, TPQ_DTYPE_F32>(x, w, M, N, K, p, eps, o, s);
    if (x_dtype == TPQ_DTYPE_F16) return launch_few_rows<Source, TPQ_DTYPE_F16>(x, w, M, N, K, p, eps, o, s);
    return launch_few_rows<Source, TPQ_DTYPE_BF16>(x, w, M, N, K, p, eps, o, s);
}

bool float_dtype(int t) { return t == TPQ_DTYPE_F32 || t == TPQ_DTYPE_F16 || t == TPQ_DTYPE_BF16; }

}  // namespace
}  // namespace tpq

using namespace tpq;

TPQ_EXPORT int tpq_int8_linear_few_takes(const void* x, const int8_t* w, int64_t M, int64_t N, int64_t K) {
    return few_rows_plan(M, N, K, FewInt8::kStep, 16).segments && aligned(x, 16) && aligned(w, 16);
}

TPQ_EXPORT int tpq_int8_linear_few_pays(int64_t M, int64_t N, int64_t K) { return few_rows_pays(few_rows_plan(M, N, K, FewInt8::kStep, 16), M, K, FewInt8::kStep); }

TPQ_EXPORT int tpq_int8_linear_few(const void* x, int x_dtype, const int8_t* w, const float* col_scale, const float* bias, int64_t M, int64_t N, int64_t K, float eps,
                                   void* out, int out_dtype, void* stream) {
    TPQ_REQUIRE(float_dtype(x_dtype) && float_dtype(out_dtype), TPQ_ERR_INVALID_TYPE, "int8_linear_few: unsupported dtype");
    TPQ_REQUIRE(col_scale, TPQ_ERR_INVALID_VALUE, "int8_linear_few: null pointer");
    return few_rows<FewInt8>(x, x_dtype, reinterpret_cast<const uint8_t*>(w), M, N, K, 16, eps, FewRowsOut{out, col_scale, bias, 0.0f, out_dtype}, stream);
}

TPQ_EXPORT int tpq_ternary_linear_few_takes(const void* x, const uint8_t* packed, int64_t M, int64_t N, int64_t K) {
    return few_rows_plan(M, N, K, FewTernary::kStep, 64).segments && aligned(x, 16) && aligned(packed, 16);
}

TPQ_EXPORT int tpq_ternary_linear_few_pays(int64_t M, int64_t N, int64_t K) { return few_rows_pays(few_rows_plan(M, N, K, FewTernary::kStep, 64), M, K, FewTernary::kStep); }

TPQ_EXPORT int tpq_ternary_linear_few(const void* x, int x_dtype, const uint8_t* packed, float w_scale, const float* bias, int64_t M, int64_t N, int64_t K, float eps,
                                      float* out, void* stream) {
    TPQ_REQUIRE(float_dtype(x_dtype), TPQ_ERR_INVALID_TYPE, "ternary_linear_few: unsupported input dtype");
    return few_rows<FewTernary>(x, x_dtype, packed, M, N, K, 64, eps, FewRowsOut{out, nullptr, bias, w_scale, TPQ_DTYPE_F32}, stream);
}

// Fused row-wise signed quantizer for gfx950.
//
// One 256-thread workgroup per row (rows of up to 1024 elements: a lane group of 8..64 lanes per
// row, several rows per workgroup).  The row is read from HBM once, kept in
// registers (8 elements per 16/32-byte vector load, up to 8 such chunks per
// lane), reduced to its absolute maximum with a 64-lane butterfly and one LDS
// exchange between the four wavefronts, and written back as int8 codes with
// 8-byte stores (rows of more than 16384 elements: 1024 threads).  Rows longer than the register budget
// (K > 65536) or rows
// that cannot be vector-loaded (K % 4 != 0) take the streaming kernel, which
// reads the row a second time (the second read comes from L2).
//
// Arithmetic (bit-exact with the reference's CPU kernel,
// p10/include/QuantNativeImpl.h:1162-1187 and
// p10/src/backend/cpu/LowBitGemmKernels.cpp:19-52):
//   absmax = max |float(x)|;  scale = fmaxf(absmax, eps) / divisor  (IEEE divide)
//   code   = clamp(rintf(float(x) / scale), qmin, qmax)              (IEEE divide, RNE)
#include "tpq_common.h"

namespace tpq {
namespace {

// -DTPQ_QUANT_STAMPS (a measuring build of its own, never the shipped library): every workgroup of the register-cached
// kernel leaves six readings of the shader clock (entry, loads issued, own data arrived and reduced, row maximum known,
// stores issued, stores acknowledged: the counters of different compute units do not share a zero, so only differences
// inside a workgroup mean something) and two of the chip-wide 100 MHz clock (entry, end).
#ifdef TPQ_QUANT_STAMPS
constexpr int kStampSlots = 8, kStampRows = 8192;
__device__ unsigned long long g_quant_stamps[kStampRows * kStampSlots];
#define TPQ_QUANT_STAMP(I)                                                                                              \
    do {                                                                                                                \
        __builtin_amdgcn_sched_barrier(0);                                                                              \
        if (threadIdx.x == 0 && blockIdx.x < kStampRows) g_quant_stamps[blockIdx.x * kStampSlots + (I)] = __builtin_amdgcn_s_memtime(); \
        __builtin_amdgcn_sched_barrier(0);                                                                              \
    } while (0)
#else
#define TPQ_QUANT_STAMP(I) do { } while (0)
#endif

}  // namespace
}  // namespace tpq

#include <type_traits>

#include "int8_gemm_kernel.h"
#include "quantize_row.h"

namespace tpq {
namespace {

constexpr int kThreads = 256;
// Rows up to this length: one wavefront (or a part of one) per row.  Longer rows on one wavefront were measured
// (2048 x 4096 bfloat16: 7.0 us against 6.6 with four wavefronts per row, 8.9 against 7.1 from HBM; two wavefronts per
// row: 8.3 against 7.9): a quarter of the wavefronts to launch, but too few loads in flight per compute unit.
constexpr int kSubwaveMaxK = 1024;

// Row cached in registers: CHUNKS * THREADS * 8 >= K >= 8, K % 4 == 0.
template <int DT, int CHUNKS, int THREADS = kThreads>
__global__ __launch_bounds__(THREADS) void quantize_rows_cached(
    const typename Elem<DT>::storage* __restrict__ x, int8_t* __restrict__ codes,
    float* __restrict__ scales, int K, QParams p) {
    __shared__ float smem[THREADS / kWave];
    const int64_t row = blockIdx.x;
    quantize_row_cached<DT, CHUNKS, THREADS>(x + row * K, codes + row * K, scales + row, K, p, smem);
}

// Short rows (8 <= K <= LANES * CHUNKS * 8, K % 4 == 0): LANES lanes of a wavefront per row, so a workgroup
// takes 256 / LANES rows and no lane idles; the maximum is found inside the lane group.
template <int DT, int LANES, int CHUNKS>
__global__ __launch_bounds__(kThreads) void quantize_rows_subwave(
    const typename Elem<DT>::storage* __restrict__ x, int8_t* __restrict__ codes,
    float* __restrict__ scales, int64_t M, int K, QParams p) {
    constexpr int kRows = kThreads / LANES;
    const int sub = threadIdx.x % LANES;
    const int64_t row = static_cast<int64_t>(blockIdx.x) * kRows + threadIdx.x / LANES;
    const bool live = row < M;  // dead lanes still take part in the butterfly
    const auto* xr = x + (live ? row : 0) * K;
    int8_t* cr = codes + (live ? row : 0) * K;

    float v[CHUNKS][kVec];
    float absmax = 0.0f;
    RawChunk<DT> raw[CHUNKS];
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) raw[c] = load_raw<DT>(xr + chunk_start((c * LANES + sub) * kVec, K));  // as in quantize_rows_cached; dead rows read row 0
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) unpack_chunk<DT>(raw[c], v[c]);
    if (live) {
#pragma unroll
        for (int c = 0; c < CHUNKS; ++c)
#pragma unroll
            for (int i = 0; i < kVec; ++i) absmax = fmaxf(absmax, fabsf(v[c][i]));
    }
    if constexpr (LANES == kWave) {
        absmax = wave_max(absmax);
    } else if constexpr (LANES >= 16) {
        over_16_lanes(absmax, [](float a, float b) { return fmaxf(a, b); });
#pragma unroll
        for (int off = LANES / 2; off >= 16; off >>= 1) absmax = fmaxf(absmax, __shfl_xor(absmax, off));
    } else {
#pragma unroll
        for (int off = LANES / 2; off >= 1; off >>= 1) absmax = fmaxf(absmax, __shfl_xor(absmax, off));
    }
    const RowScale r = scale_of_row(absmax, p);
    if (live && sub == 0) scales[row] = r.scale;

#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
        const int k0 = (c * LANES + sub) * kVec;
        if (live && k0 < K) {
            uint32_t lo, hi;
            quantize_eight(v[c], r, p, lo, hi);
            store_codes(cr + chunk_start(k0, K), lo, hi);
        }
    }
}

// The row quantizer with the preparation of the other operand of the product beside it, in one launch: workgroups 0 .. M - 1 take a row
// of x each, the others the weight.  Codes go to rows of `pitch` bytes, zeros behind K, so that a product whose K is no multiple of
// 16 reads both without a pass that copies them.  CHUNKS * 2048 >= K >= 8, K % 4 == 0.
//
// Two latency chains (load, reduce, store) that need nothing of each other: one after the other they take the sum of both and a gap.
// Measured (us, a launch each / this): training step of 512 rows, 2048 -> 4096 (the two quantizers 4.8 and 9.1) 119.1 / 116.8; of 295 rows,
// 808 -> 3840 (both operands copied to padded rows by a third launch before) 187 / 83, of 43 rows, 928 -> 2960 144 / 84 (host time,
// as it is for 85 us in every small step); int8 linear, quantizer and copies in two launches / this: 142 rows, 3640 -> 1280 38 / 20,
// 500 rows, 1060 -> 3000 33 / 15, 3000 rows, 2500 x 2500 49 / 44.
template <int DT>
struct SecondRows {  // a float matrix [N][K] quantized by rows
    const typename Elem<DT>::storage* w;
    int8_t* codes;
    float* scales;
    QParams p;
};
struct SecondCopy {  // an int8 matrix [N][K], 16-byte chunks of the copy
    const int8_t* w;
    uint4* out;
    int64_t chunks;
};

template <int DT, int CHUNKS, class Second>
__global__ __launch_bounds__(kThreads) void quantize_rows_beside(const typename Elem<DT>::storage* __restrict__ x, int8_t* __restrict__ codes,
                                                                 float* __restrict__ scales, int M, int K, int pitch, QParams p, Second second) {
    __shared__ float smem[kThreads / kWave];
    const bool of_x = blockIdx.x < static_cast<unsigned>(M);
    if constexpr (std::is_same_v<Second, SecondCopy>) {
        if (!of_x) {
            const int chunks_per_row = pitch >> 4;
            const int64_t stride = (gridDim.x - static_cast<unsigned>(M)) * static_cast<int64_t>(kThreads);
            for (int64_t j = (blockIdx.x - static_cast<unsigned>(M)) * static_cast<int64_t>(kThreads) + threadIdx.x; j < second.chunks; j += stride) {
                const int64_t row = j < 0x7FFFFFFF ? static_cast<uint32_t>(j) / static_cast<uint32_t>(chunks_per_row) : j / chunks_per_row;
                const int k = static_cast<int>(j - row * chunks_per_row) * 16;
                second.out[j] = load_k16_ragged(second.w + row * K + k, K - k);
            }
            return;
        }
    }
    const int64_t row = of_x ? blockIdx.x : blockIdx.x - static_cast<unsigned>(M);
    const auto* from = x;
    int8_t* to = codes;
    float* scale_out = scales;
    if constexpr (!std::is_same_v<Second, SecondCopy>) {
        if (!of_x) { from = second.w; to = second.codes; scale_out = second.scales; p = second.p; }
    }
    if (static_cast<int>(threadIdx.x) * 4 < pitch - K) *reinterpret_cast<uint32_t*>(to + row * pitch + K + threadIdx.x * 4) = 0;
    quantize_row_cached<DT, CHUNKS, kThreads>(from + row * K, to + row * pitch, scale_out + row, K, p, smem);
}

template <int DT, class Second>
int launch_beside(const void* x, int64_t M, int64_t K, int64_t pitch, int64_t second_blocks, const QParams& p, const Second& second, int8_t* codes, float* scales,
                  hipStream_t stream) {
    const dim3 grid(static_cast<unsigned>(M + second_blocks));
    auto run = [&](auto chunks) {
        quantize_rows_beside<DT, decltype(chunks)::value, Second><<<grid, kThreads, 0, stream>>>(static_cast<const typename Elem<DT>::storage*>(x), codes, scales,
                                                                                                 static_cast<int>(M), static_cast<int>(K), static_cast<int>(pitch), p, second);
    };
    if (K <= 2048) run(std::integral_constant<int, 1>{});
    else if (K <= 4096) run(std::integral_constant<int, 2>{});
    else if (K <= 8192) run(std::integral_constant<int, 4>{});
    else run(std::integral_constant<int, 8>{});
    return check_launch("tpq_quantize_rowwise (both operands)");
}

// (pitch - K: what 256 threads clear; M + N: a workgroup of 256 threads per row, and a launch holds fewer than 2^32 threads)
inline bool beside_takes(int64_t M, int64_t N, int64_t K, int64_t pitch) {
    return M > 0 && N > 0 && K % 4 == 0 && K >= kVec && K <= 8 * 2048 && pitch >= K && pitch - K < 4 * kThreads && pitch % 16 == 0 && M <= (int64_t{1} << 23) && N <= (int64_t{1} << 23) - 16384;
}

// Any K: two passes over the row with scalar accesses.
template <int DT>
__global__ __launch_bounds__(kThreads) void quantize_rows_streaming(
    const typename Elem<DT>::storage* __restrict__ x, int8_t* __restrict__ codes,
    float* __restrict__ scales, int64_t K, QParams p) {
    __shared__ float smem[kThreads / kWave];
    const int64_t row = blockIdx.x;
    const auto* xr = x + row * K;
    int8_t* cr = codes + row * K;
    float absmax = 0.0f;
    for (int64_t k = threadIdx.x; k < K; k += kThreads) absmax = fmaxf(absmax, fabsf(Elem<DT>::load(xr[k])));
    absmax = block_max<kThreads>(wave_max(absmax), smem);
    const float scale = __fdiv_rn(fmaxf(absmax, p.eps), p.divisor);
    if (threadIdx.x == 0) scales[row] = scale;
    for (int64_t k = threadIdx.x; k < K; k += kThreads)
        cr[k] = static_cast<int8_t>(quantize_one(Elem<DT>::load(xr[k]), scale, p));
}

template <int DT>
int launch(const void* x, int64_t M, int64_t K, const QParams& p, int8_t* codes, float* scales,
           hipStream_t stream) {
    using S = typename Elem<DT>::storage;
    const S* xp = static_cast<const S*>(x);
    const dim3 grid(static_cast<unsigned>(M)), block(kThreads);
    // K % 4 == 0: every row and its last eight elements start on a dword on both sides.  Measured (us, this / the streaming kernel):
    // 256 x 5284 float32 4.4 / 10.8, bfloat16 3.95 / 7.0; 2000 x 4100 11.1 / 16.1 and 9.6 / 14.2; 1 x 2564 float16 2.5 / 4.2.
    const bool vec_ok = K % 4 == 0 && K >= kVec && aligned(x, 16) && aligned(codes, 8) && K <= 8 * 1024 * kVec;
    if (vec_ok && K <= kSubwaveMaxK) {
        const int k = static_cast<int>(K);
        auto run = [&](auto lanes, auto chunks) {
            constexpr int L = decltype(lanes)::value, C = decltype(chunks)::value;
            const dim3 g(static_cast<unsigned>((M + kThreads / L - 1) / (kThreads / L)));
            quantize_rows_subwave<DT, L, C><<<g, block, 0, stream>>>(xp, codes, scales, M, k, p);
        };
        using std::integral_constant;
        if (K <= 64) run(integral_constant<int, 8>{}, integral_constant<int, 1>{});
        else if (K <= 128) run(integral_constant<int, 16>{}, integral_constant<int, 1>{});
        else if (K <= 256) run(integral_constant<int, 32>{}, integral_constant<int, 1>{});
        else if (K <= 512) run(integral_constant<int, 64>{}, integral_constant<int, 1>{});
        else run(integral_constant<int, 64>{}, integral_constant<int, 2>{});
    } else if (vec_ok) {
        const int chunks = static_cast<int>((K + kThreads * kVec - 1) / (kThreads * kVec));
        const int k = static_cast<int>(K);
        if (chunks <= 1) quantize_rows_cached<DT, 1><<<grid, block, 0, stream>>>(xp, codes, scales, k, p);
        else if (chunks <= 2) quantize_rows_cached<DT, 2><<<grid, block, 0, stream>>>(xp, codes, scales, k, p);
        else if (chunks <= 4) quantize_rows_cached<DT, 4><<<grid, block, 0, stream>>>(xp, codes, scales, k, p);
        else if (chunks <= 8) quantize_rows_cached<DT, 8><<<grid, block, 0, stream>>>(xp, codes, scales, k, p);
        else if (chunks <= 16) quantize_rows_cached<DT, 4, 1024><<<grid, 1024, 0, stream>>>(xp, codes, scales, k, p);
        else quantize_rows_cached<DT, 8, 1024><<<grid, 1024, 0, stream>>>(xp, codes, scales, k, p);
    } else {
        quantize_rows_streaming<DT><<<grid, block, 0, stream>>>(xp, codes, scales, K, p);
    }
    return check_launch("tpq_quantize_rowwise");
}

}  // namespace
}  // namespace tpq

#ifdef TPQ_QUANT_STAMPS
// [rows][8] clock readings of the last launch of the register-cached kernel (rows beyond 8192 are not recorded)
TPQ_EXPORT int tpq_quantize_stamps_read(unsigned long long* host, int64_t rows) {
    using namespace tpq;
    TPQ_REQUIRE(host && rows >= 0 && rows <= kStampRows, TPQ_ERR_INVALID_VALUE, "quantize stamps: at most %d rows", kStampRows);
    const hipError_t e = hipMemcpyFromSymbol(host, HIP_SYMBOL(g_quant_stamps), static_cast<size_t>(rows) * kStampSlots * sizeof(unsigned long long));
    TPQ_REQUIRE(e == hipSuccess, TPQ_ERR_RUNTIME, "quantize stamps: %s", hipGetErrorString(e));
    return TPQ_OK;
}
#endif

TPQ_EXPORT int tpq_quantize_rowwise(const void* x, int x_dtype, int64_t M, int64_t K, float eps,
                                    float divisor, int qmin, int qmax, int sign_mode,
                                    int8_t* codes, float* scales, void* stream) {
    using namespace tpq;
    TPQ_REQUIRE(M >= 0 && K >= 0, TPQ_ERR_INVALID_VALUE, "quantize_rowwise: negative shape");
    TPQ_REQUIRE(x_dtype == TPQ_DTYPE_F32 || x_dtype == TPQ_DTYPE_F16 || x_dtype == TPQ_DTYPE_BF16,
                TPQ_ERR_INVALID_TYPE, "rowwise quantize: unsupported input dtype");
    TPQ_REQUIRE(qmin >= -128 && qmax <= 127 && qmin <= qmax && divisor > 0.0f, TPQ_ERR_INVALID_VALUE,
                "quantize_rowwise: code range must fit int8 and divisor must be positive");
    if (M == 0 || K == 0) return TPQ_OK;
    TPQ_REQUIRE(x && codes && scales, TPQ_ERR_INVALID_VALUE, "quantize_rowwise: null pointer");
    TPQ_REQUIRE(M <= 0x7FFFFFFF, TPQ_ERR_INVALID_VALUE, "quantize_rowwise: more than 2^31-1 rows");
    const QParams p = row_quantizer(eps, divisor, qmin, qmax, sign_mode);
    hipStream_t s = static_cast<hipStream_t>(stream);
    switch (x_dtype) {
        case TPQ_DTYPE_F32: return launch<TPQ_DTYPE_F32>(x, M, K, p, codes, scales, s);
        case TPQ_DTYPE_F16: return launch<TPQ_DTYPE_F16>(x, M, K, p, codes, scales, s);
        default: return launch<TPQ_DTYPE_BF16>(x, M, K, p, codes, scales, s);
    }
}

TPQ_EXPORT int tpq_quantize_beside_takes(const void* x, const void* w, int64_t M, int64_t N, int64_t K, int64_t pitch) {
    return tpq::beside_takes(M, N, K, pitch) && tpq::aligned(x, 16) && tpq::aligned(w, 16);
}

TPQ_EXPORT int tpq_quantize_both_rowwise(const void* x, const void* w, int dtype, int64_t M, int64_t N, int64_t K, int64_t pitch, float x_eps, float w_eps,
                                         float w_divisor, int w_qmin, int w_qmax, int w_sign_mode, int8_t* x_codes, float* x_scales, int8_t* w_codes,
                                         float* w_scales, void* stream) {
    using namespace tpq;
    TPQ_REQUIRE(dtype == TPQ_DTYPE_F32 || dtype == TPQ_DTYPE_F16 || dtype == TPQ_DTYPE_BF16, TPQ_ERR_INVALID_TYPE, "rowwise quantize: unsupported input dtype");
    TPQ_REQUIRE(w_qmin >= -128 && w_qmax <= 127 && w_qmin <= w_qmax && w_divisor > 0.0f, TPQ_ERR_INVALID_VALUE, "quantize_both_rowwise: code range must fit int8 and divisor must be positive");
    TPQ_REQUIRE(x && w && x_codes && x_scales && w_codes && w_scales, TPQ_ERR_INVALID_VALUE, "quantize_both_rowwise: null pointer");
    TPQ_REQUIRE(beside_takes(M, N, K, pitch) && aligned(x, 16) && aligned(w, 16) && aligned(x_codes, 16) && aligned(w_codes, 16), TPQ_ERR_UNSUPPORTED,
                "quantize_both_rowwise: K a multiple of 4, 8 .. 16384, operands 16-byte aligned");
    const QParams px = row_quantizer(x_eps, 127.0f, -127, 127, 0), pw = row_quantizer(w_eps, w_divisor, w_qmin, w_qmax, w_sign_mode);
    hipStream_t s = static_cast<hipStream_t>(stream);
    auto run = [&](auto dt) {
        constexpr int DT = decltype(dt)::value;
        return launch_beside<DT>(x, M, K, pitch, N, px, SecondRows<DT>{static_cast<const typename Elem<DT>::storage*>(w), w_codes, w_scales, pw}, x_codes, x_scales, s);
    };
    if (dtype == TPQ_DTYPE_F32) return run(std::integral_constant<int, TPQ_DTYPE_F32>{});
    if (dtype == TPQ_DTYPE_F16) return run(std::integral_constant<int, TPQ_DTYPE_F16>{});
    return run(std::integral_constant<int, TPQ_DTYPE_BF16>{});
}

TPQ_EXPORT int tpq_quantize_rowwise_pad(const void* x, int dtype, int64_t M, int64_t K, float eps, const int8_t* w, int64_t N, int64_t pitch, int8_t* codes,
                                        float* scales, int8_t* w_out, void* stream) {
    using namespace tpq;
    TPQ_REQUIRE(dtype == TPQ_DTYPE_F32 || dtype == TPQ_DTYPE_F16 || dtype == TPQ_DTYPE_BF16, TPQ_ERR_INVALID_TYPE, "rowwise quantize: unsupported input dtype");
    TPQ_REQUIRE(x && w && codes && scales && w_out, TPQ_ERR_INVALID_VALUE, "quantize_rowwise_pad: null pointer");
    TPQ_REQUIRE(beside_takes(M, N, K, pitch) && aligned(x, 16) && aligned(codes, 16) && aligned(w_out, 16), TPQ_ERR_UNSUPPORTED,
                "quantize_rowwise_pad: K a multiple of 4, 8 .. 16384, operands 16-byte aligned");
    const QParams p = row_quantizer(eps, 127.0f, -127, 127, 0);
    const SecondCopy copy{w, reinterpret_cast<uint4*>(w_out), N * (pitch / 16)};
    const int64_t wanted = (copy.chunks + kThreads - 1) / kThreads, blocks = wanted > 16384 ? 16384 : wanted;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (dtype == TPQ_DTYPE_F32) return launch_beside<TPQ_DTYPE_F32>(x, M, K, pitch, blocks, p, copy, codes, scales, s);
    if (dtype == TPQ_DTYPE_F16) return launch_beside<TPQ_DTYPE_F16>(x, M, K, pitch, blocks, p, copy, codes, scales, s);
    return launch_beside<TPQ_DTYPE_BF16>(x, M, K, pitch, blocks, p, copy, codes, scales, s);
}

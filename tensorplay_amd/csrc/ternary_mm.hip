// BitNet b1.58 packed linear: int8 activations x 2-bit packed ternary weights.
//
//   acc[m,n] = sum_k x[m,k] * code[n,k],  code = sign-extended 2-bit field
//   out[m,n] = cast((float(acc) * row_scale[m]) * w_scale (+ bias[n]))
//
// The packed matrix [N, ceil(K/4)] is streamed as it is; no int8 copy of the
// weight is ever materialised (the reference unpacks to int8 on every call,
// tensorplay/ao/quantization/bitnet.py:233).
//
// One row, K % 64 == 0, K <= 8192: the flat dot-product kernel of ternary_row_kernel.h.
// Up to 32 rows with K % 256 == 0: the matrix-core decode kernel of ternary_decode_mfma.h.
//
// Dot-product decode kernel (M <= 8, other K % 64 == 0): one wavefront per 4 weight rows, lane l owns the
// 16-byte chunks l, l+64, ... of each row (64 codes per chunk, 1 KB per
// wavefront load).  For field position q of every byte,
//   f = (w >> (6-2q)) & 0x03030303  are four unsigned codes, and
//   sext(f) = f - 4*(f >> 1), so  sum x*code = dot4(x_q, f) - 4*dot4(x_q, f>>1)
// with x_q the activations of that field position gathered into one register
// (a 4x4 byte transpose of the activation chunk, done once per wavefront and
// reused for its rows).  v_dot4_i32_i8 does the multiply-adds.
//
// More rows: the tile kernel of ternary_gemm_kernel.h (K % 256 == 0), else (K % 16 == 0) the int8
// matrix-core GEMM with a loader that expands the 2-bit chunks to int8 on their way into LDS.
//
// Anything else: one thread per output.
#include <cstdlib>

#include "int8_gemm_kernel.h"
#include "ternary_gemm_kernel.h"
#include "ternary_decode_mfma.h"
#include "ternary_row_kernel.h"
#include "ternary_slab_kernel.h"

namespace tpq {

// int8_gemm.hip: tpq_int8_mm_workspace_bytes and tpq_int8_mm_dequant_ws for a weight that the launch before wrote
int64_t int8_mm_workspace_bytes(int64_t M, int64_t N, int64_t K, bool weight_cached);
int int8_mm_dequant_ws(const int8_t* a, const int8_t* w, const float* row_scale, const float* col_scale, const float* bias, void* out, int out_dtype,
                       int64_t M, int64_t N, int64_t K, void* workspace, int64_t workspace_bytes, void* stream, bool weight_cached);

namespace {

constexpr int kRowsPerWave = 4;

template <int MROWS, class Epilogue>
__global__ __launch_bounds__(256) void ternary_decode_kernel(const int8_t* __restrict__ x,
                                                             const uint8_t* __restrict__ packed,
                                                             int m_base, int N, int K, Epilogue ep) {
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int n0 = wave * kRowsPerWave;
    if (n0 >= N) return;
    const int chunks = K >> 6;  // K % 64 == 0
    const size_t bpr = static_cast<size_t>(K) >> 2;

    int acc_f[kRowsPerWave][MROWS], acc_h[kRowsPerWave][MROWS];
#pragma unroll
    for (int r = 0; r < kRowsPerWave; ++r)
#pragma unroll
        for (int m = 0; m < MROWS; ++m) acc_f[r][m] = acc_h[r][m] = 0;

    for (int chunk = lane; chunk < chunks; chunk += kWave) {
        uint4 w[kRowsPerWave];
#pragma unroll
        for (int r = 0; r < kRowsPerWave; ++r) {
            const int n = n0 + r < N ? n0 + r : N - 1;
            w[r] = *reinterpret_cast<const uint4*>(packed + n * bpr + static_cast<size_t>(chunk) * 16);
        }
        // activations of this chunk, regrouped by field position: xq[m][d][q]
        uint32_t xq[MROWS][4][4];
#pragma unroll
        for (int m = 0; m < MROWS; ++m) {
            const uint4* xp = reinterpret_cast<const uint4*>(x + static_cast<size_t>(m_base + m) * K + static_cast<size_t>(chunk) * 64);
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                const uint4 v = xp[d];
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    xq[m][d][q] = ((v.x >> (8 * q)) & 0xFFu) | (((v.y >> (8 * q)) & 0xFFu) << 8) |
                                  (((v.z >> (8 * q)) & 0xFFu) << 16) | (((v.w >> (8 * q)) & 0xFFu) << 24);
            }
        }
#pragma unroll
        for (int r = 0; r < kRowsPerWave; ++r) {
            const uint32_t wd[4] = {w[r].x, w[r].y, w[r].z, w[r].w};
#pragma unroll
            for (int d = 0; d < 4; ++d)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint32_t f = (wd[d] >> (6 - 2 * q)) & 0x03030303u;
                    const uint32_t h = (wd[d] >> (7 - 2 * q)) & 0x01010101u;
#pragma unroll
                    for (int m = 0; m < MROWS; ++m) {
                        acc_f[r][m] = __builtin_amdgcn_sdot4(static_cast<int>(xq[m][d][q]), static_cast<int>(f), acc_f[r][m], false);
                        acc_h[r][m] = __builtin_amdgcn_sdot4(static_cast<int>(xq[m][d][q]), static_cast<int>(h), acc_h[r][m], false);
                    }
                }
        }
    }
#pragma unroll
    for (int r = 0; r < kRowsPerWave; ++r)
#pragma unroll
        for (int m = 0; m < MROWS; ++m) {
            const int total = wave_sum(acc_f[r][m] - 4 * acc_h[r][m]);
            const int n = n0 + r;
            if (lane == 0 && n < N) ep.store(static_cast<int64_t>(m_base + m) * N + n, m_base + m, n, total);
        }
}

template <class Epilogue>
__global__ __launch_bounds__(256) void ternary_generic_kernel(const int8_t* __restrict__ x,
                                                              const uint8_t* __restrict__ packed,
                                                              int64_t M, int64_t N, int64_t K, Epilogue ep) {
    const int64_t bpr = (K + 3) / 4;
    const int64_t total = M * N;
    for (int64_t idx = blockIdx.x * 256ll + threadIdx.x; idx < total; idx += gridDim.x * 256ll) {
        const int64_t m = idx / N, n = idx - m * N;
        int acc = 0;
        for (int64_t k = 0; k < K; ++k) {
            const uint32_t b = static_cast<uint32_t>(packed[n * bpr + (k >> 2)]) << 24;
            const int code = static_cast<int32_t>(b << (2 * (k & 3))) >> 30;
            acc += static_cast<int>(x[m * K + k]) * code;
        }
        ep.store(idx, static_cast<int>(m), static_cast<int>(n), acc);
    }
}

// ---- the expanded route --------------------------------------------------------------------------------
// The packed weight written out once per call as int8 rows of kp bytes (zeros behind K), the weight's one scale as a column
// of scales, and, where K is no multiple of the tile stage, the activation codes copied to rows of kp bytes as well; the
// int8 GEMM does the rest with the same sums and the same float operations.  It pays where the GEMM's rate is worth more
// than the pass (N K bytes written: 7 us at 2560 x 6912), and wherever K fits none of the packed kernels.  Measured (us,
// expanded / packed kernels): 2560 -> 6912 at 384, 777, 2048 rows 24.5 / 22.3, 31 / 42, 51 / 90; 6912 -> 2560 33 / 21,
// 40 / 45, 45 / 81; 1024 -> 2048 11 / 6, 12.5 / 10.5, 13 / 19.  K that is no multiple of 256 (the tile kernel's stage):
// 1920 -> 5504 at 256 rows 20 / 45; K % 64 != 0, where one thread computed an output: 3412 <-> 7872 at 759 rows (both
// linears) 0.1 ms / 90 ms.
// In the linear, whose row quantizer runs beside the expansion, that is 3 - 5 us less and pays earlier.  Measured with the quantizer (us,
// expanded / packed kernels, weights from HBM, bfloat16; the packed kernels step up behind every 128 rows): 256 rows 2560 -> 6912 23.0 / 20.6,
// 4096 -> 8192 30 / 28.4, 8192 -> 4096 41 / 32; 384 rows 23.6 / 27.7, 32.5 / 40, 38.6 / 46.4, 3072 -> 8192 27.8 / 33.4, but 6912 -> 2560 33 / 28.5,
// 4096 x 4096 26.4 / 26.9; 512 rows 6912 -> 2560 33.7 / 39, 4096 x 4096 28.7 / 29.2, 1024 -> 4096 13.9 / 14.3, 1536 -> 2048 14.5 / 11.1; 640
// rows 1024 -> 4096 15.9 / 19, 4096 x 4096 29.3 / 38.8, 1536 -> 2048 16.4 / 16.1; 1024 rows 2048 -> 1024 16.8 / 13.9.
inline int64_t ternary_padded_k(int64_t K) { return (K + 127) / 128 * 128; }
inline int64_t round_up_256(int64_t v) { return (v + 255) / 256 * 256; }

// The int8 rows come out of the last-level cache, as far as that holds them: the tiles of the product are planned for that.  Planned for a
// weight from HBM / from the caches (us, the linear): 513 rows 5120 -> 11008 80 / 69, 577 rows 8192 -> 11008 116 / 104, 321 rows 11008 ->
// 21760 (240 MB) 216 / 204, 12288 -> 21760 (267 MB) 224 / 218, 11008 -> 28672 (316 MB) 277 / 291.
inline bool expanded_weight_cached(int64_t N, int64_t kp) { return N * kp <= (int64_t{1} << 28); }

struct ExpandedPlan {
    int64_t kp, x_at, scale_at, gemm_at, gemm_bytes, total;  // byte offsets into the workspace, the weight at 0
};
inline ExpandedPlan plan_expanded(int64_t M, int64_t N, int64_t K) {
    ExpandedPlan p;
    p.kp = ternary_padded_k(K);
    p.x_at = round_up_256(N * p.kp);
    p.scale_at = p.x_at + (p.kp == K ? 0 : round_up_256(M * p.kp));
    p.gemm_at = p.scale_at + round_up_256(N * 4);
    p.gemm_bytes = int8_mm_workspace_bytes(M, N, p.kp, expanded_weight_cached(N, p.kp));
    p.total = p.gemm_at + p.gemm_bytes;
    return p;
}

// Does a kernel that reads the packed weight take this shape (operands aligned)?
inline bool ternary_packed_kernel_takes(int64_t M, int64_t N, int64_t K) {
    if (M == 1 && ternary_row_rows_per_workgroup(M, N, K)) return true;
    if (M <= 32) return K % 256 == 0 || (M <= 8 && K % 64 == 0);
    return ternary_slab_splits(M, N, K) >= 1 || K % kTgStage == 0;
}

inline bool ternary_wants_expanded(int64_t M, int64_t N, int64_t K, bool linear) {
    if (M < 1 || N < 1 || K < 1 || M > 0x7FFFFFFF || N > 0x7FFFFFF0 || K > 0x7FFFFF00) return false;
    if (!ternary_packed_kernel_takes(M, N, K)) return true;
    if (const char* e = tuning_env("TPQ_TERNARY_EXPAND")) return M >= std::atoll(e);
    const int64_t weights = N * K;
    if (M >= 1280 || (M > 640 && weights >= (int64_t{1} << 23))) return true;
    return linear && ((M > 512 && weights >= (int64_t{1} << 22)) || (M > 384 && weights >= (int64_t{1} << 24)) ||
                      (M > 256 && (weights >= (int64_t{3} << 23) || (weights >= (int64_t{1} << 24) && N >= 2 * K))));
}

// Chunks first, first + stride, ... of the weight's int8 rows (16 bytes, a packed 32-bit word each).  Rows without padding are one
// flat run of words: no row to find, and four words are requested before the first is written out.
__device__ __forceinline__ void expand_weight(const uint8_t* __restrict__ packed, int64_t chunks_w, int K, int chunks_per_row, int64_t first, int64_t stride,
                                              uint4* __restrict__ w_out) {
    typedef uint32_t word_unaligned __attribute__((aligned(1)));
    if (chunks_per_row * 16 == K) {
        const word_unaligned* const words = reinterpret_cast<const word_unaligned*>(packed);
        for (int64_t i = first; i < chunks_w; i += 4 * stride) {
            uint32_t word[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) word[j] = words[i + j * stride < chunks_w ? i + j * stride : i];
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (i + j * stride < chunks_w) w_out[i + j * stride] = ternary_word_to_i8x16(word[j]);
        }
        return;
    }
    const int64_t bpr = (K + 3) >> 2;
    for (int64_t i = first; i < chunks_w; i += stride) {
        const int64_t row = i < 0x7FFFFFFF ? static_cast<uint32_t>(i) / static_cast<uint32_t>(chunks_per_row) : i / chunks_per_row;
        const int k = static_cast<int>(i - row * chunks_per_row) * 16, left = K - k;
        uint4 codes = make_uint4(0, 0, 0, 0);
        if (left >= 16) {
            codes = ternary_word_to_i8x16(*reinterpret_cast<const word_unaligned*>(packed + row * bpr + (k >> 2)));
        } else if (left > 0) {
            uint32_t word = 0;
            for (int b = 0; 4 * b < left; ++b) {
                uint32_t byte = packed[row * bpr + (k >> 2) + b];
                const int live = left - 4 * b;  // codes of this byte inside the row
                if (live < 4) byte &= 0xFFu << (8 - 2 * live);
                word |= (byte & 0xFFu) << (8 * b);
            }
            codes = ternary_word_to_i8x16(word);
        }
        w_out[i] = codes;
    }
}

// the weight and its scales, then the activation codes in rows of chunks_per_row chunks (if x_out)
__global__ __launch_bounds__(256) void ternary_expand_kernel(const uint8_t* __restrict__ packed, const int8_t* __restrict__ x, int64_t chunks_w,
                                                             int64_t chunks_x, int N, int K, int chunks_per_row, float w_scale, uint4* __restrict__ w_out,
                                                             uint4* __restrict__ x_out, float* __restrict__ scales) {
    const int64_t first = blockIdx.x * 256ll + threadIdx.x, stride = gridDim.x * 256ll;
    for (int64_t i = first; i < N; i += stride) scales[i] = w_scale;
    expand_weight(packed, chunks_w, K, chunks_per_row, first, stride, w_out);
    for (int64_t i = first; i < chunks_x; i += stride) {
        const int64_t row = i < 0x7FFFFFFF ? static_cast<uint32_t>(i) / static_cast<uint32_t>(chunks_per_row) : i / chunks_per_row;
        const int k = static_cast<int>(i - row * chunks_per_row) * 16;
        x_out[i] = load_k16_ragged(x + row * K + k, K - k);
    }
}

// workgroups that write the weight out: four chunks a thread
inline unsigned expand_blocks(int64_t chunks) {
    const int64_t blocks = (chunks + 1023) / 1024;
    return static_cast<unsigned>(blocks > 16384 ? 16384 : blocks);
}

// The row quantizer and the expansion in one launch: neither needs the other, and each by itself leaves the chip waiting (a row is a
// round trip, a reduction and a write; the expansion 7 us of stores).  Workgroups 0 .. M - 1 quantize a row each, straight into rows of
// kp bytes (what lies behind K meets the weight's zeros), the others expand.  CHUNKS * 2048 >= K >= 8, K % 4 == 0.
template <int DT, int CHUNKS>
__global__ __launch_bounds__(256) void ternary_quantize_expand_kernel(const typename Elem<DT>::storage* __restrict__ x, int M, int K, int kp, QParams p,
                                                                      int8_t* __restrict__ codes, float* __restrict__ row_scales,
                                                                      const uint8_t* __restrict__ packed, int64_t chunks_w, int N, float w_scale,
                                                                      uint4* __restrict__ w_out, float* __restrict__ scales) {
    __shared__ float smem[4];
    if (blockIdx.x < static_cast<unsigned>(M)) {
        const int64_t row = blockIdx.x;
        quantize_row_cached<DT, CHUNKS, 256>(x + row * K, codes + row * kp, row_scales + row, K, p, smem);
        return;
    }
    const int64_t first = (blockIdx.x - static_cast<unsigned>(M)) * 256ll + threadIdx.x, stride = (gridDim.x - static_cast<unsigned>(M)) * 256ll;
    for (int64_t i = first; i < N; i += stride) scales[i] = w_scale;
    expand_weight(packed, chunks_w, K, kp / 16, first, stride, w_out);
}

// (a workgroup of 256 threads per row: a launch holds fewer than 2^32 threads)
constexpr int64_t kQuantizeExpandMaxK = 8 * 2048, kQuantizeExpandMaxRows = int64_t{1} << 23;

template <int DT>
int launch_quantize_expand(const void* x, int64_t M, int64_t N, int64_t K, const ExpandedPlan& p, const QParams& q, int8_t* codes, float* row_scales,
                           const uint8_t* packed, float w_scale, int8_t* w8, float* scales, hipStream_t s) {
    const int64_t chunks_w = N * (p.kp / 16);
    const dim3 grid(static_cast<unsigned>(M) + expand_blocks(chunks_w));
    auto run = [&](auto chunks) {
        ternary_quantize_expand_kernel<DT, decltype(chunks)::value><<<grid, 256, 0, s>>>(
            static_cast<const typename Elem<DT>::storage*>(x), static_cast<int>(M), static_cast<int>(K), static_cast<int>(p.kp), q, codes, row_scales, packed, chunks_w,
            static_cast<int>(N), w_scale, reinterpret_cast<uint4*>(w8), scales);
    };
    if (K <= 2048) run(std::integral_constant<int, 1>{});
    else if (K <= 2 * 2048) run(std::integral_constant<int, 2>{});
    else if (K <= 4 * 2048) run(std::integral_constant<int, 4>{});
    else run(std::integral_constant<int, 8>{});
    return check_launch("tpq_ternary_linear (quantize, expand)");
}

// the int8 product of rows of kp codes with the weight written out in the workspace
int multiply_expanded(const int8_t* x, const float* row_scale, const float* bias, int64_t M, int64_t N, void* out, int out_dtype, const ExpandedPlan& p,
                      char* ws, hipStream_t s) {
    return int8_mm_dequant_ws(x, reinterpret_cast<const int8_t*>(ws), row_scale, reinterpret_cast<const float*>(ws + p.scale_at), bias, out, out_dtype, M, N, p.kp,
                              p.gemm_bytes ? ws + p.gemm_at : nullptr, p.gemm_bytes, s, expanded_weight_cached(N, p.kp));
}

int launch_ternary_expanded(const int8_t* x, const float* row_scale, const uint8_t* packed, float w_scale, const float* bias, int64_t M, int64_t N,
                            int64_t K, void* out, int out_dtype, const ExpandedPlan& p, void* workspace, hipStream_t s) {
    char* const ws = static_cast<char*>(workspace);
    const bool copy_x = p.kp != K;
    const int64_t chunks_w = N * (p.kp / 16), chunks_x = copy_x ? M * (p.kp / 16) : 0;
    int8_t* const w8 = reinterpret_cast<int8_t*>(ws);
    int8_t* const x8 = reinterpret_cast<int8_t*>(ws + p.x_at);
    float* const scales = reinterpret_cast<float*>(ws + p.scale_at);
    ternary_expand_kernel<<<expand_blocks(chunks_w + chunks_x), 256, 0, s>>>(
        packed, x, chunks_w, chunks_x, static_cast<int>(N), static_cast<int>(K), static_cast<int>(p.kp / 16), w_scale, reinterpret_cast<uint4*>(w8),
        reinterpret_cast<uint4*>(x8), scales);
    if (int rc = check_launch("tpq_ternary_mm (expand)")) return rc;
    return multiply_expanded(copy_x ? x8 : x, row_scale, bias, M, N, out, out_dtype, p, ws, s);
}

template <class Epilogue>
int launch_ternary(const int8_t* x, const uint8_t* packed, int64_t M, int64_t N, int64_t K,
                   Epilogue ep, hipStream_t s, void* workspace, int64_t workspace_bytes) {
    const bool sizes_ok = M <= 0x7FFFFFFF && N <= 0x7FFFFFFF && K <= 0x7FFFFFFF;
    // the tile kernel below takes over where it is faster and its shape conditions hold
    // Measured at 2560 -> 6912 / 6912 -> 2560 (216 / 80 tiles of 32 channels): the decode kernel takes 7, 7.5, 9.4, 11.4 us
    // for 1..4 rows and twice that for 5..8, the tile kernel 9.3 / 18.3 us for any row count up to 128.
    static const int forced_decode_rows = [] { const char* e = tuning_env("TPQ_TERNARY_DECODE_ROWS"); return e ? std::atoi(e) : -1; }();
    // ... and stays ahead of the 256 x 128-tile kernel at every larger row count tried (512 rows: 30 / 33 us against
    // 54 / 103 us; 2048 rows: 100 / 85 us against 111 / 112 us), so there is no upper limit by default.
    static const int64_t gemm_rows = [] { const char* e = tuning_env("TPQ_TERNARY_GEMM_ROWS"); return e ? std::atoll(e) : int64_t{1} << 40; }();
    const int decode_rows = forced_decode_rows >= 0 ? forced_decode_rows : ((N + kTgN - 1) / kTgN >= 128 ? 3 : 6);
    // Up to 32 rows, in slabs of 16: the weight streamed once per slab through the matrix cores.  Measured against the
    // kernels below over K, N = 1024..28672: one row 4.3..19.8 us (the dot-product kernel 4.7..19.2), 16 rows
    // 5.2..29.6 us (the tile kernel 9.3..75 us for any row count up to 128; two slabs stay below it, three do not).
    static const int mfma_min = [] { const char* e = tuning_env("TPQ_TERNARY_MFMA_MIN"); return e ? std::atoi(e) : 1; }();
    static const int mfma_rows = [] { const char* e = tuning_env("TPQ_TERNARY_MFMA_ROWS"); return e ? std::atoi(e) : 32; }();
    // One row, K up to 8192: the flat dot-product kernel (every wave-level load 1 KB of whole lines)
    if (forced_decode_rows < 0 && M == 1 && aligned(x, 16) && aligned(packed, 16) && !tuning_env("TPQ_TERNARY_NO_ROW")) {
        if (const int rows_wg = ternary_row_rows_per_workgroup(M, N, K)) return launch_ternary_row(x, packed, N, K, rows_wg, ep, s);
    }
    if (forced_decode_rows < 0 && M >= mfma_min && M <= mfma_rows && ternary_decode_mfma_ok(x, packed, M, N, K))
        return launch_ternary_decode_mfma(x, packed, M, N, K, ep, s);
    // 33 rows and more: the slab kernel (every load of a workgroup in flight at once); K beyond 2560 is split and
    // needs the caller's workspace for the exact partial sums
    if (forced_decode_rows < 0 && !tuning_env("TPQ_TERNARY_NO_SLAB") && aligned(x, 16) && aligned(packed, 16)) {
        const int splits = ternary_slab_splits(M, N, K);
        const bool room = splits == 1 || (workspace != nullptr && aligned(workspace, 16) && workspace_bytes >= static_cast<int64_t>(splits) * M * N * 4);
        if (splits >= 1 && room) return launch_ternary_slab(x, packed, M, N, K, splits, static_cast<int32_t*>(workspace), ep, s);
    }
    const bool gemm_ok = sizes_ok && M <= gemm_rows && K % kTgStage == 0 && aligned(x, 16) && aligned(packed, 4);
    if (sizes_ok && M <= 8 && (M <= decode_rows || !gemm_ok) && K % 64 == 0 && aligned(x, 16) && aligned(packed, 16)) {
        const int waves = static_cast<int>((N + kRowsPerWave - 1) / kRowsPerWave);
        const dim3 grid((waves + 3) / 4);
        for (int m0 = 0; m0 < M; m0 += 4) {
            const int rows = static_cast<int>(M - m0 < 4 ? M - m0 : 4);
            switch (rows) {
                case 1: ternary_decode_kernel<1, Epilogue><<<grid, 256, 0, s>>>(x, packed, m0, (int)N, (int)K, ep); break;
                case 2: ternary_decode_kernel<2, Epilogue><<<grid, 256, 0, s>>>(x, packed, m0, (int)N, (int)K, ep); break;
                case 3: ternary_decode_kernel<3, Epilogue><<<grid, 256, 0, s>>>(x, packed, m0, (int)N, (int)K, ep); break;
                default: ternary_decode_kernel<4, Epilogue><<<grid, 256, 0, s>>>(x, packed, m0, (int)N, (int)K, ep); break;
            }
        }
        return check_launch("tpq_ternary_mm (decode)");
    }
    if (gemm_ok) return launch_ternary_gemm_m128(x, packed, M, N, K, ep, s);
    if (sizes_ok && K % 16 == 0 && aligned(x, 16) && aligned(packed, 4))
        return launch_mfma<true>(x, packed, M, N, K, ep, s);
    const int64_t blocks = (M * N + 255) / 256;
    ternary_generic_kernel<Epilogue><<<static_cast<unsigned>(blocks > 65535 ? 65535 : blocks), 256, 0, s>>>(
        x, packed, M, N, K, ep);
    return check_launch("tpq_ternary_mm (generic)");
}

}  // namespace
}  // namespace tpq

using namespace tpq;

namespace tpq {
namespace {
// Does the row quantizer go with the expansion?  (its codes and x are aligned as allocations are)
inline bool quantize_expand_takes(int64_t M, int64_t K) { return K % 4 == 0 && K >= kVec && K <= kQuantizeExpandMaxK && M <= kQuantizeExpandMaxRows; }

inline int64_t ternary_workspace_bytes(int64_t M, int64_t N, int64_t K, bool linear) {
    if (ternary_wants_expanded(M, N, K, linear)) return plan_expanded(M, N, K).total;
    const int splits = M > 0 && N > 0 && K > 0 ? ternary_slab_splits(M, N, K) : 0;
    return splits > 1 ? static_cast<int64_t>(splits) * M * N * 4 : 0;
}
}  // namespace
}  // namespace tpq

TPQ_EXPORT int64_t tpq_ternary_mm_workspace_bytes(int64_t M, int64_t N, int64_t K) { return ternary_workspace_bytes(M, N, K, false); }

TPQ_EXPORT int64_t tpq_ternary_linear_workspace_bytes(int64_t M, int64_t N, int64_t K) { return ternary_workspace_bytes(M, N, K, quantize_expand_takes(M, K)); }

TPQ_EXPORT int tpq_ternary_mm(const int8_t* x, const float* row_scale, const uint8_t* packed,
                              float w_scale, const float* bias, int64_t M, int64_t N, int64_t K,
                              void* out, int out_dtype, int32_t* acc_out, void* stream) {
    return tpq_ternary_mm_ws(x, row_scale, packed, w_scale, bias, M, N, K, out, out_dtype, acc_out, nullptr, 0, stream);
}

TPQ_EXPORT int tpq_ternary_mm_ws(const int8_t* x, const float* row_scale, const uint8_t* packed,
                                 float w_scale, const float* bias, int64_t M, int64_t N, int64_t K,
                                 void* out, int out_dtype, int32_t* acc_out, void* workspace, int64_t workspace_bytes,
                                 void* stream) {
    TPQ_REQUIRE(M >= 0 && N >= 0 && K >= 0, TPQ_ERR_INVALID_VALUE, "bitnet_linear_packed: negative shape");
    TPQ_REQUIRE(out_dtype == TPQ_DTYPE_F32 || out_dtype == TPQ_DTYPE_F16 || out_dtype == TPQ_DTYPE_BF16,
                TPQ_ERR_INVALID_TYPE, "bitnet_linear_packed: unsupported output dtype");
    if (M == 0 || N == 0) return TPQ_OK;
    TPQ_REQUIRE(out || acc_out, TPQ_ERR_INVALID_VALUE, "bitnet_linear_packed: no destination");
    TPQ_REQUIRE((K == 0 || (x && packed)) && (!out || row_scale), TPQ_ERR_INVALID_VALUE,
                "bitnet_linear_packed: null pointer");
    hipStream_t s = static_cast<hipStream_t>(stream);
    // (the raw sums are an output of the packed kernels only)
    if (workspace != nullptr && !acc_out && K > 0 && aligned(workspace, 16) && aligned(x, 16) && ternary_wants_expanded(M, N, K, false)) {
        const ExpandedPlan plan = plan_expanded(M, N, K);
        if (workspace_bytes >= plan.total)
            return launch_ternary_expanded(x, row_scale, packed, w_scale, bias, M, N, K, out, out_dtype, plan, workspace, s);
    }
    switch (out_dtype) {
        case TPQ_DTYPE_F32: {
            const EpilogueTernary<TPQ_DTYPE_F32> ep{static_cast<float*>(out), acc_out, row_scale, bias, w_scale};
            return launch_ternary(x, packed, M, N, K, ep, s, workspace, workspace_bytes);
        }
        case TPQ_DTYPE_F16: {
            const EpilogueTernary<TPQ_DTYPE_F16> ep{static_cast<uint16_t*>(out), acc_out, row_scale, bias, w_scale};
            return launch_ternary(x, packed, M, N, K, ep, s, workspace, workspace_bytes);
        }
        default: {
            const EpilogueTernary<TPQ_DTYPE_BF16> ep{static_cast<uint16_t*>(out), acc_out, row_scale, bias, w_scale};
            return launch_ternary(x, packed, M, N, K, ep, s, workspace, workspace_bytes);
        }
    }
}

TPQ_EXPORT int tpq_ternary_linear(const void* x, int x_dtype, const uint8_t* packed, float w_scale, const float* bias, int64_t M, int64_t N,
                                  int64_t K, float eps, int8_t* codes, float* row_scales, float* out, void* workspace, int64_t workspace_bytes,
                                  void* stream) {
    TPQ_REQUIRE(M > 0 && N > 0 && K > 0 && x && packed && codes && row_scales && out, TPQ_ERR_INVALID_VALUE, "ternary_linear: empty shape or null pointer");
    TPQ_REQUIRE(x_dtype == TPQ_DTYPE_F32 || x_dtype == TPQ_DTYPE_F16 || x_dtype == TPQ_DTYPE_BF16, TPQ_ERR_INVALID_TYPE, "ternary_linear: unsupported input dtype");
    if (workspace != nullptr && aligned(workspace, 16) && aligned(x, 16) && aligned(codes, 16) && quantize_expand_takes(M, K) &&
        ternary_wants_expanded(M, N, K, true)) {
        const ExpandedPlan plan = plan_expanded(M, N, K);
        if (workspace_bytes >= plan.total) {
            char* const ws = static_cast<char*>(workspace);
            int8_t* const w8 = reinterpret_cast<int8_t*>(ws);
            int8_t* const x8 = plan.kp == K ? codes : reinterpret_cast<int8_t*>(ws + plan.x_at);
            float* const scales = reinterpret_cast<float*>(ws + plan.scale_at);
            hipStream_t s = static_cast<hipStream_t>(stream);
            const QParams quantizer = row_quantizer(eps, 127.0f, -127, 127, 0);
            const auto launch = x_dtype == TPQ_DTYPE_F32 ? launch_quantize_expand<TPQ_DTYPE_F32> : x_dtype == TPQ_DTYPE_F16 ? launch_quantize_expand<TPQ_DTYPE_F16> : launch_quantize_expand<TPQ_DTYPE_BF16>;
            if (int rc = launch(x, M, N, K, plan, quantizer, x8, row_scales, packed, w_scale, w8, scales, s)) return rc;
            return multiply_expanded(x8, row_scales, bias, M, N, out, TPQ_DTYPE_F32, plan, ws, s);
        }
    }
    if (int rc = tpq_quantize_rowwise(x, x_dtype, M, K, eps, 127.0f, -127, 127, 0, codes, row_scales, stream)) return rc;
    return tpq_ternary_mm_ws(codes, row_scales, packed, w_scale, bias, M, N, K, out, TPQ_DTYPE_F32, nullptr, workspace, workspace_bytes, stream);
}

TPQ_EXPORT int tpq_ternary_linear_row(const void* x, int x_dtype, const uint8_t* packed, float w_scale, const float* bias, int64_t N, int64_t K,
                                      float eps, float* out, void* stream) {
    TPQ_REQUIRE(x_dtype == TPQ_DTYPE_F32 || x_dtype == TPQ_DTYPE_F16 || x_dtype == TPQ_DTYPE_BF16, TPQ_ERR_INVALID_TYPE, "ternary_linear_row: unsupported input dtype");
    TPQ_REQUIRE(x && packed && out, TPQ_ERR_INVALID_VALUE, "ternary_linear_row: null pointer");
    const int rows_wg = ternary_row_rows_per_workgroup(1, N, K);
    TPQ_REQUIRE(rows_wg > 0 && aligned(x, 16) && aligned(packed, 16), TPQ_ERR_UNSUPPORTED, "ternary_linear_row: K must be a multiple of 64 up to %d, operands 16-byte aligned", kTernaryRowMaxK);
    const EpilogueTernary<TPQ_DTYPE_F32> ep{out, nullptr, nullptr, bias, w_scale};
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (x_dtype == TPQ_DTYPE_F32) return launch_ternary_row<TPQ_DTYPE_F32>(x, packed, N, K, rows_wg, ep, s, eps);
    if (x_dtype == TPQ_DTYPE_F16) return launch_ternary_row<TPQ_DTYPE_F16>(x, packed, N, K, rows_wg, ep, s, eps);
    return launch_ternary_row<TPQ_DTYPE_BF16>(x, packed, N, K, rows_wg, ep, s, eps);
}

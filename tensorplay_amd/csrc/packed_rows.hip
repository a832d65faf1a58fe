// Entry points of the packed-weight products for a block of activation rows (packed_rows_kernel.h).
#include <algorithm>

#include "int4_gemm_kernel.h"
#include "packed_rows_bits.h"

namespace tpq {
namespace {

// int4 device layout
template <int DT>
int run_int4(const PackedRowsArgs& a, const PackedRowsPlan& p, hipStream_t s) { return launch_packed_rows<DT, SourceInt4>(a, p, s); }

// Between the decode kernels and the dense route.  Upper limit, measured (us, this kernel / what runs above it, groups of 128, weights
// from HBM): float16, N < 16384: up to 2^24 weights, 768 rows of 4096 x 4096 30 / 44, 1024 rows 41 / 47; up to 2^26, 512 rows of 4096 ->
// 11008 66 / 67, 8192 x 8192 71 / 102, 14336 -> 4096 69 / 111, 768 rows 109 / 122 and 91 / 119; beyond, 384 rows of 5120 -> 13824 69 /
// 98, 512 rows 90 / 100.  Wider weights, 4096 -> 32000: 256, 384, 512 rows 81 / 112, 120 / 137, 158 / 154; bfloat16 384 and 512 rows
// 119 / 172, 155 / 182.  So the lines lie where a tile of 64 rows, which this kernel had when they were drawn, stopped paying; with the
// tiles of up to 128 rows the first rows above most of them are the shorter ones here too.  float32: 192 rows of 4096 -> 11008 217 / 228,
// 4096 -> 16384 257 / 251, at 256 rows of the first 256 / 222.  K that is no multiple of 128 has the narrow tiles only: 4768 -> 13544 at 192
// rows 111, at 256 150 (float32 at 96 rows 185 / 182, at 128 258 / 215).
int64_t rows_limit(int64_t N, int64_t K, int dtype) {
    if (dtype == TPQ_DTYPE_F32) return K % 128 ? 96 : 192;
    if (K % 128) return 192;
    if (N >= 16384) return dtype == TPQ_DTYPE_F16 ? 256 : 384;
    return N * K <= (int64_t{1} << 24) ? 768 : N * K <= (int64_t{1} << 26) ? 512 : 384;
}

// Where the kernels that take any K or (groups of 128) the decode kernels on the matrix cores ran: they keep the weight in float32
// or apply the scales to sums of whole codes.  With groups of 32 and 64 the latter dequantize to 16 bits, as the tiled kernel and
// the dense route above those rows do.
bool int4_weights_unrounded(int dtype, int64_t M, int64_t N, int64_t K, int64_t group) {
    if (dtype == TPQ_DTYPE_F32) return false;
    if (K % 128) return dtype == TPQ_DTYPE_F16 || M <= 112 || N >= 16384;
    return group == 128 && !int4_gemm_takes(M, N, K, ~size_t{0});
}

// n-bit rows: the kernel's offsets into the weight and into the (scale, zero) pairs are 32-bit.  The pairs are the larger tensor with
// few bits and short groups (1 bit in groups of 32: twice the weight).
bool lowbit_offsets_fit(int64_t N, int64_t K, int bits, int64_t group) {
    return N * K / (8 / bits) < (int64_t{1} << 32) && K / group * N * 8 <= (int64_t{1} << 32);
}

}  // namespace
}  // namespace tpq

using namespace tpq;

// Lower limit, measured (us, this kernel / decode kernels): groups of 128 (weights unrounded): 24 rows of 4096 -> 16384 17.5 / 15.4,
// 33 of 4096 x 4096 10.8 / 15.1, 48 of 4096 -> 11008 18.5 / 20.2; groups of 64, 17 rows:
// 11008 -> 4096 12.0 / 23.1, 16 rows 11.3 / 12.0.  K % 128 != 0 (slabs of four rows): 4768 -> 13544 at 3 / 33 rows 19.4 /
// 92, 31 / 868.  float32, all rows (up to eight in blocks of four): one row of 2048 x 2048
// 5.7 / 7.2, 4096 x 4096 9.2 / 14.3, 8192 x 8192 15.5 / 29.5, 4768 -> 1264 6.8 / 15.2, 1024 x 1024 4.4 / 4.7 (in a graph); 4096 -> 11008 at 2
// and 64 rows 15 / 45, 68 / 110.  bfloat16 stops at 256 rows although this kernel is the faster one beyond (384 rows of 8192 x 8192 52 / 104, 512 of
// 4096 x 4096 24 / 42): from 257 rows on the results are those of the dense route, the reference's device formulation with a weight
// rounded to bfloat16 twice, and are held to it within 1e-2, element by element, by tests.  A weight rounded once lies closer to
// the exact product and misses that on single elements; below 257 rows, where the tiled kernel and the slabs ran, the comparison
// is with the exact product.
// Operands off the alignment that the kernel wants stay with the kernels that take any address.
TPQ_EXPORT int tpq_int4_mm_rows_takes(const void* x, int dtype, int64_t M, int64_t N, int64_t K, int64_t group, const int32_t* packed,
                                      const void* scales_and_zeros) {
    if (M <= 0 || N <= 0 || K <= 0 || K % 32 || N % 8 || N * K >= (int64_t{1} << 33) || K >= (1 << 24) || M > rows_limit(N, K, dtype)) return 0;
    if (!aligned(x, 16) || !aligned(packed, 16) || !aligned(scales_and_zeros, dtype == TPQ_DTYPE_F32 ? 8 : 4)) return 0;
    if (dtype == TPQ_DTYPE_BF16 && M > 256) return 0;
    if (dtype == TPQ_DTYPE_F32) return 1;
    if (K % 128) return 1;
    return M >= (group < 128 ? 17 : 33);
}

// Lower limit, measured (us, this kernel with unrounded weights / what ran below): groups of 128, where the decode kernels are at
// home: 4096 x 4096 at 19 rows, 1 / 2 / 4 / 8 bits 10.7 / 10.0, 10.8 / 10.5, 11.4 / 11.9, 13.1 / 16.9; 4096 -> 11008, 2 bits, 24 / 32 /
// 40 rows 21.7 / 20.6, 21.6 / 21.5, 20 / 31; 1024 -> 512 at 18 rows 7.3 / 6.0.  Other groups, 4096 x 4096 in groups of 32, 2 bits:
// 1 / 16 / 80 rows 10.1 / 25, 10.4 / 46, 17.6 / 175; one row of 4 bits stays with the row kernel (8.6 / 6.1).  float32
// 4096 -> 11008: 8 / 64 rows 26 / 57, 84 / 99.  8 bits are twice the bytes: 4096 -> 11008 at 300 rows 75 / 86, at
// 384 81 / 85, at 512 90 / 84; 4096 x 4096 at 512 31 / 42.
TPQ_EXPORT int tpq_lowbit_mm_rows_takes(const void* x, int dtype, int64_t M, int64_t N, int64_t K, int bits, int lsb_first, int64_t group,
                                        const uint8_t* packed, const float* scales_and_zeros) {
    if (M <= 0 || N <= 0 || K <= 0 || group <= 0 || (bits != 1 && bits != 2 && bits != 4 && bits != 8) || (lsb_first && bits != 1)) return 0;
    if (K % 32 || group % 32 || N % 4 || !lowbit_offsets_fit(N, K, bits, group) || K >= (1 << 24)) return 0;
    if (!aligned(x, 16) || !aligned(packed, 16) || !aligned(scales_and_zeros, 8)) return 0;
    int64_t limit = rows_limit(N, K, dtype);
    if (bits == 8 && dtype != TPQ_DTYPE_F32) {
        const int64_t wide = N * K <= (int64_t{1} << 24) ? 512 : 300;
        limit = limit < wide ? limit : wide;
    }
    if (M > limit) return 0;
    if (dtype == TPQ_DTYPE_F32) return 1;
    const int64_t step = bits == 8 ? 64 : 128, steps = group / step;
    const bool at_home = K % step == 0 && group % step == 0 && (steps & (steps - 1)) == 0;
    if (M == 1) {
        const int64_t chunk = bits == 8 ? 16 : bits == 4 ? 32 : 64;
        const bool row_kernel = K % chunk == 0 && group % chunk == 0 && K <= (bits == 8 ? 32768 : 65536) && (bits != 8 || dtype == TPQ_DTYPE_F16);
        return !(at_home || row_kernel);
    }
    return M >= (bits == 8 ? 17 : 33) || !at_home;
}

static PackedRowsPlan int4_rows_plan(int dtype, int64_t M, int64_t N, int64_t K, int64_t group, int64_t room_floats) {
    return packed_rows_plan(dtype, M, N, K, room_floats, int4_weights_unrounded(dtype, M, N, K, group) ? kRowsUnrounded : kRowsRounded);
}

static int64_t slices_bytes(const PackedRowsPlan& p, int64_t M, int64_t N) { return p.slices > 1 ? static_cast<int64_t>(p.slices) * M * N * 4 : 0; }

TPQ_EXPORT int64_t tpq_packed_rows_workspace_bytes(int dtype, int64_t M, int64_t N, int64_t K) {
    return M <= 0 || N <= 0 || K <= 0 ? 0 : slices_bytes(packed_rows_plan(dtype, M, N, K, kRowsAnyRoom), M, N);
}

TPQ_EXPORT int64_t tpq_lowbit_mm_rows_workspace_bytes(int dtype, int64_t M, int64_t N, int64_t K) {  // of any width: those that cost alike
    return std::max(tpq_packed_rows_call_workspace_bytes(dtype, M, N, K, 1, 32), tpq_packed_rows_call_workspace_bytes(dtype, M, N, K, 8, 32));
}

// The plan of a call (bits 0: the int4 layout): what the launches below go by, so a workspace of its size is what they cut k for.
static PackedRowsPlan call_plan(int dtype, int64_t M, int64_t N, int64_t K, int bits, int64_t group, int64_t room_floats) {
    return bits == 0 ? int4_rows_plan(dtype, M, N, K, group, room_floats) : packed_rows_plan(dtype, M, N, K, room_floats, lowbit_rows_weights(M, N, K, bits), bits);
}

TPQ_EXPORT int64_t tpq_packed_rows_call_workspace_bytes(int dtype, int64_t M, int64_t N, int64_t K, int bits, int64_t group) {
    return M <= 0 || N <= 0 || K <= 0 ? 0 : slices_bytes(call_plan(dtype, M, N, K, bits, group, kRowsAnyRoom), M, N);
}

TPQ_EXPORT int tpq_packed_rows_call_plan(int dtype, int64_t M, int64_t N, int64_t K, int bits, int64_t group, int64_t workspace_bytes, int32_t* plan) {
    TPQ_REQUIRE(M > 0 && N > 0 && K > 0 && plan, TPQ_ERR_INVALID_VALUE, "packed_rows_call_plan: bad shape or null pointer");
    const PackedRowsPlan p = call_plan(dtype, M, N, K, bits, group, workspace_bytes < 0 ? kRowsAnyRoom : workspace_bytes / 4);
    plan[0] = p.quads == 0 ? TPQ_ROWS_STAGED : p.cw == 0 ? TPQ_ROWS_LANES : TPQ_ROWS_QUADS;
    plan[1] = p.quads ? 4 * p.quads : 16 * p.mb;
    plan[2] = p.quads && p.cw == 0 ? kWave : 32 * p.cw;
    plan[3] = p.slices;
    return TPQ_OK;
}

TPQ_EXPORT int tpq_packed_rows_tile_rows(int dtype, int64_t M, int64_t N, int64_t K) {
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    const PackedRowsPlan p = packed_rows_plan(dtype, M, N, K, kRowsAnyRoom);
    return p.quads ? 4 * p.quads : 16 * p.mb;
}

TPQ_EXPORT int tpq_int4_mm_rows(const void* x, int dtype, int64_t M, int64_t K, const int32_t* packed, int64_t N, int64_t group,
                                const void* scales_and_zeros, void* out, void* workspace, int64_t workspace_bytes, void* stream) {
    return tpq_int4_mm_rows_bias(x, dtype, M, K, packed, N, group, scales_and_zeros, nullptr, out, workspace, workspace_bytes, stream);
}

TPQ_EXPORT int tpq_int4_mm_rows_bias(const void* x, int dtype, int64_t M, int64_t K, const int32_t* packed, int64_t N, int64_t group,
                                     const void* scales_and_zeros, const void* bias, void* out, void* workspace, int64_t workspace_bytes,
                                     void* stream) {
    TPQ_REQUIRE(dtype == TPQ_DTYPE_F32 || dtype == TPQ_DTYPE_F16 || dtype == TPQ_DTYPE_BF16, TPQ_ERR_INVALID_TYPE, "int4_mm_rows: unsupported activation dtype");
    TPQ_REQUIRE(M >= 0 && N >= 0 && K >= 0 && N % 8 == 0, TPQ_ERR_INVALID_VALUE, "int4_mm_rows: bad shape");
    TPQ_REQUIRE(group == 32 || group == 64 || group == 128, TPQ_ERR_INVALID_VALUE, "int4_mm_rows: qGroupSize must be 32, 64 or 128");
    if (M == 0 || N == 0) return TPQ_OK;
    TPQ_REQUIRE(K > 0 && K % 32 == 0 && K < (1 << 24) && M < (1 << 22) && N * K / 2 < (int64_t{1} << 32), TPQ_ERR_UNSUPPORTED, "int4_mm_rows: K must be a positive multiple of 32, the weight below 4 GB");
    TPQ_REQUIRE(x && packed && scales_and_zeros && out, TPQ_ERR_INVALID_VALUE, "int4_mm_rows: null pointer");
    const bool wide = dtype == TPQ_DTYPE_F32;
    TPQ_REQUIRE(aligned(x, 16) && aligned(packed, 16) && aligned(scales_and_zeros, wide ? 8 : 4) && aligned(out, wide ? 16 : 8) && aligned(bias, wide ? 4 : 2), TPQ_ERR_UNSUPPORTED,
                "int4_mm_rows: unaligned operand");
    const bool room = workspace != nullptr && aligned(workspace, 16);
    const PackedRowsPlan p = int4_rows_plan(dtype, M, N, K, group, room ? workspace_bytes / 4 : 0);
    if (p.quads)
        return packed_rows_f32({x, packed, scales_and_zeros, nullptr, bias, out, workspace, M, N, K, group, 0, 0, 0, static_cast<hipStream_t>(stream)}, p.quads, p.cw,
                                 p.slices, p.steps_per_slice);
    PackedRowsArgs a{};
    a.x = x; a.w = packed; a.sz = scales_and_zeros; a.y = out; a.after = bias; a.partial = static_cast<float*>(workspace);
    a.M = static_cast<int>(M); a.N = static_cast<int>(N); a.K = static_cast<int>(K); a.tiles_per_group = static_cast<int>(group / 32);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (dtype == TPQ_DTYPE_F32) return run_int4<TPQ_DTYPE_F32>(a, p, s);
    if (dtype == TPQ_DTYPE_F16) return run_int4<TPQ_DTYPE_F16>(a, p, s);
    return run_int4<TPQ_DTYPE_BF16>(a, p, s);
}

TPQ_EXPORT int tpq_lowbit_mm_rows(const void* x, int dtype, int64_t M, int64_t K, const uint8_t* packed, int bits, int lsb_first,
                                  int64_t N, int64_t group, const float* scales_and_zeros, const float* bias, void* out,
                                  void* workspace, int64_t workspace_bytes, void* stream) {
    TPQ_REQUIRE(dtype == TPQ_DTYPE_F32 || dtype == TPQ_DTYPE_F16 || dtype == TPQ_DTYPE_BF16, TPQ_ERR_INVALID_TYPE, "lowbit_mm_rows: unsupported activation dtype");
    TPQ_REQUIRE(M >= 0 && N >= 0 && K >= 0 && group > 0 && K % group == 0, TPQ_ERR_INVALID_VALUE, "lowbit_mm_rows: bad shape");
    TPQ_REQUIRE(lsb_first == 0 || lsb_first == 1, TPQ_ERR_INVALID_VALUE, "lowbit_mm_rows: lsb_first must be 0 or 1");
    if (M == 0 || N == 0) return TPQ_OK;
    TPQ_REQUIRE((bits == 1 || bits == 2 || bits == 4 || bits == 8) && (!lsb_first || bits == 1 || bits == 8), TPQ_ERR_UNSUPPORTED,
                "lowbit_mm_rows: 1, 2, 4 or 8 bits, first code in the most significant bits (1 bit: either order)");
    TPQ_REQUIRE(K > 0 && K % 32 == 0 && group % 32 == 0 && N % 4 == 0 && K < (1 << 24) && M < (1 << 22) && lowbit_offsets_fit(N, K, bits, group), TPQ_ERR_UNSUPPORTED,
                "lowbit_mm_rows: K and the group must be multiples of 32, N of 4, the weight below 4 GB and the (scale, zero) pairs within it");
    TPQ_REQUIRE(x && packed && scales_and_zeros && out, TPQ_ERR_INVALID_VALUE, "lowbit_mm_rows: null pointer");
    TPQ_REQUIRE(aligned(x, 16) && aligned(packed, 16) && aligned(scales_and_zeros, 8) && aligned(out, dtype == TPQ_DTYPE_F32 ? 16 : 8), TPQ_ERR_UNSUPPORTED,
                "lowbit_mm_rows: unaligned operand");
    const bool room = workspace != nullptr && aligned(workspace, 16);
    const PackedRowsBits call{x, packed, scales_and_zeros, bias, nullptr, out, workspace, M, N, K, group, room ? workspace_bytes / 4 : 0, bits, lsb_first,
                              static_cast<hipStream_t>(stream)};
    if (dtype == TPQ_DTYPE_F32) return packed_rows_bits_f32(call);
    return dtype == TPQ_DTYPE_F16 ? packed_rows_bits_f16(call) : packed_rows_bits_bf16(call);
}

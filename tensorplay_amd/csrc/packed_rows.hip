// Entry points of the packed-weight products for a block of activation rows (packed_rows_kernel.h).
#include "packed_rows_bits.h"

namespace tpq {
namespace {

// int4 device layout
template <int DT>
int run_int4(const PackedRowsArgs& a, const PackedRowsPlan& p, hipStream_t s) { return launch_packed_rows<DT, SourceInt4>(a, p, s); }

}  // namespace
}  // namespace tpq

using namespace tpq;

TPQ_EXPORT int64_t tpq_packed_rows_workspace_bytes(int dtype, int64_t M, int64_t N, int64_t K) {
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    const PackedRowsPlan p = packed_rows_plan(dtype, M, N, K, int64_t{1} << 60);
    return p.slices > 1 ? static_cast<int64_t>(p.slices) * M * N * 4 : 0;
}

TPQ_EXPORT int tpq_int4_mm_rows(const void* x, int dtype, int64_t M, int64_t K, const int32_t* packed, int64_t N, int64_t group,
                                const void* scales_and_zeros, void* out, void* workspace, int64_t workspace_bytes, void* stream) {
    TPQ_REQUIRE(dtype == TPQ_DTYPE_F32 || dtype == TPQ_DTYPE_F16 || dtype == TPQ_DTYPE_BF16, TPQ_ERR_INVALID_TYPE, "int4_mm_rows: unsupported activation dtype");
    TPQ_REQUIRE(M >= 0 && N >= 0 && K >= 0 && N % 8 == 0, TPQ_ERR_INVALID_VALUE, "int4_mm_rows: bad shape");
    TPQ_REQUIRE(group == 32 || group == 64 || group == 128, TPQ_ERR_INVALID_VALUE, "int4_mm_rows: qGroupSize must be 32, 64 or 128");
    if (M == 0 || N == 0) return TPQ_OK;
    TPQ_REQUIRE(K > 0 && K % 32 == 0 && K < (1 << 24) && M < (1 << 22) && N * K / 2 < (int64_t{1} << 32), TPQ_ERR_UNSUPPORTED, "int4_mm_rows: K must be a positive multiple of 32, the weight below 4 GB");
    TPQ_REQUIRE(x && packed && scales_and_zeros && out, TPQ_ERR_INVALID_VALUE, "int4_mm_rows: null pointer");
    const bool wide = dtype == TPQ_DTYPE_F32;
    TPQ_REQUIRE(aligned(x, 16) && aligned(packed, 16) && aligned(scales_and_zeros, wide ? 8 : 4) && aligned(out, wide ? 16 : 8), TPQ_ERR_UNSUPPORTED,
                "int4_mm_rows: unaligned operand");
    const bool room = workspace != nullptr && aligned(workspace, 16);
    const PackedRowsPlan p = packed_rows_plan(dtype, M, N, K, room ? workspace_bytes / 4 : 0);
    PackedRowsArgs a{};
    a.x = x; a.w = packed; a.sz = scales_and_zeros; a.y = out; a.partial = static_cast<float*>(workspace);
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
    TPQ_REQUIRE(K > 0 && K % 32 == 0 && group % 32 == 0 && N % 4 == 0 && K < (1 << 24) && M < (1 << 22) && N * K / (8 / bits) < (int64_t{1} << 32), TPQ_ERR_UNSUPPORTED,
                "lowbit_mm_rows: K and the group must be multiples of 32, N of 4");
    TPQ_REQUIRE(x && packed && scales_and_zeros && out, TPQ_ERR_INVALID_VALUE, "lowbit_mm_rows: null pointer");
    TPQ_REQUIRE(aligned(x, 16) && aligned(packed, 16) && aligned(scales_and_zeros, 8) && aligned(out, dtype == TPQ_DTYPE_F32 ? 16 : 8), TPQ_ERR_UNSUPPORTED,
                "lowbit_mm_rows: unaligned operand");
    const bool room = workspace != nullptr && aligned(workspace, 16);
    const PackedRowsBits call{x, packed, scales_and_zeros, bias, out, workspace, M, N, K, group, room ? workspace_bytes / 4 : 0, bits, lsb_first,
                              static_cast<hipStream_t>(stream)};
    if (dtype == TPQ_DTYPE_F32) return packed_rows_bits_f32(call);
    return dtype == TPQ_DTYPE_F16 ? packed_rows_bits_f16(call) : packed_rows_bits_bf16(call);
}

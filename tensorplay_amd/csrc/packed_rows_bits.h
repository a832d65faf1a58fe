// Call of the n-bit packed product for a block of activation rows, between its entry point and the translation units of
// the activation types.
#pragma once

#include "packed_rows_kernel.h"

namespace tpq {

struct PackedRowsBits {
    const void *x, *packed, *sz;
    const float* bias;  // (n-bit rows)
    const void* after;  // (int4)
    void *out, *workspace;
    int64_t M, N, K, group, room_floats;
    int bits, lsb_first;  // 0 bits: the int4 layout
    hipStream_t stream;
};

int packed_rows_bits_f32(const PackedRowsBits& call);
int packed_rows_bits_f16(const PackedRowsBits& call);
int packed_rows_bits_bf16(const PackedRowsBits& call);
int packed_rows_f32(const PackedRowsBits& call, int quads, int cw, int slices, int steps_per_slice);  // float32, the kernels without LDS for the activations

namespace {

// up to these rows the decode kernels ran, which apply the scales to sums of whole codes: no weight is rounded to 16 bits; above, the
// dense route's 16-bit weight
inline RowsWeights lowbit_rows_weights(int64_t M, int64_t N, int64_t K, int bits) {
    return M <= (N * K <= (int64_t{1} << 24) ? 80 : 56) ? kRowsUnroundedBits : bits == 8 ? kRowsRoundedBytes : kRowsRoundedBits;
}

template <int DT>
int run_packed_rows_bits(const PackedRowsBits& c) {
    const PackedRowsPlan p = packed_rows_plan(DT, c.M, c.N, c.K, c.room_floats, lowbit_rows_weights(c.M, c.N, c.K, c.bits), c.bits);
    if constexpr (DT == TPQ_DTYPE_F32)
        if (p.quads) return packed_rows_f32(c, p.quads, p.cw, p.slices, p.steps_per_slice);
    PackedRowsArgs a{};
    a.x = c.x; a.w = c.packed; a.sz = c.sz; a.bias = c.bias; a.y = c.out; a.partial = static_cast<float*>(c.workspace);
    a.M = static_cast<int>(c.M); a.N = static_cast<int>(c.N); a.K = static_cast<int>(c.K); a.tiles_per_group = static_cast<int>(c.group / 32);
    switch (c.bits) {
        case 1: return c.lsb_first ? launch_packed_rows<DT, SourceBits<1, true>>(a, p, c.stream) : launch_packed_rows<DT, SourceBits<1, false>>(a, p, c.stream);
        case 2: return launch_packed_rows<DT, SourceBits<2, false>>(a, p, c.stream);
        case 4: return launch_packed_rows<DT, SourceBits<4, false>>(a, p, c.stream);
        default: return launch_packed_rows<DT, SourceBits<8, false>>(a, p, c.stream);  // one code per byte: the bit order does not matter
    }
}

}  // namespace
}  // namespace tpq

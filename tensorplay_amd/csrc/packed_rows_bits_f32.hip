// The n-bit packed product for a block of activation rows, float32 activations (one translation unit per type: they are
// many kernels).
#include "packed_rows_bits.h"

namespace tpq {

int packed_rows_bits_f32(const PackedRowsBits& call) { return run_packed_rows_bits<TPQ_DTYPE_F32>(call); }

}  // namespace tpq

// The n-bit packed product for a block of activation rows, bfloat16 activations (one translation unit per type: they are
// many kernels).
#include "packed_rows_bits.h"

namespace tpq {

int packed_rows_bits_bf16(const PackedRowsBits& call) { return run_packed_rows_bits<TPQ_DTYPE_BF16>(call); }

}  // namespace tpq

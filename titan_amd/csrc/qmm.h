// Batched dense quantized matmul (qmm.hip), for qmoe_quantized_matmul.
#pragma once

#include "common.h"

namespace qmoe_qmm {

// Does the batched kernel take M rows of this shape?  (The caller has checked
// K against the group size, the pointers and their alignment.)
bool takes(int64_t M, int64_t N, int64_t K, int group_size, int bits);

int launch(const uint16_t* x, int64_t M, int64_t K, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
           int64_t N, int group_size, int bits, uint16_t* out, hipStream_t st);

}  // namespace qmoe_qmm

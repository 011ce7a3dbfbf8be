// gemm256.h -- the many-row Q8 GEMM (gemm256.hip), called from madi_q8_gemm.
#pragma once

#include "common.h"

namespace madi {

// Whether the shape takes the 256 x 256 tiles.
bool gemm256_suits(uint32_t m, uint32_t n, uint32_t k);
// The array that holds the dequantised weight during a call, on the current
// device; nullptr if its address is not to be had.  It holds nothing else: the
// split-K partials of a captured call, replayed on a stream of its own, must
// not meet an eager call's weight.  Calls that use it are ordered by the
// library's one stream.
f16 *gemm256_weight();
// Operands checked by madi_q8_gemm.
int gemm256(const void *a, const uint8_t *qs, const f16 *sc, void *c, const float *bias, uint32_t m,
            uint32_t n, uint32_t k, int epilogue, f16 *w);

}  // namespace madi

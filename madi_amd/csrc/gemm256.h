// gemm256.h -- the many-row Q8 GEMM (gemm256.hip), called from madi_q8_gemm.
#pragma once

#include "common.h"

namespace madi {

// Whether the shape takes the 256 x 256 tiles, with at most max_scratch bytes
// of scratch memory (16-byte aligned) for its dequantised weight, and how
// many it needs.
bool gemm256_suits(uint32_t m, uint32_t n, uint32_t k, size_t max_scratch);
size_t gemm256_bytes(uint32_t n, uint32_t k);
// Operands checked by madi_q8_gemm.
int gemm256(const void *a, const uint8_t *qs, const f16 *sc, void *c, const float *bias, uint32_t m,
            uint32_t n, uint32_t k, int epilogue, void *w16);

}  // namespace madi

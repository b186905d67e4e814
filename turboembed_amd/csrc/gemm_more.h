// The GEMM launchers that gemm.hip's dispatch takes from other sources.
#pragma once

#include "gemm_tile.h"

namespace rocm {

// K shared among a workgroup's waves, on 32 x 32 output tiles
// (gemm_direct.hip): F32, F16 and BF16 operands, K and lda multiples of 16
// bytes.
hipError_t gemm_direct(hipStream_t s, Dt dt, const GemmRows &gr, int M, int N, int K, const void *A, int lda,
                       const void *W, const EpiArgs &e);

// Whether the rule takes a product of at most M rows there.
bool gemm_is_direct(Dt dt, int M, int N, int K, const EpiArgs &e);

// F32 operands as three BF16 terms each (gemm_f32.hip), on 64 x 64 output
// tiles or (wide) 128 x 128 ones: K and lda multiples of 4.
hipError_t gemm_f32_split(hipStream_t s, bool wide, const GemmRows &gr, int M, int N, int K, const void *A, int lda,
                          const void *W, const EpiArgs &e);

}  // namespace rocm

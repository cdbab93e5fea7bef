// smoe_gemm_small.h — host entry of the grouped GEMM for few rows per expert
// (smoe_gemm_small.hip), called by the GEMM entry points after they have
// checked their arguments.
#pragma once

#include "smoe_common.h"

namespace smoe {

enum class SmallWeights { kPacked, kPlain };

// Whether a grouped GEMM of R rows over E experts, [N, K = Kdim] weights, takes
// the small-row kernel (N = 2I in the fused SwiGLU form).
bool small_gemm_rows(SmallWeights lay, bool e8m0, bool swiglu, int E, int R, int N, int Kdim);

// The GEMM (hq == nullptr: c [R, N]) or, with hq, the fc1 GEMM with SwiGLU +
// 1x128 requantisation (N = 2I; c1 into c when c is not null).  e8m0: every
// scale is a power of two, applied by the MFMA (packed weights only).
int small_gemm_launch(SmallWeights lay, bool e8m0, const uint8_t* a, const float* as,
                      const uint8_t* b, const float* bs, const int32_t* offsets, int E, int R,
                      int N, int Kdim, uint16_t* c, uint8_t* hq, float* hs, hipStream_t stream);

}  // namespace smoe

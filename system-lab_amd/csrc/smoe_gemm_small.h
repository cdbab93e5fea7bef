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

// Its column tiles are 64 times this many columns wide.
int small_gemm_cols(bool swiglu, int E, int R, int N);

// Whether the 256-row kernels should skip the empty 16-row blocks of an
// expert's last tile (kShort): the launch has more than one round of 256 x 256
// tiles, NT column tiles wide (in one round the fullest tile decides, and the
// longer code costs 3 - 5%), and the experts few enough rows that short tiles are
// a share of them.  lo, hi: rows per expert between which hardly any tile is
// short; to: the highest average measured to gain.
inline bool short_tiles(int E, int R, long long NT, int lo, int hi, int to) {
  const long long r = R;
  return (r / 256 + E / 2) * NT >= 256 && r <= (long long)to * E && (r <= (long long)lo * E || r >= (long long)hi * E);
}

// The GEMM (hq == nullptr: c [R, N]) or, with hq, the fc1 GEMM with SwiGLU +
// 1x128 requantisation (N = 2I; c1 into c when c is not null).  e8m0: every
// scale is a power of two, applied by the MFMA (packed weights only).
int small_gemm_launch(SmallWeights lay, bool e8m0, const uint8_t* a, const float* as,
                      const uint8_t* b, const float* bs, const int32_t* offsets, int E, int R,
                      int N, int Kdim, uint16_t* c, uint8_t* hq, float* hs, hipStream_t stream);

}  // namespace smoe

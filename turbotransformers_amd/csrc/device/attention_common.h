// What the one-kernel attention forms (attention.hip, attention_f32.hip, attention_split.hip) share: masks and scores far
// from zero.
#pragma once

#include <cfloat>

#include "common.h"

namespace ttmi {

// Scores are kept in raw units: q . k + mask / scale, and a probability is 2^(s * c - m * c) with c = scale * log2(e), one
// multiply-add, m the running maximum.  A wholly masked row is the mean of V, as a softmax over mask + score gives it, so
// the mask of a valid key stays finite however low it is (the lowest float over the scale would be -inf, every probability
// of such a row 0 and the row 0 / 0), and keys past the end carry -inf, below any mask.  A mask of -inf stays -inf.
constexpr float kFarthestScore = 0x1p127f;  // the running maximum starts at its negative
__device__ __forceinline__ float mask_in_scores(float mask, float inv_scale) {
  const float x = mask * inv_scale;
  return fabsf(mask) <= FLT_MAX ? fminf(fmaxf(x, -kFarthestScore), kFarthestScore) : x;
}

// m * c is rounded.  The error is the same for all keys of a row and cancels in the division by the row's sum, but from
// |m * c| = 2^30 on it is 64 and more: the probabilities of a row masked with -1e10 would be 0 or infinite.  Beyond 2^12
// (error 2^-13; no row with an unmasked key comes near) the maximum is subtracted from the scores first, exactly.
// The test is three instructions per 32 keys: us per launch without / with it, 12 heads, fp16 64 x 512 tokens 83.8 / 83.0, 8 x
// 256 7.6 / 7.7, 1 x 387 6.8 / 6.8, fp32 1 x 128 6.5 / 6.5, 20 x 100 14.8 / 14.8, 16 x 512 147.2 / 148.1.
template <typename Scores>
__device__ __forceinline__ float relative_scores(Scores& st, float m_run, float scale_log2e) {
  const float neg_m = -m_run * scale_log2e;
  const bool far = fabsf(neg_m) > 0x1p12f;
  if (__builtin_expect(!__any(far), 1)) return neg_m;
  const float shift = far ? m_run : 0.f;
#pragma unroll
  for (int e = 0; e < 16; ++e) st[e] -= shift;
  return far ? 0.f : neg_m;
}

}  // namespace ttmi

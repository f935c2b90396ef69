// fp32 Flat scores from bf16 x 3 splits formed in the score kernel (flat_resident.hip).
#pragma once
#include "coarse.h"

namespace ixa {

// Whether launch_resident_f32 has a kernel for rows of d numbers.
bool resident_f32_serves(int d);

// Scores of nq row-major queries against nb row-major base rows (nb >= 1), approximately: the products of the operands' bf16 x 3
// splits, accumulated in fp32 from -|b|^2 / 2 (score = |q|^2 - 2 u) or from 0 (inner product, score = -u).  Every base element
// must be finite, and bn readable up to a multiple of four rows.
//   filter = false: out[row * ldo + col] = score
//   filter = true:  scores <= flt.tau[row] are appended to flt.cand[row][flt.cnt[row]++] as keys (score, flt.col_base + col)
// Returns false, with nothing launched, for dimensions without a kernel and for operands that are not 16-byte aligned.
bool launch_resident_f32(const float *Q, int64_t nq, const float *B, int64_t nb, int d, const float *qn, const float *bn,
                         int metric, float *out, int64_t ldo, bool filter, ScoreFilter<float> flt, hipStream_t s);

}  // namespace ixa

// fp32 scores from bf16 x 3 splits formed in the score kernel (resident_f32.hip): Flat search and assignment to centroids.
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

// The centroids as the assignment kernel reads them: relative to a centre (about their mean), so that what vectors and centroids
// have in common does not widen its error bound.
struct AssignCentroids {
    DeviceBuffer<float> centre;   // [d]
    DeviceBuffer<float> rows;     // [nc][d]
    DeviceBuffer<float> norms;    // [nc]
    float longest = 0.f;          // the largest |c - centre|
    void borrow(const AssignCentroids &o)
    {
        centre.borrow(o.centre);
        rows.borrow(o.rows);
        norms.borrow(o.norms);
        longest = o.longest;
    }
};
// cn: canonical squared norms.  lengths[nc] (device): |c - centre|^2, from which the caller sets `longest`.
void launch_centre_centroids(const float *C, int64_t nc, int d, const float *cn, AssignCentroids &out, float *lengths, hipStream_t s);

// out[i] = the centroid with the smallest canonical L2 score of vector i (the smallest number among equal ones; -1 where every
// score is a NaN).  The score kernel keeps each tile's best two centroids and its third value per vector, so nothing of the
// n x nc scores is written; what its error bound cannot decide is decided by canonical scores, all on the stream, with nothing
// for the host to read.  cn: canonical squared norms; cmax: the largest centroid length; scratch: memory that nothing queued behind
// the call relies on, resized to at most scratch_bytes (or what 256 vectors take).
bool resident_assign_serves(const float *X, const float *C, int64_t nc, int d);
bool resident_assign_pays(int64_t n, int64_t nc, int d);
void launch_resident_assign(const float *X, int64_t n, const float *C, int64_t nc, int d, const float *cn, float cmax,
                            const AssignCentroids &centred, int32_t *out, DeviceBuffer<float> &scratch, int64_t scratch_bytes,
                            hipStream_t s);

}  // namespace ixa

// Host launchers of the product-quantizer kernels (codeword norms, exact encode).
#pragma once
#include "common.h"

namespace ixa {

// codes[i][m] = first argmin_k sum_t (x[i][m*dsub+t] - codebook[m][k][t])^2, fp32, left to right.
void launch_pq_encode(const float *x, int64_t n, int d, int M, const float *codebook, uint8_t *codes, hipStream_t s);

// ---- training of sub-quantizers -----------------------------------------------------------------------------
// Sub-vectors m0 .. m0 + M - 1 of a sample x [ns][d], sub-vector-major: out[(m * ns + i) * dsub + t].
void launch_pq_subvectors(const float *x, int64_t ns, int d, int m0, int M, int dsub, float *out, hipStream_t s);
// launch_pq_encode on such sub-vectors; codes[m * ns + i].
void launch_pq_encode_subvectors(const float *subs, int64_t ns, int M, int dsub, const float *codebook, uint8_t *codes,
                                 hipStream_t s);
struct PqUpdateWorkspace {
    DeviceBuffer<uint32_t> starts;   // [M][chunks][256]
    DeviceBuffer<uint32_t> first;    // [M][257]: first member of every codeword in `order`
    DeviceBuffer<uint32_t> order;    // [M][ns]: the samples of every codeword, in sample order
};
// One Lloyd update of M codebooks [M][256][dsub]: every codeword with members becomes their mean, the sum taken in
// float64 in sample order; cnt[m][k] = its number of members.
void launch_pq_update(const float *subs, const uint8_t *codes, int64_t ns, int M, int dsub, float *codebook,
                      unsigned long long *cnt, PqUpdateWorkspace &ws, hipStream_t s);

}  // namespace ixa

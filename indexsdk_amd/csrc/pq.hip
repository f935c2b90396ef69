// PQ encode on the GPU, bit-exact to the reference's host encoder
// (FR/ascend/impl/AscendIndexIVFPQImpl.cpp:879-921: encodeSingleVectorPQ /
// findCentroidInSubQuantizer / calDistance): the RAW vector is encoded (by_residual = false),
// distance = sum (a-b)^2 accumulated left to right in fp32 without FMA, strict '<' so the first
// minimum wins.  This is plain VALU work: the arithmetic order is the contract, so it is not
// reshaped into a GEMM.
#include "pq.h"

#include <algorithm>

namespace ixa {

// One workgroup finds the codes of 256 vectors for ONE sub-quantizer (blockIdx.y): its 256 x dsub codeword
// slab is staged in LDS and every lane walks all 256 codewords for its own vector (all lanes read the same
// LDS address per step: a broadcast, no bank conflicts).  A small batch still fills the GPU this way: the
// walk is a serial chain per lane, and 10000 vectors x 32 sub-quantizers are 1280 workgroups instead of 40.
//
// Sub-vector m of vector i starts at x + i * xi + m * xm, its code is codes[i * ci + m * cm].
struct PqStrides {
    int64_t xi, xm, ci, cm;
};

template <int DSUB>
__global__ __launch_bounds__(256) void pq_encode_kernel(const float *__restrict__ x, int64_t n, PqStrides st,
                                                        const float *__restrict__ codebook,
                                                        uint8_t *__restrict__ codes)
{
    __shared__ float cb[256 * DSUB];
    const int tid = threadIdx.x;
    const int m = blockIdx.y;
    const int64_t i = (int64_t)blockIdx.x * 256 + tid;
    const float *src = codebook + (int64_t)m * 256 * DSUB;
    for (int e = tid; e < 256 * DSUB; e += 256) {
        cb[e] = src[e];
    }
    __syncthreads();
    if (i < n) {
        float sub[DSUB];
#pragma unroll
        for (int t = 0; t < DSUB; t++) {
            sub[t] = x[i * st.xi + m * st.xm + t];
        }
        float best = 3.402823466e+38f;
        int arg = 0;
        for (int k = 0; k < 256; k++) {
            float dist = 0.f;
#pragma unroll
            for (int t = 0; t < DSUB; t++) {
                float diff = __fsub_rn(sub[t], cb[k * DSUB + t]);
                dist = __fadd_rn(dist, __fmul_rn(diff, diff));
            }
            if (dist < best) {
                best = dist;
                arg = k;
            }
        }
        codes[i * st.ci + m * st.cm] = (uint8_t)arg;
    }
}

// Any dsub: the sub-vector is re-read from global memory (cached) instead of living in registers.
__global__ __launch_bounds__(256) void pq_encode_generic_kernel(const float *__restrict__ x, int64_t n, PqStrides st,
                                                                int dsub, const float *__restrict__ codebook,
                                                                uint8_t *__restrict__ codes)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int m = blockIdx.y;
    if (i >= n) {
        return;
    }
    const float *sub = x + i * st.xi + m * st.xm;
    const float *cb = codebook + (int64_t)m * 256 * dsub;
    float best = 3.402823466e+38f;
    int arg = 0;
    for (int k = 0; k < 256; k++) {
        float dist = 0.f;
        for (int t = 0; t < dsub; t++) {
            float diff = __fsub_rn(sub[t], cb[k * dsub + t]);
            dist = __fadd_rn(dist, __fmul_rn(diff, diff));
        }
        if (dist < best) {
            best = dist;
            arg = k;
        }
    }
    codes[i * st.ci + m * st.cm] = (uint8_t)arg;
}

namespace {

void launch_encode(const float *x, int64_t n, int M, int dsub, PqStrides st, const float *codebook, uint8_t *codes,
                   hipStream_t s)
{
    if (n == 0) {
        return;
    }
    dim3 grid((unsigned)((n + 255) / 256), (unsigned)M), block(256);
#define IXA_ENC(D)                                                                                             \
    case D:                                                                                                    \
        hipLaunchKernelGGL(pq_encode_kernel<D>, grid, block, 0, s, x, n, st, codebook, codes);                \
        break;
    switch (dsub) {
        IXA_ENC(1)
        IXA_ENC(2)
        IXA_ENC(3)
        IXA_ENC(4)
        IXA_ENC(5)
        IXA_ENC(6)
        IXA_ENC(8)
        IXA_ENC(10)
        IXA_ENC(12)
        IXA_ENC(16)
        IXA_ENC(24)
        IXA_ENC(32)
        default:
            hipLaunchKernelGGL(pq_encode_generic_kernel, grid, block, 0, s, x, n, st, dsub, codebook, codes);
    }
#undef IXA_ENC
}

// ---- training -------------------------------------------------------------------------------------------------------

// 64 rows x C columns (whole sub-vectors, C <= 64) through LDS: read along the rows, written along the sub-vectors, both
// in whole lines (read straight from the rows, a 16-byte sub-vector would fetch 128 bytes).
__global__ __launch_bounds__(256) void pq_subvectors_kernel(const float *__restrict__ x, int64_t ns, int d, int m0, int M,
                                                            int dsub, int per_tile, float *__restrict__ out)
{
    __shared__ float tile[64][65];
    const int mt = blockIdx.y * per_tile;   // first sub-vector of the tile, counted from m0
    const int nm = M - mt < per_tile ? M - mt : per_tile, cols = nm * dsub;
    const int64_t i0 = (int64_t)blockIdx.x * 64;
    const int rows = (int)(ns - i0 < 64 ? ns - i0 : 64);
    const float *src = x + i0 * d + (int64_t)(m0 + mt) * dsub;
    for (int r = threadIdx.x >> 6; r < rows; r += 4) {
        const int c = threadIdx.x & 63;
        if (c < cols) {
            tile[r][c] = src[(int64_t)r * d + c];
        }
    }
    __syncthreads();
    for (int m = 0; m < nm; m++) {
        float *dst = out + ((int64_t)(mt + m) * ns + i0) * dsub;
        for (int e = threadIdx.x; e < rows * dsub; e += 256) {
            dst[e] = tile[e / dsub][m * dsub + e % dsub];
        }
    }
}

// sub-vectors of more than 64 components: their rows are whole lines as they stand
__global__ __launch_bounds__(256) void pq_subvectors_long_kernel(const float *__restrict__ x, int64_t ns, int d, int m0,
                                                                 int dsub, float *__restrict__ out)
{
    const int m = blockIdx.y;
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e < ns * dsub) {
        const int64_t i = e / dsub;
        out[(int64_t)m * ns * dsub + e] = x[i * d + (int64_t)(m0 + m) * dsub + (e - i * dsub)];
    }
}

// A Lloyd update needs, for every (sub-quantizer, codeword), the sum of its samples' sub-vectors in float64 and in
// sample order.  The samples are first sorted by code, stably: `chunks` pieces of the sample are counted by one
// wavefront each, the counts turned into starting positions, and the same wavefronts place their samples (64 at a time,
// ranked among equal codes by ballots).  Then every component of every codeword is one lane's chain of additions over
// a list it reads ahead of, which is what bounds the update (the latency of two dependent L2 reads per 16 additions).
// 131072 samples x 32 sub-quantizers of 4 components: count 7, starts 11, place 41, means 99 us per update.  One
// workgroup per sub-quantizer walking the whole sample for all 256 codewords (M workgroups on the GPU, 256 comparisons
// per sample) took 8.7 ms.
__device__ __forceinline__ unsigned long long same_code_lanes(int code, bool valid)
{
    unsigned long long mask = __builtin_amdgcn_ballot_w64(valid);
#pragma unroll
    for (int b = 0; b < 8; b++) {
        const bool bit = (code >> b) & 1;
        const unsigned long long set = __builtin_amdgcn_ballot_w64(bit);
        mask &= bit ? set : ~set;
    }
    return mask;
}

// counts[(m * chunks + c) * 256 + code]
__global__ __launch_bounds__(256) void pq_count_kernel(const uint8_t *__restrict__ codes, int64_t ns, int chunk, int chunks,
                                                       uint32_t *__restrict__ counts)
{
    __shared__ uint32_t n[4][256];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, m = blockIdx.y;
    const int c = blockIdx.x * 4 + wave;
#pragma unroll
    for (int k = lane; k < 256; k += 64) {
        n[wave][k] = 0;
    }
    __syncthreads();
    const uint8_t *src = codes + (int64_t)m * ns;
    const int64_t b = (int64_t)c * chunk, e = b + chunk < ns ? b + chunk : ns;
    for (int64_t i = b + lane; i < e; i += 64) {
        atomicAdd(&n[wave][src[i]], 1u);
    }
    __syncthreads();
    if (c < chunks) {
        for (int k = lane; k < 256; k += 64) {
            counts[((int64_t)m * chunks + c) * 256 + k] = n[wave][k];
        }
    }
}

// counts become positions in the sub-quantizer's `order`; first[m][k] = start of codeword k, first[m][256] = ns
__global__ __launch_bounds__(256) void pq_starts_kernel(uint32_t *__restrict__ counts, int chunks,
                                                        uint32_t *__restrict__ first, unsigned long long *__restrict__ cnt)
{
    __shared__ uint32_t part[256];
    const int m = blockIdx.x, k = threadIdx.x;
    uint32_t *mine = counts + (int64_t)m * chunks * 256 + k;
    uint32_t sum = 0;
#pragma unroll 8
    for (int c = 0; c < chunks; c++) {
        sum += mine[(int64_t)c * 256];
    }
    part[k] = sum;
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {
        const uint32_t add = k >= off ? part[k - off] : 0;
        __syncthreads();
        part[k] += add;
        __syncthreads();
    }
    uint32_t run = part[k] - sum;
    first[m * 257 + k] = run;
    if (k == 255) {
        first[m * 257 + 256] = part[255];
    }
    cnt[m * 256 + k] = sum;
#pragma unroll 8
    for (int c = 0; c < chunks; c++) {
        const uint32_t n = mine[(int64_t)c * 256];
        mine[(int64_t)c * 256] = run;
        run += n;
    }
}

__global__ __launch_bounds__(256) void pq_place_kernel(const uint8_t *__restrict__ codes, int64_t ns, int chunk, int chunks,
                                                       const uint32_t *__restrict__ starts, uint32_t *__restrict__ order)
{
    __shared__ volatile uint32_t cursor[4][256];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, m = blockIdx.y;
    const int c = blockIdx.x * 4 + wave;
    if (c < chunks) {
        for (int k = lane; k < 256; k += 64) {
            cursor[wave][k] = starts[((int64_t)m * chunks + c) * 256 + k];
        }
    }
    __syncthreads();
    const uint8_t *src = codes + (int64_t)m * ns;
    uint32_t *dst = order + (int64_t)m * ns;
    const int64_t b = (int64_t)c * chunk, e = b + chunk < ns ? b + chunk : ns;
    for (int64_t i0 = b; i0 < e; i0 += 64) {
        const bool valid = i0 + lane < e;
        const int code = valid ? src[i0 + lane] : 0;
        const unsigned long long same = same_code_lanes(code, valid);
        const uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(same >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)same, 0));
        if (valid) {
            // one wavefront's LDS operations complete in order: every lane has read its cursor before the last of its
            // equals moves it, and the next step reads it afterwards
            const uint32_t at = cursor[wave][code];
            dst[at + rank] = (uint32_t)(i0 + lane);
            if ((same >> lane) == 1ull) {
                cursor[wave][code] = at + rank + 1;
            }
        }
    }
}

// G lanes per codeword (a power of two that covers the sub-vector, at most 64), one component each.
template <int G>
__global__ __launch_bounds__(256) void pq_mean_kernel(const float *__restrict__ subs, int64_t ns, int dsub,
                                                      const uint32_t *__restrict__ first, const uint32_t *__restrict__ order,
                                                      float *__restrict__ codebook)
{
    constexpr int kAhead = 16;
    const int m = blockIdx.y, k = blockIdx.x * (256 / G) + threadIdx.x / G, t = blockIdx.z * G + threadIdx.x % G;
    if (t >= dsub) {
        return;
    }
    const uint32_t b = first[m * 257 + k], e = first[m * 257 + k + 1];
    if (b == e) {
        return;   // keeps its value; split_empty_kernel re-seeds it
    }
    const uint32_t *list = order + (int64_t)m * ns;
    const float *src = subs + (int64_t)m * ns * dsub + t;
    double sum = 0.0;
    uint32_t idx[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; u++) {
        idx[u] = list[b + u < e ? b + u : e - 1];
    }
    for (uint32_t i = b; i < e; i += kAhead) {
        float v[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; u++) {
            v[u] = src[(int64_t)idx[u] * dsub];
        }
#pragma unroll
        for (int u = 0; u < kAhead; u++) {   // the next positions, while the values are on their way
            const uint32_t at = i + kAhead + u;
            idx[u] = list[at < e ? at : e - 1];
        }
#pragma unroll
        for (int u = 0; u < kAhead; u++) {
            sum += i + u < e ? (double)v[u] : 0.0;   // (the sum is never -0, so adding 0 past the end leaves it as it is)
        }
    }
    codebook[((int64_t)m * 256 + k) * dsub + t] = (float)(sum / (double)(e - b));
}

template <int G>
void launch_mean(const float *subs, int64_t ns, int M, int dsub, const PqUpdateWorkspace &ws, float *codebook, hipStream_t s)
{
    hipLaunchKernelGGL(pq_mean_kernel<G>, dim3(G, (unsigned)M, (unsigned)((dsub + G - 1) / G)), dim3(256), 0, s, subs, ns,
                       dsub, ws.first.data(), ws.order.data(), codebook);
}

}  // namespace

void launch_pq_encode(const float *x, int64_t n, int d, int M, const float *codebook, uint8_t *codes, hipStream_t s)
{
    launch_encode(x, n, M, d / M, PqStrides{d, d / M, M, 1}, codebook, codes, s);
}

void launch_pq_subvectors(const float *x, int64_t ns, int d, int m0, int M, int dsub, float *out, hipStream_t s)
{
    if (dsub > 64) {
        hipLaunchKernelGGL(pq_subvectors_long_kernel, dim3((unsigned)((ns * dsub + 255) / 256), (unsigned)M), dim3(256), 0,
                           s, x, ns, d, m0, dsub, out);
        return;
    }
    const int per_tile = 64 / dsub;
    hipLaunchKernelGGL(pq_subvectors_kernel, dim3((unsigned)((ns + 63) / 64), (unsigned)((M + per_tile - 1) / per_tile)),
                       dim3(256), 0, s, x, ns, d, m0, M, dsub, per_tile, out);
}

void launch_pq_encode_subvectors(const float *subs, int64_t ns, int M, int dsub, const float *codebook, uint8_t *codes,
                                 hipStream_t s)
{
    launch_encode(subs, ns, M, dsub, PqStrides{dsub, ns * dsub, 1, ns}, codebook, codes, s);
}

void launch_pq_update(const float *subs, const uint8_t *codes, int64_t ns, int M, int dsub, float *codebook,
                      unsigned long long *cnt, PqUpdateWorkspace &ws, hipStream_t s)
{
    // pieces of 1024 samples, longer ones where there would be more than 512 of them (pq_starts_kernel walks them)
    const int chunk = (int)std::max<int64_t>(1024, round_up((ns + 511) / 512, 64));
    const int chunks = (int)((ns + chunk - 1) / chunk);
    ws.starts.resize((size_t)M * chunks * 256);
    ws.first.resize((size_t)M * 257);
    ws.order.resize((size_t)M * ns);
    const dim3 grid((unsigned)((chunks + 3) / 4), (unsigned)M);
    hipLaunchKernelGGL(pq_count_kernel, grid, dim3(256), 0, s, codes, ns, chunk, chunks, ws.starts.data());
    hipLaunchKernelGGL(pq_starts_kernel, dim3((unsigned)M), dim3(256), 0, s, ws.starts.data(), chunks, ws.first.data(), cnt);
    hipLaunchKernelGGL(pq_place_kernel, grid, dim3(256), 0, s, codes, ns, chunk, chunks, ws.starts.data(), ws.order.data());
    switch (pow2_ceil(std::min(dsub, 64))) {
    case 1: launch_mean<1>(subs, ns, M, dsub, ws, codebook, s); break;
    case 2: launch_mean<2>(subs, ns, M, dsub, ws, codebook, s); break;
    case 4: launch_mean<4>(subs, ns, M, dsub, ws, codebook, s); break;
    case 8: launch_mean<8>(subs, ns, M, dsub, ws, codebook, s); break;
    case 16: launch_mean<16>(subs, ns, M, dsub, ws, codebook, s); break;
    case 32: launch_mean<32>(subs, ns, M, dsub, ws, codebook, s); break;
    default: launch_mean<64>(subs, ns, M, dsub, ws, codebook, s); break;
    }
}

}  // namespace ixa

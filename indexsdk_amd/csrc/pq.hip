// PQ encode on the GPU, bit-exact to the reference's host encoder
// (FR/ascend/impl/AscendIndexIVFPQImpl.cpp:879-921: encodeSingleVectorPQ /
// findCentroidInSubQuantizer / calDistance): the RAW vector is encoded (by_residual = false),
// distance = sum (a-b)^2 accumulated left to right in fp32 without FMA, strict '<' so the first
// minimum wins.  That arithmetic decides every code; the matrix cores only say which 16 of a sub-quantizer's 256
// codewords it has to be applied to.
#include "pq.h"

#include <algorithm>

#include "resident_tile.h"

namespace ixa {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

// Sub-vector m of vector i starts at x + i * xi + m * xm, its code is codes[i * ci + m * cm].
struct PqStrides {
    int64_t xi, xm, ci, cm;
};

constexpr float kPqFar = 3.402823466e+38f;   // a codeword at this distance or farther is never chosen

// A workgroup of four wavefronts encodes one sub-quantizer of a block of vectors, 32 vectors of a wavefront at a time.
//   1. u = x.c - |c|^2 / 2 of 32 vectors and all 256 codewords on the bf16 matrix cores, both relative to a centre (the mean of
//      eight codewords), so that what sub-vectors have in common does not widen the error bound.  Vectors and codewords are split
//      into hi + lo (x = hi + lo + rest, |rest| <= 2^-18 |x|) and laid side by side in K: [hi | hi | lo | 1 1 1] against
//      [hi | lo | hi | the three parts of -|c|^2 / 2], so up to four dimensions are ONE matrix instruction per 32 codewords.
//      The codewords' fragments are made once per workgroup and stay in registers (in LDS above eight dimensions).
//   2. A lane owns one vector and 16 codewords of each block of 32 (the other half of the wavefront the others): it keeps the
//      largest u of every 16.  A group of 16 whose largest u is within the error bound of the vector's largest is in reach.
//   3. The reference's arithmetic decides among the groups in reach, one (eight codewords by either half) in most vectors.  Where
//      some vector of the wavefront has more than kPqWalk of its 16 groups in reach (codewords that are equal, or nearly so), the
//      wavefront walks through all 256 instead, and through those of its next kPqWalks steps without asking the matrix cores.
// The bound: distances decide by |x|^2 - 2 u, so a lead of u decides when twice it exceeds the errors of both sides:
//   a u misses at most 3 x 2^-18 |x||c| and its K + dsub sums (2^-24 of at most |x||c| + |c|^2 / 2 each), a canonical
//   distance (dsub + 2) 2^-24 of itself, at most (|x| + |c|)^2, and the differences from the centre, rounded once, move a squared
//   distance by 2 x 2^-24 (|x| + |c|)^2.  Lengths below 1e-15, where products may vanish, decide nothing.
// Per 32 vectors: KS matrix instructions and a maximum over 16 per block, and 16 distances, where every lane walking 256
// codewords for its own vector took 256 of them: 20000 x 32 sub-quantizers of 4 dimensions 55 -> 20 us,
//   131072 x 32 280 -> 70 (88 on the sub-vectors of a training), 20000 x 4 of 32 dimensions 75 -> 34.  Adding 100000 x 64 of 2
//   dimensions to two lists, every lane walking / this: 864 / 303 us; an offset of 30 851 / 305; codewords in runs of eight equal
//   ones 920 / 395 (4 of 32 dimensions: 858 / 352, 805 / 290, 832 / 368).
// What bounds it at 4 dimensions: the LDS pipe, active in 71 % of a CU's cycles, three quarters of that with bank conflicts of the lanes'
// codewords (each lane reads those of its own group); matrix cores busy 21 %, 45 vector instructions to a matrix instruction.
constexpr int kPqWalk = 11, kPqWalks = 7;

template <int DSUB>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(DSUB > 24 ? 1 : 2))) void pq_encode_kernel(
    const float *__restrict__ x, int64_t n, PqStrides st, int M, const float *__restrict__ codebook, uint8_t *__restrict__ codes,
    int64_t per_block)
{
    constexpr int K = 3 * DSUB + 3, KS = (K + 15) / 16;
    constexpr bool kInRegisters = KS <= 2;
    __shared__ __align__(16) float cb[256 * DSUB];
    __shared__ __align__(16) bf16x8 frag[8][KS][64];   // [block of 32 codewords][K-step][lane]
    __shared__ float wave_max[4];
    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5, l32 = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // the sub-quantizers of a block of vectors run on one XCD, whose L2 then has the lines their sub-vectors share
    const int64_t vb = (blockIdx.x >> 3) / M * 8 + (blockIdx.x & 7), i_first = vb * per_block;
    const int m = (blockIdx.x >> 3) % M;
    if (i_first >= n) {
        return;
    }
    const int64_t i_end = i_first + per_block < n ? i_first + per_block : n;
    // element `slot` of K for a vector (hi, hi, lo, ones) or codeword (hi, lo, hi, parts of the norm)
    auto slot_of = [](int slot, const __bf16 *first, const __bf16 *second, const __bf16 *third, const __bf16 *tail) {
        return slot < DSUB ? first[slot] : (slot < 2 * DSUB ? second[slot - DSUB]
               : (slot < 3 * DSUB ? third[slot - 2 * DSUB] : (slot < K ? tail[slot - 3 * DSUB] : (__bf16)0.f)));
    };
    float centre[DSUB];   // the same in every lane: scalar registers
#pragma unroll
    for (int t = 0; t < DSUB; t++) {
        float sum = 0.f;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            sum += codebook[((int64_t)m * 256 + 32 * j) * DSUB + t];
        }
        sum = fabsf(sum) < 1e38f ? 0.125f * sum : 0.f;
        centre[t] = __uint_as_float((uint32_t)__builtin_amdgcn_readfirstlane((int)__float_as_uint(sum)));
    }
    {
        const float *src = codebook + ((int64_t)m * 256 + tid) * DSUB;
        __bf16 hi[DSUB], lo[DSUB], part[3];
        float sq = 0.f;
#pragma unroll
        for (int t = 0; t < DSUB; t++) {
            cb[tid * DSUB + t] = src[t];
            const float c = src[t] - centre[t];
            sq += c * c;
            hi[t] = (__bf16)c;
            lo[t] = (__bf16)(c - (float)hi[t]);
        }
        float rest = -0.5f * sq;
#pragma unroll
        for (int t = 0; t < 3; t++) {
            part[t] = (__bf16)rest;
            rest -= (float)part[t];
        }
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
#pragma unroll
            for (int h = 0; h < 2; h++) {
                bf16x8 f;
#pragma unroll
                for (int t = 0; t < 8; t++) {
                    f[t] = slot_of(ks * 16 + h * 8 + t, hi, lo, hi, part);
                }
                frag[tid >> 5][ks][h * 32 + (tid & 31)] = f;
            }
        }
        for (int o = 32; o > 0; o >>= 1) {
            sq = fmaxf(sq, __shfl_xor(sq, o));
        }
        if (lane == 0) {
            wave_max[wave] = sq;
        }
    }
    __syncthreads();
    const float cmax = sqrtf(fmaxf(fmaxf(wave_max[0], wave_max[1]), fmaxf(wave_max[2], wave_max[3])));
    bf16x8 own[kInRegisters ? 8 : 1][KS];
    if constexpr (kInRegisters) {
#pragma unroll
        for (int b = 0; b < 8; b++) {
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                own[b][ks] = frag[b][ks][lane];
            }
        }
    }
    const float *xm = x + m * st.xm;
    float next[DSUB];
    auto fetch = [&](int64_t i0) {
        const float *src = xm + (i0 + l32 < n ? i0 + l32 : n - 1) * st.xi;
#pragma unroll
        for (int t = 0; t < DSUB; t++) {
            next[t] = src[t];
        }
    };
    fetch(i_first + wave * 32);
    int walks = 0;   // steps that are walked without asking first (the same in every lane)
    for (int64_t i0 = i_first + wave * 32; i0 < i_end; i0 += 128) {
        float sub[DSUB];
#pragma unroll
        for (int t = 0; t < DSUB; t++) {
            sub[t] = next[t];
        }
        fetch(i0 + 128);
        float best = kPqFar;
        int arg = 0;
        auto distance = [&](int k) {
            float dist = 0.f;
#pragma unroll
            for (int j = 0; j < DSUB; j++) {
                const float diff = __fsub_rn(sub[j], cb[k * DSUB + j]);
                dist = __fadd_rn(dist, __fmul_rn(diff, diff));
            }
            return dist;
        };
        bool walk = walks > 0;
        walks -= walk ? 1 : 0;
        if (!walk) {
            __bf16 hi[DSUB], lo[DSUB];
            const __bf16 ones[3] = {(__bf16)1.f, (__bf16)1.f, (__bf16)1.f};
            float sq = 0.f;
#pragma unroll
            for (int t = 0; t < DSUB; t++) {
                const float v = sub[t] - centre[t];
                sq += v * v;
                hi[t] = (__bf16)v;
                lo[t] = (__bf16)(v - (float)hi[t]);
            }
            bf16x8 vec[KS];
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                bf16x8 f0, f1;
#pragma unroll
                for (int t = 0; t < 8; t++) {
                    f0[t] = slot_of(ks * 16 + t, hi, hi, lo, ones);
                    f1[t] = slot_of(ks * 16 + 8 + t, hi, hi, lo, ones);
                }
                vec[ks] = half ? f1 : f0;
            }
            float top[8];   // the largest u of the lane's 16 codewords of each block
#pragma unroll
            for (int b = 0; b < 8; b++) {
                if constexpr (!kInRegisters) {
                    asm volatile("" ::: "memory");   // the fragments stay in LDS
                }
                v16f acc{};
#pragma unroll
                for (int ks = 0; ks < KS; ks++) {
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kInRegisters ? own[kInRegisters ? b : 0][ks] : frag[b][ks][lane], vec[ks],
                                                                  acc, 0, 0, 0);
                }
                top[b] = acc[0];
#pragma unroll
                for (int r = 1; r < 16; r++) {
                    top[b] = fmaxf(top[b], acc[r]);
                }
            }
            float lead = top[0];
#pragma unroll
            for (int b = 1; b < 8; b++) {
                lead = fmaxf(lead, top[b]);
            }
            lead = fmaxf(lead, __shfl_xor(lead, 32));
            const float len = sqrtf(sq), mag = len * cmax + 0.5f * cmax * cmax, far = len + cmax;
            const float need = 2.f * (3.f / 262144.f * len * cmax + (float)(K + DSUB + 4) * 5.9604645e-8f * mag) +
                               (float)(DSUB + 7) * 5.9604645e-8f * far * far;
            // (written so that a bound or a u that is undefined, and a bound that is infinite, leave no group out)
            const float reach = far > 1e-15f ? lead - need : -__builtin_inff();
            uint32_t todo = 0;   // groups in reach: bit = block, + 8 where the upper half of the wavefront has them
#pragma unroll
            for (int b = 0; b < 8; b++) {
                todo |= top[b] < reach ? 0u : 1u << b;
            }
            todo = i0 + l32 < i_end ? todo << (8 * half) : 0u;
            todo |= (uint32_t)__shfl_xor((int)todo, 32);
            walk = __ballot(__popc(todo) > kPqWalk) != 0;
            walks = walk ? kPqWalks : 0;
            while (!walk && __ballot(todo != 0) != 0) {
                if (todo != 0) {
                    const int at = __builtin_ctz(todo);
                    const int first = (at & 7) * 32 + (at >> 3) * 4;   // the 16: first + 8 g + t, g < 4, t < 4
                    float near = kPqFar;
                    int k_near = 256;
#pragma unroll
                    for (int g = 0; g < 2; g++) {
#pragma unroll
                        for (int t = 0; t < 4; t++) {
                            const int k = first + 8 * (2 * half + g) + t;
                            const float dist = distance(k);
                            if (dist < near) {
                                near = dist;
                                k_near = k;
                            }
                        }
                    }
                    const bool nearer = near < best || (near == best && k_near < arg);
                    best = nearer ? near : best;
                    arg = nearer ? k_near : arg;
                    todo &= todo - 1;
                }
            }
        }
        if (walk) {   // all codewords, the even ones by the lower half of the wavefront
#pragma unroll 4
            for (int j = 0; j < 128; j++) {
                const int k = 2 * j + half;
                const float dist = distance(k);
                if (dist < best) {
                    best = dist;
                    arg = k;
                }
            }
        }
        {   // what the other half found; of equal distances the smaller codeword
            const float ob = __shfl_xor(best, 32);
            const int oa = __shfl_xor(arg, 32);
            arg = ob < best || (ob == best && oa < arg) ? oa : arg;
        }
        if (half == 0 && i0 + l32 < i_end) {
            codes[(i0 + l32) * st.ci + m * st.cm] = (uint8_t)arg;
        }
    }
}

// One dimension: a lane walks the 256 codewords for its own vector (three instructions each; 3000 x 64 sub-quantizers 12 us,
// with the kernel above 27).
__global__ __launch_bounds__(256) void pq_encode_scalar_kernel(const float *__restrict__ x, int64_t n, PqStrides st,
                                                               const float *__restrict__ codebook, uint8_t *__restrict__ codes)
{
    __shared__ float cb[256];
    const int m = blockIdx.y;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    cb[threadIdx.x] = codebook[(int64_t)m * 256 + threadIdx.x];
    __syncthreads();
    if (i < n) {
        const float v = x[i * st.xi + m * st.xm];
        float best = kPqFar;
        int arg = 0;
        for (int k = 0; k < 256; k++) {
            const float diff = __fsub_rn(v, cb[k]);
            const float dist = __fmul_rn(diff, diff);
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
    // vectors per workgroup: 2048 (16 per wavefront and codeword fragment made), fewer while that leaves CUs without four
    const int64_t per_block = std::min<int64_t>(2048, std::max<int64_t>(128, round_up(n * M / (4 * device_cus()), 128)));
    const int64_t blocks = round_up((n + per_block - 1) / per_block, 8) * M;
    IXA_REQUIRE(blocks < (int64_t)1 << 31, kErrInvalidParam, "encode grid too large");
#define IXA_ENC(D)                                                                                             \
    case D:                                                                                                    \
        hipLaunchKernelGGL(pq_encode_kernel<D>, dim3((unsigned)blocks), block, 0, s, x, n, st, M, codebook, codes, per_block); \
        break;
    switch (dsub) {
    case 1:
        hipLaunchKernelGGL(pq_encode_scalar_kernel, grid, block, 0, s, x, n, st, codebook, codes);
        break;
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

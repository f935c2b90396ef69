// fp32 scores on the bf16 matrix cores, the streamed operand read as it lies: Flat search (queries in LDS, base streamed) and
// assignment (centroids in LDS, vectors streamed).
//
// resident_f32_kernel has the structure of the int8 kernel (flat_i8.hip): a persistent workgroup of 8 wavefronts keeps a tile
// of QT = 32 RA queries in LDS, wavefront w owns rows 32 w .. 32 w + 31 of every tile of 256 base rows, and no workgroup barrier
// stands in the main loop.  What differs:
//   * operands are fp32.  x = hi + lo + rest with hi = bf16(x), lo = bf16(x - hi), and a score is formed from the three products
//     hi.hi + hi.lo + lo.hi (coarse.hip has the bound of what they miss).  The queries are split when their tile is copied into
//     LDS; the base rows are split IN REGISTERS, between their load and the matrix instructions: 24 vector instructions per
//     K-step of 16 dimensions beside 3 RA matrix instructions of 32 cycles.  So the base is read once, as the fp32 rows that
//     it is kept in: no split copy of it is written and read (10 bytes of traffic per element and, at 1M x 128, 0.28 of the 1.8 ms
//     of a search), and none needs room;
//   * the rows are row-major.  Per two K-steps a row's 128 bytes are fetched by four 16-byte loads of two lanes, issued together
//     so that the cache line is used while it is there.  The lane half h of K-step s holds elements 16 s + 4 h .. + 3 and
//     16 s + 8 + 4 h .. + 3 (neighbouring halves read 32 contiguous bytes): the matrix instruction sums over k in whatever
//     order, and the query tile is written to LDS in the same one;
//   * the K loop is a run-time loop over batches of SPB K-steps (dimensions need only be a multiple of 4: query elements past the
//     end are zero in LDS, and the loads of the base stay inside the row by reading its last elements again; the caller
//     sees to it that every base element is finite).  A batch is converted at once, which frees its registers for the next
//     batch's loads: they have SPB K-steps to arrive.
//
// 1M x 128, 1000 queries: a search 1763 -> 964 us on the device; 1.23 PFLOP/s of bf16 products in the longest launch (the ring kernel
// that reads split rows: 0.71), matrix cores busy 70 % of the CU's cycles at the 1.9 GHz that they hold, the LDS pipe 28 %, wavefronts
// waiting a quarter of theirs; with few queries the base's bytes (512 MB in 100 us of the 207 of one query).  Assignment of 1M x 128 to
// 1024 centroids, where scores, selections and the refinement took 7.6 ms: norms and bounds 94 us, the score launch 655 us (1.20 PFLOP/s,
// matrix cores busy 65 %: five vector instructions per matrix instruction, most of them the three largest of every sum), the tiles' best
// 96 us, what they leave open 17 us.
//
// Score arithmetic: the accumulators start from -|b|^2 / 2 (L2; 0 for inner product) and end as u = q.b - |b|^2 / 2, and the
// score is fma(-2, u, |q|^2), or -u.  The admission test of a block of 16 rows is one compare of the largest u with a value
// that lies below every u whose score reaches the bound (test_value); what passes is tested again by its score.
#include <cmath>

#include "coarse.h"
#include "resident_f32.h"
#include "resident_tile.h"
#include "topk.h"

namespace ixa {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float v8f __attribute__((ext_vector_type(8)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int kWaves = 8;
constexpr int kTileRows = 256;       // base rows of a tile
constexpr int kQueueKeys = 128;      // per-wavefront queue of admitted keys (16 bytes each); flushed above 64
constexpr float kNoRow = -__builtin_inff();   // accumulator start of a row outside the launch: it reaches no test value
constexpr float kNoCentroid = -3e38f;   // of a centroid past the last one (a number: low bits are put into the sums)
// LDS behind the query tile of a filtered launch: {bound, norm, test value, -} per query, the wavefronts' queues
constexpr int filter_lds(int qt) { return qt * 16 + kWaves * kQueueKeys * 16; }
constexpr int assign_lds(int qt, int k) { return (qt + k) * 4; }   // a start per centroid; the centre, k = dimensions of whole batches
constexpr int kLdsLimit = 160 * 1024;

// hi and lo of eight numbers
__device__ __forceinline__ void split8(const v4f &a, const v4f &b, bf16x8 &hi, bf16x8 &lo)
{
    const v8f v = __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
    hi = __builtin_convertvector(v, bf16x8);
    const v4u h = __builtin_bit_cast(v4u, hi);
    v8f rest;
#pragma unroll
    for (int t = 0; t < 4; t++) {
        rest[2 * t] = v[2 * t] - __uint_as_float(h[t] << 16);
        rest[2 * t + 1] = v[2 * t + 1] - __uint_as_float(h[t] & 0xffff0000u);
    }
    lo = __builtin_convertvector(rest, bf16x8);
}

__device__ __forceinline__ float max16(const v16f &a)
{
    const float m0 = fmaxf(fmaxf(a[0], a[1]), a[2]), m1 = fmaxf(fmaxf(a[3], a[4]), a[5]);
    const float m2 = fmaxf(fmaxf(a[6], a[7]), a[8]), m3 = fmaxf(fmaxf(a[9], a[10]), a[11]);
    const float m4 = fmaxf(fmaxf(a[12], a[13]), a[14]);
    return fmaxf(fmaxf(fmaxf(m0, m1), m2), fmaxf(fmaxf(m3, m4), a[15]));
}

// A value below every u whose score is at or below tau.  L2: fl(qn - 2 u) <= tau implies qn - 2 u <= tau + 2^-24 |tau| or so,
// hence u >= (qn - tau) / 2 - 2^-25 |tau|; the difference is rounded once more, and 4.8e-7 (2^-21) of the magnitudes covers
// both several times over.  Inner product: -u <= tau is u >= -tau.  Never -inf: rows outside the launch have u = -inf.
__device__ __forceinline__ float test_value(float qn, float tau, bool l2)
{
    const float t = l2 ? 0.5f * (qn - tau) - 4.8e-7f * (qn + fabsf(tau)) : -tau;
    return fmaxf(t, -3.402823466e+38f);
}

// The larger of two numbers, or the number where the other is a NaN.  (fmaxf would make v a quiet number first, an instruction
// each.  The operands are results of vector instructions, never of a matrix instruction, whose results an inline instruction
// would not wait for.  A signalling NaN takes m away instead: AssignBound rules the sums out that could become one.)
__device__ __forceinline__ float max_number(float m, float v)
{
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(m), "v"(v));
    return r;
}

// Three largest values, the places of two.  (A NaN among the values is passed over: med3 of it and two numbers is the smaller.)
struct Best {
    float v1, v2, v3;
    uint32_t p1, p2;
    __device__ __forceinline__ void merge(const Best &o)
    {
        const bool first = o.v1 > v1;
        const float a1 = first ? o.v1 : v1, a2 = first ? o.v2 : v2, a3 = first ? o.v3 : v3, b1 = first ? v1 : o.v1, b2 = first ? v2 : o.v2;
        const uint32_t ap1 = first ? o.p1 : p1, ap2 = first ? o.p2 : p2, bp1 = first ? p1 : o.p1;
        const bool second = b1 > a2;   // of the list with the smaller best
        v1 = a1;
        p1 = ap1;
        v2 = second ? b1 : a2;
        p2 = second ? bp1 : ap2;
        v3 = second ? fmaxf(a2, b2) : fmaxf(a3, b1);
    }
};

enum { kStore = 0, kFilter = 1, kAssign = 2 };

// Words of a (tile, vector) that say which of the tile's centroids are within the vector's bound of the tile's best: half of them from
// either half of the wavefront, bit 16 (ra % 2) + r of word ra / 2 for the half's centroid of block ra in accumulator r.
constexpr int within_words(int qt) { return qt >= 64 ? qt / 32 : 2; }

// What a kAssign launch reads and writes per vector: the bound; the best two centroids of every tile and the third value; and, where
// the third value is within the bound of the best (crowded), all centroids that are.
struct AssignTiles {
    const float *need;
    float4 *top;        // [tile][vector] {best, second, third u, places}
    uint32_t *within;   // [tile][vector][within_words]
};
__device__ __forceinline__ bool crowded(float best, float third, float need) { return !(best - third > need); }

// RA: query blocks of 32 per tile; SPB: K-steps of 16 dimensions per batch; nbat >= 2 batches cover the d dimensions.  MODE:
//   kStore   every score is stored;
//   kFilter  admitted keys are appended;
//   kAssign  the "queries" are centroids, the base rows vectors: of every tile of centroids the best two of each vector and the
//            third value.  The matrix operands change places, so that a lane owns ONE vector and 16 centroids per block, and
//            the accumulators start from -qn / 2 of the centroid, kept in LDS.  The centroids are relative to a centre (bn: its
//            d numbers), which is taken from the vectors between their load and their split.
template <int RA, int SPB, int MODE>
__global__ __launch_bounds__(kWaves * 64) __attribute__((amdgpu_waves_per_eu(2, 2))) void resident_f32_kernel(
    const float *__restrict__ Q, int64_t nq, const float *__restrict__ B, int64_t nb, int d, int nbat,
    const float *__restrict__ qn, const float *__restrict__ bn, int metric, float *__restrict__ out, int64_t ldo,
    ScoreFilter<float> flt, AssignTiles assign, int tiles_m, int ntiles, int seg_tiles, int own_resident)
{
    constexpr bool FILTER = MODE == kFilter, ASSIGN = MODE == kAssign;
    constexpr int QT = RA * 32;
    // LDS of a K-step: [half][RA blocks of hi, RA of lo][32 queries][16 B]
    constexpr int kStepLds = QT * 64;
    constexpr int kBatchLds = SPB * kStepLds;
    constexpr int G = RA >= 2 ? 4 : 2;     // blocks of a read group
    constexpr int UPS = 2 * RA / G;        // groups of a K-step
    constexpr int UPB = SPB * UPS;
    static_assert(UPB % 2 == 0, "groups alternate between two register sets");
    static_assert(kBatchLds + G * 512 <= 65536, "offset field of an LDS read");
    extern __shared__ __align__(16) unsigned char lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = lane >> 5, l32 = lane & 31;
    const bool l2 = metric == kMetricL2;

    const int xcd = blockIdx.x & 7, wi = blockIdx.x >> 3, wpx = gridDim.x >> 3;
    const ResidentItems sched(tiles_m, ntiles, seg_tiles, xcd, wpx, own_resident != 0);
    const int S = sched.S;
    const int first_item = sched.next(wi);
    if (first_item < 0) {
        return;
    }
    const uint32_t lds_base = (uint32_t)reinterpret_cast<size_t>((__attribute__((address_space(3))) unsigned char *)lds);
    const uint32_t a_lane = lds_base + (uint32_t)(half * (QT * 32) + l32 * 16);
    float4 *meta = reinterpret_cast<float4 *>(lds + (size_t)nbat * kBatchLds);   // {tau, |q|^2, test value, -}
    float *start = reinterpret_cast<float *>(meta);   // kAssign: the starts of the centroids' sums, and the centre
    float *centre = start + QT;
    uint4 *queue = reinterpret_cast<uint4 *>(meta + QT) + wave * kQueueKeys;
    int qcount = 0;   // keys in this wavefront's queue (wave-uniform)
    // every queued key takes its place in its query's candidate buffer; 64 lanes, one key each
    auto flush_queue = [&]() {
        wave_lds_fence();
        for (int i0 = 0; i0 < qcount; i0 += 64) {
            if (i0 + lane < qcount) {
                const uint4 e = queue[i0 + lane];   // {base row, ordered score, query row, -}
                const int pos = atomicAdd(&flt.cnt[e.z], 1);
                if (pos < flt.cap) {
                    flt.cand[(int64_t)e.z * flt.cap + pos] = ((key_t)e.y << 32) | e.x;
                }
            }
        }
        wave_lds_fence();
        qcount = 0;
    };
    // tile j of this XCD's share: first of this wave's 32 rows, and the lane's row of them (past the end: the last row)
    auto block_row0 = [&](int j) { return sched.streamed_tile(j) * kTileRows + wave * 32; };
    auto row_ptr = [&](int j) {
        const int64_t r = block_row0(j) + l32;
        return B + (r < nb ? r : nb - 1) * d;
    };
    const int dlast = d - 4;
    v4f raw[2 * SPB];   // a batch of the lane's row: two runs of four elements per K-step
    auto load_batch = [&](const float *row, int b) {
#pragma unroll
        for (int t = 0; t < 2 * SPB; t++) {
            const int k = (b * (2 * SPB) + t) * 8 + 4 * half;
            raw[t] = *reinterpret_cast<const v4f *>(row + (k < dlast ? k : dlast));
        }
        asm volatile("" ::: "memory");
    };
    const int64_t bn_last = (nb + 3) / 4 * 4 - 4;
    v4f bnv[4];   // norms of the lane's 16 rows (four runs of four) of a block
    auto load_norms = [&](int j) {
        const int64_t r = block_row0(j) + 4 * half;
#pragma unroll
        for (int g = 0; g < 4; g++) {
            bnv[g] = *reinterpret_cast<const v4f *>(bn + (r + 8 * g < bn_last ? r + 8 * g : bn_last));
        }
        asm volatile("" ::: "memory");
    };

    v16f acc[RA];
    int cur_tm = -1;
    int it_t = first_item;
    int tm, j, jend;
    sched.range(it_t, tm, j, jend);
    const float *cur = row_ptr(j);
    // Loads are issued in the same order here and in the loop: norms of a tile before its first batch.
    if constexpr (!ASSIGN) {
        load_norms(j);
    }
    load_batch(cur, 0);
    bool staggered = false;
    while (true) {
        if (tm != cur_tm) {
            if (cur_tm >= 0) {
                __syncthreads();
            }
            // The query tile: a wavefront step moves 16 queries x 2 K-steps (128 contiguous bytes of a row); queries past the
            // end of the batch repeat its last one.
            const int qq = lane & 15, s2 = lane >> 5, h = (lane >> 4) & 1;
            const int steps = (QT / 16) * (nbat * SPB / 2);
            constexpr int kIn = 4;   // steps in flight
            for (int st0 = wave; st0 < steps; st0 += kWaves * kIn) {
                v4f a[kIn], b[kIn];
#pragma unroll
                for (int i = 0; i < kIn; i++) {
                    const int st = st0 + i * kWaves;
                    const int64_t qrow = (int64_t)tm * QT + (st % (QT / 16)) * 16 + qq;
                    const float *src = Q + (qrow < nq ? qrow : nq - 1) * d;
                    const int k = (st / (QT / 16) * 2 + s2) * 16 + 4 * h;
                    a[i] = v4f{0.f, 0.f, 0.f, 0.f};
                    b[i] = v4f{0.f, 0.f, 0.f, 0.f};
                    if (st < steps && k < d) {
                        a[i] = *reinterpret_cast<const v4f *>(src + k);
                    }
                    if (st < steps && k + 8 < d) {
                        b[i] = *reinterpret_cast<const v4f *>(src + k + 8);
                    }
                }
#pragma unroll
                for (int i = 0; i < kIn; i++) {
                    const int st = st0 + i * kWaves;
                    if (st < steps) {
                        bf16x8 hi, lo;
                        split8(a[i], b[i], hi, lo);
                        unsigned char *dst = lds + (size_t)(st / (QT / 16) * 2 + s2) * kStepLds + h * (QT * 32) +
                                             ((st % (QT / 16)) * 16 + qq) * 16;
                        *reinterpret_cast<bf16x8 *>(dst) = hi;
                        *reinterpret_cast<bf16x8 *>(dst + QT * 16) = lo;
                    }
                }
            }
            if constexpr (FILTER) {
                if (tid < QT) {
                    const int64_t row = (int64_t)tm * QT + tid;
                    const float tau = row < nq ? flt.tau[row] : 0.f, norm = row < nq && l2 ? qn[row] : 0.f;
                    // no score compares as at or below the NaN of a query past the end of the batch
                    meta[tid] = row < nq ? make_float4(tau, norm, test_value(norm, tau, l2), 0.f)
                                         : make_float4(__builtin_nanf(""), 0.f, __builtin_inff(), 0.f);
                }
            }
            if constexpr (ASSIGN) {
                if (tid < QT) {
                    const int64_t c = (int64_t)tm * QT + tid;
                    start[tid] = c < nq ? -0.5f * qn[c] : kNoCentroid;
                }
                if (cur_tm < 0) {
                    for (int k = tid; k < nbat * SPB * 16; k += kWaves * 64) {
                        centre[k] = k < d ? bn[k] : 0.f;
                    }
                }
            }
            cur_tm = tm;
            __syncthreads();
            // The second wavefront of every SIMD starts half a tile late, once: from then on each one's epilogue runs under the
            // other's matrix instructions (a tile is nbat SPB 3 RA of them, 32 cycles each; s_sleep counts 64).
            if (!staggered && wave >= kWaves / 2) {
                for (int t = 0; t < nbat; t++) {
                    __builtin_amdgcn_s_sleep((3 * SPB * RA + 1) / 2);
                }
            }
            staggered = true;
        }
        // the tile after this one (the last tile names itself: its loads are harmless repeats)
        int n_it = it_t, n_tm = tm, n_j = j + S, n_jend = jend;
        bool has_next = true;
        if (n_j >= jend) {
            n_it = sched.next(it_t + wpx);
            if (n_it >= 0) {
                sched.range(n_it, n_tm, n_j, n_jend);
            } else {
                has_next = false;
                n_it = it_t;
                n_j = j;
            }
        }
        const float *nxt = row_ptr(n_j);
        const int64_t row0 = block_row0(j);
        v16f c0;
        if constexpr (ASSIGN) {
#pragma unroll
            for (int ra = 0; ra < RA; ra++) {
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const v4f c = *reinterpret_cast<const v4f *>(start + ra * 32 + 8 * g + 4 * half);
#pragma unroll
                    for (int t = 0; t < 4; t++) {
                        acc[ra][4 * g + t] = c[t];
                    }
                }
            }
        } else {
#pragma unroll
            for (int r = 0; r < 16; r++) {
                c0[r] = l2 ? -0.5f * bnv[r >> 2][r & 3] : 0.f;
            }
        }
        float need = 0.f;
        if constexpr (ASSIGN) {
            need = assign.need[row0 + l32 < nb ? row0 + l32 : nb - 1];
        }
        if (!ASSIGN && row0 + 32 > nb) {   // the last tile of the launch: rows past its end take no part
#pragma unroll
            for (int r = 0; r < 16; r++) {
                c0[r] = row0 + 4 * half + 8 * (r >> 2) + (r & 3) < nb ? c0[r] : kNoRow;
            }
        }
        uint32_t addr = a_lane;
        const float *centre_at = centre + 4 * half;
        // one batch: its rows are split, the loads that follow it sent for, the products added
        auto batch = [&](auto first, auto last, const float *next_row, int next_batch) {
            constexpr bool FIRST = decltype(first)::value, LAST = decltype(last)::value;
            // the batch's first fragments arrive behind the split; no read is in flight where batches meet (a register copy
            // at a loop's edge would not wait for it)
            bf16x8 fa[2][G];
            lds_read_group<G, 0>(addr, fa[0]);
            bf16x8 bh[SPB], bl[SPB];
#pragma unroll
            for (int t = 0; t < SPB; t++) {
                if constexpr (ASSIGN) {
                    raw[2 * t] -= *reinterpret_cast<const v4f *>(centre_at + 16 * t);
                    raw[2 * t + 1] -= *reinterpret_cast<const v4f *>(centre_at + 16 * t + 8);
                }
                split8(raw[2 * t], raw[2 * t + 1], bh[t], bl[t]);
            }
            centre_at += 16 * SPB;
            if constexpr (LAST && !ASSIGN) {
                load_norms(n_j);
            }
            load_batch(next_row, next_batch);
            static_for<0, UPB>([&](auto uc) {
                constexpr int u = decltype(uc)::value;
                constexpr int st = u / UPS, p = u % UPS;
                if constexpr (u + 1 < UPB) {
                    lds_read_group<G, (u + 1) / UPS * kStepLds + (u + 1) % UPS * (G * 512)>(addr, fa[(u + 1) & 1]);
                    lds_wait_group<G, G>(fa[u & 1]);
                } else {
                    lds_wait_group<G, 0>(fa[u & 1]);
                }
                static_for<0, G>([&](auto tc) {
                    constexpr int t = decltype(tc)::value, f = p * G + t, ra = f % RA;
                    if constexpr (ASSIGN) {
                        acc[ra] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[u & 1][t], bh[st], acc[ra], 0, 0, 0);
                    } else if constexpr (FIRST && st == 0 && f < RA) {
                        acc[ra] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bh[st], fa[u & 1][t], c0, 0, 0, 0);
                    } else {
                        acc[ra] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bh[st], fa[u & 1][t], acc[ra], 0, 0, 0);
                    }
                });
                static_for<0, G>([&](auto tc) {
                    constexpr int t = decltype(tc)::value, f = p * G + t;
                    if constexpr (f < RA && ASSIGN) {
                        acc[f] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[u & 1][t], bl[st], acc[f], 0, 0, 0);
                    } else if constexpr (f < RA) {
                        acc[f] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bl[st], fa[u & 1][t], acc[f], 0, 0, 0);
                    }
                });
            });
            addr += kBatchLds;
        };
        constexpr std::true_type yes{};
        constexpr std::false_type no{};
        batch(yes, no, cur, 1);
        for (int b = 1; b < nbat - 1; b++) {
            batch(no, no, cur, b + 1);
        }
        batch(no, yes, nxt, 0);
        // a lane owns query (block ra, l32) and base rows row0 + 8 g + 4 half + t of the wave's block
        const int64_t col0 = row0 + 4 * half;
        if constexpr (FILTER) {
            unsigned long long hit[RA], any = 0;
#pragma unroll
            for (int ra = 0; ra < RA; ra++) {
                hit[ra] = __builtin_amdgcn_ballot_w64(max16(acc[ra]) >= meta[ra * 32 + l32].z);
                any |= hit[ra];
            }
            if (any != 0) {
                const uint32_t colv = (uint32_t)(col0 + flt.col_base);
#pragma unroll
                for (int ra = 0; ra < RA; ra++) {
                    if (hit[ra] != 0) {
                        const float4 mt = meta[ra * 32 + l32];
                        const uint32_t row = (uint32_t)(tm * QT + ra * 32 + l32);
#pragma unroll
                        for (int r = 0; r < 16; r++) {
                            const float u = acc[ra][r];
                            if (__builtin_amdgcn_ballot_w64(u >= mt.z) != 0) {
                                const float score = l2 ? __builtin_fmaf(-2.f, u, mt.y) : -u;
                                const bool pass = u >= mt.z && score <= mt.x;
                                const unsigned long long mask = __builtin_amdgcn_ballot_w64(pass);
                                if (mask != 0) {
                                    const int pre = __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                                                              __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0));
                                    if (pass) {
                                        queue[qcount + pre] = make_uint4(colv + 8 * (r >> 2) + (r & 3), ordered_bits(score),
                                                                         row, 0u);
                                    }
                                    qcount += __builtin_popcountll(mask);
                                    if (qcount > kQueueKeys - 64) {
                                        flush_queue();
                                    }
                                }
                            }
                        }
                    }
                }
            }
        } else if constexpr (ASSIGN) {
            // Largest, second and third u of four blocks at a time, their places 16 ra + r in the low six bits (which moves a value
            // by at most 2^-17 of it); then of all blocks, and of both halves, which hold different centroids of the same vector.
            constexpr int SETS = RA > 4 ? RA / 4 : 1, BLOCKS = RA / SETS;
            Best best[SETS];
#pragma unroll
            for (int set = 0; set < SETS; set++) {
                float m1 = kNoCentroid, m2 = kNoCentroid, m3 = kNoCentroid;
#pragma unroll
                for (int i = 0; i < BLOCKS * 16; i++) {
                    const float v = __uint_as_float((__float_as_uint(acc[set * BLOCKS + i / 16][i % 16]) & ~63u) | (uint32_t)i);
                    m3 = __builtin_amdgcn_fmed3f(m2, m3, v);
                    m2 = __builtin_amdgcn_fmed3f(m1, m2, v);
                    m1 = max_number(m1, v);
                }
                auto place = [&](float v) {
                    const uint32_t i = __float_as_uint(v) & 63u;
                    return set * (BLOCKS * 32) + (i >> 4) * 32 + ((i >> 2) & 3) * 8 + half * 4 + (i & 3);
                };
                best[set] = Best{m1, m2, m3, place(m1), place(m2)};
            }
            if constexpr (SETS == 2) {
                best[0].merge(best[1]);
            }
            const Best &own = best[0];
            best[0].merge(Best{__shfl_xor(own.v1, 32), __shfl_xor(own.v2, 32), __shfl_xor(own.v3, 32),
                               (uint32_t)__shfl_xor((int)own.p1, 32), (uint32_t)__shfl_xor((int)own.p2, 32)});
            const int64_t at = (int64_t)tm * nb + row0 + l32;
            const bool there = row0 + l32 < nb;
            if (half == 0 && there) {
                assign.top[at] = make_float4(own.v1, own.v2, own.v3, __uint_as_float(own.p1 | own.p2 << 16));
            }
            if (__builtin_amdgcn_ballot_w64(there && crowded(own.v1, own.v3, need)) != 0) {
                constexpr int WORDS = within_words(QT) / 2;
                const float reach = own.v1 - need;
                uint32_t *out_words = assign.within + (at * 2 + half) * WORDS;
#pragma unroll
                for (int w = 0; w < WORDS; w++) {
                    uint32_t word = 0;
                    // (written so that an undefined reach or u leaves nothing out)
#pragma unroll
                    for (int i = (RA > 1 ? 31 : 15); i >= 0; i--) {
                        word = word << 1 | (acc[2 * w + i / 16][i % 16] < reach ? 0u : 1u);
                    }
                    if (there) {
                        out_words[w] = word;
                    }
                }
            }
        } else {
#pragma unroll
            for (int ra = 0; ra < RA; ra++) {
                const int64_t row = (int64_t)tm * QT + ra * 32 + l32;
                if (row < nq) {
                    const float norm = l2 ? qn[row] : 0.f;
                    float *o = out + row * ldo + col0;
#pragma unroll
                    for (int g = 0; g < 4; g++) {
                        v4f v;
#pragma unroll
                        for (int t = 0; t < 4; t++) {
                            v[t] = l2 ? __builtin_fmaf(-2.f, acc[ra][4 * g + t], norm) : -acc[ra][4 * g + t];
                        }
                        if (col0 + 8 * g + 4 <= nb) {
                            *reinterpret_cast<v4f *>(o + 8 * g) = v;
                        } else {
#pragma unroll
                            for (int t = 0; t < 4; t++) {
                                if (col0 + 8 * g + t < nb) {
                                    o[8 * g + t] = v[t];
                                }
                            }
                        }
                    }
                }
            }
        }
        if (!has_next) {
            break;
        }
        it_t = n_it;
        tm = n_tm;
        j = n_j;
        jend = n_jend;
        cur = nxt;
    }
    if constexpr (FILTER) {
        flush_queue();
    }
}

struct Args {
    const float *Q;
    int64_t nq;
    const float *B;
    int64_t nb;
    int d;
    const float *qn, *bn;
    int metric;
    float *out;
    int64_t ldo;
    ScoreFilter<float> flt;
    AssignTiles assign;
    hipStream_t s;
};

constexpr int extra_lds(int mode, int qt, int k) { return mode == kFilter ? filter_lds(qt) : (mode == kAssign ? assign_lds(qt, k) : 0); }

template <int RA, int SPB, int MODE>
void launch_shape(const Args &a, int nbat)
{
    constexpr int QT = RA * 32;
    const size_t smem = (size_t)nbat * SPB * QT * 64 + extra_lds(MODE, QT, nbat * SPB * 16);
    auto kern = resident_f32_kernel<RA, SPB, MODE>;
    static std::atomic<bool> configured{false};   // per instantiation
    if (!configured) {
        hipFuncAttributes attr;
        IXA_HIP(hipFuncGetAttributes(&attr, reinterpret_cast<const void *>(kern)));
        // the fragment reads address the query tile from LDS offset 0 of the dynamic allocation only
        IXA_REQUIRE(attr.sharedSizeBytes == 0, kErrInner, "resident fp32 kernel: unexpected static LDS of %zu bytes",
                    (size_t)attr.sharedSizeBytes);
        IXA_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kLdsLimit));
        configured = true;
    }
    const int64_t tiles_m = (a.nq + QT - 1) / QT, ntiles = (a.nb + kTileRows - 1) / kTileRows;
    IXA_REQUIRE(tiles_m < (1 << 20) && ntiles < ((int64_t)1 << 30), kErrInvalidParam, "fp32 score launch too large");
    const unsigned grid = (unsigned)((device_cus() + 7) / 8 * 8);   // one persistent workgroup per CU
    const int64_t wpx = grid / 8;
    // Which operand's tiles an XCD owns.  The streamed one's, so that its L2 serves a tile to every query tile; but where an
    // XCD's share of few streamed tiles is uneven, the resident one's (both counted in rounds of tiles per workgroup).
    const int64_t rounds_b = (tiles_m * ((ntiles + 7) / 8) + wpx - 1) / wpx, rounds_q = ((tiles_m + 7) / 8 * ntiles + wpx - 1) / wpx;
    const bool own_q = MODE == kAssign && rounds_q < rounds_b;
    const int64_t tm = own_q ? (tiles_m + 7) / 8 : tiles_m, tn = own_q ? ntiles : (ntiles + 7) / 8;
    // segments: enough items for an even share per workgroup, long enough to pay for a query tile that changes
    const int seg = (int)std::min<int64_t>(16, std::max<int64_t>(1, (tn * tm + wpx * 8 - 1) / (wpx * 8)));
    hipLaunchKernelGGL(kern, dim3(grid), dim3(kWaves * 64), smem, a.s, a.Q, a.nq, a.B, a.nb, a.d, nbat, a.qn, a.bn, a.metric,
                       a.out, a.ldo, a.flt, a.assign, (int)tiles_m, (int)ntiles, seg, own_q ? 1 : 0);
}

// batches of a row: of four K-steps where that does not add padding, else of two
int batch_steps(int d) { return (d + 31) / 32 % 2 == 0 && d > 64 ? 4 : 2; }
int batches(int d, int spb) { return (d + 16 * spb - 1) / (16 * spb); }
bool fits(int d, int ra) { return (d + 31) / 32 * 32 * 4 * ra * 32 + filter_lds(ra * 32) <= kLdsLimit; }

// query blocks per tile: tiles x (blocks + 1), the one for loading and splitting a base row and for the epilogue
int tile_blocks(int64_t nq, int d)
{
    int ra = 1;
    int64_t best = INT64_MAX;
    for (int c = 8; c >= 1; c /= 2) {
        const int64_t cost = (nq + 32 * c - 1) / (32 * c) * (c + 1);
        if (fits(d, c) && cost < best) {
            best = cost;
            ra = c;
        }
    }
    return ra;
}

template <int MODE>
void launch_mode(const Args &a)
{
    const int ra = tile_blocks(a.nq, a.d), spb = ra == 8 ? 2 : batch_steps(a.d), nbat = batches(a.d, spb);
    if (ra == 8) {
        launch_shape<8, 2, MODE>(a, nbat);
    } else if (ra == 4) {
        spb == 4 ? launch_shape<4, 4, MODE>(a, nbat) : launch_shape<4, 2, MODE>(a, nbat);
    } else if (ra == 2) {
        spb == 4 ? launch_shape<2, 4, MODE>(a, nbat) : launch_shape<2, 2, MODE>(a, nbat);
    } else {
        spb == 4 ? launch_shape<1, 4, MODE>(a, nbat) : launch_shape<1, 2, MODE>(a, nbat);
    }
}

// ---- what the tiles' best become ------------------------------------------------------------------------------------------

// The best two of every vector over all tiles and the third value; a lead of more than the error bound decides, a tie of two
// goes to `pairs` (vector, two centroids), of more (or an undefined length) to `rows`.  count: the two lists' lengths.
__global__ __launch_bounds__(256) void assign_combine_kernel(const float4 *__restrict__ top, int tiles, int tile_centroids, int64_t n,
                                                             const float *__restrict__ bound, int32_t *__restrict__ out,
                                                             int4 *__restrict__ pairs,
                                                             int32_t *__restrict__ rows, int32_t *__restrict__ count)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int lane = threadIdx.x & 63;
    Best best{kNoCentroid, kNoCentroid, kNoCentroid, 0u, 0u};
    if (i < n) {
        for (int t = 0; t < tiles; t++) {
            const float4 v = top[(int64_t)t * n + i];
            const uint32_t p = __float_as_uint(v.w), c0 = (uint32_t)(t * tile_centroids);
            best.merge(Best{v.x, v.y, v.z, c0 + (p & 0xffffu), c0 + (p >> 16)});
        }
    }
    const float need = bound[i < n ? i : n - 1];
    const bool decided = i >= n || best.v1 - best.v2 > need, pair = !decided && best.v1 - best.v3 > need;
    if (i < n) {
        out[i] = (int32_t)best.p1;
    }
    const unsigned long long mp = __ballot(pair), mr = __ballot(!decided && !pair);
    if ((mp | mr) != 0) {
        int at = 0;
        if (lane == 0 && mp) {
            at = atomicAdd(count, (int)__popcll(mp));
        }
        if (lane == 1 && mr) {
            at = atomicAdd(count + 1, (int)__popcll(mr));
        }
        const int at_p = __builtin_amdgcn_readlane(at, 0), at_r = __builtin_amdgcn_readlane(at, 1);
        const unsigned long long below = (1ull << lane) - 1;
        if (pair) {
            pairs[at_p + __popcll(mp & below)] = make_int4((int)i, (int)best.p1, (int)best.p2, 0);
        } else if (!decided) {
            rows[at_r + __popcll(mr & below)] = (int32_t)i;
        }
    }
}

// the score of the exact plans: dot product left to right without FMA, then (|x|^2 + |c|^2) - g - g
__device__ __forceinline__ float canonical_l2(const float *__restrict__ x, const float *__restrict__ c, int d, float xn, float cn)
{
    float g = 0.f;
#pragma unroll 8
    for (int t = 0; t < d; t += 4) {
        const float4 a = *reinterpret_cast<const float4 *>(x + t), b = *reinterpret_cast<const float4 *>(c + t);
        g = __fadd_rn(g, __fmul_rn(a.x, b.x));
        g = __fadd_rn(g, __fmul_rn(a.y, b.y));
        g = __fadd_rn(g, __fmul_rn(a.z, b.z));
        g = __fadd_rn(g, __fmul_rn(a.w, b.w));
    }
    return __fsub_rn(__fsub_rn(__fadd_rn(xn, cn), g), g);
}

constexpr int kResolveRows = 16;   // vectors that a wavefront of the next kernel takes at a time, at most

// What assign_combine_kernel has left open, from canonical scores: first the pairs, a lane for each of the two centroids; then the
// vectors with more.  A wavefront takes up to sixteen of them, and a lane a word of a tile's centroids: where the tile's best is
// within reach of the vector's best, the best and the second if they are, or all that are within reach of the tile's best where
// the third is.  The (vector, centroid) items are gathered in LDS and scored 64 at a time, a lane for each, whatever vectors they
// belong to; the least key of every vector is kept in LDS.  Adding 200000 x 128 of 64 components of deviation 0.25 to 1024 lists, us
// (every centroid of a crowded tile scored / this): component centres of deviation 1 691 / 671, 3 3643 / 860, 10 9329 / 980; of
// deviation 1 with an offset of 24 9036 / 897.
// Equal scores: the smaller number.  A NaN is never chosen; -1 where nothing else is left.
__global__ __launch_bounds__(256) void assign_resolve_kernel(const float *__restrict__ X, const float *__restrict__ xn, int64_t n,
                                                             const float *__restrict__ C, const float *__restrict__ cn, int64_t nc,
                                                             int d, AssignTiles assign, int tiles, int tile_centroids,
                                                             const int4 *__restrict__ pairs, const int32_t *__restrict__ rows,
                                                             const int32_t *__restrict__ count, int32_t *__restrict__ out)
{
    __shared__ unsigned long long least_all[4][kResolveRows];
    __shared__ uint2 items_all[4][128];   // {vector among the wavefront's, centroid}
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t wave = (int64_t)blockIdx.x * 4 + wv, waves = (int64_t)gridDim.x * 4;
    const int npairs = count[0], nrows = count[1];
    auto key_of = [&](int64_t row, int64_t c) {
        const float v = canonical_l2(X + row * d, C + c * d, d, xn[row], cn[c]);
        return v == v ? make_key(v, (uint32_t)c) : kEmptyKey;
    };
    for (int64_t p0 = wave * 32; p0 < npairs; p0 += waves * 32) {
        const int64_t p = p0 + (lane >> 1);
        const int4 e = pairs[p < npairs ? p : npairs - 1];
        const key_t mine = key_of(e.x, lane & 1 ? e.z : e.y), other = __shfl_xor(mine, 1);
        const key_t best = mine < other ? mine : other;
        if (p < npairs && (lane & 1) == 0) {
            out[e.x] = best == kEmptyKey ? -1 : (int32_t)key_index(best);
        }
    }
    unsigned long long *least = least_all[wv];
    uint2 *items = items_all[wv];
    const int words = within_words(tile_centroids), words_log2 = __builtin_ctz(words), all_words = tiles * words;
    // few vectors: a wavefront takes fewer at a time
    const int64_t per_wave = (nrows + waves - 1) / waves;
    const int take = (int)(per_wave < kResolveRows ? per_wave : kResolveRows);
    for (int64_t r0 = wave * take; r0 < nrows; r0 += waves * take) {
        const int here = (int)(nrows - r0 < take ? nrows - r0 : take);
        const int my_row = rows[r0 + (lane < here ? lane : here - 1)];
        if (lane < kResolveRows) {
            least[lane] = kEmptyKey;
        }
        int queued = 0;   // the same in every lane
        auto score = [&](int m) {   // the first m items, at most 64; those behind them move up
            wave_lds_fence();
            const uint2 e = items[lane];
            const uint2 behind = items[64 + lane];
            const int row = __shfl(my_row, lane < m ? (int)e.x : 0);
            if (lane < m) {
                atomicMin(least + e.x, key_of(row, e.y));
            }
            wave_lds_fence();
            items[lane] = behind;
            queued -= m;
        };
        for (int v = 0; v < here; v++) {
            const int64_t row = __builtin_amdgcn_readlane(my_row, v);
            const float need = assign.need[row];
            float lead = kNoCentroid;
            for (int t = lane; t < tiles; t += 64) {
                lead = fmaxf(lead, assign.top[(int64_t)t * n + row].x);
            }
            for (int o = 32; o > 0; o >>= 1) {
                lead = fmaxf(lead, __shfl_xor(lead, o));
            }
            const float reach = lead - need;
            for (int w0 = 0; w0 < all_words; w0 += 64) {
                const int w = w0 + lane, t = w >> words_log2, j = w & (words - 1);
                const int jh = j / (words / 2), jw = j % (words / 2);   // half of the wavefront, its word
                uint32_t bits = 0;
                // (written so that an undefined reach leaves nothing out)
                if (w < all_words) {
                    const int64_t at = (int64_t)t * n + row;
                    const float4 best = assign.top[at];
                    if (!(best.x < reach)) {
                        if (crowded(best.x, best.z, need)) {
                            bits = assign.within[at * words + j];
                        } else {
                            const uint32_t p = __float_as_uint(best.w);
                            auto bit_of = [&](uint32_t place) {   // 32 ra + 8 (r / 4) + 4 half + r % 4
                                const bool mine = (int)(place >> 6) == jw && (int)(place >> 2 & 1) == jh;
                                return mine ? 1u << ((place >> 5 & 1) * 16 + (place >> 3 & 3) * 4 + (place & 3)) : 0u;
                            };
                            bits = bit_of(p & 0xffffu) | (best.y < reach ? 0u : bit_of(p >> 16));
                        }
                    }
                }
                while (__ballot(bits != 0) != 0) {
                    const int bit = bits != 0 ? __builtin_ctz(bits) : 0;
                    const int64_t c = (int64_t)t * tile_centroids + (2 * jw + (bit >> 4)) * 32 + (bit >> 2 & 3) * 8 + jh * 4 + (bit & 3);
                    const bool has = bits != 0 && c < nc;
                    const unsigned long long m = __ballot(has);
                    if (has) {
                        items[queued + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0))] =
                            make_uint2((uint32_t)v, (uint32_t)c);
                    }
                    queued += __popcll(m);
                    if (queued >= 64) {
                        score(64);
                    }
                    bits &= bits - 1;
                }
            }
        }
        score(queued);
        wave_lds_fence();
        if (lane < here) {
            const unsigned long long best = least[lane];
            out[my_row] = best == kEmptyKey ? -1 : (int32_t)key_index(best);
        }
    }
}

}  // namespace

bool resident_f32_serves(int d) { return d % 4 == 0 && d > 32 && fits(d, 1); }

bool launch_resident_f32(const float *Q, int64_t nq, const float *B, int64_t nb, int d, const float *qn, const float *bn,
                         int metric, float *out, int64_t ldo, bool filter, ScoreFilter<float> flt, hipStream_t s)
{
    if (!resident_f32_serves(d) || nq < 1 || nb < 1 || reinterpret_cast<uintptr_t>(Q) % 16 != 0 ||
        reinterpret_cast<uintptr_t>(B) % 16 != 0 || reinterpret_cast<uintptr_t>(bn) % 16 != 0 ||
        (!filter && (ldo % 4 != 0 || reinterpret_cast<uintptr_t>(out) % 16 != 0))) {
        return false;
    }
    const Args a{Q, nq, B, nb, d, qn, bn, metric, out, ldo, flt, AssignTiles{}, s};
    if (filter) {
        launch_mode<kFilter>(a);
    } else {
        launch_mode<kStore>(a);
    }
    return true;
}

// Above 512 dimensions a tile holds 32 centroids and every vector is read once per tile (adding 40000 x 768, score matrix / this in
// us: 1500 lists 2271 / 1125, 2048 1887 / 1308, 8192 3121 / 3794; 512 dimensions, 4096 lists 1909 / 997, 384, 8192 1769 / 1272).
bool resident_assign_serves(const float *X, const float *C, int64_t nc, int d)
{
    return resident_f32_serves(d) && (d <= 512 || nc <= 4096) && reinterpret_cast<uintptr_t>(X) % 16 == 0 &&
           reinterpret_cast<uintptr_t>(C) % 16 == 0;
}

// Whether n vectors are assigned faster than from the score matrix, or by the sampled bound.  Many centroids of many dimensions are
// read for every tile of vectors, and some thousand vectors are too few to share that (adding, us, the older plans / this):
//   16384 x 512: 30 vectors 145 / 155, 1000 203 / 274, 5000 537 / 557, 20000 1753 / 1670, 100000 8292 / 7020;
//   50000 x 128: 30 104 / 117, 1000 166 / 186, 5000 378 / 380, 20000 1236 / 973; 16384 x 256: 30 114 / 101, 1000 161 / 156;
//   4096 x 1024, with 32 centroids to a tile: 300 235 / 210, 1000 250 / 283, 5000 538 / 579, 20000 1598 / 1644, 100000 7470 / 6553;
//   4096 x 768: 300 204 / 176, 1000 216 / 232, 5000 458 / 462, 20000 1299 / 1261.
bool resident_assign_pays(int64_t n, int64_t nc, int d)
{
    if (d > 512 && nc * d > 2500000) {
        return n <= 512 || n >= 32768;
    }
    return nc * d <= 5000000 || n >= 16384;
}

// Every workgroup adds up the mean of up to 64 of the centroids for itself (a component without one: 0), then takes the centroids
// wave by wave: rows = c - centre, lengths = |rows|^2, norms = the number that a sum of products with it starts from, times -2:
// |rows|^2 plus what the rounding of cn = |c|^2 has added to it.  Bound by the round trips of the mean's loads: 6 us for 1024
// centroids of 128 dimensions.
__global__ __launch_bounds__(256) void centre_centroids_kernel(const float *__restrict__ C, int64_t nc, int d, const float *__restrict__ cn,
                                                               float *__restrict__ centre, float *__restrict__ rows,
                                                               float *__restrict__ norms, float *__restrict__ lengths)
{
    extern __shared__ float mean[];   // [d]
    const int count = nc < 64 ? (int)nc : 64;
    const int64_t step = nc / count * d;
    for (int t = threadIdx.x; t < d; t += 256) {
        float sum = 0.f;
#pragma unroll 16
        for (int r = 0; r < count; r++) {
            sum += C[r * step + t];
        }
        sum /= (float)count;
        sum = fabsf(sum) < 1e38f ? sum : 0.f;
        mean[t] = sum;
        if (blockIdx.x == 0) {
            centre[t] = sum;
        }
    }
    __syncthreads();
    const int lane = threadIdx.x & 63;
    for (int64_t c = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); c < nc; c += (int64_t)gridDim.x * 4) {
        double apart = 0.0, whole = 0.0;
        for (int t = lane; t < d; t += 64) {
            const float v = C[c * d + t], r = v - mean[t];
            rows[c * d + t] = r;
            apart += (double)r * r;
            whole += (double)v * v;
        }
        for (int o = 32; o > 0; o >>= 1) {
            apart += __shfl_xor(apart, o);
            whole += __shfl_xor(whole, o);
        }
        if (lane == 0) {
            norms[c] = (float)(apart + ((double)cn[c] - whole));
            lengths[c] = (float)apart;
        }
    }
}

void launch_centre_centroids(const float *C, int64_t nc, int d, const float *cn, AssignCentroids &out, float *lengths, hipStream_t s)
{
    out.centre.resize((size_t)d);
    out.rows.resize((size_t)nc * d);
    out.norms.resize((size_t)nc);
    hipLaunchKernelGGL(centre_centroids_kernel, dim3((unsigned)std::min<int64_t>((nc + 3) / 4, device_cus() * 4)), dim3(256),
                       (size_t)d * sizeof(float), s, C, nc, d, cn, out.centre.data(), out.rows.data(), out.norms.data(), lengths);
}

void launch_resident_assign(const float *X, int64_t n, const float *C, int64_t nc, int d, const float *cn, float cmax,
                            const AssignCentroids &centred, int32_t *out, DeviceBuffer<float> &scratch, int64_t scratch_bytes,
                            hipStream_t s)
{
    if (n <= 0) {
        return;
    }
    IXA_REQUIRE(resident_assign_serves(X, C, nc, d) && nc >= 1 && n < ((int64_t)1 << 31), kErrInner,
                "assignment kernel does not serve these operands");
    const int qt = 32 * tile_blocks(nc, d);
    const int64_t tiles = (nc + qt - 1) / qt;
    // vectors per pass, and what the scratch holds of them, the widest first: of every tile the best two centroids and its crowd; what
    // is left open (pairs: {vector, two centroids}; rows: vectors with more; the lengths of the two lists); |x|^2 and the bounds
    const int words = within_words(qt);
    const int64_t per_vector = (16 + 4 * words) * tiles + 28;
    const int64_t page = std::min<int64_t>(n, std::max<int64_t>(kTileRows, (scratch_bytes - 8) / per_vector / kTileRows * kTileRows));
    scratch.resize((size_t)(page * per_vector + 8) / 4);
    float4 *top = reinterpret_cast<float4 *>(scratch.data());
    int4 *pairs = reinterpret_cast<int4 *>(top + page * tiles);
    uint32_t *within = reinterpret_cast<uint32_t *>(pairs + page);
    float *xn = reinterpret_cast<float *>(within + page * tiles * words), *need = xn + page;
    int32_t *rows = reinterpret_cast<int32_t *>(need + page), *count = rows + page;
    const AssignTiles assign{need, top, within};
    const float u = 5.9604645e-8f;
    const AssignBound bound{cmax, centred.longest, 2.f * (float)(d + 8) * u, 6.f / 262144.f,
                            (float)(3 * ((d + 31) / 32 * 32) + 6) * u};
    for (int64_t i0 = 0; i0 < n; i0 += page) {
        const int64_t m = std::min(page, n - i0);
        const float *xi = X + i0 * d;
        launch_assign_bounds(xi, m, d, centred.centre.data(), bound, xn, need, count, s);
        launch_mode<kAssign>(Args{centred.rows.data(), nc, xi, m, d, centred.norms.data(), centred.centre.data(), kMetricL2, nullptr, 0,
                                  ScoreFilter<float>{}, assign, s});
        hipLaunchKernelGGL(assign_combine_kernel, dim3((unsigned)((m + 255) / 256)), dim3(256), 0, s, top, (int)tiles, qt, m, need,
                           out + i0, pairs, rows, count);
        hipLaunchKernelGGL(assign_resolve_kernel, dim3((unsigned)std::min<int64_t>(m, device_cus() * 4)), dim3(256), 0, s, xi, xn, m, C,
                           cn, nc, d, assign, (int)tiles, qt, pairs, rows, count, out + i0);
    }
}

}  // namespace ixa

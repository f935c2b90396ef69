// fp32 Flat scores on the bf16 matrix cores, the base read as it lies.
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
// 1M x 128, 1000 queries: 1.23 PFLOP/s of bf16 products in the longest launch (0.71 of the ring kernel that reads split rows); a
// search 1763 -> 964 us.  What bounds it is what bounds the int8 kernel: the clock under dense matrix work, and LDS reads (85
// bytes per cycle and CU of 128); with few queries the base's bytes (512 MB in 100 us of the 207 of one query over 1M x 128).
//
// Score arithmetic: the accumulators start from -|b|^2 / 2 (L2; 0 for inner product) and end as u = q.b - |b|^2 / 2, and the
// score is fma(-2, u, |q|^2), or -u.  The admission test of a block of 16 rows is one compare of the largest u with a value
// that lies below every u whose score reaches the bound (test_value); what passes is tested again by its score.
#include <cmath>

#include "coarse.h"
#include "flat_resident.h"
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
// LDS behind the query tile of a filtered launch: {bound, norm, test value, -} per query, the wavefronts' queues
constexpr int filter_lds(int qt) { return qt * 16 + kWaves * kQueueKeys * 16; }
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

// RA: query blocks of 32 per tile; SPB: K-steps of 16 dimensions per batch; FILTER: append admitted keys, otherwise store
// every score.  nbat >= 2 batches cover the d dimensions.
template <int RA, int SPB, bool FILTER>
__global__ __launch_bounds__(kWaves * 64) __attribute__((amdgpu_waves_per_eu(2, 2))) void resident_f32_kernel(
    const float *__restrict__ Q, int64_t nq, const float *__restrict__ B, int64_t nb, int d, int nbat,
    const float *__restrict__ qn, const float *__restrict__ bn, int metric, float *__restrict__ out, int64_t ldo,
    ScoreFilter<float> flt, int tiles_m, int ntiles, int seg_tiles)
{
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
    const ResidentItems sched(tiles_m, ntiles, seg_tiles, xcd, wpx);
    const int S = sched.S;
    const int first_item = sched.next(wi);
    if (first_item < 0) {
        return;
    }
    const uint32_t lds_base = (uint32_t)reinterpret_cast<size_t>((__attribute__((address_space(3))) unsigned char *)lds);
    const uint32_t a_lane = lds_base + (uint32_t)(half * (QT * 32) + l32 * 16);
    float4 *meta = reinterpret_cast<float4 *>(lds + (size_t)nbat * kBatchLds);   // {tau, |q|^2, test value, -}
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
    load_norms(j);
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
#pragma unroll
        for (int r = 0; r < 16; r++) {
            c0[r] = l2 ? -0.5f * bnv[r >> 2][r & 3] : 0.f;
        }
        if (row0 + 32 > nb) {   // the last tile of the launch: rows past its end take no part
#pragma unroll
            for (int r = 0; r < 16; r++) {
                c0[r] = row0 + 4 * half + 8 * (r >> 2) + (r & 3) < nb ? c0[r] : kNoRow;
            }
        }
        uint32_t addr = a_lane;
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
                split8(raw[2 * t], raw[2 * t + 1], bh[t], bl[t]);
            }
            if constexpr (LAST) {
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
                    if constexpr (FIRST && st == 0 && f < RA) {
                        acc[ra] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bh[st], fa[u & 1][t], c0, 0, 0, 0);
                    } else {
                        acc[ra] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bh[st], fa[u & 1][t], acc[ra], 0, 0, 0);
                    }
                });
                static_for<0, G>([&](auto tc) {
                    constexpr int t = decltype(tc)::value, f = p * G + t;
                    if constexpr (f < RA) {
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
    hipStream_t s;
};

template <int RA, int SPB, bool FILTER>
void launch_shape(const Args &a, int nbat)
{
    constexpr int QT = RA * 32;
    const size_t smem = (size_t)nbat * SPB * QT * 64 + (FILTER ? filter_lds(QT) : 0);
    auto kern = resident_f32_kernel<RA, SPB, FILTER>;
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
    const int64_t wpx = grid / 8, own_n = (ntiles + 7) / 8;
    // segments: enough items for an even share per workgroup, long enough to pay for a query tile that changes
    const int seg = (int)std::min<int64_t>(16, std::max<int64_t>(1, (own_n * tiles_m + wpx * 8 - 1) / (wpx * 8)));
    hipLaunchKernelGGL(kern, dim3(grid), dim3(kWaves * 64), smem, a.s, a.Q, a.nq, a.B, a.nb, a.d, nbat, a.qn, a.bn, a.metric,
                       a.out, a.ldo, a.flt, (int)tiles_m, (int)ntiles, seg);
}

// batches of a row: of four K-steps where that does not add padding, else of two
int batch_steps(int d) { return (d + 31) / 32 % 2 == 0 && d > 64 ? 4 : 2; }
int batches(int d, int spb) { return (d + 16 * spb - 1) / (16 * spb); }
bool fits(int d, int ra)
{
    return (d + 31) / 32 * 32 * 4 * ra * 32 + filter_lds(ra * 32) <= kLdsLimit;
}

template <bool FILTER>
void launch_filter(const Args &a)
{
    // query blocks per tile: tiles x (blocks + 1), the one for loading and splitting a base row and for the epilogue
    int ra = 1;
    int64_t best = INT64_MAX;
    for (int c = 8; c >= 1; c /= 2) {
        const int64_t cost = (a.nq + 32 * c - 1) / (32 * c) * (c + 1);
        if (fits(a.d, c) && cost < best) {
            best = cost;
            ra = c;
        }
    }
    const int spb = ra == 8 ? 2 : batch_steps(a.d);
    const int nbat = batches(a.d, spb);
    if (ra == 8) {
        launch_shape<8, 2, FILTER>(a, nbat);
    } else if (ra == 4) {
        spb == 4 ? launch_shape<4, 4, FILTER>(a, nbat) : launch_shape<4, 2, FILTER>(a, nbat);
    } else if (ra == 2) {
        spb == 4 ? launch_shape<2, 4, FILTER>(a, nbat) : launch_shape<2, 2, FILTER>(a, nbat);
    } else {
        spb == 4 ? launch_shape<1, 4, FILTER>(a, nbat) : launch_shape<1, 2, FILTER>(a, nbat);
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
    const Args a{Q, nq, B, nb, d, qn, bn, metric, out, ldo, flt, s};
    if (filter) {
        launch_filter<true>(a);
    } else {
        launch_filter<false>(a);
    }
    return true;
}

}  // namespace ixa

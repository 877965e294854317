// Exact GEMM (AIONHIP_GEMM_EXACT_I8) and the few-row calls that share its kernel: C[m,n] = alpha * A[m,:] . W[n,:] + beta * C in
// aion's CPU arithmetic (cpu/kernels/matmul_q_i8.zig:384-497): activations int8 per (row, 32-block), exact i32 block dots, then
// acc += f32(dot) * (a_scale * w_scale). The kernel is in gemm_i8_kernel.h; here are the choice of its workgroup shape and the
// launches.
#include "gemm_i8_kernel.h"

#include <cmath>

namespace {

// C = alpha * (p[0] + p[1] + ...) + beta * C over the K slices in slice order, one thread per (row, four columns of a tile)
__global__ __launch_bounds__(256) void gemm_i8_slices_kernel(GemmSegs segs, const float *__restrict__ partial, int M, int slices, int partial_ld,
                                                             int bn, float alpha, float beta) {
    const int quads = partial_ld >> 2;
    const size_t id = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (id >= (size_t)M * quads) return;
    const int row = (int)(id / quads), pc = (int)(id % quads) * 4, tile = pc / bn;
    int si = 0;
#pragma unroll
    for (int i = 1; i < 4; ++i)
        if (i < segs.count && tile >= segs.first_tile[i]) si = i;
    const int col = pc - segs.first_tile[si] * bn;
    if (col >= segs.n[si]) return;
    f32x4 sum = *(const f32x4 *)(partial + (size_t)row * partial_ld + pc);
    for (int z = 1; z < slices; ++z) sum += *(const f32x4 *)(partial + ((size_t)z * M + row) * partial_ld + pc);
    float *dst = segs.c[si] + (size_t)row * segs.ldc[si] + col;
    const float e[4] = {sum.x, sum.y, sum.z, sum.w};
#pragma unroll
    for (int t = 0; t < 4; ++t)
        if (col + t < segs.n[si]) dst[t] = beta == 0.f ? alpha * e[t] : alpha * e[t] + beta * dst[t];
}

// How the K of a weight is divided, which fixes the order its sums are taken in: across the 1, 2, 4 or 8 wavefronts of a workgroup that
// share a tile, and across `slices` workgroups. It depends on the rows, the weight itself, the device's CUs and on whether the call may use
// scratch memory, not on the weights beside it, so that a weight that shares a launch with siblings gives the bits it gives by itself;
// the tile is chosen freely below.
struct KSplit {
    int wavefronts, slices;
    bool fewer;                                  // fewer wavefronts than a longer K would get, see k_split
    bool operator==(const KSplit &o) const { return wavefronts == o.wavefronts && slices == o.slices && fewer == o.fewer; }
};

// The workgroup shapes, and a model of their times: t = t0 + (blocks + e) * us * max(1, b * ((1 - q) * r + q * whole)), where r is the
// workgroups per CU and `whole` the same in whole rounds of `resident` workgroups per CU - a lone workgroup costs us per quant
// block of K, a filled device b * us per workgroup and CU, and what a tile costs beside its K counts as e blocks. Three sets of constants
// per block format (no t0: not a shape of that set), all of whole calls:
//   [0]  K past SHORT_BLOCKS, from a sweep of every shape over 17 .. 2048 rows x N = 1024 .. 32768 x K = 4096 .. 14336 (rms 3 .. 10 % a shape); the
//        tiles whose K is shared as far as it pays for a long K are chosen by it
//   [1]  a shorter K, the same rows and columns x K = 512, 1056, 2048 (rms 6 .. 9 %); [2] up to 16 rows x N = 1024 .. 131072. Here those tiles are
//        weighed against wide tiles whose wavefronts share K less as well: at a short K a tile's start and end weigh as much as its K, and
//        these halve them. 512 x 32768 x 512 q4 61.9 -> 42.9 us with 128 x 128 tiles, 512 x 131072 x 1056 q8 386 -> 280; 8 x 131072 x 512 q8
//        26.3 -> 20.5 with 32 x 256.
// Choosing by them costs 0.9 % over the fastest shape of each of the 1806 measured cells. The constants before these were fitted to the kernel that
// multiplied its scales on the vector ALU and did not weigh 32 x 64 tiles past 32 rows, three wavefronts to a SIMD now: 2.4 %, 356 cells more than 3 %
// slower and 31 faster (160 x 6144 x 14336 q4 69.3 -> 52.5 us, 160 x 22016 x 2048 39.8 -> 31.7, q8 41.5 -> 33.8; 700 x 11008 x 512 q8 31.0 -> 24.6).
struct I8Shape {
    int bm, bn, ks;
};
constexpr I8Shape I8_SHAPES[] = {
    {32, 32, 8}, {32, 32, 4}, {64, 32, 4}, {96, 32, 4}, {64, 64, 4}, {128, 64, 2}, {32, 64, 2}, {128, 128, 1}, {32, 128, 2}, {32, 256, 1}, {32, 64, 4},
};
constexpr int I8_COUNT = 11;
constexpr int I8_LONE4 = 1, I8_SQUARE4 = 4, I8_WIDE4 = 10;
struct I8Fit {
    int resident;
    float t0, us, b, q, e;
};
constexpr size_t SHORT_BLOCKS = 80;              // between the measured K = 2080 and 4096
constexpr I8Fit I8_FITS[3][2][I8_COUNT] = {      // [set][q4_0, q8_0][shape]
    {{{2, 5.43f, 0.0300f, 1.446f, 0.00f, 0.f}, {1, 6.60f, 0.0435f, 0.709f, 0.82f, 0.0f}, {1, 7.06f, 0.0659f, 0.777f, 0.69f, 0.1f},
      {1, 5.95f, 0.0957f, 0.765f, 0.78f, 15.8f}, {1, 6.93f, 0.1099f, 0.832f, 0.74f, 10.9f}, {1, 10.00f, 0.2451f, 0.755f, 0.75f, 3.2f}, {}, {}, {}, {},
      {1, 7.15f, 0.0648f, 0.802f, 0.76f, 0.8f}},
     {{}, {1, 6.38f, 0.0418f, 0.820f, 0.96f, 0.0f}, {1, 6.85f, 0.0647f, 0.853f, 0.74f, 0.0f}, {1, 6.35f, 0.0937f, 0.837f, 0.68f, 8.1f},
      {1, 7.58f, 0.1109f, 0.877f, 0.67f, 5.2f}, {1, 10.00f, 0.2428f, 0.773f, 0.66f, 2.9f}, {}, {}, {}, {}, {1, 6.81f, 0.0645f, 0.910f, 0.78f, 0.6f}}},
    {{{1, 5.15f, 0.0330f, 1.156f, 0.67f, 26.2f}, {1, 6.03f, 0.0388f, 0.769f, 0.79f, 14.4f}, {1, 6.06f, 0.0633f, 0.805f, 0.71f, 15.7f},
      {1, 5.56f, 0.0962f, 0.791f, 0.84f, 21.5f}, {1, 5.71f, 0.1124f, 0.832f, 0.77f, 20.0f}, {1, 5.72f, 0.2286f, 0.805f, 0.82f, 13.0f},
      {1, 6.20f, 0.0824f, 0.752f, 0.80f, 6.2f}, {1, 5.74f, 0.4557f, 0.827f, 0.82f, 6.7f}, {1, 6.57f, 0.1289f, 0.831f, 0.82f, 6.8f},
      {1, 6.55f, 0.2661f, 0.834f, 0.78f, 3.3f}, {1, 6.08f, 0.0633f, 0.811f, 0.78f, 14.7f}},
     {{}, {1, 6.24f, 0.0361f, 0.854f, 0.61f, 12.4f}, {1, 6.25f, 0.0629f, 0.847f, 0.61f, 14.3f}, {1, 5.69f, 0.0940f, 0.821f, 0.76f, 19.4f},
      {2, 6.15f, 0.1091f, 0.910f, 0.39f, 16.4f}, {1, 5.89f, 0.2293f, 0.819f, 0.76f, 12.1f}, {1, 6.30f, 0.0771f, 0.842f, 0.65f, 4.4f},
      {1, 5.31f, 0.4575f, 0.817f, 0.77f, 7.2f}, {1, 5.70f, 0.1319f, 0.848f, 0.79f, 12.0f}, {2, 6.34f, 0.2526f, 0.929f, 0.37f, 3.7f},
      {2, 5.74f, 0.0612f, 0.896f, 0.38f, 21.3f}}},
    {{{1, 5.12f, 0.0264f, 1.467f, 0.50f, 17.f}, {4, 4.86f, 0.0426f, 0.818f, 0.24f, 10.3f}, {}, {}, {}, {}, {3, 4.99f, 0.0804f, 0.938f, 0.34f, 2.1f},
      {}, {4, 4.72f, 0.1529f, 0.933f, 0.11f, 4.6f}, {2, 5.18f, 0.2571f, 1.286f, 0.22f, 2.f}},
     {{}, {3, 5.10f, 0.0416f, 1.259f, 0.22f, 7.6f}, {}, {}, {}, {}, {3, 4.91f, 0.0829f, 1.253f, 0.25f, 4.1f},
      {}, {3, 3.33f, 0.1636f, 1.093f, 0.26f, 10.5f}, {1, 6.76f, 0.1922f, 2.286f, 0.43f, 0.1f}}},
};
constexpr float I8_SLICE_US = 4.5f;              // the launch that adds K slices

float shape_us(const aionhip_ctx *ctx, int i, const I8Fit &f, size_t m, const size_t *ns, int count, size_t k, int slices) {
    const I8Shape &s = I8_SHAPES[i];
    const float cus = (float)(ctx->cu_count > 0 ? ctx->cu_count : 256), blocks = (float)(k / QK) / (float)slices;
    size_t tiles = 0;
    for (int w = 0; w < count; ++w) tiles += (ns[w] + s.bn - 1) / s.bn;
    const float r = (float)(tiles * ((m + s.bm - 1) / s.bm) * (size_t)slices) / cus;
    const float whole = ceilf(r / (float)f.resident) * (float)f.resident;
    return f.t0 + (blocks + f.e) * f.us * fmaxf(1.f, f.b * ((1.f - f.q) * r + f.q * whole)) + (slices > 1 ? I8_SLICE_US : 0.f);
}

int fit_set(size_t m, size_t k) { return k / QK > SHORT_BLOCKS ? 0 : m > 16 ? 1 : 2; }

// the fastest shape of a K split (-1: there is none) for m rows against weights of ns[0 .. count - 1] columns
int pick_shape(const aionhip_ctx *ctx, int dtype, size_t m, const size_t *ns, int count, size_t k, const KSplit &split, float *us) {
    const I8Fit *fits = I8_FITS[fit_set(m, k)][dtype == AIONHIP_Q8_0];
    int best = -1;
    float best_us = 0.f;
    for (int i = 0; i < I8_COUNT; ++i) {
        if (fits[i].t0 == 0.f || I8_SHAPES[i].ks != split.wavefronts) continue;
        const float t = shape_us(ctx, i, fits[i], m, ns, count, k, split.slices);
        if (best < 0 || t < best_us) {
            best = i;
            best_us = t;
        }
    }
    // Up to 16 rows the kernel keeps half of a tile, which the sets for more rows do not price. Three 32 x 32 tiles per CU or more: two of them to a
    // wavefront, half the starts and ends and half the reads of the activation (16 x 32768 x 8192: q4 50.9 -> 46.1 us, q8 69.2 -> 61.0; x 4096 27.9 -> 25.9,
    // 39.1 -> 36.0; x 2080 19.4 -> 18.4, 24.9 -> 23.9; level at two tiles per CU, and at K = 512).
    if (m <= 16 && split.wavefronts == 4 && !split.fewer) {
        size_t tiles = 0;
        for (int w = 0; w < count; ++w) tiles += (ns[w] + 31) / 32;
        best = k >= 1024 && tiles >= 3 * (ctx->cu_count > 0 ? (size_t)ctx->cu_count : 256) ? I8_WIDE4 : I8_LONE4;
        best_us = shape_us(ctx, I8_LONE4, fits[I8_LONE4], m, ns, count, k, split.slices);
    }
    if (us) *us = best_us;
    return best;
}

//   8 wavefronts: q4 against a grid of at most one 32 x 32 tile per CU, K >= 2048 (16 x 4096 x 4096: 7.0 us against 8.6 with 4; q8,
//                 twice the bytes per block, is level or better with 4)
//   2 wavefronts: from 1024 rows and two 128 x 64 tiles per CU on (2048 x 14336 x 2048: q4 188 against 213 us, q8 210 against 243;
//                 512 x 14336 x 4096 the other way, 101 against 95)
//   fewer:        a K of up to SHORT_BLOCKS, where the model finds that 5 % ahead (never more: siblings of different widths seldom differ)
//   4 slices:     few tiles against a long K, a second launch adds them in order (q4 16 x 2048 x 8192: 9.7 against 10.7 us,
//                 16 x 2048 x 14336: 11.8 against 15.0; q8, twice the bytes a tile, from K = 6144 and up to half a tile per CU on:
//                 16 x 2048 x 6144 14.9 -> 12.4 us, 16 x 4096 x 8192 20.2 -> 17.1, 16 x 3072 x 11008 25.3 -> 18.8; past K = 11008 up to
//                 three quarters: 16 x 6144 x 11008 28.8 -> 26.6, 64 x 3072 x 14336 31.1 -> 28.7)
//   3, 2 slices:  up to 32 rows against a little more than one tile per CU, where a few CUs have two and the rest wait (up to five quarters:
//                 8 x 9664 x 14336 q4 37.1 -> 31.9 us, q8 48.1 -> 40.9, 16 x 9664 x 8192 25.1 -> 23.6, 30.1 -> 28.6; up to six quarters 16 x 11008 x
//                 11008 33.1 -> 30.8, 42.8 -> 38.9, x 8192 level; at two tiles per CU slices cost 7 % and more)
KSplit k_split(const aionhip_ctx *ctx, int dtype, size_t m, size_t n, size_t k) {
    const size_t cus = ctx->cu_count > 0 ? (size_t)ctx->cu_count : 256, blocks = k / QK;
    const size_t small = ((m + 31) / 32) * ((n + 31) / 32), large = ((m + 127) / 128) * ((n + 63) / 64);
    const bool sliced = dtype == AIONHIP_Q4_0 ? (blocks >= 256 && small <= cus / 4) || (blocks >= 448 && small <= cus / 2)
                                              : (blocks >= 192 && small <= cus / 2) || (blocks >= 344 && small <= cus * 3 / 4);
    const bool uneven = m <= 32 && small > cus;
    const int slices = ctx->no_scratch_paths ? 1 : sliced ? 4
                       : uneven && small * 4 <= cus * 5 && blocks >= (dtype == AIONHIP_Q4_0 ? 256 : 204) ? 3
                       : uneven && small * 2 <= cus * 3 && blocks >= 344 ? 2 : 1;
    KSplit split{dtype == AIONHIP_Q4_0 && blocks >= 64 && small <= cus ? 8 : m >= 1024 && large >= 2 * cus ? 2 : 4, slices, false};
    if (blocks > SHORT_BLOCKS) return split;
    const I8Fit *fits = I8_FITS[fit_set(m, k)][dtype == AIONHIP_Q8_0];
    const int own = pick_shape(ctx, dtype, m, &n, 1, k, split, nullptr);
    if (fits[own].t0 == 0.f) return split;
    float best_us = 0.95f * shape_us(ctx, own, fits[own], m, &n, 1, k, 1);
    for (int ks = split.wavefronts / 2; ks >= 1; ks /= 2) {
        const KSplit fewer{ks, 1, true};
        float us = 0.f;
        if (pick_shape(ctx, dtype, m, &n, 1, k, fewer, &us) < 0 || us >= best_us) continue;
        split = fewer;
        best_us = us;
    }
    return split;
}

template <int DT, int MT, int NT, int KS, int WGM, int WGN, int SHAPE, int RQ, bool WHOLE>
int launch_kernel(aionhip_ctx *ctx, const aionhip_weight *const *ws, float *const *cs, const size_t *ldcs, int count, size_t m, PreparedAct act,
                 float alpha, float beta, int slices) {
    constexpr int BM = 32 * MT * WGM, BN = 32 * NT * WGN, LDS = gemm_i8_lds_bytes<DT == AIONHIP_Q8_0, MT, NT, KS, WGM, WGN, RQ>();
    static_assert(I8_SHAPES[SHAPE].bm == BM && I8_SHAPES[SHAPE].bn == BN && I8_SHAPES[SHAPE].ks == KS, "shape table order");
    static_assert(LDS <= 80 * 1024, "two workgroups per CU");
    static_assert((uint64_t)32 * NT * GEMM_I8_MAX_K <= (uint64_t)1 << 32, "a lane's weight offset and the group's behind it fit 32 bits");
    GemmSegs segs{};
    segs.count = count;
    int tiles = 0;
    for (int i = 0; i < count; ++i) {
        segs.qs[i] = ws[i]->qs;
        segs.sc[i] = ws[i]->sc;
        segs.c[i] = cs[i];
        segs.ldc[i] = ldcs[i];
        segs.n[i] = (int)ws[i]->n;
        segs.first_tile[i] = tiles;
        tiles += (int)((ws[i]->n + BN - 1) / BN);
    }
    const int row_tiles = (int)((m + BM - 1) / BM), groups = (int)(((ws[0]->k >> 5) + 3) / 4);
    while (slices > 1 && (groups + slices - 1) / slices * (slices - 1) >= groups) --slices;      // no empty slice
    float *partial = nullptr;
    const int partial_ld = tiles * BN;
    if (slices > 1) {
        const int rc = ensure_scratch2(ctx, (size_t)slices * m * partial_ld * sizeof(float));
        if (rc) return rc;
        partial = (float *)ctx->scratch2;
    }
    // The kernel deals tiles out in groups of eight row tiles (256 .. 1024 rows), columns within: the activation rows and weight columns that run on an XCD
    // at the same time then fit its L2 (2048 x 14336 x 4096, 64 x 64 tiles: 409 -> 387 us for q4, 524 -> 465 for q8).
    // All workgroups at once, two per CU at most: wavefronts give way to those behind them, see the kernel (128 x 16384 x 2048 q4 22.0 -> 21.3 us, q8
    // 24.2 -> 23.1; q8 512 x 4096 x 4096 35.9 -> 35.0, 256 x 4096 x 4096 23.4 -> 22.8; 48 x 9000 x 2080 q4 14.8 -> 13.9).
    const int one_round = (size_t)tiles * row_tiles * slices <= 2 * (size_t)(ctx->cu_count > 0 ? ctx->cu_count : 256);
    const auto launch = [&](auto many, const auto &form) {
        constexpr bool MANY = decltype(many)::value;
        using Segs = typename GemmSegsOf<GEMM_PLAIN, MANY>::type;
        auto *kern = gemm_i8_kernel<DT, MT, NT, KS, WGM, WGN, RQ, WHOLE, GEMM_PLAIN, MANY>;
        static std::atomic<uint64_t> attr{0};
        if (const int rc = allow_lds(ctx, attr, (const void *)kern, LDS)) return rc;
        launch_k(ctx, kern, dim3((unsigned)(tiles * row_tiles), 1, (unsigned)slices), dim3(64 * KS * WGM * WGN), LDS, (const uint8_t *)act.q, (const float *)act.scale, ws[0]->qs,
                 ws[0]->sc, (int)m, (int)ws[0]->k, (int)ws[0]->n, gemm_i8_form(one_round, slices, tiles), nullptr, GemmTail<Segs>{form, alpha, beta, partial, partial_ld});
        return (int)AIONHIP_OK;
    };
    if (const int rc = count > 1 ? launch(std::true_type{}, segs) : launch(std::false_type{}, GemmOne{{cs[0]}, {ldcs[0]}})) return rc;
    if (slices > 1) {
        const size_t threads = m * (size_t)(partial_ld >> 2);
        launch_k(ctx, gemm_i8_slices_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, segs, partial, (int)m, slices, partial_ld, BN, alpha, beta);
    }
    return AIONHIP_OK;
}

// WHOLE: K is whole groups of four blocks, as the projections of models are. The checks for blocks past the end of K cost a lone wavefront
// up to 80 ns a group (32 x 1024 x 4096 q8 11.0 -> 11.7 us, 256 x 1024 x 8192 20.0 -> 21.5).
template <int DT, int MT, int NT, int KS, int WGM, int WGN, int SHAPE, int RQ = 4>
int launch_shape(aionhip_ctx *ctx, const aionhip_weight *const *ws, float *const *cs, const size_t *ldcs, int count, size_t m, PreparedAct act,
                 float alpha, float beta, int slices) {
    if (ws[0]->k % (4 * QK) == 0) return launch_kernel<DT, MT, NT, KS, WGM, WGN, SHAPE, RQ, true>(ctx, ws, cs, ldcs, count, m, act, alpha, beta, slices);
    return launch_kernel<DT, MT, NT, KS, WGM, WGN, SHAPE, RQ, false>(ctx, ws, cs, ldcs, count, m, act, alpha, beta, slices);
}

// a shape of one row tile: up to 16 rows its kernel keeps half the sums
template <int DT, int NT, int KS, int WGN, int SHAPE>
int launch_rows32(aionhip_ctx *ctx, const aionhip_weight *const *ws, float *const *cs, const size_t *ldcs, int count, size_t m, PreparedAct act,
                  float alpha, float beta, int slices) {
    if (m <= 16) return launch_shape<DT, 1, NT, KS, 1, WGN, SHAPE, 2>(ctx, ws, cs, ldcs, count, m, act, alpha, beta, slices);
    return launch_shape<DT, 1, NT, KS, 1, WGN, SHAPE>(ctx, ws, cs, ldcs, count, m, act, alpha, beta, slices);
}

template <int DT>
int launch_split(aionhip_ctx *ctx, const aionhip_weight *const *ws, float *const *cs, const size_t *ldcs, int count, size_t m, PreparedAct act,
                 float alpha, float beta, KSplit split) {
    size_t ns[4];
    for (int i = 0; i < count; ++i) ns[i] = ws[i]->n;
    const int slices = split.slices;
    switch (pick_shape(ctx, DT, m, ns, count, ws[0]->k, split, nullptr)) {
    case 0:
        if constexpr (DT == AIONHIP_Q4_0) return launch_rows32<DT, 1, 8, 1, 0>(ctx, ws, cs, ldcs, count, m, act, alpha, beta, slices);
        break;
    case 1: return launch_rows32<DT, 1, 4, 1, 1>(ctx, ws, cs, ldcs, count, m, act, alpha, beta, slices);
    case 2: return launch_shape<DT, 2, 1, 4, 1, 1, 2>(ctx, ws, cs, ldcs, count, m, act, alpha, beta, slices);
    case 3: return launch_shape<DT, 3, 1, 4, 1, 1, 3>(ctx, ws, cs, ldcs, count, m, act, alpha, beta, slices);
    case 4: return launch_shape<DT, 2, 2, 4, 1, 1, 4>(ctx, ws, cs, ldcs, count, m, act, alpha, beta, slices);
    case 5: return launch_shape<DT, 2, 2, 2, 2, 1, 5>(ctx, ws, cs, ldcs, count, m, act, alpha, beta, slices);
    case 6: return launch_rows32<DT, 1, 2, 2, 6>(ctx, ws, cs, ldcs, count, m, act, alpha, beta, slices);
    case 7: return launch_shape<DT, 2, 2, 1, 2, 2, 7>(ctx, ws, cs, ldcs, count, m, act, alpha, beta, slices);
    case 8: return launch_rows32<DT, 2, 2, 2, 8>(ctx, ws, cs, ldcs, count, m, act, alpha, beta, slices);
    case 9: return launch_rows32<DT, 2, 1, 4, 9>(ctx, ws, cs, ldcs, count, m, act, alpha, beta, slices);
    case I8_WIDE4: return launch_rows32<DT, 2, 4, 1, I8_WIDE4>(ctx, ws, cs, ldcs, count, m, act, alpha, beta, slices);
    }
    return set_err(ctx, AIONHIP_EXECUTION_FAILED, "gemm: no tile shape for m=%zu, n=%zu, k=%zu", m, ns[0], (size_t)ws[0]->k);
}

// one launch for the weights of each K split (siblings of one model nearly always share it)
template <int DT>
int launch_dt(aionhip_ctx *ctx, const aionhip_weight *const *ws, float *const *cs, const size_t *ldcs, int count, size_t m, PreparedAct act,
              float alpha, float beta) {
    bool done[4] = {};
    for (int i = 0; i < count; ++i) {
        if (done[i]) continue;
        const KSplit split = k_split(ctx, DT, m, ws[i]->n, ws[i]->k);
        const aionhip_weight *w[4];
        float *c[4];
        size_t ld[4];
        int cnt = 0;
        for (int j = i; j < count; ++j) {
            if (done[j] || !(k_split(ctx, DT, m, ws[j]->n, ws[j]->k) == split)) continue;
            done[j] = true;
            w[cnt] = ws[j];
            c[cnt] = cs[j];
            ld[cnt++] = ldcs[j];
        }
        const int rc = launch_split<DT>(ctx, w, c, ld, cnt, m, act, alpha, beta, split);
        if (rc) return rc;
    }
    return AIONHIP_OK;
}

}  // namespace

float gemm_i8_us(const aionhip_ctx *ctx, int dtype, size_t m, size_t n, size_t k) {
    float us = 0.f;
    pick_shape(ctx, dtype, m, &n, 1, k, k_split(ctx, dtype, m, n, k), &us);
    return us;
}

bool gemm_i8_unsliced(const aionhip_ctx *ctx, int dtype, size_t m, size_t n, size_t k, int *wavefronts) {
    const KSplit split = k_split(ctx, dtype, m, n, k);
    *wavefronts = split.wavefronts;
    return split.slices == 1;
}
float gemm_i8_wide_behind_us(const aionhip_ctx *ctx, int dtype, size_t m, const size_t *ns, int count, size_t k) {
    const I8Fit *fits = I8_FITS[fit_set(m, k)][dtype == AIONHIP_Q8_0];
    float best = 0.f;
    pick_shape(ctx, dtype, m, ns, count, k, KSplit{4, 1, false}, &best);
    return fminf(shape_us(ctx, I8_SQUARE4, fits[I8_SQUARE4], m, ns, count, k, 1), shape_us(ctx, I8_WIDE4, fits[I8_WIDE4], m, ns, count, k, 1)) - best;
}
bool gemm_i8_tall(const aionhip_ctx *ctx, int dtype, size_t m, const size_t *ns, int count, size_t k) {
    const I8Fit *fits = I8_FITS[fit_set(m, k)][dtype == AIONHIP_Q8_0];
    return m > 32 && shape_us(ctx, I8_SQUARE4, fits[I8_SQUARE4], m, ns, count, k, 1) < shape_us(ctx, I8_WIDE4, fits[I8_WIDE4], m, ns, count, k, 1);
}

int launch_gemm_i8_few_rows(aionhip_ctx *ctx, const aionhip_weight *w, size_t m, PreparedAct act, float *c, size_t ldc, float alpha, float beta) {
    return w->dtype == AIONHIP_Q8_0 ? launch_dt<AIONHIP_Q8_0>(ctx, &w, &c, &ldc, 1, m, act, alpha, beta)
                                    : launch_dt<AIONHIP_Q4_0>(ctx, &w, &c, &ldc, 1, m, act, alpha, beta);
}

// 1..4 weights of one dtype, layout and K against the same prepared rows, one launch
int launch_gemm_i8_batch(aionhip_ctx *ctx, const aionhip_weight *const *ws, float *const *cs, const size_t *ldcs, int count, size_t m,
                         PreparedAct act, float alpha, float beta) {
    if (count < 1 || count > 4) return set_err(ctx, AIONHIP_INVALID_ARGUMENT, "gemm: %d weights in one launch (1..4)", count);
    const char *name = ws[0]->dtype == AIONHIP_Q8_0 ? "gemm_i8_q8" : "gemm_i8_q4";
    ProfScope scope(ctx, name);
    const int rc = ws[0]->dtype == AIONHIP_Q8_0 ? launch_dt<AIONHIP_Q8_0>(ctx, ws, cs, ldcs, count, m, act, alpha, beta)
                                                 : launch_dt<AIONHIP_Q4_0>(ctx, ws, cs, ldcs, count, m, act, alpha, beta);
    if (rc) return rc;
    LAUNCH_CHECK(ctx, name);
    return AIONHIP_OK;
}

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

// How the K of a weight is divided, which fixes the order its sums are taken in: across the 2, 4 or 8 wavefronts of a workgroup that
// share a tile, and across `slices` workgroups. It depends on the rows, K and the weight's own columns alone, so that a weight that
// shares a launch with siblings gives the bits it gives by itself; the tile is chosen freely below.
//   8 wavefronts: q4 against a grid of at most one 32 x 32 tile per CU, K >= 2048 (16 x 4096 x 4096: 7.0 us against 8.6 with 4; q8,
//                 twice the bytes per block, is level or better with 4)
//   2 wavefronts: from 1024 rows and two 128 x 64 tiles per CU on (2048 x 14336 x 2048: q4 188 against 213 us, q8 210 against 243;
//                 512 x 14336 x 4096 the other way, 101 against 95)
//   4 slices:     few tiles against a long K, a second launch adds them in order (q4 16 x 2048 x 8192: 9.7 against 10.7 us,
//                 16 x 2048 x 14336: 11.8 against 15.0; q8, twice the bytes a tile, from K = 6144 and up to half a tile per CU on:
//                 16 x 2048 x 6144 14.9 -> 12.4 us, 16 x 4096 x 8192 20.2 -> 17.1, 16 x 3072 x 11008 25.3 -> 18.8; past K = 11008 up to
//                 three quarters: 16 x 6144 x 11008 28.8 -> 26.6, 64 x 3072 x 14336 31.1 -> 28.7)
struct KSplit {
    int wavefronts, slices;
    bool operator==(const KSplit &o) const { return wavefronts == o.wavefronts && slices == o.slices; }
};
KSplit k_split(const aionhip_ctx *ctx, int dtype, size_t m, size_t n, size_t k) {
    const size_t cus = ctx->cu_count > 0 ? (size_t)ctx->cu_count : 256, blocks = k / QK;
    const size_t small = ((m + 31) / 32) * ((n + 31) / 32), large = ((m + 127) / 128) * ((n + 63) / 64);
    const bool sliced = dtype == AIONHIP_Q4_0 ? (blocks >= 256 && small <= cus / 4) || (blocks >= 448 && small <= cus / 2)
                                              : (blocks >= 192 && small <= cus / 2) || (blocks >= 344 && small <= cus * 3 / 4);
    const int slices = !ctx->no_scratch_paths && sliced ? 4 : 1;
    if (dtype == AIONHIP_Q4_0 && blocks >= 64 && small <= cus) return KSplit{8, slices};
    if (m >= 1024 && large >= 2 * cus) return KSplit{2, slices};
    return KSplit{4, slices};
}

// The workgroup shapes, and a model of their times: t = t0 + blocks * us * max(1, b * ((1 - q) * r + q * whole)), where r is the
// workgroups per CU and `whole` the same in whole rounds of `resident` workgroups per CU - a lone workgroup costs us per quant
// block of K, a filled device b * us per workgroup and CU. Fitted per block format to a sweep of 5 .. 2048 rows x N = 1024 ..
// 32768 x K = 1024 .. 14336 (rms 4 .. 11 % a shape); choosing by it costs 1 % on average over always taking the fastest.
struct I8Shape {
    int bm, bn, ks, resident;
    float t0[2], us[2], b[2], q[2];              // [0] q4_0, [1] q8_0
};
constexpr I8Shape I8_SHAPES[] = {
    {32, 32, 8, 2, {3.43f, 3.27f}, {0.0300f, 0.0468f}, {1.446f, 1.267f}, {0.00f, 0.09f}},
    {32, 32, 4, 4, {3.12f, 2.85f}, {0.0437f, 0.0449f}, {0.903f, 1.213f}, {0.07f, 0.05f}},
    {64, 32, 4, 3, {3.61f, 3.54f}, {0.0709f, 0.0686f}, {0.858f, 1.082f}, {0.15f, 0.10f}},
    {96, 32, 4, 2, {4.03f, 4.01f}, {0.1034f, 0.0993f}, {0.938f, 1.082f}, {0.16f, 0.07f}},
    {64, 64, 4, 2, {4.32f, 4.41f}, {0.1240f, 0.1187f}, {0.941f, 1.135f}, {0.28f, 0.18f}},
    {128, 64, 2, 2, {5.71f, 5.61f}, {0.2479f, 0.2357f}, {0.875f, 1.050f}, {0.27f, 0.10f}},
};
constexpr int I8_COUNT = (int)(sizeof(I8_SHAPES) / sizeof(I8_SHAPES[0]));
constexpr float I8_SLICE_US = 4.5f;              // the launch that adds K slices

// the fastest shape of a K split for m rows against weights of ns[0 .. count - 1] columns
int pick_shape(const aionhip_ctx *ctx, int dtype, size_t m, const size_t *ns, int count, size_t k, KSplit split, float *us) {
    const float cus = (float)(ctx->cu_count > 0 ? ctx->cu_count : 256), blocks = (float)(k / QK) / (float)split.slices;
    const int f = dtype == AIONHIP_Q8_0;
    int best = -1;
    float best_us = 0.f;
    for (int i = 0; i < I8_COUNT; ++i) {
        const I8Shape &s = I8_SHAPES[i];
        if (s.ks != split.wavefronts) continue;
        size_t tiles = 0;
        for (int w = 0; w < count; ++w) tiles += (ns[w] + s.bn - 1) / s.bn;
        const float r = (float)(tiles * ((m + s.bm - 1) / s.bm) * (size_t)split.slices) / cus;
        const float whole = ceilf(r / (float)s.resident) * (float)s.resident;
        const float t = s.t0[f] + blocks * s.us[f] * fmaxf(1.f, s.b[f] * ((1.f - s.q[f]) * r + s.q[f] * whole)) + (split.slices > 1 ? I8_SLICE_US : 0.f);
        if (best < 0 || t < best_us) {
            best = i;
            best_us = t;
        }
    }
    if (us) *us = best_us;
    return best;
}

template <int DT, int MT, int NT, int KS, int WGM, int SHAPE, bool WHOLE>
int launch_kernel(aionhip_ctx *ctx, const aionhip_weight *const *ws, float *const *cs, const size_t *ldcs, int count, size_t m, PreparedAct act,
                 float alpha, float beta, int slices) {
    constexpr int BM = 32 * MT * WGM, BN = 32 * NT, LDS = gemm_i8_lds_bytes<DT == AIONHIP_Q8_0, MT, NT, KS, WGM, 1, 4>();
    static_assert(I8_SHAPES[SHAPE].bm == BM && I8_SHAPES[SHAPE].bn == BN && I8_SHAPES[SHAPE].ks == KS, "shape table order");
    static_assert(LDS <= 80 * 1024, "two workgroups per CU");
    if (LDS > 64 * 1024)
        HIP_TRY(ctx, hipFuncSetAttribute((const void *)gemm_i8_kernel<DT, MT, NT, KS, WGM, 1, 4, WHOLE>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS));
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
    // Tiles are dealt out in groups of 512 or 1024 rows, columns within: the activation rows and weight columns that run on an XCD
    // at the same time then fit its L2 (2048 x 14336 x 4096, 64 x 64 tiles: 409 -> 387 us for q4, 524 -> 465 for q8).
    const int row_group = row_tiles < 8 ? row_tiles : 8;
    launch_k(ctx, gemm_i8_kernel<DT, MT, NT, KS, WGM, 1, 4, WHOLE>, dim3((unsigned)(tiles * row_tiles), 1, (unsigned)slices), dim3(64 * KS * WGM), LDS, segs,
             (const uint8_t *)act.q, (const float *)act.scale, (int)m, (int)ws[0]->k, row_tiles, row_group, tiles, alpha, beta, partial, partial_ld);
    if (slices > 1) {
        const size_t threads = m * (size_t)(partial_ld >> 2);
        launch_k(ctx, gemm_i8_slices_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, segs, partial, (int)m, slices, partial_ld, BN, alpha, beta);
    }
    return AIONHIP_OK;
}

// WHOLE: K is whole groups of four blocks, as the projections of models are. The checks for blocks past the end of K cost a lone wavefront
// up to 80 ns a group (32 x 1024 x 4096 q8 11.0 -> 11.7 us, 256 x 1024 x 8192 20.0 -> 21.5).
template <int DT, int MT, int NT, int KS, int WGM, int SHAPE>
int launch_shape(aionhip_ctx *ctx, const aionhip_weight *const *ws, float *const *cs, const size_t *ldcs, int count, size_t m, PreparedAct act,
                 float alpha, float beta, int slices) {
    if (ws[0]->k % (4 * QK) == 0) return launch_kernel<DT, MT, NT, KS, WGM, SHAPE, true>(ctx, ws, cs, ldcs, count, m, act, alpha, beta, slices);
    return launch_kernel<DT, MT, NT, KS, WGM, SHAPE, false>(ctx, ws, cs, ldcs, count, m, act, alpha, beta, slices);
}

template <int DT>
int launch_split(aionhip_ctx *ctx, const aionhip_weight *const *ws, float *const *cs, const size_t *ldcs, int count, size_t m, PreparedAct act,
                 float alpha, float beta, KSplit split) {
    size_t ns[4];
    for (int i = 0; i < count; ++i) ns[i] = ws[i]->n;
    switch (pick_shape(ctx, DT, m, ns, count, ws[0]->k, split, nullptr)) {
    case 0: return launch_shape<DT, 1, 1, 8, 1, 0>(ctx, ws, cs, ldcs, count, m, act, alpha, beta, split.slices);
    case 1: return launch_shape<DT, 1, 1, 4, 1, 1>(ctx, ws, cs, ldcs, count, m, act, alpha, beta, split.slices);
    case 2: return launch_shape<DT, 2, 1, 4, 1, 2>(ctx, ws, cs, ldcs, count, m, act, alpha, beta, split.slices);
    case 3: return launch_shape<DT, 3, 1, 4, 1, 3>(ctx, ws, cs, ldcs, count, m, act, alpha, beta, split.slices);
    case 4: return launch_shape<DT, 2, 2, 4, 1, 4>(ctx, ws, cs, ldcs, count, m, act, alpha, beta, split.slices);
    default: return launch_shape<DT, 2, 2, 2, 2, 5>(ctx, ws, cs, ldcs, count, m, act, alpha, beta, split.slices);
    }
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

// 2..8 activation rows against a weight of few columns, the dots on the matrix pipe: gemv_slim_kernel.
//
// Such a weight gives the lane-per-row kernel (gemv_rows_kernel) two workgroups per CU that each copy all rows' K into LDS before the first dot
// and read it back for every two weight rows. Here a workgroup has 16 weight rows and its 16 (8, 4) wavefronts divide K: each takes
// contiguous stages of four quant blocks, with the activation's codes of those alone, and no wavefront waits for another before the
// partial sums meet in LDS. K is always summed as 16 runs of stages (the i-th ends at stage i * stages / 16) that are added as a binary tree, one, two or
// four runs to a wavefront: the bits of a weight's results depend on its K alone, not on the wavefronts that its siblings in the launch leave
// it. 4096 rows are one workgroup per CU. The arithmetic per stage is gemv_mfma_kernel's: v_mfma_i32_16x16x64_i8
// with a block-diagonal activation operand gives the exact dots of two blocks, 16 weight rows and 8 activation rows, every lane rescales four.
// q4 nibbles stay 0..15 and a second MFMA against a constant -8 supplies their offset, which costs the vector ALU nothing.
#include "gemm_i8_kernel.h"

namespace {

using u32x2 = __attribute__((ext_vector_type(2))) unsigned int;

constexpr int SL_ROWS = 16, SL_RUN = 8, SL_PARTS = 16;      // weight rows of a workgroup; stages whose scales are held at a time; runs of K
template <int DT> struct SlCfg {
    static constexpr bool Q8 = DT == AIONHIP_Q8_0;
    static constexpr int ROWB = Q8 ? 128 : 64;                   // bytes of a weight row per stage
    static constexpr int LPR = ROWB / 16, WL = SL_ROWS * LPR / 64;      // lanes to a row of a load, loads per stage
    static constexpr int W_BYTES = SL_ROWS * ROWB, STAGE = W_BYTES + 1024;      // + the activation codes [8 rows][128]
    static constexpr int NSTG = Q8 ? 2 : 3;
    static constexpr int WAVE = NSTG * STAGE + 2048;             // + activation scales [32 blocks][8 rows], weight scales [8 stages][16 rows][4]
};

// workgroup `bid` of the kernel's grid (GemmSegs: tiles of SL_ROWS weight rows)
template <int DT, int KS, class Segs>
__device__ __forceinline__ void gemv_slim_body(const Segs &segs, int bid, const uint8_t *__restrict__ aq, const float *__restrict__ a_scale, const uint8_t *__restrict__ qs0,
                                               const __half *__restrict__ sc0, int n0, int a_tiled, int K, int m, float alpha, float beta) {
    using Cfg = SlCfg<DT>;
    constexpr bool Q8 = Cfg::Q8;
    extern __shared__ __attribute__((aligned(1024))) unsigned char s_sl[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = lane & 15, g = lane >> 4, hb = g >> 1, hh = g & 1;
    int si = 0, first_tile = 0, N = n0;
    [[maybe_unused]] const uint8_t *__restrict__ qs = qs0;       // (in the device pass only)
    const __half *__restrict__ sc = sc0;
    if constexpr (std::is_same<Segs, GemmSegs>::value) {
        if (bid >= (n0 + SL_ROWS - 1) / SL_ROWS) {       // (the second weight's first workgroup)
            si = 1;
#pragma unroll
            for (int i = 2; i < 4; ++i)
                if (i < segs.count && bid >= segs.first_tile[i]) si = i;
            qs = segs.qs[si];
            sc = segs.sc[si];
            N = segs.n[si];
            first_tile = segs.first_tile[si];
        }
    }
    float *__restrict__ c = segs.c[si];
    const size_t ldc = segs.ldc[si];
    const int row0 = (bid - first_tile) * SL_ROWS;
    constexpr int RUNS = SL_PARTS / KS;                          // of a wavefront
    const int KB = K >> 5, stages = K >> 7;
    auto run_end = [&](int i) { return (wave * RUNS + i) * stages / SL_PARTS; };
    const int s_lo = run_end(0), count = run_end(RUNS) - s_lo;
    unsigned char *ring = s_sl + wave * Cfg::WAVE;
    float *s_as = (float *)(ring + Cfg::NSTG * Cfg::STAGE);
    __half *s_ws = (__half *)(s_as + 256);

    // Loads of a stage: the weight rows, a row's lanes side by side (its 16-byte piece c in slot c ^ swz: operand reads of 16 rows then cover the
    // banks), and the activation rows, eight lanes each (rows past m: the last one again, never stored). An activation in the exact GEMM's order
    // (a_tiled: per block [half][row][16 codes]) is kept in it: lanes on neighbouring rows of one piece.
    const int w_row = lane / Cfg::LPR;
    auto swz = [](int row) { return Q8 ? row & 7 : (row >> 1) & 3; };
    const size_t pitch = Q8 ? (size_t)K : (size_t)(K >> 1);
    const int first = min(row0, N - 1);
    unsigned wo[Cfg::WL];
#pragma unroll
    for (int l = 0; l < Cfg::WL; ++l) {
        const int row = l * (64 / Cfg::LPR) + w_row;
        wo[l] = (unsigned)(min(row0 + row, N - 1) - first) * (unsigned)pitch + (unsigned)((lane % Cfg::LPR) ^ swz(row)) * 16;
    }
    const int a_row = a_tiled ? lane & 7 : lane >> 3, a_src = min(a_row, m - 1), a_stage = a_tiled ? lane >> 3 : lane & 7;
    [[maybe_unused]] const int a_step = a_tiled ? m * 128 : 128;
    [[maybe_unused]] const unsigned ao = a_tiled ? (unsigned)(a_stage * m + a_src) * 16 : (unsigned)a_src * (unsigned)K + (unsigned)(a_stage ^ a_row) * 16;
    // where piece p of row n & 7 lies
    const int a_at = a_tiled ? (n & 7) * 16 : (n & 7) * 128, a_mul = a_tiled ? 128 : 16, a_xor = a_tiled ? 0 : n & 7;
#if defined(__HIP_DEVICE_COMPILE__)   // (buffer loads: a global LDS-writing load makes the compiler wait for everything in flight before the next LDS read)
    const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)(qs + (size_t)first * pitch + (size_t)s_lo * Cfg::ROWB), 0, 0xFFFFFFFFu, 0x00027000);
    const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)(aq + (size_t)s_lo * a_step), 0, 0xFFFFFFFFu, 0x00027000);
#endif
    auto issue = [&](int s, int slot) {                          // (s past the run: its last stage again, never used)
#if defined(__HIP_DEVICE_COMPILE__)
        const int st = min(s, count - 1);
        unsigned char *dst = ring + slot * Cfg::STAGE;
#pragma unroll
        for (int l = 0; l < Cfg::WL; ++l) __builtin_amdgcn_raw_ptr_buffer_load_lds(w_rsrc, (lds_void *)(dst + l * 1024), 16, wo[l], st * Cfg::ROWB, 0, 0);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, (lds_void *)(dst + Cfg::W_BYTES), 16, ao, st * a_step, 0, 0);
#endif
    };
    constexpr int LPS = Cfg::WL + 1;
    // Scales of the next eight stages: a lane's activation row and stage, and its weight row (lane >> 2) and two stages
    f32x4 as_next;
    u32x2 ws_next[2];
    const float *asp = a_scale + (a_tiled ? (size_t)a_src : (size_t)a_src * KB);
    const __half *wsp = sc + (size_t)min(row0 + (lane >> 2), N - 1) * KB;
    auto load_scales = [&](int s) {
        const size_t kb = (size_t)min(s_lo + s + a_stage, stages - 1) * 4;
        if (a_tiled) {
#pragma unroll
            for (int i = 0; i < 4; ++i) as_next[i] = asp[(kb + i) * m];
        } else {
            as_next = *(const f32x4 *)(asp + kb);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) ws_next[i] = *(const u32x2 *)(wsp + (size_t)min(s_lo + s + i * 4 + (lane & 3), stages - 1) * 4);
    };
    f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
    [[maybe_unused]] f32x4 pair = acc, third = acc;              // runs 0 and 1 (of two: 0), run 2
    [[maybe_unused]] const int end0 = run_end(1) - s_lo, end1 = run_end(RUNS > 2 ? 2 : 1) - s_lo, end2 = run_end(RUNS > 2 ? 3 : 1) - s_lo;
    if (count > 0) {
        load_scales(0);
#pragma unroll
        for (int s = 0; s < Cfg::NSTG - 1; ++s) issue(s, s);
        int slot = 0;
        const bool a_real = (n >> 3) == hb;                      // block-diagonal: rows 0..7 the pair's first block, rows 8..15 its second
        for (int s = 0; s < count; ++s) {
            if ((s & (SL_RUN - 1)) == 0) {
#pragma unroll
                for (int i = 0; i < 4; ++i) s_as[(a_stage * 4 + i) * 8 + a_row] = as_next[i];
#pragma unroll
                for (int i = 0; i < 2; ++i) *(u32x2 *)(s_ws + ((i * 4 + (lane & 3)) * 16 + (lane >> 2)) * 4) = ws_next[i];
                load_scales(s + SL_RUN);
            }
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(vmcnt_imm(63) & ~(15 << 8));      // the slot about to be filled has been read
            issue(s + Cfg::NSTG - 1, slot == 0 ? Cfg::NSTG - 1 : slot - 1);
            __builtin_amdgcn_s_waitcnt(vmcnt_imm((Cfg::NSTG - 1) * LPS));
            asm volatile("" ::: "memory");
            const unsigned char *st = ring + slot * Cfg::STAGE;
            slot = slot + 1 == Cfg::NSTG ? 0 : slot + 1;
            const u32x2 wsv = *(const u32x2 *)(s_ws + ((s & (SL_RUN - 1)) * 16 + n) * 4);
            i32x4 A[2], B[2], d[2];
            u32x2 nib[2];
            f32x4 as4[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                A[j] = *(const i32x4 *)(st + Cfg::W_BYTES + a_at + ((j * 4 + g) ^ a_xor) * a_mul);
                if (Q8) B[j] = *(const i32x4 *)(st + n * Cfg::ROWB + ((j * 4 + g) ^ swz(n)) * 16);
                else nib[j] = *(const u32x2 *)(st + n * Cfg::ROWB + ((j * 2 + hb) ^ swz(n)) * 16 + hh * 8);
                as4[j] = *(const f32x4 *)(s_as + ((s & (SL_RUN - 1)) * 4 + 2 * j + hb) * 8 + hh * 4);
            }
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                if (!a_real) A[j] = i32x4{0, 0, 0, 0};
                if (Q8) d[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[j], B[j], i32x4{0, 0, 0, 0}, 0, 0, 0);
                else {
                    B[j] = i32x4{(int)(nib[j].x & 0x0F0F0F0Fu), (int)(nib[j].x >> 4 & 0x0F0F0F0Fu), (int)(nib[j].y & 0x0F0F0F0Fu), (int)(nib[j].y >> 4 & 0x0F0F0F0Fu)};
                    constexpr int M8 = (int)0xF8F8F8F8u;
                    d[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[j], i32x4{M8, M8, M8, M8}, i32x4{0, 0, 0, 0}, 0, 0, 0);
                    d[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[j], B[j], d[j], 0, 0, 0);
                }
            }
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const float w = __half2float(__ushort_as_half((unsigned short)((j ? wsv.y : wsv.x) >> (16 * hb))));
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[e] += (float)d[j][e] * (as4[j][e] * w);
            }
            // (a run without stages ends where the one before it does)
            if constexpr (RUNS > 1)
                if (s + 1 == end0) {
                    pair = acc;
                    acc = f32x4{0.f, 0.f, 0.f, 0.f};
                }
            if constexpr (RUNS > 2) {
                if (s + 1 == end1) {
                    pair += acc;
                    acc = f32x4{0.f, 0.f, 0.f, 0.f};
                }
                if (s + 1 == end2) {
                    third = acc;
                    acc = f32x4{0.f, 0.f, 0.f, 0.f};
                }
            }
        }
    }
    if constexpr (RUNS > 2) acc = third + acc;
    if constexpr (RUNS > 1) acc = pair + acc;
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));                    // no LDS-writing load may outlive the ring
    __syncthreads();
    f32x4 *red = (f32x4 *)s_sl;
    red[wave * 64 + lane] = acc;
    __syncthreads();
    if (threadIdx.x >= 128) return;
    const int col = threadIdx.x & 15, row = threadIdx.x >> 4;
    if (row >= m || row0 + col >= N) return;
    float sum[2][KS];                                            // the two blocks of the pairs: lanes 32 apart
#pragma unroll
    for (int w = 0; w < KS; ++w) {
        const float *p = (const float *)(red + w * 64 + (row >> 2) * 16 + col) + (row & 3);
        sum[0][w] = p[0];
        sum[1][w] = p[128];
    }
#pragma unroll
    for (int half = KS / 2; half >= 1; half /= 2)
#pragma unroll
        for (int w = 0; w < half; ++w)
#pragma unroll
            for (int i = 0; i < 2; ++i) sum[i][w] = sum[i][2 * w] + sum[i][2 * w + 1];
    const float v = alpha * (sum[0][0] + sum[1][0]);
    float *dst = c + (size_t)row * ldc + row0 + col;
    *dst = beta == 0.f ? v : v + beta * *dst;
}

// (the arguments' order: see GemmTail)
template <int DT, int KS, class Segs>
__global__ __launch_bounds__(64 * KS, 4) void gemv_slim_kernel(const uint8_t *__restrict__ aq, const float *__restrict__ a_scale, const uint8_t *__restrict__ qs0,
                                                               const __half *__restrict__ sc0, int K, int m, int n0, int a_tiled, GemmTail<Segs> tail) {
    gemv_slim_body<DT, KS>(tail.segs, (int)blockIdx.x, aq, a_scale, qs0, sc0, n0, a_tiled, K, m, tail.alpha, tail.beta);
}

// Siblings of both kinds in one grid, q4: the exact GEMM's tiles of eight wavefronts first, then this kernel's workgroups of as many. Two launches one
// after the other would leave half of the CUs to each: 8 x (5120 + 1024 + 1024) x 5120 17.6 -> 14.3 us (all
// three on the exact GEMM 11.2, with other bits for the narrow ones than they have by themselves), 8 x (8192 + 1024 + 1024) x 8192 21.7 -> 19.0 (23.2).
constexpr int GS_KS = 8;
__global__ __launch_bounds__(64 * GS_KS, 4) void gemm_slim_q4_kernel(const uint8_t *__restrict__ aq, const float *__restrict__ a_scale, int K, int m, int gemm_tiles, float alpha,
                                                                     float beta, GemmSegs gemm, GemmSegs slim) {
    if ((int)blockIdx.x < gemm_tiles)
        gemm_i8_body<AIONHIP_Q4_0, 1, 1, GS_KS, 1, 1, 2, true, GEMM_PLAIN, true>(gemm, (int)blockIdx.x, aq, a_scale, gemm.qs[0], gemm.sc[0], m, K, gemm.n[0], nullptr, gemm_tiles, 1, 0,
                                                                                 alpha, beta, nullptr, 0);
    else
        gemv_slim_body<AIONHIP_Q4_0, GS_KS>(slim, (int)blockIdx.x - gemm_tiles, aq, a_scale, slim.qs[0], slim.sc[0], slim.n[0], 1, K, m, alpha, beta);
}

int fill_segs(GemmSegs &segs, const aionhip_weight *const *ws, float *const *cs, const size_t *ldcs, int count, int rows) {
    segs = GemmSegs{};
    segs.count = count;
    int tiles = 0;
    for (int i = 0; i < count; ++i) {
        segs.qs[i] = ws[i]->qs;
        segs.sc[i] = ws[i]->sc;
        segs.c[i] = cs[i];
        segs.ldc[i] = ldcs[i];
        segs.n[i] = (int)ws[i]->n;
        segs.first_tile[i] = tiles;
        tiles += (int)((ws[i]->n + rows - 1) / rows);
    }
    return tiles;
}

template <int DT, int KS>
int launch_ks(aionhip_ctx *ctx, const aionhip_weight *const *ws, float *const *cs, const size_t *ldcs, int count, int m, PreparedAct act, float alpha, float beta) {
    constexpr int LDS = KS * SlCfg<DT>::WAVE;
    static_assert(LDS <= 160 * 1024 / (16 / KS), "16 wavefronts per CU");
    static_assert(KS * 1024 <= LDS && (KS == 4 || KS == 8 || KS == 16), "partial sums in the rings; one, two or four runs of K to a wavefront");
    GemmSegs segs;
    const int tiles = fill_segs(segs, ws, cs, ldcs, count, SL_ROWS);
    const auto launch = [&](const auto &form) {
        using Segs = typename std::decay<decltype(form)>::type;
        auto *kern = gemv_slim_kernel<DT, KS, Segs>;
        static std::atomic<uint64_t> attr{0};
        if (const int rc = allow_lds(ctx, attr, (const void *)kern, LDS)) return rc;
        launch_k(ctx, kern, dim3((unsigned)tiles), dim3(64 * KS), LDS, (const uint8_t *)act.q, (const float *)act.scale, ws[0]->qs, ws[0]->sc, (int)ws[0]->k, m, (int)ws[0]->n,
                 (int)act.tiled, GemmTail<Segs>{form, alpha, beta, nullptr, 0});
        return (int)AIONHIP_OK;
    };
    return count > 1 ? launch(segs) : launch(GemmOne{{cs[0]}, {ldcs[0]}});
}

}  // namespace

// Where it is the fastest kernel, from timing 2..8 rows against every other kernel over K = 512 .. 28672 x N = 256 .. 131072, both block formats,
// preparation included, weights rotated past the memory-side cache (the kernel it replaces / this one, us):
//   up to three workgroups per CU (12288 weight rows). q4 4 x 4096 x 14336 16.3 / 12.8, 4 x 9664 x 14336 1.6 times as fast, 3 x 3072 x 11008 1.46; 2 x
//     6144 x 8192 1.2; q8 4 x 4096 x 4096 1.2, 4 x 256 x 28672 1.5. Past them it has no fewer workgroups than its rivals have better tiles: 14336 rows
//     level, 32768 0.85 .. 1.1.
//   5..8 rows, where the exact GEMM is the rival: K up to 16384 (8 x 2048 x 28672 q4 0.82), and for q4 not between one and two workgroups per CU (8 x
//     7680 x 11008 0.85). q8 5 x 3072 x 4096 1.47, 8 x 2048 x 8192 1.31, 8 x 4096 x 14336 1.21; q4 8 x 3072 x 4096 1.33, 8 x 9664 x 8192 1.21.
// Two rows up to K = 4096 stay with gemv_rows_kernel, whose sums are the one-row kernel's to the bit.
bool gemv_slim_applies(const aionhip_ctx *ctx, const aionhip_weight *w, int m) {
    const size_t cus = ctx->cu_count > 0 ? (size_t)ctx->cu_count : 256, tiles = (w->n + SL_ROWS - 1) / SL_ROWS;
    if (m < 2 || m > 8 || w->dtype == AIONHIP_F32 || w->k % 128 != 0 || w->k < 512 || w->k > GEMM_I8_MAX_K || tiles > 3 * cus) return false;
    if (m <= 4) return m > 2 || w->k > FUSED_PAYS_K;
    return w->k <= 16384 && !(w->dtype == AIONHIP_Q4_0 && tiles > cus && tiles <= 2 * cus);
}

template <int DT>
static int launch_slim(aionhip_ctx *ctx, const aionhip_weight *const *ws, float *const *cs, const size_t *ldcs, int count, int m, PreparedAct act, float alpha, float beta) {
    // 16 wavefronts to a CU, in as few workgroups as the tiles allow
    const size_t cus = ctx->cu_count > 0 ? (size_t)ctx->cu_count : 256;
    size_t tiles = 0;
    for (int i = 0; i < count; ++i) tiles += (ws[i]->n + SL_ROWS - 1) / SL_ROWS;
    if (tiles <= cus) return launch_ks<DT, 16>(ctx, ws, cs, ldcs, count, m, act, alpha, beta);
    if (tiles <= 2 * cus) return launch_ks<DT, 8>(ctx, ws, cs, ldcs, count, m, act, alpha, beta);
    return launch_ks<DT, 4>(ctx, ws, cs, ldcs, count, m, act, alpha, beta);
}

int launch_gemv_slim(aionhip_ctx *ctx, const aionhip_weight *const *ws, float *const *cs, const size_t *ldcs, int count, int m, PreparedAct act, float alpha, float beta) {
    const char *name = ws[0]->dtype == AIONHIP_Q8_0 ? "gemv_q8_slim" : "gemv_q4_slim";
    ProfScope scope(ctx, name);
    const int rc = ws[0]->dtype == AIONHIP_Q8_0 ? launch_slim<AIONHIP_Q8_0>(ctx, ws, cs, ldcs, count, m, act, alpha, beta)
                                                : launch_slim<AIONHIP_Q4_0>(ctx, ws, cs, ldcs, count, m, act, alpha, beta);
    if (rc) return rc;
    LAUNCH_CHECK(ctx, name);
    return AIONHIP_OK;
}

bool gemm_slim_applies(const aionhip_ctx *ctx, const aionhip_weight *const *gemm, int count, int m) {
    for (int i = 0; i < count; ++i) {
        int wavefronts = 0;
        if (gemm[i]->dtype != AIONHIP_Q4_0 || !gemm_i8_unsliced(ctx, AIONHIP_Q4_0, (size_t)m, gemm[i]->n, gemm[i]->k, &wavefronts) || wavefronts != GS_KS) return false;
    }
    return true;
}

int launch_gemm_slim(aionhip_ctx *ctx, const aionhip_weight *const *gemm, float *const *gemm_cs, const size_t *gemm_ldcs, int gemm_count, const aionhip_weight *const *slim,
                     float *const *slim_cs, const size_t *slim_ldcs, int slim_count, int m, PreparedAct act, float alpha, float beta) {
    constexpr int GEMM_LDS = gemm_i8_lds_bytes<false, 1, 1, GS_KS, 1, 1, 2>(), SLIM_LDS = GS_KS * SlCfg<AIONHIP_Q4_0>::WAVE, LDS = GEMM_LDS > SLIM_LDS ? GEMM_LDS : SLIM_LDS;
    static_assert(LDS <= 64 * 1024, "no attribute to set");
    GemmSegs segs, slim_segs;
    const int gemm_tiles = fill_segs(segs, gemm, gemm_cs, gemm_ldcs, gemm_count, 32), slim_tiles = fill_segs(slim_segs, slim, slim_cs, slim_ldcs, slim_count, SL_ROWS);
    ProfScope scope(ctx, "gemm_i8_q4_slim");
    launch_k(ctx, gemm_slim_q4_kernel, dim3((unsigned)(gemm_tiles + slim_tiles)), dim3(64 * GS_KS), LDS, (const uint8_t *)act.q, (const float *)act.scale, (int)gemm[0]->k, m,
             gemm_tiles, alpha, beta, segs, slim_segs);
    LAUNCH_CHECK(ctx, "gemm_i8_q4_slim");
    return AIONHIP_OK;
}

// Launches of the exact GEMM's kernel whose wavefronts finish what belongs to a pair of columns (EPI, see gemm_i8_kernel.h):
//   GEMM_GATE  gate and up projections of a GeGLU block, the gate and the int8 preparation of the gated rows: the f32 rows of both projections and
//              their launch of gate + preparation (4.8 us for 128 rows of 8192) fall away. A workgroup's tile is 32 columns of both weights, which is a
//              quant block of the gated row.
//   GEMM_ROPE  q, k and v projections, the rotation of q and k, the f16 cast and append of k and v: likewise (3.9 us for 128 rows of 8 + 1 + 1 heads of
//              256). A workgroup's tile is 32 columns of a head and the 32 that they are rotated with.
// K is divided among as many wavefronts as the separate launches would divide it (k_split in gemm_i8.hip), so that the results are theirs to the bit.
#include "gemm_i8_kernel.h"

namespace {

template <int EPI, int DT, int MT, int KS, int WGM, int RQ, bool WHOLE, class Segs>
int launch_kernel(aionhip_ctx *ctx, const Segs &segs, int tiles, size_t k, size_t m, PreparedAct in) {
    constexpr int LDS = gemm_i8_lds_bytes<DT == AIONHIP_Q8_0, MT, 2, KS, WGM, 1, RQ>();
    static_assert(LDS <= 80 * 1024, "two workgroups per CU");
    auto *kern = gemm_i8_kernel<DT, MT, 2, KS, WGM, 1, RQ, WHOLE, EPI, true>;
    static std::atomic<uint64_t> attr{0};
    if (const int rc = allow_lds(ctx, attr, (const void *)kern, LDS)) return rc;
    const int row_tiles = (int)((m + 32 * MT * WGM - 1) / (32 * MT * WGM));
    const int one_round = (size_t)tiles * row_tiles <= 2 * (size_t)(ctx->cu_count > 0 ? ctx->cu_count : 256);
    launch_k(ctx, kern, dim3((unsigned)(tiles * row_tiles)), dim3(64 * KS * WGM), LDS, (const uint8_t *)in.q, (const float *)in.scale, segs.qs[0], segs.sc[0], (int)m, (int)k,
             segs.n[0], gemm_i8_form(one_round, 1, tiles), segs.qs[1], GemmTail<Segs>{segs, 1.f, 0.f, nullptr, 0});
    return AIONHIP_OK;
}

template <int EPI, int DT, int MT, int KS, int WGM, int RQ = 4, class Segs>
int launch_shape(aionhip_ctx *ctx, const Segs &segs, int tiles, size_t k, size_t m, PreparedAct in) {
    if (k % (4 * QK) == 0) return launch_kernel<EPI, DT, MT, KS, WGM, RQ, true>(ctx, segs, tiles, k, m, in);
    return launch_kernel<EPI, DT, MT, KS, WGM, RQ, false>(ctx, segs, tiles, k, m, in);
}

template <int EPI, int DT, class Segs>
int launch_dt(aionhip_ctx *ctx, const Segs &segs, int tiles, size_t k, size_t m, PreparedAct in, int wavefronts, bool tall) {
    if constexpr (DT == AIONHIP_Q4_0)
        if (wavefronts == 8) {
            if (m <= 16) return launch_shape<EPI, DT, 1, 8, 1, 2>(ctx, segs, tiles, k, m, in);
            return launch_shape<EPI, DT, 1, 8, 1>(ctx, segs, tiles, k, m, in);
        }
    if (wavefronts == 2) return launch_shape<EPI, DT, 2, 2, 2>(ctx, segs, tiles, k, m, in);
    if (wavefronts == 1) return launch_shape<EPI, DT, 2, 1, 2>(ctx, segs, tiles, k, m, in);
    if (m <= 16) return launch_shape<EPI, DT, 1, 4, 1, 2>(ctx, segs, tiles, k, m, in);
    if (tall) return launch_shape<EPI, DT, 2, 4, 1>(ctx, segs, tiles, k, m, in);
    return launch_shape<EPI, DT, 1, 4, 1>(ctx, segs, tiles, k, m, in);
}

// The divisions of K that have an instance: up to eight wavefronts for q4 as for the separate launches, two and one from 65 rows on (128-row
// tiles). All weights have to be divided alike.
bool pair_plan(const aionhip_ctx *ctx, const aionhip_weight *const *ws, int count, size_t m, int *wavefronts, bool *tall) {
    size_t ns[3];
    for (int i = 0; i < count; ++i) {
        int own = 0;
        if (!gemm_i8_unsliced(ctx, ws[i]->dtype, m, ws[i]->n, ws[i]->k, &own) || (i && own != *wavefronts)) return false;
        *wavefronts = own;
        ns[i] = ws[i]->n;
    }
    *tall = gemm_i8_tall(ctx, ws[0]->dtype, m, ns, count, ws[0]->k);
    return m <= 0x7FFFFFFFu && ws[0]->k <= GEMM_I8_MAX_K && (*wavefronts >= 4 || m > 64);
}

constexpr size_t LONG_K = 2560;                  // (between the measured 2048 and 4096)
size_t cus_of(const aionhip_ctx *ctx) { return ctx->cu_count > 0 ? (size_t)ctx->cu_count : 256; }

}  // namespace

// The launch is worth 2 .. 11 us less (9 .. 512 rows x 4096 .. 14336 x 1024 .. 4096, both block formats, timed behind each other in a stream) but
// for two places where the separate launches' tiles are the better ones by more than it saves, us separate -> this launch:
//   a long K, one row tile and between one and one and a half pair tiles per CU, a nearly empty second round where 32 x 32 tiles fill more of theirs: 9 and
//     16 rows x 11008 x 4096 q4 41.9 -> 43.3, 44.2 -> 45.0, q8 50.7 -> 51.7, 52.2 -> 53.6, x 8704 q8 2.6 and 2.1 us, at 32 rows level; over K = 2048 the
//     launch is level (q8) or 1 .. 2 us ahead (q4)
//   where the model of the shapes (gemm_i8.hip) has them ahead by more than 3.25 us: q8, three row tiles as one of 96 rows, 96 x 11008 x 4096 84.2 -> 86.1, x
//     14336 104.5 -> 105.8; 2.99 us of the model are 41.5 -> 40.4 at 96 x 8192 x 2048
bool gemm_i8_gate_applies(const aionhip_ctx *ctx, const aionhip_weight *gate, size_t m) {
    int wavefronts = 0;
    bool tall = false;
    const aionhip_weight *ws[2] = {gate, gate};
    if (!pair_plan(ctx, ws, 2, m, &wavefronts, &tall)) return false;
    const size_t cus = cus_of(ctx), pairs = (gate->n + 31) / 32, ns[2] = {gate->n, gate->n};
    if (gate->k > LONG_K && m <= 32 && pairs > cus && pairs * 2 < cus * 3) return false;
    return wavefronts != 4 || m <= 32 || gemm_i8_wide_behind_us(ctx, gate->dtype, m, ns, 2, gate->k) <= 3.25f;
}

int launch_gemm_i8_gate(aionhip_ctx *ctx, const aionhip_weight *gate, const aionhip_weight *up, size_t m, PreparedAct in, PreparedAct out) {
    int wavefronts = 0;
    bool tall = false;
    const aionhip_weight *ws[2] = {gate, up};
    pair_plan(ctx, ws, 2, m, &wavefronts, &tall);
    GemmSegs segs{};
    segs.count = 1;
    for (int i = 0; i < 2; ++i) {
        segs.qs[i] = ws[i]->qs;
        segs.sc[i] = ws[i]->sc;
    }
    segs.c[0] = (float *)out.q;
    segs.c[1] = out.scale;
    segs.n[0] = (int)gate->n;
    const int tiles = (int)(gate->n / 32);
    ProfScope scope(ctx, "gemm_i8_gate");
    const int rc = gate->dtype == AIONHIP_Q8_0 ? launch_dt<GEMM_GATE, AIONHIP_Q8_0>(ctx, segs, tiles, gate->k, m, in, wavefronts, tall)
                                               : launch_dt<GEMM_GATE, AIONHIP_Q4_0>(ctx, segs, tiles, gate->k, m, in, wavefronts, tall);
    if (rc) return rc;
    LAUNCH_CHECK(ctx, "gemm_i8_gate");
    return AIONHIP_OK;
}

// Microseconds of preparation + projections + rotation and append, separate launches -> these, behind each other in a stream: 128 x 2048 into 8 + 1 + 1
// heads of 256 q4 15.4 -> 13.5, q8 15.8 -> 14.5; 4096 into 32 + 8 + 8 heads of 128 64 rows 22.5 -> 19.6, 27.0 -> 24.0, 512 rows 61.7 -> 59.4; 512 x 1024 into
// 16 + 4 + 4 of 64 15.7 -> 13.3. Where q and k, v divide K differently (q4, hidden 4096, 77 .. 200 rows: few columns of k and v) the separate launches
// stay: one launch for q and one for k and v would be 28.8 -> 31.7 at 100 rows. They stay too where a pair of tiles to a workgroup costs more than the launch:
//   up to one 32 x 32 tile per CU, which pairs would leave half of the CUs: 32 rows of 4096 into 32 + 8 + 8 of 128 q4 18.2 -> 19.7, q8 21.4 -> 23.2, of 3072
//     into 24 + 8 + 8 15.2 -> 16.6, 17.1 -> 19.5; 96 x 2048 into 8 + 1 + 1 of 256 12.6 -> 13.2, 13.7 -> 14.4
//   a long K and more than one pair per CU where wide weights meet few rows, up to 96 of q8 or a K among eight wavefronts: 33 and 64 rows of 4096 into
//     32 + 32 + 32 of 128 q8 30.8 -> 33.3, 34.1 -> 34.9, q4 28.6 -> 29.8 and 32.1 -> 31.6; q8 96 rows into 32 + 8 + 8 30.0 -> 31.1, 128 rows 33.2 -> 31.7; over
//     K = 2048 the launch is 1 .. 3 us ahead there
bool gemm_i8_rope_applies(const aionhip_ctx *ctx, const aionhip_weight *const *qkv, size_t m, size_t d) {
    int wavefronts = 0;
    bool tall = false;
    if (d % 64 != 0 || !pair_plan(ctx, qkv, 3, m, &wavefronts, &tall)) return false;
    const size_t cus = cus_of(ctx), tiles = (m + 31) / 32 * ((qkv[0]->n + qkv[1]->n + qkv[2]->n) / 32);
    return tiles > cus && (tiles <= 2 * cus || qkv[0]->k <= LONG_K || (wavefronts < 8 && (qkv[0]->dtype != AIONHIP_Q8_0 || m > 96)));
}

int launch_gemm_i8_rope(aionhip_ctx *ctx, const aionhip_weight *const *qkv, size_t m, PreparedAct in, float *q_out, RopeAppend rope) {
    int wavefronts = 0;
    bool tall = false;
    pair_plan(ctx, qkv, 3, m, &wavefronts, &tall);
    GemmRopeSegs segs{};
    segs.count = 3;
    int tiles = 0;
    for (int i = 0; i < 3; ++i) {
        segs.qs[i] = qkv[i]->qs;
        segs.sc[i] = qkv[i]->sc;
        segs.n[i] = (int)qkv[i]->n;
        segs.first_tile[i] = tiles;
        tiles += (int)(qkv[i]->n / 64);
    }
    segs.q_out = q_out;
    segs.kcache = rope.kcache;
    segs.vcache = rope.vcache;
    segs.positions = rope.positions;
    segs.write_index = rope.write_index;
    segs.freq = rope.freq;
    segs.s_len = rope.s_len;
    segs.t_cap = rope.t_cap;
    segs.h_q = rope.h_q;
    segs.h_kv = rope.h_kv;
    segs.d = rope.d;
    segs.rope_pairs = rope.rope_pairs;
    ProfScope scope(ctx, "gemm_i8_rope");
    const int rc = qkv[0]->dtype == AIONHIP_Q8_0 ? launch_dt<GEMM_ROPE, AIONHIP_Q8_0>(ctx, segs, tiles, qkv[0]->k, m, in, wavefronts, tall)
                                                 : launch_dt<GEMM_ROPE, AIONHIP_Q4_0>(ctx, segs, tiles, qkv[0]->k, m, in, wavefronts, tall);
    if (rc) return rc;
    LAUNCH_CHECK(ctx, "gemm_i8_rope");
    return AIONHIP_OK;
}

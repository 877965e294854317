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
    auto *kern = gemm_i8_kernel<DT, MT, 2, KS, WGM, 1, RQ, WHOLE, EPI>;
    static std::atomic<uint64_t> attr{0};
    if (const int rc = allow_lds(ctx, attr, (const void *)kern, LDS)) return rc;
    const int row_tiles = (int)((m + 32 * MT * WGM - 1) / (32 * MT * WGM));
    const int one_round = (size_t)tiles * row_tiles <= 2 * (size_t)(ctx->cu_count > 0 ? ctx->cu_count : 256);
    launch_k(ctx, kern, dim3((unsigned)(tiles * row_tiles)), dim3(64 * KS * WGM), LDS, segs, (const uint8_t *)in.q, (const float *)in.scale, (int)m,
             (int)k, row_tiles, row_tiles < 8 ? row_tiles : 8, tiles, one_round, 1.f, 0.f, (float *)nullptr, 0);
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

}  // namespace

bool gemm_i8_gate_applies(const aionhip_ctx *ctx, const aionhip_weight *gate, size_t m) {
    int wavefronts = 0;
    bool tall = false;
    const aionhip_weight *ws[2] = {gate, gate};
    return pair_plan(ctx, ws, 2, m, &wavefronts, &tall);
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

// Microseconds of preparation + projections + rotation and append, separate launches -> these (q4 unless said): 128 x 2048 into 8 + 1 + 1 heads of
// 256 15.7 -> 13.1 (q8 15.5 -> 13.7); hidden 1024 1.25 .. 1.44 times; hidden 4096 into 32 + 8 + 8 heads of 128: 16 rows 16.0 -> 15.8, 64 rows
// 21.2 -> 17.8, 512 rows 59.5 -> 56.2; the least is q8 at 24 rows of 4096, 18.9 -> 19.4. Where q and k, v divide K differently (q4, hidden 4096, 77 .. 200
// rows: few columns of k and v) the separate launches stay: one launch for q and one for k and v would be 28.8 -> 31.7 at 100 rows.
bool gemm_i8_rope_applies(const aionhip_ctx *ctx, const aionhip_weight *const *qkv, size_t m, size_t d) {
    int wavefronts = 0;
    bool tall = false;
    return d % 64 == 0 && pair_plan(ctx, qkv, 3, m, &wavefronts, &tall);
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

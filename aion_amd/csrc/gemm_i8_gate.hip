// Gate and up projections of a GeGLU block, the gate and the int8 preparation of the gated rows as one launch of the exact GEMM's kernel (GATE, see
// gemm_i8_kernel.h): the f32 rows of both projections and their launch of gate + preparation (4.8 us for 128 rows of 8192) fall away. A
// workgroup's tile is 32 columns of both weights, which is a quant block of the gated row. K is divided among as many wavefronts as the separate
// launches would divide it (k_split in gemm_i8.hip), so that the codes and scales are theirs to the bit.
#include "gemm_i8_kernel.h"

#include <atomic>

namespace {

template <int DT, int MT, int KS, int WGM, int RQ, bool WHOLE>
int launch_kernel(aionhip_ctx *ctx, const aionhip_weight *gate, const aionhip_weight *up, size_t m, PreparedAct in, PreparedAct out) {
    constexpr int LDS = gemm_i8_lds_bytes<DT == AIONHIP_Q8_0, MT, 2, KS, WGM, 1, RQ>();
    static_assert(LDS <= 80 * 1024, "two workgroups per CU");
    auto *kern = gemm_i8_kernel<DT, MT, 2, KS, WGM, 1, RQ, WHOLE, true>;
    if (LDS > 64 * 1024) {
        static std::atomic<uint64_t> attr{0};                // devices (by number, of the first 64) that have it; per instance
        const uint64_t bit = ctx->device < 64 ? (uint64_t)1 << ctx->device : 0;
        if (!(attr.load() & bit)) {
            HIP_TRY(ctx, hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, LDS));
            attr.fetch_or(bit);
        }
    }
    GemmSegs segs{};
    segs.count = 1;
    segs.qs[0] = gate->qs;
    segs.qs[1] = up->qs;
    segs.sc[0] = gate->sc;
    segs.sc[1] = up->sc;
    segs.c[0] = (float *)out.q;
    segs.c[1] = out.scale;
    segs.n[0] = (int)gate->n;
    const int tiles = (int)(gate->n / 32), row_tiles = (int)((m + 32 * MT * WGM - 1) / (32 * MT * WGM));
    const int one_round = (size_t)tiles * row_tiles <= 2 * (size_t)(ctx->cu_count > 0 ? ctx->cu_count : 256);
    launch_k(ctx, kern, dim3((unsigned)(tiles * row_tiles)), dim3(64 * KS * WGM), LDS, segs, (const uint8_t *)in.q, (const float *)in.scale, (int)m,
             (int)gate->k, row_tiles, row_tiles < 8 ? row_tiles : 8, tiles, one_round, 1.f, 0.f, (float *)nullptr, 0);
    return AIONHIP_OK;
}

template <int DT, int MT, int KS, int WGM, int RQ = 4>
int launch_shape(aionhip_ctx *ctx, const aionhip_weight *gate, const aionhip_weight *up, size_t m, PreparedAct in, PreparedAct out) {
    if (gate->k % (4 * QK) == 0) return launch_kernel<DT, MT, KS, WGM, RQ, true>(ctx, gate, up, m, in, out);
    return launch_kernel<DT, MT, KS, WGM, RQ, false>(ctx, gate, up, m, in, out);
}

template <int DT> int launch_dt(aionhip_ctx *ctx, const aionhip_weight *gate, const aionhip_weight *up, size_t m, PreparedAct in, PreparedAct out, int wavefronts, bool tall) {
    if constexpr (DT == AIONHIP_Q4_0)
        if (wavefronts == 8) {
            if (m <= 16) return launch_shape<DT, 1, 8, 1, 2>(ctx, gate, up, m, in, out);
            return launch_shape<DT, 1, 8, 1>(ctx, gate, up, m, in, out);
        }
    if (wavefronts == 2) return launch_shape<DT, 2, 2, 2>(ctx, gate, up, m, in, out);
    if (wavefronts == 1) return launch_shape<DT, 2, 1, 2>(ctx, gate, up, m, in, out);
    if (m <= 16) return launch_shape<DT, 1, 4, 1, 2>(ctx, gate, up, m, in, out);
    if (tall) return launch_shape<DT, 2, 4, 1>(ctx, gate, up, m, in, out);
    return launch_shape<DT, 1, 4, 1>(ctx, gate, up, m, in, out);
}

}  // namespace

// The divisions of K that have a GATE instance: up to eight wavefronts for q4 as for the separate launches, two and one from 65 rows on (128-row tiles).
bool gemm_i8_gate_applies(const aionhip_ctx *ctx, const aionhip_weight *gate, size_t m) {
    int wavefronts = 0;
    bool tall = false;
    if (m > 0x7FFFFFFFu || gate->k > GEMM_I8_MAX_K || !gemm_i8_pair_plan(ctx, gate->dtype, m, gate->n, gate->k, &wavefronts, &tall)) return false;
    return wavefronts >= 4 || m > 64;
}

int launch_gemm_i8_gate(aionhip_ctx *ctx, const aionhip_weight *gate, const aionhip_weight *up, size_t m, PreparedAct in, PreparedAct out) {
    int wavefronts = 0;
    bool tall = false;
    gemm_i8_pair_plan(ctx, gate->dtype, m, gate->n, gate->k, &wavefronts, &tall);
    ProfScope scope(ctx, "gemm_i8_gate");
    const int rc = gate->dtype == AIONHIP_Q8_0 ? launch_dt<AIONHIP_Q8_0>(ctx, gate, up, m, in, out, wavefronts, tall)
                                               : launch_dt<AIONHIP_Q4_0>(ctx, gate, up, m, in, out, wavefronts, tall);
    if (rc) return rc;
    LAUNCH_CHECK(ctx, "gemm_i8_gate");
    return AIONHIP_OK;
}

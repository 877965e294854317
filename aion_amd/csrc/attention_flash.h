// The 16-row flash attention body (split mode: a decode or a short prompt; per-wavefront mode: the hi+lo precise path over
// many rows), shared by attn_flash_kernel (attention.hip) and the one-launch decoder stack (decode_stack.hip), which runs
// it as one phase of a longer kernel with the queries arriving late and the output going to its exchange buffers. The
// formulation is described at the top of attention.hip.
#pragma once
#include "attention_common.h"

namespace attn {

// NW = wavefronts per workgroup: 4 in prefill mode, 8 in split mode (a decode over a short cache
// is one workgroup whose eight wavefronts take one 32-key tile each)
template <int D, int NW, int DVS = 1>
struct FlashCfg {
    static constexpr int DV = D / DVS;                           // the workgroup's share of a value row
    static constexpr int ROW_BYTES = DV * 2;                     // unpadded: the tile is filled by LDS-writing loads
    static constexpr int WAVE_LDS = TILE_KEYS * ROW_BYTES;       // one V tile per wavefront
    static constexpr int WG_LDS = NW * WAVE_LDS;
    static constexpr int MERGE_LDS = NW * (16 * (DV + 4) + 32) * 4;   // split mode: NW x (acc[16][DV+4], ref[16], l[16]) f32
    static constexpr int Q_ROW = D * 2 + 64;                     // split mode: the 16 query rows in the K/V element type
    static constexpr int Q_OFF = WG_LDS > MERGE_LDS ? WG_LDS : MERGE_LDS;
    static constexpr int LDS_BYTES = Q_OFF + 16 * Q_ROW;
};
constexpr int SPLIT_NW = 8;
constexpr float REF_NONE = -3.402823466e38f;      // the reference of what holds no key
constexpr int MEET_PARTS = 32;     // parts that the merging workgroup adds in one tree, with all of their loads in flight

// HILO: q and the probabilities are fed to the MFMAs as a high and a low half-precision part
// (x = hi + lo, ~2x the mantissa), which keeps an f32 query path at f32-level accuracy; used when
// q arrives as f32 (aion's cached decode: f32 q over an f16 cache). K and V are exact either way.
// RING: the caches are rolling rings (a.ring = T). A template flag, not a run-time test: the identity instances
// must not carry the ring's extra live values (both kernels sit at their register limit).
// DVS (split mode): DVS workgroups share a row tile and key segment, each computing all of its scores and a DVS-th of the value
// columns (the slice_dv-th); an output element is the same sum in the same order whatever DVS is.
// What bounds it: for one token over a short cache the chain index operands -> K, V -> scores -> softmax -> product -> merge, each link
// a latency; over a long one HBM, with the wavefronts' own chains under it. The chain is kept short: one memory round trip for the
// index operands and the queries, reductions by DPP and lane swaps instead of LDS permutes, hardware exp2 (the arguments are <= 0 and
// results under 2^-126 vanish in a sum that holds a 1), V in flight under the scores. One token, one KV head of size 256, 144 keys:
// 8.0 -> 6.75 us, 6.1 with the operands in SGPRs; 1531 keys, 8 KV heads of size 128: 7.6 -> 6.0 us with eight tiles to a segment (+ 3.6 for the merge as a
// launch), 5.9 with four and the merge inside; eight sequences over 16384 keys, one KV head of size 256: 25.7 -> 23.5 us = 5.7 TB/s.
template <int KV, int D, bool SPLIT, bool HILO, bool RING, int DVS = 1, class Hooks>
__device__ __forceinline__ void attn_flash_body(const AttnArgs &a, unsigned char *lds, const int rt_block, const int seg, const int b, const int hk, Hooks &hooks,
                                                const int slice_dv = 0) {
    const int ring = RING ? a.ring : 0;
    constexpr int NW = SPLIT ? SPLIT_NW : 4;
    using Cfg = FlashCfg<D, NW, DVS>;
    static_assert(SPLIT || DVS == 1, "value columns are divided in split mode only");
    constexpr int DV = Cfg::DV;
    constexpr int KK = D / 32;   // MFMA k-steps over the head dim
    constexpr int MT = DV / 16;  // 16-wide dv tiles
    const int dv0 = DVS == 1 ? 0 : slice_dv * DV;

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = lane & 15, g = lane >> 4;
    const int unit = b * a.Hkv + hk;
    const int rt = SPLIT ? rt_block : rt_block * 4 + wave;

    // ---- this lane's query row. Loads are requested in dependency order and consumed late: the index
    // operands first, then q (its address needs no loaded value), so one memory round trip covers both.
    const int r = rt * 16 + n;
    const bool row_ok = rt < a.row_tiles && r < a.rows_total;
    // (one query per sequence: no division, some 20 dependent instructions ahead of the first load)
    const int li = row_ok && a.L > 1 ? (int)((unsigned)r / (unsigned)a.groups) : 0, gi = row_ok ? r - li * a.groups : 0;
    const int hq = hk * a.groups + gi;
    // The cache length is read with a vector load (a per-lane zero in the address keeps the compiler from
    // turning it into a scalar load, which it would wait for on the spot): it is then in flight together with
    // the position and the query loads instead of ahead of them.
    // Both loads are unconditional (an absent operand reads a word of q instead and is replaced afterwards): a
    // load under a branch is waited for at the end of its block.
    const int lane_zero = (int)__builtin_amdgcn_mbcnt_lo(0u, 0u);
    const int *len_p = a.kv_lengths ? a.kv_lengths + b : (const int *)a.q;
    const int *pos_p = a.positions ? a.positions + ((size_t)b * a.L + li) : (const int *)a.q;
    const int len_ld = len_p[lane_zero], pos_ld = *pos_p;
    // (chosen by masks the compiler cannot see through: a select it would turn back into a branch around the load)
    int len_mask = a.kv_lengths ? -1 : 0, pos_mask = a.positions ? -1 : 0;
    asm("" : "+v"(len_mask), "+v"(pos_mask));
    const int kv_end_raw = (len_ld & len_mask) | (a.T & ~len_mask);
    const int pos_raw = (pos_ld & pos_mask) | (li & ~pos_mask);

    const size_t qbase = (((size_t)b * a.L + li) * a.Hq + hq) * D;
    const bool q_f32_vec = a.q_dtype == AIONHIP_F32 && (((uintptr_t)a.q) & 15) == 0;
    const bool q_same = a.q_dtype == KV && (((uintptr_t)a.q) & 15) == 0;
    u32x4 qf[KK], qf_lo[HILO ? KK : 1];
    f32x4 qx0[KK], qx1[KK];
    // split mode, f32 queries: every wavefront needs the same 16 rows, so the workgroup fetches them once
    // (two 16-byte loads per thread instead of 2*KK per lane of every wavefront through the one L1), converts
    // and shares them through LDS; the fragments are read back after the first tile's K/V loads are issued.
    const bool q_shared = SPLIT && !HILO && q_f32_vec && D * 16 / 8 <= NW * 64;
    f32x4 qs0 = f32x4{0.f, 0.f, 0.f, 0.f}, qs1 = qs0;
    constexpr int QT = D / 8;                                    // threads per staged row (8 elements each)
    const int qs_row = threadIdx.x / QT, qs_col = (threadIdx.x % QT) * 8;
    if (q_shared && Hooks::Q_LATE) {
        // the queries are not there yet (they arrive while the first K/V tile is in flight): hooks.late_q below
    } else if (q_shared) {
        const int r2 = rt * 16 + qs_row;
        if (qs_row < 16 && rt < a.row_tiles && r2 < a.rows_total) {
            const int l2 = a.L > 1 ? (int)((unsigned)r2 / (unsigned)a.groups) : 0, g2 = r2 - l2 * a.groups;
            const f32x4 *qp = (const f32x4 *)((const float *)a.q + (((size_t)b * a.L + l2) * a.Hq + hk * a.groups + g2) * D + qs_col);
            qs0 = qp[0];
            qs1 = qp[1];
        }
    } else
    if (q_same) {                    // already in the MFMA element type: one 16-byte load per k-step
#pragma unroll
        for (int kk = 0; kk < KK; ++kk)
            qf[kk] = *(const u32x4 *)((const unsigned short *)a.q + qbase + kk * 32 + g * 8);
    } else if (q_f32_vec) {
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
            const f32x4 *qp = (const f32x4 *)((const float *)a.q + qbase + kk * 32 + g * 8);
            qx0[kk] = qp[0];
            qx1[kk] = qp[1];
        }
    }

    int kv_end = clip_kv_end(ring, a.T, kv_end_raw);
    int lo, hi;
    window_keys(a.win_left, a.win_right, a.win_chunk, max(pos_raw, 0), kv_end, lo, hi);
    clip_to_ring(ring, kv_end, lo, hi);
    lo = row_ok ? lo : 0;                                        // (a padding row's position is row 0's)
    hi = row_ok ? hi : 0;
    const int uni_lo = rows16_min_i(hi > lo ? lo : INT_MAX);
    const int uni_hi = rows16_max_i(hi > lo ? hi : 0);

    // ---- Q^T operand: 8 consecutive d of row n per k-step, converted to the K/V element type
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
        if (q_shared) break;
        if (q_same) {
            if (!row_ok) qf[kk] = u32x4{0u, 0u, 0u, 0u};
            if (HILO) qf_lo[kk] = u32x4{0u, 0u, 0u, 0u};
            continue;
        }
        float x[8];
        if (q_f32_vec) {
            x[0] = qx0[kk].x; x[1] = qx0[kk].y; x[2] = qx0[kk].z; x[3] = qx0[kk].w;
            x[4] = qx1[kk].x; x[5] = qx1[kk].y; x[6] = qx1[kk].z; x[7] = qx1[kk].w;
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j) x[j] = load_scalar(a.q, a.q_dtype, qbase + kk * 32 + g * 8 + j);
        }
        if (!HILO) {
#pragma unroll
            for (int j = 0; j < 8; ++j) x[j] = row_ok ? x[j] : 0.f;
            qf[kk] = u32x4{pack2<KV>(x[0], x[1]), pack2<KV>(x[2], x[3]), pack2<KV>(x[4], x[5]), pack2<KV>(x[6], x[7])};
            continue;
        }
        unsigned short h[8], lo8[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float xv = row_ok ? x[j] : 0.f;
            h[j] = to_half_bits<KV>(xv);
            lo8[j] = HILO ? to_half_bits<KV>(xv - from_half_bits<KV>(h[j])) : (unsigned short)0;
        }
        qf[kk] = u32x4{(unsigned)h[0] | ((unsigned)h[1] << 16), (unsigned)h[2] | ((unsigned)h[3] << 16),
                       (unsigned)h[4] | ((unsigned)h[5] << 16), (unsigned)h[6] | ((unsigned)h[7] << 16)};
        if (HILO)
            qf_lo[kk] = u32x4{(unsigned)lo8[0] | ((unsigned)lo8[1] << 16), (unsigned)lo8[2] | ((unsigned)lo8[3] << 16),
                              (unsigned)lo8[4] | ((unsigned)lo8[5] << 16), (unsigned)lo8[6] | ((unsigned)lo8[7] << 16)};
    }

    f32x4 acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;
    [[maybe_unused]] float ref_run = REF_NONE, to_ref = 1.f;         // split mode, of the last tile

    // ---- key tiles of this wavefront
    int t_begin = 0, t_end = 0, t_step = 1;
    if (uni_hi > uni_lo) {
        const int tb = uni_lo / TILE_KEYS, te = (uni_hi + TILE_KEYS - 1) / TILE_KEYS;
        if (SPLIT) {
            // a segment's tiles go round robin to eight wavefronts, which 1, 2 or 4 workgroups hold
            const int segs = a.nseg >> a.sub, mine = NW >> a.sub, whole = seg >> a.sub;
            const int per = (te - tb + segs - 1) / segs;
            t_begin = tb + whole * per + (seg - (whole << a.sub)) * mine + wave;
            t_end = wave < mine ? min(tb + (whole + 1) * per, te) : t_begin;
            t_step = NW;
        } else {
            t_begin = tb;
            t_end = te;
        }
    }

    unsigned char *vs = lds + wave * Cfg::WAVE_LDS;
    const unsigned short *kp = (const unsigned short *)a.k;
    const unsigned short *vp = (const unsigned short *)a.v;
    const size_t kv_row = (size_t)a.Hkv * D;                     // elements between consecutive tokens
    const size_t kv_base = ((size_t)b * a.T * a.Hkv + hk) * D;

    // K (MFMA operand layout, registers) of a tile is requested one tile ahead, right after the S MFMAs
    // have released the registers. V goes global -> LDS directly (global_load_lds_dwordx4, 1 KiB per
    // instruction) into this wavefront's tile, requested as soon as the previous tile's gathers are done.
    // Tile layout: key row of DV*2 bytes, 16-byte chunk c of key k at slot c ^ (2 * ((k >> 2) & 3)) ^ (8 * (k & 1)) (the
    // last term for rows of 256 bytes and more; 128-byte rows alternate bank halves by themselves): the sixteen keys
    // one transposing read of the second product covers (four key groups x four keys) then fall on eight distinct
    // 32-byte bank ranges, two keys each - 512 bytes in the two passes they need anyway. Keys outside the union interval are read from
    // a clamped in-range key instead (their probabilities are exact zeros, and the cache tail may hold
    // anything, so the value must only be finite).
    constexpr int NVI = TILE_KEYS * DV * 2 / 1024;
    constexpr int KEYS_PER_VI = 1024 / (DV * 2);
    // A row is reached by one 32 x 32 + 64-bit multiply-add; no second form for small caches, whose branch would blur the
    // compiler's count of the loads in flight (see the tile loop).
    const unsigned row_bytes = (unsigned)(kv_row * 2);
    const unsigned char *kb8 = (const unsigned char *)(kp + kv_base), *vb8 = (const unsigned char *)(vp + kv_base + dv0);
    const int k_last = RING ? max(uni_hi - 1, 0) : a.T - 1;        // the last key a K load may name
    u32x4 kf[2][KK];
    auto load_k = [&](int t) __attribute__((always_inline)) {
        const int key0 = t * TILE_KEYS;
        const TileMap tm(ring, key0);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int kabs = tm.row(min(key0 + h * 16 + n, k_last));
            const unsigned char *krow = kb8 + (size_t)(unsigned)kabs * row_bytes + (unsigned)g * 16u;
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) kf[h][kk] = *(const u32x4 *)(krow + kk * 64);
        }
    };
    const int v_key_in = (lane * 16) / (DV * 2);                     // key of this lane within one V load
    const int v_slot = ((lane * 16) % (DV * 2)) / 16;                // its 16-byte slot within the key row
    const int v_hi_key = max(uni_hi - 1, 0);
    (void)NVI; (void)KEYS_PER_VI; (void)vb8; (void)v_key_in; (void)v_slot; (void)v_hi_key;   // (used by the V loads, which exist in the device pass only)
    auto load_v = [&](int t) __attribute__((always_inline)) {
#if defined(__HIP_DEVICE_COMPILE__)   // the builtin exists in the device pass only
        const int key0 = t * TILE_KEYS;
        const TileMap tm(ring, key0);
        // As buffer loads: a global LDS-writing load counts as an LDS access too, and with one in flight the compiler waits for every
        // load before it uses any - the scores for this tile's V. Keys past the clamps fall back into the tile (it holds a visible key),
        // so an offset from the tile's first row stays below 32 rows: < 2^31 at the largest row. A ring's rows may lie before it.
        [[maybe_unused]] const __amdgpu_buffer_rsrc_t v_rsrc =
            __builtin_amdgcn_make_buffer_rsrc((void *)(vb8 + (size_t)(unsigned)key0 * row_bytes), 0, 0xFFFFFFFFu, 0x00027000);
#pragma unroll
        for (int i = 0; i < NVI; ++i) {
            const int key = i * KEYS_PER_VI + v_key_in;
            // (key >> 2) & 3 does not depend on the lane while an instruction covers at most four keys
            const int grp = KEYS_PER_VI <= 4 ? ((i * KEYS_PER_VI) >> 2) & 3 : (key >> 2) & 3;
            const int chunk = v_slot ^ (2 * grp) ^ (DV >= 128 ? 8 * (key & 1) : 0);
            const int kabs = tm.row(min(max(key0 + key, uni_lo), v_hi_key));
            if constexpr (RING)
                __builtin_amdgcn_global_load_lds(vb8 + (size_t)(unsigned)kabs * row_bytes + (unsigned)chunk * 16u, (lds_void *)(vs + i * 1024), 16, 0, 0);
            else
                __builtin_amdgcn_raw_ptr_buffer_load_lds(v_rsrc, (lds_void *)(vs + i * 1024), 16, (int)((unsigned)(kabs - key0) * row_bytes + (unsigned)chunk * 16u), 0, 0, 0);
        }
#endif
    };
    // V^T operand addresses (second product): lane = 16*g + 4*r + q reads key 4g+r (and 16+4g+r), dv 16*mt + 4q .. +3
    const int tr_r = (lane >> 2) & 3, tr_q = lane & 3;
    const unsigned v_rowaddr = (unsigned)(size_t)(lds_void *)vs + (unsigned)((4 * g + tr_r) * Cfg::ROW_BYTES + (tr_q & 1) * 8);
    const unsigned v_slot_l = (unsigned)(((tr_q >> 1) ^ (2 * g) ^ (DV >= 128 ? 8 * (tr_r & 1) : 0)) << 4);
    // The queries go through LDS between the requests for K and those for V: they arrived with the index operands, and behind the
    // LDS-writing loads the compiler would wait for V before it reads them back. Late queries arrive behind both.
    if (t_begin < t_end) {
        load_k(t_begin);
        if (Hooks::Q_LATE) load_v(t_begin);
    }
    if (q_shared) {
        unsigned char *qsm = lds + Cfg::Q_OFF;
        if (Hooks::Q_LATE) {
            const int r2 = rt * 16 + qs_row;
            const bool live = qs_row < 16 && rt < a.row_tiles && r2 < a.rows_total;
            hooks.late_q(live ? (((size_t)b * a.L + r2 / a.groups) * a.Hq + hk * a.groups + r2 % a.groups) * D + qs_col : (size_t)0, live, qs0, qs1);
        }
        if (qs_row < 16)
            *(u32x4 *)(qsm + qs_row * Cfg::Q_ROW + qs_col * 2) =
                u32x4{pack2<KV>(qs0.x, qs0.y), pack2<KV>(qs0.z, qs0.w), pack2<KV>(qs1.x, qs1.y), pack2<KV>(qs1.z, qs1.w)};
        if (Hooks::Q_LATE) __syncthreads();
        else asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");      // (no wait for the K loads in flight)
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) qf[kk] = *(const u32x4 *)(qsm + n * Cfg::Q_ROW + kk * 64 + g * 16);
    }
    if constexpr (Hooks::Q_LATE) {
        // The first tile was requested before the caller's late operands arrived; a key row written since then (the row a
        // decode step appends) is stale in it. K: the lane that holds that key takes the row from the caller instead.
        const int rel = hooks.new_key() - t_begin * TILE_KEYS;
        if (t_begin < t_end && rel >= 0 && rel < TILE_KEYS && n == (rel & 15)) {
#pragma unroll
            for (int h = 0; h < 2; ++h)
                if (h == (rel >> 4)) {
#pragma unroll
                    for (int kk = 0; kk < KK; ++kk) kf[h][kk] = hooks.new_k(hk * D + kk * 32 + g * 8);
                }
        }
    }
    // MORE: another tile of this wavefront follows. Two copies of the body rather than a test in one: every path then requests K
    // and V in the same order, and the compiler's count of the loads in flight behind K (which lets V of the same tile arrive under
    // the scores and the softmax) holds; with the test in the body it waited for everything at every tile.
    auto tile = [&](int t, auto more_c) __attribute__((always_inline)) {
        constexpr bool more = decltype(more_c)::value;
        const int key0 = t * TILE_KEYS;
        // -- S^T = K . Q^T for two 16-key halves
        f32x4 s[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int kk = 0; kk < KK; ++kk)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                s[h] = mfma16<KV>(kf[h][kk], qf[kk], s[h]);
                if (HILO) s[h] = mfma16<KV>(kf[h][kk], qf_lo[kk], s[h]);
            }
        if (more) {
            load_k(t + t_step);
            asm volatile("" ::: "memory");         // requested here, ahead of the counted wait for V below
        }
        // -- scale, soft cap, interval mask; lane holds keys key0 + h*16 + g*4 + i of row n
        float p[8];
        float mx = -INFINITY;
#pragma unroll
        for (int j = 0; j < 8; ++j) p[j] = s[j >> 2][j & 3] * a.scale;
        if (a.soft_cap > 0.f) {
#pragma unroll
            for (int j = 0; j < 8; ++j) p[j] = a.soft_cap * tanhf(p[j] / a.soft_cap);
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int key = key0 + (j >> 2) * 16 + g * 4 + (j & 3);
            p[j] = key >= lo && key < hi ? p[j] : -INFINITY;
            mx = fmaxf(mx, p[j]);
        }
        mx = groups4_max(mx);
        const float m_new = fmaxf(m_run, mx);
        float alpha = 1.f, rowsum = 0.f;
        if (m_new > -INFINITY) {
            alpha = m_run > -INFINITY ? __builtin_amdgcn_exp2f((m_run - m_new) * LOG2E) : 1.f;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                p[j] = p[j] > -INFINITY ? __builtin_amdgcn_exp2f((p[j] - m_new) * LOG2E) : 0.f;
                rowsum += p[j];
            }
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j) p[j] = 0.f;
        }
        rowsum = groups4_sum(rowsum);
        l_run = l_run * alpha + rowsum;
        m_run = m_new;
        if (SPLIT && !more) {
            // The wavefronts' results meet under references that are powers of four (of two would leave the range of floats before m does), 4^ref >= e^m: to_ref =
            // e^m / 4^ref, at most one. (Here, under the wait for V. Past 2^24, where floats are coarser than the grid, clamped; without a visible key the sums are
            // zeros under the lowest reference.)
            const float half = ceilf(m_run * (0.5f * LOG2E));
            to_ref = __builtin_amdgcn_exp2f(-2.f * fminf(fmaxf(fmaf(m_run, -0.5f * LOG2E, half), 0.f), 1.f));
            ref_run = fmaxf(half, REF_NONE);
        }
        const u32x4 pf = u32x4{pack2<KV>(p[0], p[1]), pack2<KV>(p[2], p[3]), pack2<KV>(p[4], p[5]), pack2<KV>(p[6], p[7])};
        u32x4 pf_lo = u32x4{0u, 0u, 0u, 0u};
        if (HILO) {
            const unsigned ph[4] = {pf.x, pf.y, pf.z, pf.w};
            float lo8[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) lo8[j] = p[j] - from_half_bits<KV>((unsigned short)(ph[j >> 1] >> (16 * (j & 1))));
            pf_lo = u32x4{pack2<KV>(lo8[0], lo8[1]), pack2<KV>(lo8[2], lo8[3]), pack2<KV>(lo8[4], lo8[5]), pack2<KV>(lo8[6], lo8[7])};
        }

        // -- this tile's V has landed in the wavefront's LDS tile once only the younger K loads are
        //    outstanding (loads complete in order); the tile is written and read by this wavefront only
        if (more) __builtin_amdgcn_s_waitcnt(vmcnt_imm(2 * KK));
        else __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
        if constexpr (Hooks::Q_LATE) {
            // V: the same stale row, overwritten in the wavefront's LDS tile (16-byte chunk c of key k sits in slot
            // c ^ 2 * ((k >> 2) & 3) ^ 8 * (k & 1), the last term for rows of 256 bytes and more) before any operand read
            const int rel = hooks.new_key() - key0;
            if (t == t_begin && rel >= 0 && rel < TILE_KEYS && lane < DV / 8) {
                const int slot = lane ^ (2 * ((rel >> 2) & 3)) ^ (DV >= 128 ? 8 * (rel & 1) : 0);
                *(u32x4 *)(vs + rel * Cfg::ROW_BYTES + slot * 16) = hooks.new_v(hk * D + dv0 + lane * 8);
            }
        }

        // -- O^T += V^T . P^T ; operand slot j of lane group g is key g*4+j (j<4) / 16+g*4+j-4
        const bool rescale = __any(alpha != 1.f);     // wavefront-uniform: skip 4*MT multiplies when no row's max moved
        // The V^T operand of a 16-dv tile comes by two transposing LDS reads (ds_read_b64_tr_b16: within 16 lanes, lane
        // 4r+q supplies the address of 4 consecutive dv of key r, lane i receives keys 0..3 of dv i): keys 4g+r and
        // 16+4g+r of row-major V, dv 16*mt + 4q .. +3, which is the slot order above. Written as assembly and waited for
        // by count: as a builtin the compiler would wait for every load in flight - the next tile's K - before the first.
        constexpr int VA = HILO ? 2 : MT < 4 ? MT : 4;               // operands requested ahead
        u32x4 vop[VA];
        auto v_operand = [&](auto mt_c) __attribute__((always_inline)) {
            constexpr int mt = decltype(mt_c)::value;
            const unsigned addr = v_rowaddr + (v_slot_l ^ (unsigned)(mt << 5));
            u32x2 a0, a1;
            asm volatile("ds_read_b64_tr_b16 %0, %2\n\tds_read_b64_tr_b16 %1, %2 offset:%3"
                         : "=&v"(a0), "=&v"(a1) : "v"(addr), "n"(16 * Cfg::ROW_BYTES) : "memory");
            return u32x4{a0.x, a0.y, a1.x, a1.y};
        };
        static_for<0, VA>([&](auto mc) __attribute__((always_inline)) { vop[decltype(mc)::value] = v_operand(mc); });
        static_for<0, MT>([&](auto mc) __attribute__((always_inline)) {
            constexpr int mt = decltype(mc)::value;
            constexpr int later = MT - 1 - mt < VA - 1 ? MT - 1 - mt : VA - 1;
            asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(vop[mt % VA]) : "n"(2 * later));
            f32x4 c = acc[mt];
            if (rescale) c *= alpha;
            c = mfma16<KV>(vop[mt % VA], pf, c);
            if (HILO) c = mfma16<KV>(vop[mt % VA], pf_lo, c);
            acc[mt] = c;
            if constexpr (mt + VA < MT) vop[mt % VA] = v_operand(std::integral_constant<int, mt + VA>{});
        });
        if (more) {
            asm volatile("" ::: "memory");         // the operand reads above are complete: each was waited for before its MFMA
            load_v(t + t_step);
        }
    };
    if (t_begin < t_end) {
        if (!Hooks::Q_LATE) load_v(t_begin);
        int t = t_begin;
        for (; t + t_step < t_end; t += t_step) tile(t, std::true_type{});
        tile(t, std::false_type{});
    }

    if (!SPLIT) {
        if (row_ok) {
            const float inv = l_run > 0.f ? 1.f / l_run : 0.f;      // empty interval -> zeros
            float *o = a.out + (((size_t)b * a.L + li) * a.Hq + hq) * D + g * 4;
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) *(f32x4 *)(o + mt * 16) = acc[mt] * inv;
        }
        return;
    }

    // ---- split mode: merge the wavefronts through LDS. Rows are DV+4 floats apart so that the sixteen
    // lanes of a row group write their 16-byte pieces to distinct banks.
    __syncthreads();
    float *mg = (float *)lds;
    constexpr int RS = DV + 4;                // padded row stride (floats)
    constexpr int WSTRIDE = 16 * RS + 32;     // one wavefront's slot: acc[16][RS], ref[16], l[16]
    // From here on a row's reference is 4^ref (see the last tile): the factors between wavefronts and between segments, 4^(ref - ref'), are exact (v_exp_f32 of a
    // whole number), and what a row sums to depends on the order of the sums alone. That order is one tree - a segment's eight wavefronts pairwise, then the
    // parts pairwise, a segment's parts being neighbours, 32 of them at a time - whichever workgroups hold the wavefronts and whoever merges: a sequence has the
    // same bits in every batch whose segments fit the CUs, and in the merge by the last workgroup and by the launch (down to the subnormal numbers).
    {
        float *w = mg + wave * WSTRIDE;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) *(f32x4 *)(w + n * RS + mt * 16 + g * 4) = acc[mt] * to_ref;
        if (g == 0) { w[16 * RS + n] = ref_run; w[16 * RS + 16 + n] = l_run * to_ref; }
    }
    __syncthreads();
    // every thread derives the weights 4^(ref_w - ref) of its own row from the NW references (NW LDS reads that
    // the sixteen lanes of a row share, NW exp2): cheaper than a serial pass by sixteen threads and a third barrier
    // partial slot layout in global memory (read by attn_merge_kernel): [16][D] o, [16] ref, [16] l; where the last workgroup merges, each share of the value
    // columns has slots of its own, [16][DV] o, [16] (ref, l)
    constexpr int PSTRIDE = 16 * D + 32, SSTRIDE = 16 * DV + 32;
    const size_t pslot = ((size_t)(unit * a.row_tiles + rt) * a.nseg + seg) * PSTRIDE;
    [[maybe_unused]] const unsigned meeting = (unsigned)(unit * a.row_tiles + rt) * DVS + (unsigned)slice_dv;
    [[maybe_unused]] float *const slots = a.partial + (size_t)meeting * a.nseg * SSTRIDE;
    const bool last_merges = !Hooks::Q_LATE && a.tickets;
    // Device-scope accesses: written through, read at the point where the XCDs' caches agree. As buffer accesses: 16 bytes each, and a lane past the last slot
    // gets zeros without a request.
    [[maybe_unused]] constexpr int DEVICE_SCOPE = 16;                                // the sc1 bit of a buffer access
#if defined(__HIP_DEVICE_COMPILE__)
    [[maybe_unused]] const __amdgpu_buffer_rsrc_t slots_rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)slots, 0, (unsigned)(a.nseg * SSTRIDE * 4), 0x00027000);
#endif
    for (int e = threadIdx.x; e < 16 * DV / 4; e += NW * 64) {
        const int row = e / (DV / 4), col = (e % (DV / 4)) * 4;
        float ref_w[NW], lw[NW];
        f32x4 ow[NW];
        float ref = REF_NONE;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            ref_w[w] = mg[w * WSTRIDE + 16 * RS + row];
            ref = fmaxf(ref, ref_w[w]);
        }
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            const float f = pow4(ref_w[w] - ref);
            lw[w] = mg[w * WSTRIDE + 16 * RS + 16 + row] * f;
            ow[w] = *(const f32x4 *)(mg + w * WSTRIDE + row * RS + col) * f;
        }
#pragma unroll
        for (int s = 1; s < NW; s *= 2)
#pragma unroll
            for (int w = 0; w < NW; w += 2 * s) {
                lw[w] += lw[w + s];
                ow[w] += ow[w + s];
            }
        const f32x4 o = ow[0];
        const float l_all = lw[0];
        if (a.nseg == 1) {
            const int rr = rt * 16 + row;
            if (rr < a.rows_total) {
                const int l2 = rr / a.groups, g2 = rr % a.groups;
                const float inv = l_all > 0.f ? 1.f / l_all : 0.f;
                hooks.store_out(a.out, (((size_t)b * a.L + l2) * a.Hq + hk * a.groups + g2) * D + dv0 + col, o * inv);
            }
        } else if (last_merges) {
            if (rt * 16 + row < a.rows_total) {
#if defined(__HIP_DEVICE_COMPILE__)
                const int at = (seg * SSTRIDE + row * DV + col) * 4;
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, o), slots_rsrc, at, 0, DEVICE_SCOPE);
                if (col == 0)
                    __builtin_amdgcn_raw_buffer_store_b64(u32x2{__float_as_uint(ref), __float_as_uint(l_all)}, slots_rsrc, (seg * SSTRIDE + 16 * DV + row * 2) * 4, 0, DEVICE_SCOPE);
#endif
            }
        } else if (rt * 16 + row < a.rows_total) {        // (rows past the last query row are padding: nobody reads them)
            *(f32x4 *)(a.partial + pslot + row * D + dv0 + col) = o;
            if (col == 0 && dv0 == 0) {
                a.partial[pslot + 16 * D + row] = ref;
                a.partial[pslot + 16 * D + 16 + row] = l_all;
            }
        }
    }
    if constexpr (!Hooks::Q_LATE) {
        // The workgroup that ends last merges the segments: each publishes its partial result, waits until the stores have been acknowledged and takes a
        // ticket; whoever draws the last one finds all of them. Nobody waits for anybody. No device-scope fence: it would write back and
        // invalidate the L2 of the XCD.
        if (!last_merges) return;
        int *s_ticket = (int *)(lds + Cfg::Q_OFF);                  // (the queries are dead)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (threadIdx.x == 0) *s_ticket = (int)__hip_atomic_fetch_add(a.tickets + meeting * MEET_TICKET_WORDS, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (*s_ticket != a.nseg - 1) return;
        if (threadIdx.x == 0) __hip_atomic_store(a.tickets + meeting * MEET_TICKET_WORDS, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // A wavefront merges a row: lane s has the reference and sum of part s (there are at most 64, the launcher sees to that); a lane has four columns
        // and 8 of every 8 G consecutive parts, the G lanes of a column meet by lane swaps.
        constexpr int TPR = DV / 4, G = 64 / TPR, RUNS = 4 / G;
        const int grp = lane / TPR, col = (lane % TPR) * 4, rows = min(16, a.rows_total - rt * 16);
        for (int row = wave; row < rows; row += NW) {
            u32x2 stat = {};
#if defined(__HIP_DEVICE_COMPILE__)
            stat = __builtin_amdgcn_raw_buffer_load_b64(slots_rsrc, (lane * SSTRIDE + 16 * DV + row * 2) * 4, 0, DEVICE_SCOPE);
#endif
            f32x4 o = f32x4{0.f, 0.f, 0.f, 0.f};
            float f_lane = 0.f, l_all = 0.f;
            for (int s0 = 0; s0 < a.nseg; s0 += MEET_PARTS) {
                u32x4 os[RUNS][8] = {};
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
                for (int c = 0; c < RUNS; ++c)
                    if (c == 0 || s0 + c * 8 * G < a.nseg) {
#pragma unroll
                        for (int u = 0; u < 8; ++u)
                            os[c][u] = __builtin_amdgcn_raw_buffer_load_b128(slots_rsrc, ((s0 + (c * G + grp) * 8 + u) * SSTRIDE + row * DV + col) * 4, 0, DEVICE_SCOPE);
                    }
#endif
                if (s0 == 0) {
                    const float ref = lane < a.nseg ? __uint_as_float(stat.x) : REF_NONE;
                    f_lane = pow4(ref - lanes_max(ref));
                    l_all = lanes_sum(__uint_as_float(stat.y) * f_lane);
                }
                f32x4 run[RUNS];
#pragma unroll
                for (int c = 0; c < RUNS; ++c) {
                    run[c] = f32x4{0.f, 0.f, 0.f, 0.f};
                    if (c == 0 || s0 + c * 8 * G < a.nseg) {
                        f32x4 part[8];
#pragma unroll
                        for (int u = 0; u < 8; ++u) {
                            const int s = (s0 + (c * G + grp) * 8 + u) & 63;                    // (past the last part: a factor, times zeros)
                            const float f = G == 1 ? __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(f_lane), s)) : __shfl(f_lane, s, 64);
                            part[u] = __builtin_bit_cast(f32x4, os[c][u]) * f;
                        }
#pragma unroll
                        for (int i = 1; i < 8; i *= 2)
#pragma unroll
                            for (int u = 0; u < 8; u += 2 * i) part[u] += part[u + i];
                        run[c] = part[0];
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            if constexpr (G == 4) run[c][i] = groups4_sum(run[c][i]);
                            else if constexpr (G == 2) run[c][i] += half_swap(run[c][i]);
                        }
                    }
                }
                if constexpr (RUNS == 1) o += run[0];
                else if constexpr (RUNS == 2) o += run[0] + run[1];
                else o += (run[0] + run[1]) + (run[2] + run[3]);
            }
            if (grp > 0) continue;
            const int rr = rt * 16 + row, l2 = a.L > 1 ? (int)((unsigned)rr / (unsigned)a.groups) : 0, g2 = rr - l2 * a.groups;
            const float inv = l_all > 0.f ? 1.f / l_all : 0.f;
            hooks.store_out(a.out, (((size_t)b * a.L + l2) * a.Hq + hk * a.groups + g2) * D + dv0 + col, o * inv);
        }
    }
}

}  // namespace attn

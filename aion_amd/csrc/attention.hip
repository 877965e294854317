// Attention step: grouped-query attention over token-major K/V with an interval window per query
// (aion graph/graph.zig:130-181,365-393; CPU executor cpu/exec/attention.zig:627-815,1347-1442).
//
// attn_flash_kernel - d_k = d_v in {64,128,256}, K/V f16 or bf16. Flash-style online softmax with
//   MFMA for both products, written in the transposed form so that no cross-lane shuffle of the
//   probabilities is needed:
//       S^T[keys x rows] = K_tile[keys x d] . Q^T[d x rows]          (A = K rows straight from HBM)
//       O^T[dv x rows]  += V_tile^T[dv x keys] . P^T[keys x rows]    (A = V^T gathered through LDS)
//   A wavefront owns 16 query rows (row = position-major, GQA head fastest, all sharing one K/V
//   head); each lane's accumulators, running max and sum belong to ONE query row, so the softmax
//   bookkeeping is per-lane scalar work. Two launch shapes:
//     split mode (few query rows: decode) - a workgroup is one 16-row tile x one key segment, its
//       eight wavefronts interleave 32-key tiles and merge through LDS; where CUs are idle two or four workgroups hold a segment's
//       eight wavefronts. The parts are merged by the workgroup that ends last, many of them by attn_merge_kernel (the flash-decoding split of
//       cpu/exec/attention.zig:879-962).
//       Where that leaves CUs idle, the value columns are divided over up to D / 64 workgroups as well.
//     per-wavefront mode - a workgroup is four 16-row tiles, each wavefront walks its own key range; used
//       for many query rows only when the hi+lo precise mode is on (see attn_prefill_kernel otherwise).
// attn_prefill_kernel (attention_prefill.hip) - many query rows: 128 rows per workgroup, K/V tiles shared through LDS,
//   32x32x16 MFMA (described at the kernel).
// attn_generic_kernel - any head size / f32 K,V: one wavefront per query row, scores staged in
//   global scratch. Slow; it exists so that every shape the op allows has a GPU path.
//
// Softmax uses exp2 on (s - m) * log2(e); aion's CPU path uses a 4th-order polynomial exp
// (cpu/kernels/fast_math.zig:79-92, rel. err 4e-5), so results agree to ~1e-4, not bitwise.
#include "attention_flash.h"

#include <type_traits>

namespace {
using namespace attn;

// What the body does at its two seams when it is a kernel of its own: the queries are in global memory from the start,
// the output rows go to global memory as they are.
struct FlashKernelHooks {
    static constexpr bool Q_LATE = false;
    __device__ __forceinline__ void late_q(size_t, bool, f32x4 &, f32x4 &) {}
    __device__ __forceinline__ int new_key() { return -1; }
    __device__ __forceinline__ u32x4 new_k(int) { return u32x4{0u, 0u, 0u, 0u}; }
    __device__ __forceinline__ u32x4 new_v(int) { return u32x4{0u, 0u, 0u, 0u}; }
    __device__ __forceinline__ void store_out(float *out, size_t index, f32x4 v) { *(f32x4 *)(out + index) = v; }
};

// The output rows prepared for the matmul behind them: a row of the body's last loop is written by 16 lanes or more, four columns each, so eight
// neighbours hold a quant block, as prepare_act_block8 wants it. 32-bit indices: the launcher has seen to it. What it saves is the f32 rows' way through
// memory to a launch of their own: a 128-token prompt, 26 blocks of 8 + 1 + 1 heads of 256, 1948 -> 1886 us (2.4 us a block).
struct FlashPrepareHooks : FlashKernelHooks {
    int *codes;
    float *scales;
    unsigned rows, width;
    __device__ __forceinline__ void store_out(float *, size_t index, f32x4 v) {
        const unsigned row = (unsigned)index / width, col = (unsigned)index - row * width;
        int word, sum;
        float scale;
        prepare_act_block8(v.x, v.y, v.z, v.w, word, scale, sum);
        const unsigned mt = row >> 5, r = row & 31, tile_rows = min(rows - mt * 32, 32u), block = mt * width + (col >> 5) * tile_rows;
        codes[block * 8 + (col >> 4 & 1) * tile_rows * 4 + r * 4 + (col >> 2 & 3)] = word;
        if ((col & 31) == 0) scales[block + r] = scale;
    }
};

// The leading arguments, 14 words, arrive in SGPRs with the wavefront and are what the index operands, the queries and the first K tile are addressed by;
// a structure by value (all of AttnArgs came in one) is read from memory first, and so is gridDim. heads: KV heads, query heads of each << 16; form: key
// segments, their subdivision << 12, query type << 16. One token over 1531 keys, 8 KV heads of 128, 9.03 -> 8.56 us with the merge. The grid is (row tiles x segments x shares of the value columns, KV heads, sequences).
struct FlashTail {
    float *out, *partial;
    unsigned *tickets;
    float scale, soft_cap;
    unsigned win_left, win_right, win_chunk;
    int ring, B;
    int *codes;
    float *code_scales;
};
template <int KV, int D, bool SPLIT, bool HILO, bool RING = false, int DVS = 1, bool PREPARE = false>
__global__ __launch_bounds__(SPLIT ? SPLIT_NW * 64 : 256) void attn_flash_kernel(const void *q, const int *kv_lengths, const int *positions, const void *k, const void *v, int T, int L,
                                                                                 unsigned heads, unsigned form, FlashTail tail) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    AttnArgs a{};
    a.q = q;
    a.k = k;
    a.v = v;
    a.kv_lengths = kv_lengths;
    a.positions = positions;
    a.T = T;
    a.L = L;
    a.Hkv = (int)(heads & 0xFFFFu);
    a.groups = (int)(heads >> 16);
    a.Hq = a.Hkv * a.groups;
    a.rows_total = L * a.groups;
    a.row_tiles = (a.rows_total + 15) >> 4;
    a.nseg = (int)(form & 0xFFFu);
    a.sub = (int)(form >> 12 & 0xFu);
    a.q_dtype = (int)(form >> 16);
    a.kv_dtype = KV;
    a.out = tail.out;
    a.partial = tail.partial;
    a.tickets = tail.tickets;
    a.scale = tail.scale;
    a.soft_cap = tail.soft_cap;
    a.win_left = tail.win_left;
    a.win_right = tail.win_right;
    a.win_chunk = tail.win_chunk;
    a.ring = tail.ring;
    a.B = tail.B;
    a.codes = tail.codes;
    a.code_scales = tail.code_scales;
    typename std::conditional<PREPARE, FlashPrepareHooks, FlashKernelHooks>::type hooks;
    if constexpr (PREPARE) {
        hooks.codes = a.codes;
        hooks.scales = a.code_scales;
        hooks.rows = (unsigned)(a.B * a.L);
        hooks.width = (unsigned)(a.Hq * D);
    }
    int bx = (int)blockIdx.x, slice = 0, rt = bx, seg = 0;
    if constexpr (SPLIT) {
        const int tiles = a.row_tiles * a.nseg;
        if constexpr (DVS > 1) {
#pragma unroll
            for (int i = 1; i < DVS; ++i) slice += bx >= i * tiles;
            bx -= slice * tiles;
        }
        // one row tile or one segment, the common forms, need no division
        rt = a.nseg == 1 ? bx : a.row_tiles == 1 ? 0 : (int)((unsigned)bx / (unsigned)a.nseg);
        seg = bx - rt * a.nseg;
    }
    attn_flash_body<KV, D, SPLIT, HILO, RING, DVS>(a, lds, rt, seg, (int)blockIdx.z, (int)blockIdx.y, hooks, slice);
}

inline unsigned flash_heads(const AttnArgs &a) { return (unsigned)a.Hkv | (unsigned)a.groups << 16; }
inline unsigned flash_form(const AttnArgs &a) { return (unsigned)a.nseg | (unsigned)a.sub << 12 | (unsigned)a.q_dtype << 16; }
inline FlashTail flash_tail(const AttnArgs &a) {
    return FlashTail{a.out, a.partial, a.tickets, a.scale, a.soft_cap, a.win_left, a.win_right, a.win_chunk, a.ring, a.B, a.codes, a.code_scales};
}

// Merge of the key segments as a launch: one workgroup per (row tile, 16-wide dv slice, unit). A wavefront derives the segments' exact factors for every
// fourth row, a lane to a segment (there are at most 256); thread = (8 segments of every 32, row of 16, 4 consecutive dv) adds its segments, with all
// of a round's loads in flight at once, the first round's ahead of the factors, and the four groups meet through LDS - the order of the sums in attn_flash_body.
constexpr int MERGE_DV = 16, MERGE_SG = MEET_PARTS / 8, MERGE_MOST = 256;
template <int D>
__global__ __launch_bounds__(256) void attn_merge_kernel(AttnArgs a) {
    constexpr int WSTRIDE = 16 * D + 32;
    constexpr int SLICES = D / MERGE_DV;
    __shared__ float s_f[16][MERGE_MOST], s_l[16];
    __shared__ __attribute__((aligned(16))) float s_o[MERGE_MOST / MEET_PARTS][MERGE_SG][16][MERGE_DV];
    const int unit = blockIdx.y, rt = blockIdx.x / SLICES, slice = blockIdx.x % SLICES;
    const int b = unit / a.Hkv, hk = unit % a.Hkv;
    const int tid = threadIdx.x, lane = tid & 63, q4 = tid & 3, row = (tid >> 2) & 15, sg = __builtin_amdgcn_readfirstlane(tid >> 6);
    const float *base = a.partial + (size_t)(unit * a.row_tiles + rt) * a.nseg * WSTRIDE;
    const int dv = slice * MERGE_DV + q4 * 4, rows = min(16, a.rows_total - rt * 16);
    // padding rows of the last tile were never stored: their threads read the tile's last real row instead (the same lines
    // its own threads fetch) and drop the result below
    const int row_ld = min(row, rows - 1);
    f32x4 os[8];
    auto request = [&](int s0) {
#pragma unroll
        for (int u = 0; u < 8; ++u)                                   // clamped: every load is unconditional
            os[u] = *(const f32x4 *)(base + (size_t)min(s0 + sg * 8 + u, a.nseg - 1) * WSTRIDE + row_ld * D + dv);
    };
    request(0);
    for (int r = sg; r < rows; r += 4) {
        float ref[MERGE_MOST / 64], l[MERGE_MOST / 64], top = REF_NONE, sum = 0.f;
#pragma unroll
        for (int j = 0; j < MERGE_MOST / 64; ++j) {
            const int s = lane + 64 * j;
            const float *p = base + (size_t)min(s, a.nseg - 1) * WSTRIDE + 16 * D + r;
            ref[j] = s < a.nseg ? p[0] : REF_NONE;
            l[j] = s < a.nseg ? p[16] : 0.f;
            top = fmaxf(top, ref[j]);
        }
        top = lanes_max(top);
#pragma unroll
        for (int j = 0; j < MERGE_MOST / 64; ++j) {
            const float f = pow4(ref[j] - top);
            s_f[r][lane + 64 * j] = f;
            sum += l[j] * f;
        }
        sum = lanes_sum(sum);
        if (lane == 0) s_l[r] = sum;
    }
    __syncthreads();
    for (int s0 = 0; s0 < a.nseg; s0 += MEET_PARTS) {
        if (s0) request(s0);
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int s = s0 + sg * 8 + u;                             // (past the last: that one again, and zero times an infinite value is no zero)
            os[u] = (s < a.nseg ? os[u] : f32x4{0.f, 0.f, 0.f, 0.f}) * s_f[row_ld][s];
        }
#pragma unroll
        for (int i = 1; i < 8; i *= 2)
#pragma unroll
            for (int u = 0; u < 8; u += 2 * i) os[u] += os[u + i];
        *(f32x4 *)&s_o[s0 / MEET_PARTS][sg][row][q4 * 4] = os[0];
    }
    __syncthreads();
    if (sg == 0 && row < rows) {
        f32x4 o = f32x4{0.f, 0.f, 0.f, 0.f};
        for (int c = 0; c * MEET_PARTS < a.nseg; ++c) {
            auto run = [&](int i) { return *(const f32x4 *)&s_o[c][i][row][q4 * 4]; };
            o += (run(0) + run(1)) + (run(2) + run(3));
        }
        const int rr = rt * 16 + row, l2 = rr / a.groups, g3 = rr % a.groups;
        const float l_all = s_l[row], inv = l_all > 0.f ? 1.f / l_all : 0.f;
        *(f32x4 *)(a.out + (((size_t)b * a.L + l2) * a.Hq + hk * a.groups + g3) * D + dv) = o * inv;
    }
}

// One wavefront per query row; any head sizes and element types. scores: [rows][T] f32 scratch.
__global__ __launch_bounds__(256) void attn_generic_kernel(AttnArgs a, int d_k, int d_v, float *scores) {
    const int lane = threadIdx.x & 63;
    const size_t row = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const size_t total_rows = (size_t)a.B * a.L * a.Hq;
    if (row >= total_rows) return;
    const int hq = (int)(row % a.Hq);
    const int li = (int)((row / a.Hq) % a.L);
    const int b = (int)(row / ((size_t)a.Hq * a.L));
    const int hk = hq / a.groups;
    const int kv_end = clip_kv_end(a.ring, a.T, a.kv_lengths ? a.kv_lengths[b] : a.T);
    const int pos = a.positions ? a.positions[(size_t)b * a.L + li] : li;
    int lo, hi;
    window_keys(a.win_left, a.win_right, a.win_chunk, max(pos, 0), kv_end, lo, hi);
    clip_to_ring(a.ring, kv_end, lo, hi);
    float *o = a.out + row * d_v;
    if (hi <= lo) {
        for (int j = lane; j < d_v; j += 64) o[j] = 0.f;
        return;
    }
    float *sc = scores + row * a.T;
    const size_t qb = row * d_k;
    float mx = -INFINITY;
    // scores are kept at the key's physical row: a ring's visible keys span at most T steps
    for (int t = lo + lane; t < hi; t += 64) {
        const int tp = phys_key(a.ring, t);
        const size_t kb = (((size_t)b * a.T + tp) * a.Hkv + hk) * d_k;
        float d = 0.f;
        for (int j = 0; j < d_k; ++j) d += (load_scalar(a.q, a.q_dtype, qb + j) * a.scale) * load_scalar(a.k, a.kv_dtype, kb + j);
        if (a.soft_cap > 0.f) d = a.soft_cap * tanhf(d / a.soft_cap);
        sc[tp] = d;
        mx = fmaxf(mx, d);
    }
    mx = wave_max(mx);
    float sum = 0.f;
    for (int t = lo + lane; t < hi; t += 64) {
        const int tp = phys_key(a.ring, t);
        const float p = exp2f((sc[tp] - mx) * LOG2E);
        sc[tp] = p;
        sum += p;
    }
    sum = wave_sum(sum);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    const float inv = 1.f / sum;
    for (int j = lane; j < d_v; j += 64) {
        float acc = 0.f;
        for (int t = lo; t < hi; ++t) {
            const int tp = phys_key(a.ring, t);
            acc += sc[tp] * load_scalar(a.v, a.kv_dtype, (((size_t)b * a.T + tp) * a.Hkv + hk) * d_v + j);
        }
        o[j] = acc * inv;
    }
}

template <int KV, int D, bool HILO, bool RING, int DVS, bool PREPARE = false>
int launch_flash_split(aionhip_ctx *ctx, AttnArgs &a) {
    if constexpr (!HILO && !RING && !PREPARE)
        if (a.codes) return launch_flash_split<KV, D, HILO, RING, DVS, true>(ctx, a);
    constexpr int LDS = FlashCfg<D, SPLIT_NW, DVS>::LDS_BYTES;
    static std::atomic<uint64_t> attr{0};
    if (const int rc = allow_lds(ctx, attr, (const void *)attn_flash_kernel<KV, D, true, HILO, RING, DVS, PREPARE>, LDS)) return rc;
    ProfScope scope(ctx, "attn_flash_split");
    launch_k(ctx, attn_flash_kernel<KV, D, true, HILO, RING, DVS, PREPARE>, dim3((unsigned)(a.row_tiles * a.nseg * DVS), (unsigned)a.Hkv, (unsigned)a.B),
             dim3(SPLIT_NW * 64), LDS, a.q, a.kv_lengths, a.positions, a.k, a.v, a.T, a.L, flash_heads(a), flash_form(a), flash_tail(a));
    return AIONHIP_OK;
}

// Whether the parts are merged by the workgroup that ends last instead of a launch of their own: a wavefront of it adds a row's parts, 32 with all of their
// loads in flight, and as long as those are no more than 256 columns' worth that costs less than a launch. us with the merge launch / without: 1531 keys of 8
// KV heads x 128, 6 segments, 8.6 / 7.0; 8 sequences over 4000 keys of one KV head x 256, 16 segments, 12.6 / 10.9; one over 16384, 64 segments in four shares
// of the value columns, 12.4 / 11.0; 8 x 16384, 32 in one share, 27.7 / 27.5. Past that the one workgroup reads too much: 4 x 16384, 64 in one share, 19.1 / 20.2.
bool last_merges(const AttnArgs &a, int dv) { return a.nseg <= min(64, MEET_PARTS * (256 / dv)); }

// Key segments of a 16-row tile, eight 32-key tiles each where that leaves no CU with two workgroups: what a row sums to depends on these alone (and a
// sequence's bits on the batch only from where they no longer fit the CUs). Behind a window there are no more keys than it shows to the call's consecutive queries.
// sub: a segment's eight wavefronts divided over 2^sub workgroups. How fast a short cache is read is what one CU's L1 fills (64 bytes a clock), so that two
// or four tiles to a workgroup on more CUs beat eight on fewer as long as the merge stays small: 24 parts, a quarter of a segment each only where the workgroups, with
// the value columns in all their shares, fit the CUs at once. us a token, whole segments / so: 512 keys of one KV head x 256 8.7 / 6.2, 1531 8.9 / 6.4, 3000 8.9 /
// 7.3; of 8 x 128 512 keys 6.7 / 5.6, 1531 6.8 / 5.9 (in quarters, 24 parts, 6.6), 3000 7.3 / 7.0; 4 sequences over 11378 keys, 1469 visible, 9.0 / 7.8. From 13
// segments on they stay whole (8000 keys: 32 parts 9.3, 63 9.4).
struct KeySegments { int nseg, sub; };
KeySegments key_segments(const AttnArgs &a, int d, int cus, int units) {
    long keys = a.T;
    if (!a.codes && a.win_chunk == 0 && a.win_right < (unsigned)a.T && a.win_left < (unsigned)a.T) keys = min(keys, (long)a.win_left + (long)a.win_right + a.L + TILE_KEYS);
    const long wgs = (long)units * a.row_tiles;
    // (as many segments as keep the workgroups within one per CU: a second, partial round of workgroups plus the merge
    // costs more than CUs left idle - 192 row tiles in two segments each took 26 us, in one 13)
    const int room = (int)min((long)cus / wgs, 256L), of_eight = (int)((keys + SPLIT_NW * TILE_KEYS - 1) / (SPLIT_NW * TILE_KEYS));
    KeySegments ks{max(1, min(room, of_eight)), 0};
    if (a.codes || ks.nseg == 1) return ks;
    const long full = wgs * (d / 64);
    if (ks.nseg * 2 <= min(room, 24)) ks.sub = ks.nseg * 4 <= min(room, full * 24 <= cus ? 24 : full * 16 <= cus ? 16 : 12) ? 2 : 1;
    return ks;
}

template <int KV, int D, bool HILO, bool RING = false>
int launch_flash(aionhip_ctx *ctx, AttnArgs &a) {
    using Cfg = FlashCfg<D, 4>;
    const int units = a.B * a.Hkv;
    // Few query rows, or so few 128-row prefill workgroups that they would occupy under a quarter of the CUs
    // (measured: one batch, one kv head, up to ~1024 positions x 8 heads): 16-row tiles spread the K/V reads
    // over many CUs, which outweighs re-reading K/V per row tile from L2.
    const int cus0 = ctx->cu_count > 0 ? ctx->cu_count : 256;
    // (the smaller the head, the longer the 16-row kernel stays ahead: per key it re-reads less. Crossovers measured over
    // five head layouts x L = 32 .. 2048, one and two sequences: about 112 / 40 / 32 workgroups of the 128-row kernel at head size 64 /
    // 128 / 256. 16 q / 4 kv heads x 64: 768 queries, 96 workgroups, 14.0 against 19.2 us; 1024, 128 workgroups, 19.3 against 19.3;
    // two sequences of 768, 192 workgroups, 23.5 against 19.5. 32 / 8 x 128: 128 queries 6.1 against 8.1, 192 10.6 against 9.2)
    const long pf_wgs = (long)units * ((a.rows_total + PF_ROWS - 1) / PF_ROWS);
    const long pf_min = D <= 64 ? (long)cus0 * 7 / (2 * PF_FLASH_BELOW) : D <= 128 ? (long)cus0 * 5 / (4 * PF_FLASH_BELOW) : (long)cus0 / PF_FLASH_BELOW;
    bool split = a.rows_total <= 64 || (!HILO && pf_wgs <= pf_min) ||
                 (!HILO && !prefill_takes(a, D));      // e.g. a softmax scale that is not positive: the 16-row kernel takes any
    // A chunk of queries over a cache at least four times its length (chunked prompts, speculative batches): the crossover
    // above was measured on prompts over their own keys, where few rows mean few keys. Here the keys dominate, and the 128-row
    // kernel, which can cut them into up to 16 segments, is weighed against the 16-row kernel by what both measured over
    // 1 ... 1024 queries x 1024 ... 16384 keys at head sizes 128 and 256: the 16-row kernel 13 us + 0.56 us per 32-key tile a
    // workgroup walks (head size 256; in proportion below), the 128-row kernel 16 us + 1.9 us per 64-key tile (1.2 at head
    // size 128, 0.85 at 64; 0.7 of that while half the CUs stay free). 8 heads x 256, 256 queries over 16384 keys: 159 -> 46 us.
    // The 16-row kernel has become faster since, and its segments finer; over 110 shapes, 9 ... 1024 queries x 4 ... 64 times as many keys, head sizes 64 to
    // 256, the choice is within 5 % of the faster kernel on 108 and costs at most 18 % (8 heads on one x 128, 104 queries over 4992 keys 21.2 against 17.9 us).
    if (!HILO && a.rows_total > 64 && pf_wgs <= pf_min && prefill_takes(a, D) && (long)a.T >= 4L * a.L && a.win_left >= (unsigned)a.T) {
        const float ds = (float)D / 256.f;
        const long wgs16 = (long)units * a.row_tiles;
        const int tiles32 = (a.T + TILE_KEYS - 1) / TILE_KEYS;
        const long nseg_s = max(1L, min((long)cus0 / max(wgs16, 1L), (long)(tiles32 + SPLIT_NW - 1) / SPLIT_NW));
        const long rounds_s = (wgs16 * nseg_s + cus0 - 1) / cus0;
        const float split_us = (nseg_s > 1 ? 13.f : 10.f) + (float)((tiles32 + nseg_s - 1) / nseg_s) * 0.56f * ds * (float)rounds_s;
        const int tiles64 = (a.T + PF_TK - 1) / PF_TK;
        const long nseg_p = max(1L, min(min((long)cus0 / max(pf_wgs, 1L), (long)tiles64 / (D > 128 ? 4 : 8)), 16L));
        const long rounds_p = (pf_wgs * nseg_p + cus0 - 1) / cus0;
        const float per_tile = (0.5f + 1.4f * ds) * (pf_wgs * nseg_p * 2 <= cus0 ? 0.7f : 1.f);
        const float prefill_us = (nseg_p > 1 ? 16.f : 12.f) + (float)((tiles64 + nseg_p - 1) / nseg_p) * per_tile * (float)rounds_p;
        if (prefill_us < split_us) split = false;
    }
    if (a.codes && (HILO || RING)) return rows_not_prepared(ctx, HILO ? "the precise mode" : "rolling caches");
    if (split) {
        const int cus = ctx->cu_count > 0 ? ctx->cu_count : 256;
        const KeySegments ks = key_segments(a, D, cus, units);
        if (a.codes && ks.nseg != 1) return rows_not_prepared(ctx, "keys in segments");      // (their merge writes f32 rows)
        a.sub = ks.sub;
        a.nseg = ks.nseg << ks.sub;
        const long tiles = (long)units * a.row_tiles, wgs = tiles * a.nseg;
        const int shares = D >= 256 && wgs * (D / 64) <= cus ? D / 64 : D >= 128 && wgs * 2 <= cus ? 2 : 1;      // of the value columns, see below
        const bool meet = a.nseg > 1 && last_merges(a, D / shares);
        if (meet) {
            if (const int rc = ensure_scratch2(ctx, (size_t)tiles * shares * a.nseg * (16 * (D / shares) + 32) * sizeof(float))) return rc;
            if (const int rc = ensure_tickets(ctx, (size_t)tiles * shares * MEET_TICKET_WORDS * sizeof(unsigned))) return rc;
            a.partial = (float *)ctx->scratch2;
            a.tickets = (unsigned *)ctx->tickets;
        } else if (a.nseg > 1) {
            if (const int rc = ensure_scratch2(ctx, (size_t)tiles * a.nseg * (16 * D + 32) * sizeof(float))) return rc;
            a.partial = (float *)ctx->scratch2;
        }
        // Workgroups that leave CUs idle divide the value columns as well, down to 64 each: the scores are computed by every share,
        // the loads of V, the second product and the merge of the wavefronts through LDS are divided. A short cache (one key
        // segment) is a chain of latencies in one CU, of which those three were about 2 us of 9.8: one token over 144 keys, one KV
        // head of size 256, 9.8 -> 8.0 us; over 1531 keys, 8 KV heads of size 128, 10.8 -> 10.4 with the segments' merge. Only
        // while the shares fit one workgroup per CU: past that a second round costs more than a share saves.
        int rc;
        if (D >= 256 && shares == D / 64) rc = launch_flash_split<KV, D, HILO, RING, D / 64>(ctx, a);
        else if (D >= 128 && shares == 2) rc = launch_flash_split<KV, D, HILO, RING, D >= 128 ? 2 : 1>(ctx, a);
        else rc = launch_flash_split<KV, D, HILO, RING, 1>(ctx, a);
        if (rc) return rc;
        if (a.nseg > 1 && !meet) {
            ProfScope scope(ctx, "attn_merge");
            launch_k(ctx, attn_merge_kernel<D>, dim3((unsigned)(a.row_tiles * (D / MERGE_DV)), (unsigned)units), dim3(256), 0, a);
        }
        LAUNCH_CHECK(ctx, "attn_flash_split");
    } else if (!HILO) {
        return launch_prefill(ctx, a, D);
    } else {
        a.nseg = 1;
        static std::atomic<uint64_t> attr{0};
        if (const int rc = allow_lds(ctx, attr, (const void *)attn_flash_kernel<KV, D, false, HILO>, Cfg::LDS_BYTES)) return rc;
        ProfScope scope(ctx, "attn_flash_prefill");
        launch_k(ctx, attn_flash_kernel<KV, D, false, HILO>, dim3((unsigned)((a.row_tiles + 3) / 4), (unsigned)a.Hkv, (unsigned)a.B), dim3(256), Cfg::LDS_BYTES, a.q, a.kv_lengths,
                 a.positions, a.k, a.v, a.T, a.L, flash_heads(a), flash_form(a), flash_tail(a));
        LAUNCH_CHECK(ctx, "attn_flash_prefill");
    }
    return AIONHIP_OK;
}

template <int KV>
int launch_flash_d(aionhip_ctx *ctx, AttnArgs &a, int d) {
    const bool hilo = a.q_dtype == AIONHIP_F32 && ctx->attn_precise;
    if (a.ring) {       // rolling caches: the plain instances only (precise mode and soft cap take the generic kernel)
        if (d == 64) return launch_flash<KV, 64, false, true>(ctx, a);
        if (d == 128) return launch_flash<KV, 128, false, true>(ctx, a);
        return launch_flash<KV, 256, false, true>(ctx, a);
    }
    if (d == 64) return hilo ? launch_flash<KV, 64, true>(ctx, a) : launch_flash<KV, 64, false>(ctx, a);
    if (d == 128) return hilo ? launch_flash<KV, 128, true>(ctx, a) : launch_flash<KV, 128, false>(ctx, a);
    return hilo ? launch_flash<KV, 256, true>(ctx, a) : launch_flash<KV, 256, false>(ctx, a);
}

bool dtype_ok(int d) { return d == AIONHIP_F32 || d == AIONHIP_F16 || d == AIONHIP_BF16; }

}  // namespace

int run_attention(aionhip_ctx *ctx, const aionhip_attention *p, const PreparedAct *prepared) {
    if (!ctx || !p) return AIONHIP_INVALID_ARGUMENT;
    if ((!p->out && !prepared) || !p->q || !p->k || !p->v) return set_err(ctx, AIONHIP_INVALID_ARGUMENT, "attention: null operand");
    if (!dtype_ok(p->q_dtype) || !dtype_ok(p->kv_dtype)) return set_err(ctx, AIONHIP_UNSUPPORTED, "attention: q/kv dtype must be f32, f16 or bf16");
    if (p->h_kv == 0 || p->h_q == 0 || p->h_q % p->h_kv != 0) return set_err(ctx, AIONHIP_INVALID_ARGUMENT, "attention: h_q %zu is not a multiple of h_kv %zu", p->h_q, p->h_kv);
    if (p->d_k == 0 || p->d_v == 0) return set_err(ctx, AIONHIP_INVALID_ARGUMENT, "attention: zero head size");
    if (p->batch == 0 || p->l_q == 0) return AIONHIP_OK;
    const size_t lim = 0x7FFFFFFF;
    if (p->batch > lim || p->l_q > lim || p->t_kv > lim || p->h_q > 65535 || p->d_k > 65535 || p->d_v > 65535 ||
        p->batch * p->h_kv > 65535 || p->l_q * (p->h_q / p->h_kv) > lim)
        return set_err(ctx, AIONHIP_UNSUPPORTED, "attention: dimension too large");

    AttnArgs a{};
    a.q = (const void *)(uintptr_t)p->q;
    a.k = (const void *)(uintptr_t)p->k;
    a.v = (const void *)(uintptr_t)p->v;
    if (prepared) {
        a.codes = (int *)prepared->q;
        a.code_scales = prepared->scale;
    } else {
        a.out = (float *)(uintptr_t)p->out;
    }
    a.positions = (const int *)(uintptr_t)p->query_positions;
    a.kv_lengths = (const int *)(uintptr_t)p->kv_lengths;
    a.B = (int)p->batch; a.L = (int)p->l_q; a.T = (int)p->t_kv; a.Hq = (int)p->h_q; a.Hkv = (int)p->h_kv;
    a.groups = a.Hq / a.Hkv;
    a.rows_total = a.L * a.groups;
    a.row_tiles = (a.rows_total + 15) / 16;
    a.nseg = 1;
    a.q_dtype = p->q_dtype; a.kv_dtype = p->kv_dtype;
    a.scale = p->scale; a.soft_cap = p->attn_logits_soft_cap;
    a.win_left = p->window_left; a.win_right = p->window_right; a.win_chunk = p->window_chunk;
    a.ring = p->rolling ? a.T : 0;

    if (prepared && a.T == 0) return rows_not_prepared(ctx, "no keys");
    if (a.T == 0) {
        // no keys at all: every interval is empty -> zeros (cpu/exec/attention.zig:787-815)
        return aionhip_memset(ctx, p->out, 0, 0, p->batch * p->l_q * p->h_q * p->d_v * sizeof(float));
    }

    const bool flash = p->d_k == p->d_v && (p->d_k == 64 || p->d_k == 128 || p->d_k == 256) &&
                       (p->kv_dtype == AIONHIP_F16 || p->kv_dtype == AIONHIP_BF16) &&
                       ((p->k | p->v | (prepared ? 0 : p->out)) & 15) == 0 &&
                       // a ring shorter than a key tile, or a ring in precise / soft-cap mode: generic kernel
                       (!a.ring || (a.T >= PF_TK && !(a.q_dtype == AIONHIP_F32 && ctx->attn_precise) && a.soft_cap <= 0.f));
    if (flash) {
        if (p->kv_dtype == AIONHIP_F16) return launch_flash_d<AIONHIP_F16>(ctx, a, (int)p->d_k);
        return launch_flash_d<AIONHIP_BF16>(ctx, a, (int)p->d_k);
    }
    if (prepared) return rows_not_prepared(ctx, "the generic kernel");
    const size_t rows = p->batch * p->l_q * p->h_q;
    int rc = ensure_scratch2(ctx, rows * p->t_kv * sizeof(float));
    if (rc) return rc;
    ProfScope scope(ctx, "attn_generic");
    launch_k(ctx, attn_generic_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, a, (int)p->d_k, (int)p->d_v, (float *)ctx->scratch2);
    LAUNCH_CHECK(ctx, "attn_generic");
    return AIONHIP_OK;
}

extern "C" int aionhip_step_attention(aionhip_ctx *ctx, const aionhip_attention *p) { return run_attention(ctx, p, nullptr); }

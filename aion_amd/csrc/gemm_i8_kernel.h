// The exact GEMM's kernel (see gemm_i8.hip for the launcher and the choice of shapes).
//
// v_mfma_i32_32x32x32_i8: the 32 of K are one quant block, so the i32 tile is the exact block dot; then
// acc += f32(dot) * (a_scale * w_scale), three operations per output and block, and that is the bound. Of the three the vector ALU does
// the conversion and the multiply-add; the products of scales come from v_mfma_f32_32x32x1_2b_f32, two tiles' outer products an instruction
// (one product a term, rounded as v_mul_f32 rounds it: the same bits, subnormals and infinities included), except where a wavefront has one
// tile or half of one. What the parts cost on gfx950: 48 vector instructions of a tile's rescale 52 ns a SIMD with four wavefronts on it, 57
// with two, 94 with one; with the i8 MFMA (14 ns alone) in front 62, 69, 89: the two pipes hardly overlap once both are in demand. The
// outer products cost 13.5 ns a tile, less than the 16 multiplies and four 16-byte LDS reads of a lane's 16 row scales that they replace (2 x 2
// tiles: 2048 x 4096 x 4096 q4 112.5 -> 106.0 us, q8 116.8 -> 111.0; 512 x 4096 x 4096 35.5 -> 33.9, 37.6 -> 36.1; 2048 x 14336 x 512 63.4 -> 60.9, 66 ->
// 61; 3 x 1 level; a lone tile, which takes them for two blocks at a time, loses 2 .. 4 %: 32 x 32768 x 2048, q8 64 x 4096 x 4096).
// So the shape of this kernel: wavefronts that never wait for each other, two or more per SIMD
// as soon as there are two workgroups per CU (a grid of at most one runs one per SIMD, q4 from K = 2048 on two: eight wavefronts to a
// workgroup). A wavefront owns a (32 MT) x (32 NT) tile and a share of K (every KS-th group of four blocks); the KS wavefronts of a tile
// meet once, at the end, in LDS, in a fixed order. No barrier in the loop: what a wavefront stages, it stages for itself.
//   activations: prepared in operand order, a wavefront's load of a block is 1 KiB of consecutive memory, straight to registers, three blocks
//     ahead
//   weights and activation scales: LDS-writing buffer loads, a group of four blocks ahead. The row-major weight puts a lane's operand bytes
//     (its row's 16 of a block) far from its neighbours', and the L1 takes such a load lane by lane: 64 accesses, 60 .. 85 % of its cycles
//     at 2048 x 14336 x 4096 when the operands came straight from memory. Staged, neighbouring lanes read a row's consecutive bytes: 16
//     accesses, whole lines. The scales are read from there, one word a lane and block (a lone tile: 16 rows', 4 reads)
// Other forms measured: f16 codes on v_mfma_f32_32x32x16_f16 (no conversion after the dot, 51 ns a tile, but the codes have to be
// converted and the operands are twice the bytes), scale products as 4x4x1 outer products (82 ns) and as sums of bf16 parts (the sums of six products round up to 2 ulp off), codes as fp6 digits (exact dots
// in f32, but what the conversion cost the unpacking of nibbles costs), activation scales by
// DPP broadcast (90 ns), an integer bias in place of the conversion (62 ns).
// RQ: of a tile's 32 rows the first 8 RQ are kept (2: calls of up to 16 rows, half the rescale; 131072 x 512 at 9 rows q4 22.7 -> 20.3 us).
// WHOLE: K is a multiple of 128, see the launcher.
// Measured (whole calls, weights straight from memory -> staged): q8 8 x 14336 x 4096 19.3 -> 15.5 us, 2048 x 14336 x 4096 429 -> 384,
// 512 x 4096 x 4096 41.3 -> 37.0; q4 374 -> 366, 36.8 -> 36.0, 128 x 2048 x 8192 15.5 -> 14.8 us (q4 asks for half the bytes). Since K of whole groups
// runs without checks: 8 x 14336 x 4096 14.4 us. What is left is the vector ALU, 37 .. 41 instructions a tile and block at 2048 rows, and what the loads
// take beside it: with neither loads nor LDS reads in the loop 512 x 4096 x 4096 took 25 of 35 us.
#pragma once
#include "common.h"

#include <type_traits>

using i32x2 = __attribute__((ext_vector_type(2))) int;
using i32x4 = __attribute__((ext_vector_type(4))) int;
using i32x16 = __attribute__((ext_vector_type(16))) int;
using f32x16 = __attribute__((ext_vector_type(16))) float;
using f32x32 = __attribute__((ext_vector_type(32))) float;

// up to four weights with the same K and block format against one prepared activation: column tiles first_tile[i] .. of weight i
struct GemmSegs {
    const uint8_t *qs[4];
    const __half *sc[4];
    float *c[4];
    size_t ldc[4];
    int n[4], first_tile[4];
    int count;
};

// What leaves the kernel (EPI). Past GEMM_PLAIN the two column tiles of a wavefront belong together:
//   GEMM_GATE  the same columns of weights 0 and 1 (gate and up): gelu(gate) * up, prepared for the next matmul, its codes to c[0], its scales to
//              c[1], in the order below
//   GEMM_ROPE  the two halves of a head's columns of weight 0, 1 or 2 (q, k, v): q and k rotated, q to q_out, k and v as f16 to their caches
constexpr int GEMM_PLAIN = 0, GEMM_GATE = 1, GEMM_ROPE = 2;
struct GemmRopeSegs : GemmSegs {
    float *q_out;
    __half *kcache, *vcache;
    const int *positions, *write_index;
    const float *freq;
    int s_len, t_cap, h_q, h_kv, d, rope_pairs;
};
// A launch's arguments. What a wavefront needs for its first loads - the activation, the first weight, the sizes - are plain leading arguments, which
// arrive in SGPRs with it (14 words do); a structure by value is read from memory, a round trip ahead of the first address, and so is gridDim. The rest is
// the last argument, in the form that the launch needs: one weight (c, ldc), up to four, the pair launches' own. q4 512 x 4096 x 4096 33.7 -> 33.0 us, q8 77 x
// 11008 x 4096 25.5 -> 25.1, q4 4 x 4096 x 14336 (gemv_slim_kernel) 11.4 -> 10.9; a 128-token prompt of 26 blocks 1898 -> 1856.
struct GemmOne {
    float *c[1];
    size_t ldc[1];
};
template <int EPI, bool MANY> struct GemmSegsOf { using type = GemmSegs; };
template <> struct GemmSegsOf<GEMM_PLAIN, false> { using type = GemmOne; };
template <> struct GemmSegsOf<GEMM_ROPE, true> { using type = GemmRopeSegs; };
template <class Segs> struct GemmTail {
    Segs segs;
    float alpha, beta;
    float *partial;
    int partial_ld;
};
// the sizes that ride in one word: whether all workgroups run at once, the K slices (at most 4), the column tiles of all weights
inline int gemm_i8_form(int one_round, int slices, int col_tiles) { return one_round | slices << 1 | col_tiles << 4; }

// Prepared activation in the order the kernel's operand loads want: row tiles of 32 rows (the last one may hold fewer), per
// tile and quant block [h = 0, 1][row][16 codes] - k = 16 h .. 16 h + 15 of the block - so that a wavefront's load of one
// block of a full tile is 1 KiB of consecutive memory; scales per tile and block [row].
__host__ __device__ __forceinline__ int act_tile_rows(int M, int mt) { return M - mt * 32 < 32 ? M - mt * 32 : 32; }

// LDS of a wavefront: two groups of four blocks, weight codes and activation scales
template <bool Q8, int MT, int NT> __host__ __device__ constexpr int gemm_i8_wave_lds_bytes() { return 2 * (NT * 32 * (Q8 ? 128 : 64) + MT * 512); }

// workgroup `bid` of the kernel's grid (the K slices, if any, are the grid's z). qs0, sc0, n0: the first weight; qs1: GEMM_GATE's second.
template <int DT, int MT, int NT, int KS, int WGM, int WGN, int RQ, bool WHOLE, int EPI, bool MANY>
__device__ __forceinline__ void gemm_i8_body(const typename GemmSegsOf<EPI, MANY>::type &segs, int bid, const uint8_t *__restrict__ aq, const float *__restrict__ a_scale,
                                             const uint8_t *__restrict__ qs0, const __half *__restrict__ sc0, int M, int K, int n0w, const uint8_t *__restrict__ qs1,
                                             int col_tiles, int slices, int one_round, float alpha, float beta, float *__restrict__ partial, int partial_ld) {
    constexpr bool Q8 = DT == AIONHIP_Q8_0;
    constexpr bool PAIR = EPI != GEMM_PLAIN, GATE = EPI == GEMM_GATE;
    constexpr int BM = 32 * MT * WGM, BN = 32 * NT * WGN;
    static_assert(!PAIR || (NT == 2 && WGN == 1), "a pair of tiles side by side");
    constexpr bool OUTER = RQ == 4 && MT * NT > 1;        // scale products from the matrix pipe
    static_assert(OUTER || MT == 1, "one row tile");
    static_assert(RQ == 4 || MT * WGM == 1, "fewer rows than a tile: one row tile");
    using Acc = __attribute__((ext_vector_type(4 * RQ))) float;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 31, h = lane >> 5;
    const int ks = wave / (WGM * WGN), wsub = wave % (WGM * WGN), wm = wsub / WGN, wn = wsub % WGN;
    // workgroup -> tile: ids go round-robin over the 8 XCDs; every XCD takes a contiguous run of tiles, row tiles fastest, so that
    // the workgroups that share a weight column tile run on one L2
    // (row tiles in groups of eight, columns within: see the launcher)
    const int row_tiles = (M + BM - 1) / BM, row_group = min(row_tiles, 8), tiles = row_tiles * col_tiles;
    const int xcd = bid & 7, slot = bid >> 3;
    const int t = xcd * (tiles >> 3) + min(xcd, tiles & 7) + slot;
    // (up to eight row tiles: one group. Divisions are some 20 dependent instructions each ahead of the first load)
    const int gr0 = row_tiles <= 8 ? 0 : (int)((unsigned)t / (unsigned)(row_group * col_tiles)) * row_group, gr = min(row_group, row_tiles - gr0);
    const int in_group = t - gr0 * col_tiles, ct = gr == 1 ? in_group : (int)((unsigned)in_group / (unsigned)gr), rt = gr0 + in_group - ct * gr;
    int si = 0, first_tile = 0, N = n0w;
    const uint8_t *__restrict__ qs = qs0;
    const __half *__restrict__ sc = sc0;
    if constexpr (MANY && !GATE) {
        if (ct >= (n0w + BN - 1) / BN) {                 // (the second weight's first tile)
            si = 1;
#pragma unroll
            for (int i = 2; i < 4; ++i)
                if (i < segs.count && ct >= segs.first_tile[i]) si = i;
            qs = segs.qs[si];
            sc = segs.sc[si];
            N = segs.n[si];
            first_tile = segs.first_tile[si];
        }
    }
    float *__restrict__ c = segs.c[si];
    size_t ldc = segs.ldc[si];
    const int KB = K >> 5, G = (KB + 3) >> 2;
    // (a head's columns: pair tile `head_tile` is its columns 32 head_tile .. and the same of its second half)
    [[maybe_unused]] int head = 0, head_tile = 0, pair_col = ct * 32;
    size_t partner = 0;                          // weight rows from a column of the first tile to its partner's
    if constexpr (EPI == GEMM_ROPE) {
        const int per_head = segs.d >> 6;
        head = (ct - first_tile) / per_head;
        head_tile = ct - first_tile - head * per_head;
        partner = (size_t)segs.d >> 1;
        pair_col = head * segs.d + head_tile * 32;
    }
    const int n0 = PAIR ? pair_col : (ct - first_tile) * BN + wn * (32 * NT), m0 = rt * BM + wm * (32 * MT);

    Acc acc[MT][NT];
    // q4 dots are 16 times the codes' dots. The 1/16 is taken from the sums, where it is exact down to subnormal products of scales; sums past
    // 2^124 leave the f32 range that way (a row that holds the lowest f32 as a mask), so a wavefront with one that is not finite runs
    // its share again with the 1/16 in the weight scales. (Codes without the 16 cost eight vector instructions a tile and block.)
    float code_scale = 1.f, sum_scale = Q8 ? 1.f : 0.0625f;
    for (;;) {
        // (the addresses of a second walk are computed again: kept, they would cost the first one registers)
        int lane_now = lane;
        asm volatile("" : "+v"(lane_now));
        const int lane = lane_now, r = lane & 31, h = lane >> 5;
        // this wavefront's operand rows: activation tiles mt0 .., weight rows n0 + 32 ni + r (clamped: a clamped row's results are not
        // stored). Every operand address is a uniform base that moves with K plus a 32-bit offset a lane keeps for good, so that a
        // load costs the vector ALU nothing.
        const uint8_t *ab[MT];
        const float *asb[MT];
        unsigned ao[MT], aso[MT];
        int arows[MT];
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            const int mt = min((m0 >> 5) + i, (M - 1) >> 5);
            arows[i] = act_tile_rows(M, mt);
            ab[i] = aq + (size_t)mt * 32 * K;
            ao[i] = (unsigned)(h * arows[i] + min(r, arows[i] - 1)) * 16;
            asb[i] = a_scale + (size_t)mt * 32 * KB;
            aso[i] = (unsigned)min(r, arows[i] - 1) * 4;
        }
        const int nb = min(n0, N - 1);
        const unsigned wpitch = Q8 ? (unsigned)K : (unsigned)K >> 1;
        [[maybe_unused]] const uint8_t *wb = qs + (size_t)nb * wpitch, *wb1 = (GATE ? qs1 : qs) + ((size_t)nb + partner) * wpitch;      // (used in the device pass only)
        const __half *sb = sc;
        if constexpr (GATE) sb = h ? segs.sc[1] : sc;
        sb += ((size_t)nb + (EPI == GEMM_ROPE && h ? partner : 0)) * KB;
        // weights: load l of a tile's group covers 8 (q8) or 16 (q4) rows, the lanes of a row side by side along it
        constexpr int RB = Q8 ? 128 : 64, LPR = RB / 16, WL = LPR / 2;      // bytes of a row per group, lanes per row, loads per 32 rows
        const int w_row = lane / LPR;
        unsigned wo[NT][WL];
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int l = 0; l < WL; ++l)
                wo[i][l] = (unsigned)(min(n0 + (PAIR ? 0 : i * 32) + l * (64 / LPR) + w_row, N - 1) - nb) * wpitch + (unsigned)((lane % LPR) ^ (Q8 ? w_row & 7 : (w_row >> 1) & 3)) * 16;
        // weight scales: with two tiles a lane half takes one tile's rows each and the halves are exchanged afterwards
        const unsigned so = (unsigned)(min(n0 + (NT == 2 && !PAIR ? h * 32 : 0) + r, N - 1) - nb) * (unsigned)KB;

        // groups of four quant blocks: K slice z takes a contiguous run of them, its KS wavefronts every KS-th group of the run
        const int g_per = slices == 1 ? G : (G + slices - 1) / slices;
        const int g_lo = (int)blockIdx.z * g_per, g_hi = min(G, g_lo + g_per);

        // Registers: the four blocks of a group's activations (reloaded for the next group as each is used up), the next group's weight
        // scales. LDS, private to the wavefront and written by the loads themselves: two groups of weight codes and activation scales.
        i32x4 A[4][MT];
        unsigned long sw_raw = 0, sw_now = 0;      // four f16 scales of a weight row: the next group's, this group's
        int sw_shift = 0, sw_shift_now = 0;
#if defined(__HIP_DEVICE_COMPILE__)
        const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)wb, 0, 0xFFFFFFFFu, 0x00027000);
        [[maybe_unused]] const __amdgpu_buffer_rsrc_t w_rsrc1 = __builtin_amdgcn_make_buffer_rsrc((void *)wb1, 0, 0xFFFFFFFFu, 0x00027000);
        __amdgpu_buffer_rsrc_t sa_rsrc[MT];
#pragma unroll
        for (int i = 0; i < MT; ++i) sa_rsrc[i] = __builtin_amdgcn_make_buffer_rsrc((void *)asb[i], 0, 0xFFFFFFFFu, 0x00027000);
#endif
        constexpr int LGKM0 = vmcnt_imm(63) & ~(15 << 8);        // every LDS operation has completed
        constexpr int WBUF = NT * 32 * RB;
        unsigned char *w_lds = lds + wave * gemm_i8_wave_lds_bytes<Q8, MT, NT>();
        float *sa_lds = (float *)(w_lds + 2 * WBUF);
        auto load_a = [&](int set, int kb) {
            if (!WHOLE) kb = min(kb, KB - 1);
#pragma unroll
            for (int i = 0; i < MT; ++i) A[set][i] = *(const i32x4 *)(ab[i] + (size_t)((unsigned)kb * (unsigned)(arows[i] * 32)) + ao[i]);
        };
        // Row R of a tile is at R * RB, its 16-byte piece c in slot c ^ (R & 7) (q8) or c ^ ((R >> 1) & 3) (q4): the lanes of a read,
        // consecutive rows at one piece, then cover 128 bytes of banks. (Blocks past the end of K: another row's or the slack behind the
        // weight, scale 0.)
        auto load_w = [&](int g, int buf) {
#if defined(__HIP_DEVICE_COMPILE__)   // the builtin exists in the device pass only
#pragma unroll
            for (int i = 0; i < NT; ++i)
#pragma unroll
                for (int l = 0; l < WL; ++l)
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(PAIR && i ? w_rsrc1 : w_rsrc, (lds_void *)(w_lds + buf * WBUF + (i * WL + l) * 1024), 16, wo[i][l], g * RB, 0, 0);
#endif
        };
        const int r_slot = Q8 ? h ^ (r & 7) : (r >> 1) & 3;
        using Codes = typename std::conditional<Q8, i32x4, i32x2>::type;    // what a lane's MFMA operand is made of: 16 codes, 16 nibbles
        Codes Bn[NT];
        auto read_b = [&](int buf, int j) {
#pragma unroll
            for (int i = 0; i < NT; ++i)
                Bn[i] = *(const Codes *)(w_lds + buf * WBUF + (i * 32 + r) * RB + (Q8 ? ((2 * j) ^ r_slot) * 16 : (j ^ r_slot) * 16 + h * 8));
        };
        struct __attribute__((packed, aligned(2))) U64 { unsigned long v; };
        auto load_scales = [&](int g, int buf) {
            const int kb = WHOLE ? g * 4 : min(g * 4, KB - 1), base = WHOLE ? kb : max(0, min(kb, KB - 4));
            sw_shift = (kb - base) * 16;
            sw_raw = ((const U64 *)(sb + base + so))->v;
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int q = 0; q < 2; ++q)                  // two blocks' scales of 32 rows
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(sa_rsrc[i], (lds_void *)(sa_lds + (buf * MT + i) * 128 + q * 64), 4,
                                                             aso[i] + (h && (WHOLE || g * 4 + 2 * q + 1 < KB) ? (unsigned)arows[i] * 4 : 0u),
                                                             (WHOLE ? g * 4 + 2 * q : min(g * 4 + 2 * q, KB - 1)) * arows[i] * 4, 0, 0);
#endif
        };

        // the activation scales a lane multiplies with - 16 rows of each row tile - come from the wavefront's LDS copy of the group
        float sa[MT][4 * RQ];
        auto read_sa = [&](int i, int buf, int j) {
#pragma unroll
            for (int q = 0; q < RQ; ++q) {
                const f32x4 v = *(const f32x4 *)(sa_lds + (buf * MT + i) * 128 + j * 32 + 8 * q + 4 * h);
                sa[i][4 * q] = v.x; sa[i][4 * q + 1] = v.y; sa[i][4 * q + 2] = v.z; sa[i][4 * q + 3] = v.w;
            }
        };
        // Scale products from the matrix pipe: v_mfma_f32_32x32x1_2b gives the products of two 32 x 32 tiles, here neighbouring tiles of a block
        // or, of an odd tile, two blocks. Lane half h holds the rows' scales of the pair's tile (or block) h.
        constexpr int PAIRS = MT * NT / 2;
        constexpr bool ODD = (MT * NT) % 2 == 1;
        float sp = 0.f, sp_odd = 0.f;
        auto read_sp = [&](int buf, int j) {
            if constexpr (PAIRS > 0) sp = sa_lds[(buf * MT + (MT > 1 ? h : 0)) * 128 + j * 32 + r];
            if constexpr (ODD)
                if (j % 2 == 0) sp_odd = sa_lds[(buf * MT + MT - 1) * 128 + (j + h) * 32 + r];
        };
        // Blocks past the end of K in the last group: activation scale 0 as well as weight scale 0, where a real block's infinite scale
        // would make a NaN of the product. Called as the group begins: its loads have landed, and what has been read ahead is its first
        // block's. (Writes in every group, all but the last to words nobody reads, in place of the branch: 1 % slower.)
        auto clear_tail = [&](int g, int buf) {
            if (WHOLE || g * 4 + 4 <= KB) return;
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 1; j < 4; ++j)
                    if (g * 4 + j >= KB && lane < 32) sa_lds[(buf * MT + i) * 128 + j * 32 + lane] = 0.f;
        };
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int e = 0; e < 4 * RQ; ++e) acc[i][j][e] = 0.f;
        int g = g_lo + ks;
        if (g < g_hi) {
            load_w(g, 0);
            load_scales(g, 0);
#pragma unroll
            for (int j = 0; j < 3; ++j) load_a(j, g * 4 + j);
            sw_now = sw_raw;
            sw_shift_now = sw_shift;
            __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
            asm volatile("" ::: "memory");
            read_b(0, 0);
            if constexpr (OUTER) read_sp(0, 0);
        }
#pragma unroll
        for (int e = 0; e < 4 * RQ; ++e) sa[MT - 1][e] = 0.f;      // the first rescale has no block behind it: 0 * 0, and no real block's scale
        int buf = 0;
        i32x16 d = i32x16{0};                      // the dots whose rescale is due: tile (MT - 1, NT - 1) of the previous block
        float sw_due = 0.f;
        // Of two wavefronts on a SIMD the older goes first wherever both could, ends a quarter of its time ahead and leaves the other to run alone,
        // at little more than half the SIMD's rate (512 x 4096 x 4096: workgroups end between 19 and 25 us). So a wavefront's priority falls as it
        // proceeds. Where more workgroups follow that would hold up the ones about to end: 2048 x 14336 x 512 q8 61.2 -> 66.7 us.
        const int quarter = (g_hi - g + 4 * KS - 1) / (4 * KS) * KS, quarter2 = g + quarter, quarter3 = quarter2 + quarter, quarter4 = quarter3 + quarter;
        if (MT * NT > 1 && one_round) __builtin_amdgcn_s_setprio(3);
        for (; g < g_hi; g += KS) {
            if (MT * NT > 1 && one_round) {
                if (g == quarter2) __builtin_amdgcn_s_setprio(2);
                if (g == quarter3) __builtin_amdgcn_s_setprio(1);
                if (g == quarter4) __builtin_amdgcn_s_setprio(0);
            }
            const int gn = g + KS < g_hi ? g + KS : g;      // past the last group it is repeated (never used)
            constexpr int SW = OUTER ? 1 : NT;           // (a lane's own column is what a pair of column tiles wants of it)
            float sw[4][SW];
            [[maybe_unused]] float sw_odd[2];
            {
                const unsigned long v = sw_now >> sw_shift_now;
                unsigned lo[2], hi[2];
                if constexpr (SW == 2) {
                    const auto x = __builtin_amdgcn_permlane32_swap((unsigned)v, (unsigned)v, false, false);
                    const auto y = __builtin_amdgcn_permlane32_swap((unsigned)(v >> 32), (unsigned)(v >> 32), false, false);
                    lo[0] = x[0]; lo[1] = x[1]; hi[0] = y[0]; hi[1] = y[1];
                } else {
                    lo[0] = (unsigned)v; hi[0] = (unsigned)(v >> 32);
                }
                auto scale = [&](unsigned bits) { return code_scale * __half2float(__ushort_as_half((unsigned short)bits)); };
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int i = 0; i < SW; ++i)
                        sw[j][i] = WHOLE || g * 4 + j < KB ? scale((j < 2 ? lo[i] : hi[i]) >> (16 * (j & 1))) : 0.f;
                if constexpr (OUTER && ODD) {
                    sw_odd[0] = WHOLE || g * 4 + h < KB ? scale(lo[0] >> (16 * h)) : 0.f;
                    sw_odd[1] = WHOLE || g * 4 + 2 + h < KB ? scale(hi[0] >> (16 * h)) : 0.f;
                }
            }
            [[maybe_unused]] f32x32 s_odd;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                // The other buffer was last read in the previous group (those reads have returned once lgkmcnt is 0); its loads have three
                // steps' time, and 3 MT younger ones are in flight when they are waited for. They are buffer loads: global_load_lds counts as a
                // flat access, after which the compiler waits for every load in flight before the next use of any.
                if (j == 0) {
                    asm volatile("" ::: "memory");
                    __builtin_amdgcn_sched_barrier(0);
                    __builtin_amdgcn_s_waitcnt(LGKM0);
                    __builtin_amdgcn_sched_barrier(0);
                    clear_tail(g, buf);
                    if constexpr (OUTER && ODD && !WHOLE) read_sp(buf, 0);       // (its second block may be past the end)
                    load_w(gn, buf ^ 1);
                    load_scales(gn, buf ^ 1);
                }
                load_a((j + 3) & 3, j == 0 ? g * 4 + 3 : gn * 4 + j - 1);
                __builtin_amdgcn_sched_barrier(0);
                if (j == 3) {
                    __builtin_amdgcn_s_waitcnt(vmcnt_imm(3 * MT));
                    asm volatile("" ::: "memory");
                }
                i32x4 B[NT];
#pragma unroll
                for (int i = 0; i < NT; ++i) {
                    if constexpr (Q8) {
                        B[i] = Bn[i];                        // (copied by the loop's unrolling: no instruction)
                    } else {
                        // 16 * (nibble - 8) as int8: the nibble in the upper half of its byte with the top bit flipped
                        const unsigned w0 = Bn[i].x, w1 = Bn[i].y;
                        B[i] = i32x4{(int)(((w0 << 4) & 0xF0F0F0F0u) ^ 0x80808080u), (int)((w0 & 0xF0F0F0F0u) ^ 0x80808080u),
                                     (int)(((w1 << 4) & 0xF0F0F0F0u) ^ 0x80808080u), (int)((w1 & 0xF0F0F0F0u) ^ 0x80808080u)};
                    }
                }
                read_b(j == 3 ? buf ^ 1 : buf, (j + 1) & 3);
                if constexpr (OUTER) {
                    f32x32 zero;
#pragma unroll
                    for (int e = 0; e < 32; ++e) zero[e] = 0.f;
                    const float sp_now = sp, sp_odd_now = sp_odd;
                    read_sp(j == 3 ? buf ^ 1 : buf, (j + 1) & 3);
                    auto dot = [&](int tl) { return __builtin_amdgcn_mfma_i32_32x32x32_i8(A[j][tl / NT], B[tl % NT], i32x16{0}, 0, 0, 0); };
#pragma unroll
                    for (int p = 0; p < PAIRS; ++p) {
                        const int t0 = 2 * p, t1 = 2 * p + 1;
                        // (2 x 2 tiles: the rows of tile p for both)
                        const f32x32 s = MT * NT < 4 ? __builtin_amdgcn_mfma_f32_32x32x1f32(sp_now, sw[j][0], zero, 0, 0, 0)
                                         : p == 0    ? __builtin_amdgcn_mfma_f32_32x32x1f32(sp_now, sw[j][0], zero, 1, 0, 0)
                                                     : __builtin_amdgcn_mfma_f32_32x32x1f32(sp_now, sw[j][0], zero, 1, 1, 0);
                        const i32x16 d0 = dot(t0), d1 = dot(t1);
#pragma unroll
                        for (int e = 0; e < 16; ++e) acc[t0 / NT][t0 % NT][e] += (float)d0[e] * s[e];
#pragma unroll
                        for (int e = 0; e < 16; ++e) acc[t1 / NT][t1 % NT][e] += (float)d1[e] * s[16 + e];
                    }
                    if constexpr (ODD) {
                        if (j % 2 == 0) s_odd = __builtin_amdgcn_mfma_f32_32x32x1f32(sp_odd_now, sw_odd[j / 2], zero, 0, 0, 0);
                        const i32x16 d0 = dot(MT * NT - 1);
#pragma unroll
                        for (int e = 0; e < 16; ++e) acc[MT - 1][NT - 1][e] += (float)d0[e] * s_odd[(j & 1) * 16 + e];
                    }
                } else {
                // a tile's dots are issued ahead of the previous tile's rescale (the last tile's is left to the next block); the empty
                // asm statements keep that order. A row tile's scales of the next block are read once the block's last use of them is past.
#pragma unroll
                for (int tl = 0; tl < MT * NT; ++tl) {
                    const i32x16 dn = __builtin_amdgcn_mfma_i32_32x32x32_i8(A[j][tl / NT], B[tl % NT], i32x16{0}, 0, 0, 0);
                    const int pt = (tl + MT * NT - 1) % (MT * NT), pi = pt / NT, pj = pt % NT;
                    const float s = tl == 0 ? sw_due : sw[j][pj];
#pragma unroll
                    for (int e = 0; e < 4 * RQ; ++e) acc[pi][pj][e] += (float)d[e] * (sa[pi][e] * s);
                    asm volatile("" : "+v"(acc[pi][pj]));
                    if (pj == NT - 1) read_sa(pi, tl == 0 ? buf : (j == 3 ? buf ^ 1 : buf), tl == 0 ? j : (j + 1) & 3);
                    d = dn;
                }
                sw_due = sw[j][NT - 1];
                }
            }
            buf ^= 1;
            sw_now = sw_raw;
            sw_shift_now = sw_shift;
        }
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));            // no LDS-writing load may outlive the loop: its LDS is reused, or another workgroup's
        // the last block's last tile (a wavefront without a group has none)
        if constexpr (!OUTER)
            if (g_lo + ks < g_hi)
#pragma unroll
                for (int e = 0; e < 4 * RQ; ++e) acc[MT - 1][NT - 1][e] += (float)d[e] * (sa[MT - 1][e] * sw_due);

        if constexpr (Q8) break;
        if (code_scale != 1.f) break;
        float finite = 0.f;                                  // NaN if a sum is not finite
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int e = 0; e < 4 * RQ; ++e) finite += acc[i][j][e] * 0.f;
        if (!__any(finite != finite)) break;
        code_scale = 0.0625f;
        sum_scale = 1.f;
    }
    if constexpr (!Q8) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) acc[i][j] *= sum_scale;
    }

    if (partial) {
        // a K slice leaves raw sums; gemm_i8_slices_kernel adds the slices in order and applies alpha and beta
        c = partial + (size_t)blockIdx.z * M * partial_ld + (size_t)first_tile * BN;
        ldc = partial_ld;
        alpha = 1.f;
        beta = 0.f;
    }
    auto put = [&](int mi, int ni, int e, float v) {
        const int row = m0 + mi * 32 + 8 * (e >> 2) + 4 * h + (e & 3), col = n0 + ni * 32 + r;
        if (row >= M || col >= N) return;
        float *dst = c + (size_t)row * ldc + col;
        v *= alpha;
        *dst = beta == 0.f ? v : v + beta * *dst;
    };
    // A lane has four rows of a column of both tiles. GEMM_GATE: a quant block of the gated rows is the 32 lanes of its half.
    [[maybe_unused]] auto put_pair = [&](int i, int q, f32x4 g, f32x4 u) {
        if constexpr (EPI == GEMM_ROPE) {
            // (rope_append_kernel's arithmetic and bounds)
            const int pair = head_tile * 32 + r;
            const bool rot = si < 2 && pair < segs.rope_pairs;
            const float fr = rot ? segs.freq[pair] : 0.f;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int row = m0 + i * 32 + 8 * q + 4 * h + e;
                if (row >= M) continue;
                const float xl = alpha * g[e], xh = alpha * u[e];
                float yl = xl, yh = xh;
                if (rot) {
                    float sn, cs;
                    sincosf((float)segs.positions[row] * fr, &sn, &cs);
                    rope_rotate(xl, xh, sn, cs, yl, yh);
                }
                if (si == 0) {
                    float *dst = segs.q_out + ((size_t)row * segs.h_q + head) * segs.d + pair;
                    dst[0] = yl;
                    dst[partner] = yh;
                    continue;
                }
                const int b = row / segs.s_len;
                const long t = (long)segs.write_index[b] + (long)(row - b * segs.s_len);
                if (t < 0 || t >= segs.t_cap) continue;
                __half *dst = (si == 1 ? segs.kcache : segs.vcache) + (((size_t)b * segs.t_cap + (size_t)t) * segs.h_kv + head) * segs.d + pair;
                dst[0] = __float2half_rn(yl);
                dst[partner] = __float2half_rn(yh);
            }
            return;
        }
        if constexpr (GATE) {
        const int kb = n0 >> 5, KBN = N >> 5, mt = (m0 >> 5) + i, rows = act_tile_rows(M, mt);
        uint8_t *codes = (uint8_t *)segs.c[0] + ((size_t)mt * 32 * KBN + (size_t)kb * rows) * 32 + (r >> 4) * rows * 16 + (r & 15);
        float *scales = segs.c[1] + (size_t)mt * 32 * KBN + (size_t)kb * rows;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int row = 8 * q + 4 * h + e;
            int code;
            float scale;
            prepare_act_lane32(aion_gate_gelu(g[e], u[e]), code, scale);
            if (row >= rows) continue;
            codes[row * 16] = (uint8_t)code;
            if (r == 0) scales[row] = scale;
        }
        }
    };
    if constexpr (PAIR && KS == 1) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int q = 0; q < RQ; ++q) {
                const Acc &g = acc[i][0], &u = acc[i][1];
                put_pair(i, q, f32x4{g[4 * q], g[4 * q + 1], g[4 * q + 2], g[4 * q + 3]}, f32x4{u[4 * q], u[4 * q + 1], u[4 * q + 2], u[4 * q + 3]});
            }
    } else if constexpr (KS == 1) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int e = 0; e < 4 * RQ; ++e) put(i, j, e, acc[i][j][e]);
    } else {
        // the KS partial sums of a tile through LDS, added in wavefront order by the tile's wavefronts, a share each
        constexpr int CH = MT * NT * RQ;                 // 16-byte chunks per lane
        f32x4 *red = (f32x4 *)lds + (size_t)wsub * KS * CH * 64;
        __syncthreads();                                 // (the staged activation scales are dead)
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int q = 0; q < RQ; ++q)
                    red[(ks * CH + (i * NT + j) * RQ + q) * 64 + lane] = f32x4{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
        __syncthreads();
        if constexpr (PAIR) {
#pragma unroll
            for (int p0 = 0; p0 < (MT * RQ + KS - 1) / KS; ++p0) {
                const int p = p0 * KS + ks, i = p / RQ, q = p % RQ, ch = i * 2 * RQ + q;
                if (p >= MT * RQ) break;
                f32x4 g = red[ch * 64 + lane], u = red[(ch + RQ) * 64 + lane];
#pragma unroll
                for (int k = 1; k < KS; ++k) {
                    g += red[(k * CH + ch) * 64 + lane];
                    u += red[(k * CH + ch + RQ) * 64 + lane];
                }
                put_pair(i, q, g, u);
            }
            return;
        }
#pragma unroll
        for (int c0 = 0; c0 < (CH + KS - 1) / KS; ++c0) {
            const int ch = c0 * KS + ks;
            if (ch >= CH) break;
            f32x4 s = red[ch * 64 + lane];
#pragma unroll
            for (int k = 1; k < KS; ++k) s += red[(k * CH + ch) * 64 + lane];
#pragma unroll
            for (int e = 0; e < 4; ++e) put(ch / RQ / NT, ch / RQ % NT, ch % RQ * 4 + e, s[e]);
        }
    }
}

template <int DT, int MT, int NT, int KS, int WGM, int WGN, int RQ, bool WHOLE, int EPI, bool MANY>
__global__ __launch_bounds__(64 * KS * WGM * WGN, MT * NT == 1 ? 4 : 2) void gemm_i8_kernel(const uint8_t *__restrict__ aq, const float *__restrict__ a_scale, const uint8_t *__restrict__ qs0,
                                                                         const __half *__restrict__ sc0, int M, int K, int n0, int form, const uint8_t *__restrict__ qs1,
                                                                         GemmTail<typename GemmSegsOf<EPI, MANY>::type> tail) {
    gemm_i8_body<DT, MT, NT, KS, WGM, WGN, RQ, WHOLE, EPI, MANY>(tail.segs, (int)blockIdx.x, aq, a_scale, qs0, sc0, M, K, n0, qs1, form >> 4, form >> 1 & 7, form & 1, tail.alpha,
                                                                 tail.beta, tail.partial, tail.partial_ld);
}

template <bool Q8, int MT, int NT, int KS, int WGM, int WGN, int RQ> constexpr int gemm_i8_lds_bytes() {
    const int operands = KS * WGM * WGN * gemm_i8_wave_lds_bytes<Q8, MT, NT>(), red = KS > 1 ? KS * WGM * WGN * MT * NT * RQ * 1024 : 0;
    return operands > red ? operands : red;
}

// Shared by the attention kernels: argument block, element conversions, the interval window of a query, the row map of
// rolling caches (attention.hip, attention_prefill.hip).
#pragma once
#include "common.h"

#include <climits>
#include <type_traits>

namespace attn {


using f16x8 = __attribute__((ext_vector_type(8))) _Float16;
using bf16x8 = __attribute__((ext_vector_type(8))) __bf16;

constexpr float LOG2E = 1.4426950408889634f;
constexpr int TILE_KEYS = 32;

struct AttnArgs {
    const void *q, *k, *v;
    float *out;
    const int *positions, *kv_lengths;
    float *partial;
    unsigned *tickets;        // not null: the segments are merged by the workgroup that ends last (attn_flash_body), zero between launches
    int B, L, T, Hq, Hkv, groups, rows_total, row_tiles, nseg;
    int sub;                  // 16-row kernel: the eight wavefronts of a key segment's tiles are divided over 2^sub workgroups, and nseg counts those (attn_flash_body)
    int ring;      // rolling caches: T (logical key t lives in row t % T); 0: row t is key t
    int q_dtype, kv_dtype;
    float scale, soft_cap;
    unsigned win_left, win_right, win_chunk;
    int pf_tiles, pf_first;   // 128-row kernel: row tiles; how many of them go out longest first with the unit fastest, 0: unit by unit (see launch_prefill_t)
    int pf_half;              // 128-row kernel: the segments' partial accumulators are f16 (pf_half_partials)
    int *codes;               // not null: the output leaves as rows prepared for the exact GEMM (PreparedAct::tiled) in place of `out`
    float *code_scales;
};

inline int rows_not_prepared(aionhip_ctx *ctx, const char *why) {
    return set_err(ctx, AIONHIP_UNSUPPORTED, "attention_matmul: the attention step writes f32 rows only (%s)", why);
}

__device__ __forceinline__ unsigned short f32_to_bf16_bits(float x) {
    unsigned u = __float_as_uint(x);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (unsigned short)(u >> 16);
}
__device__ __forceinline__ float bf16_bits_to_f32(unsigned short b) { return __uint_as_float((unsigned)b << 16); }

template <int KV>
__device__ __forceinline__ unsigned short to_half_bits(float x) {
    if (KV == AIONHIP_F16) return __half_as_ushort(__float2half_rn(x));
    return f32_to_bf16_bits(x);
}
template <int KV>
__device__ __forceinline__ float from_half_bits(unsigned short b) {
    if (KV == AIONHIP_F16) return __half2float(__ushort_as_half(b));
    return bf16_bits_to_f32(b);
}
// two f32 -> one 32-bit word of two halves (RNE), low half first
using f32x2 = __attribute__((ext_vector_type(2))) float;
using bf16x2 = __attribute__((ext_vector_type(2))) __bf16;
template <int KV>
__device__ __forceinline__ unsigned pack2(float a, float b) {
    if (KV == AIONHIP_F16) {
        const __half2 h = __floats2half2_rn(a, b);
        return *reinterpret_cast<const unsigned *>(&h);
    }
    // one v_cvt_pk_bf16_f32 (round to nearest even) instead of integer rounding per element
    return __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{a, b}, bf16x2));
}
template <int KV>
__device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
    if (KV == AIONHIP_F16)
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

__device__ __forceinline__ float load_scalar(const void *p, int dtype, size_t i) {
    if (dtype == AIONHIP_F32) return ((const float *)p)[i];
    if (dtype == AIONHIP_F16) return __half2float(((const __half *)p)[i]);
    return bf16_bits_to_f32(((const unsigned short *)p)[i]);
}

// AttentionWindow.keys (aion graph/graph.zig:160-167)
__device__ __forceinline__ void window_keys(unsigned left, unsigned right, unsigned chunk, int pos, int kv_end, int &lo, int &hi) {
    const long anchor = chunk > 0 ? (long)(pos / (int)chunk) * (int)chunk : pos;
    const long span = chunk > 0 ? chunk : 1;
    const long l = anchor - (anchor < (long)left ? anchor : (long)left);
    long h = right == 0xFFFFFFFFu ? (long)INT_MAX : anchor + span + (long)right;
    if (h > kv_end) h = kv_end;
    lo = (int)l;
    hi = (int)h;
}

// Rolling caches (aion storage/cache.zig:202-207, cpu/exec/attention.zig:1072-1075, 1150-1152): the cache length may
// exceed the capacity, keys older than length - capacity are gone, and key t is read from row t % capacity.
__device__ __forceinline__ int phys_key(int ring, int t) { return ring ? (int)((unsigned)t % (unsigned)ring) : t; }
// The same for the keys of one tile, whose first key key0 is uniform: one modulo per tile (base), then an add and
// a conditional subtract per key. Valid while a tile is no longer than the ring (the launcher sees to that).
struct TileMap {
    int key0, base, wrap;
    __device__ __forceinline__ TileMap(int ring, int k0) : key0(k0), base(ring ? (int)((unsigned)k0 % (unsigned)ring) : k0), wrap(ring ? ring : INT_MAX) {}
    __device__ __forceinline__ int row(int key) const {
        const int r = base + (key - key0);
        return r >= wrap ? r - wrap : r;
    }
};
__device__ __forceinline__ int clip_kv_end(int ring, int t_cap, int kv_end_raw) {
    return ring ? max(0, kv_end_raw) : max(0, min(kv_end_raw, t_cap));
}
__device__ __forceinline__ void clip_to_ring(int ring, int kv_end, int &lo, int &hi) {
    if (ring) lo = max(lo, kv_end - ring);
    if (hi < lo) hi = lo;
}

__device__ __forceinline__ int wave_min_i(int v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v = min(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ __forceinline__ int wave_max_i(int v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
    return v;
}
// Minimum / maximum over the sixteen rows of a wavefront whose lanes l, l + 16, l + 32, l + 48 hold the same value: four DPP steps on
// the vector pipe (an LDS permute is some 60 cycles of latency each), the result in a scalar register.
__device__ __forceinline__ int rows16_min_i(int v) {
    v = min(v, dpp_i<DPP_QUAD_XOR1>(v));
    v = min(v, dpp_i<DPP_QUAD_XOR2>(v));
    v = min(v, dpp_i<DPP_ROW_HALF_MIRROR>(v));
    v = min(v, dpp_i<DPP_ROW_MIRROR>(v));
    return __builtin_amdgcn_readfirstlane(v);
}
__device__ __forceinline__ int rows16_max_i(int v) {
    v = max(v, dpp_i<DPP_QUAD_XOR1>(v));
    v = max(v, dpp_i<DPP_QUAD_XOR2>(v));
    v = max(v, dpp_i<DPP_ROW_HALF_MIRROR>(v));
    v = max(v, dpp_i<DPP_ROW_MIRROR>(v));
    return __builtin_amdgcn_readfirstlane(v);
}
// Maximum / sum over the four lanes l, l + 16, l + 32, l + 48: swapped with itself, a register's halves (rows of sixteen) end up as
// both operands of one vector instruction. Sums are taken as ((r0 + r1) + (r2 + r3)), the order of an exchange across 16, then 32.
__device__ __forceinline__ float groups4_max(float v) {
    auto x = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(x[0]), __uint_as_float(x[1]));
    x = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(x[0]), __uint_as_float(x[1]));
}
// over the 64 lanes, in the order of wave_sum and wave_max, without their two LDS permutes
__device__ __forceinline__ float lanes_max(float v) {
    v = fmaxf(v, dpp_f<DPP_QUAD_XOR1>(v));
    v = fmaxf(v, dpp_f<DPP_QUAD_XOR2>(v));
    v = fmaxf(v, dpp_f<DPP_ROW_HALF_MIRROR>(v));
    return groups4_max(fmaxf(v, dpp_f<DPP_ROW_MIRROR>(v)));
}
// 4^n for a whole n <= 0: exact, zero below 2^-126
__device__ __forceinline__ float pow4(float n) { return __builtin_amdgcn_exp2f(2.f * n); }
// the value of the lane 32 away
__device__ __forceinline__ float half_swap(float v) {
    const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float((__lane_id() & 32) ? x[0] : x[1]);
}
__device__ __forceinline__ float groups4_sum(float v) {
    auto x = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(x[0]) + __uint_as_float(x[1]);
    x = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(x[0]) + __uint_as_float(x[1]);
}
__device__ __forceinline__ float lanes_sum(float v) {
    v += dpp_f<DPP_QUAD_XOR1>(v);
    v += dpp_f<DPP_QUAD_XOR2>(v);
    v += dpp_f<DPP_ROW_HALF_MIRROR>(v);
    return groups4_sum(v + dpp_f<DPP_ROW_MIRROR>(v));
}

using u32x2 = __attribute__((ext_vector_type(2))) unsigned int;
// f(integral_constant<int, I>) for I in [I0, E): a loop whose index is a constant expression in the body (immediate
// operands of assembly, if constexpr)
template <int I, int E, class F>
__device__ __forceinline__ void static_for(F &&f) {
    if constexpr (I < E) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, E>(f);
    }
}

// ---- prefill kernel (attention_prefill.hip): 128 query rows per workgroup, 64-key tiles
constexpr int PF_ROWS = 128, PF_TK = 64;
#ifndef PF_FLASH_BELOW
#define PF_FLASH_BELOW 8   // prompts whose 128-row workgroups would fill under 1/PF_FLASH_BELOW of the CUs (head size 256; more at smaller heads) run on the 16-row split kernel
#endif
// whether the prefill kernel takes this call (head size 64, 128 or 256; K/V f16 or bf16; not the hi+lo precise mode)
bool prefill_takes(const AttnArgs &a, int d);
int launch_prefill(aionhip_ctx *ctx, AttnArgs &a, int d);

}  // namespace attn

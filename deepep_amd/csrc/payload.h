// The payload of a dispatch, out[row(t,s)] = x[t], as device functions: token-major or row-major, copied or quantised to FP8.  They run as
// kernels of their own behind a layout that has ended (Mapped..., dispatch.hip), or in the layout's own grid, where they look for the
// places of their rows (Awaited..., layout.hip).
//
// Observable contract: as dispatch.hip.
#pragma once
#include "common.h"

#pragma clang fp contract(off)

namespace dpep {

constexpr int kMaxThreads = 256;
constexpr int kMaxScaleCols = 1024;  // hidden <= 131072 for the fused quantiser

template <int kPolicy>
__device__ __forceinline__ void store16_as(void* p, u32x4 v)
{
    if (kPolicy == DPEP_STORE_THROUGH) store16_through(p, v);
    else if (kPolicy == DPEP_STORE_STREAMING) store16_nt(p, v);
    else *reinterpret_cast<u32x4*>(p) = v;
}

// One payload launch.  units per row: 16-byte vectors (copy), or 16-value groups (quantise), in `parts` column parts of `per_part`;
// one token (token-major) or row (row-major) and part to `threads` threads.  (The pointers are parameters of their own: __restrict__ counts on
// those alone, and without it no load of a row overtakes a store, 0.3 us of a few hundred rows.)
struct PayloadShape {
    int num_tokens, num_topk, units, per_part, parts, threads, scale_cols;
};

// ---- where a payload's workgroups find its rows -------------------------------------------------------------------------
// LDS of a token's threads: its rows (-1: none), and whether there is any.
struct TokenLds {
    int rows[DPEP_MAX_TOPK];
    int any_valid;
};

// Token-major, in the map that an earlier launch has left.  Rows at or beyond `capacity` are dropped; with all_rows (the layout's
// count) nothing is moved unless DPEP_ROWS_KEPT.
struct MappedTokens {
    const int* route_to_row;
    int capacity;
    const int* all_rows;
    __device__ __forceinline__ int begin() const { return all_rows != nullptr ? *all_rows : capacity; }  // (travels with the values and the routes)
    // The token's rows into lds.rows; whether there is any.  Called by all threads of the workgroup.
    __device__ __forceinline__ bool find_rows(const PayloadShape& p, int all, int token, int t, TokenLds& lds) const
    {
        if (t == 0) lds.any_valid = 0;
        __syncthreads();
        if (t < p.num_topk) {
            int row = route_to_row[static_cast<size_t>(token) * p.num_topk + t];
            if (row >= capacity || !DPEP_ROWS_KEPT(all, capacity)) row = -1;  // outputs allocated before R was known
            lds.rows[t] = row;
            if (row >= 0) lds.any_valid = 1;
        }
        __syncthreads();
        return lds.any_valid != 0;
    }
};

// In the layout's own grid (layout.hip) a route's row, or a row's route, comes as a word that says itself which launch it belongs to:
// the launch's number above, the value (-1: no row) below.  The number of rows comes the same way.
__device__ __forceinline__ unsigned long long row_word(uint32_t launch, int value)
{
    return static_cast<unsigned long long>(launch) << 32 | static_cast<uint32_t>(value);
}

// ---- token-major: one token and column part to `p.threads` threads; read once, write K times ----------------------------------
// t: the thread's number among them.  Called by all threads of a workgroup whose `block` is in range.

// How far (in 16-byte vectors) an address lies behind the start of its cache line.
__device__ __forceinline__ int behind_line(const void* p) { return static_cast<int>(reinterpret_cast<uintptr_t>(p) >> 4 & 7); }

// kStaged: rows that are no whole lines.  A wave's 1 KB would begin and end inside a line of every such row, two partial writes to HBM each: the
// piece goes through LDS (`stage`, kStagedVec vectors), and each row is written from the start of a line on.
constexpr int kStagedVec = 4 * kMaxThreads;
template <int kPolicy, bool kStaged, typename Tokens>
__device__ __forceinline__ void copy_token(const u32x4* __restrict__ x, const float* __restrict__ scales, const float* __restrict__ weights,
                                           u32x4* __restrict__ out, float* __restrict__ out_scales, float* __restrict__ out_weights,
                                           const PayloadShape& p, const Tokens& tokens, unsigned block, int t, TokenLds& lds,
                                           u32x4* stage = nullptr)
{
    const int token = block / static_cast<unsigned>(p.parts), part = block % static_cast<unsigned>(p.parts);
    const int all = tokens.begin();
    const int v_begin = part * p.per_part, v_end = min(v_begin + p.per_part, p.units);
    const u32x4* src = x + static_cast<size_t>(token) * p.units;
    // The token's first values are asked for before its routes are known (see the quantising one below), and written row by row: 4 KB and
    // more of one row at a time instead of 1 KB of every row in turn (6045 tokens x top-10 of 6064 BF16 columns, dispatch and
    // combine 357 -> 353 us, 4372 x 7 of 5840 178 -> 173).
    const int v_first = v_begin + t;
    constexpr int kEarly = 2;
    u32x4 early[kEarly];
#pragma unroll
    for (int j = 0; j < kEarly; ++j)
        if (v_first + j * p.threads < v_end) early[j] = load16(src + v_first + j * p.threads);
    if constexpr (kStaged) {
#pragma unroll
        for (int j = 0; j < kEarly; ++j)
            if (v_first + j * p.threads < v_end) stage[t + j * p.threads] = early[j];
        for (int v = v_first + kEarly * p.threads; v < v_end; v += p.threads) stage[v - v_begin] = load16(src + v);
    }
    if (!tokens.find_rows(p, all, token, t, lds)) return;  // (with a barrier behind the staging)
    for (int s = 0; s < p.num_topk; ++s) {
        const int row = lds.rows[s];
        if (row < 0) continue;
        u32x4* dst = out + static_cast<size_t>(row) * p.units;
        if constexpr (kStaged) {
            for (int i = t - behind_line(dst + v_begin); i < v_end - v_begin; i += p.threads)
                if (i >= 0) store16_as<kPolicy>(dst + v_begin + i, stage[i]);
        } else {
#pragma unroll
            for (int j = 0; j < kEarly; ++j)
                if (v_first + j * p.threads < v_end) store16_as<kPolicy>(dst + v_first + j * p.threads, early[j]);
        }
    }
    for (int v = v_first + kEarly * p.threads; v < v_end && !kStaged; v += p.threads) {  // rows wider than that
        const u32x4 value = load16(src + v);
        for (int s = 0; s < p.num_topk; ++s) {
            const int row = lds.rows[s];
            if (row >= 0) store16_as<kPolicy>(out + static_cast<size_t>(row) * p.units + v, value);
        }
    }
    if (part == 0) {
        if (scales != nullptr) {
            for (int c = t; c < p.scale_cols; c += p.threads) {
                const float value = scales[static_cast<size_t>(token) * p.scale_cols + c];
                for (int s = 0; s < p.num_topk; ++s) {
                    const int row = lds.rows[s];
                    if (row >= 0) out_scales[static_cast<size_t>(row) * p.scale_cols + c] = value;
                }
            }
        }
        if (weights != nullptr && t < p.num_topk && lds.rows[t] >= 0)
            out_weights[lds.rows[t]] = weights[static_cast<size_t>(token) * p.num_topk + t];
    }
}

// ---- row-major, in the layout's grid: one output row and column part to `p.threads` threads; for sparse receive shares --------
// stride: rows between two of a workgroup.  (dispatch.hip has the same for maps that are there already: in one piece with this its prologue
// grew by 0.1 us, a fortieth of what a few hundred rows take.)
template <int kPolicy, typename Rows>
__device__ __forceinline__ void copy_rows(const u32x4* __restrict__ x, const float* __restrict__ scales, const float* __restrict__ weights,
                                          u32x4* __restrict__ out, float* __restrict__ out_scales, float* __restrict__ out_weights,
                                          const PayloadShape& p, const Rows& source, unsigned block, int stride, int t)
{
    const int part = block % static_cast<unsigned>(p.parts);
    const int v_begin = part * p.per_part, v_end = min(v_begin + p.per_part, p.units);
    int row = block / static_cast<unsigned>(p.parts);
    for (; row < source.rows; row += stride) {
        const int route = source.route_of(row);
        if (route < 0) return;
        const int token = route / p.num_topk;
        const u32x4* src = x + static_cast<size_t>(token) * p.units;
        u32x4* dst = out + static_cast<size_t>(row) * p.units;
        for (int v = v_begin + t; v < v_end; v += p.threads) store16_as<kPolicy>(dst + v, load16(src + v));
        if (part == 0) {
            if (scales != nullptr)
                for (int c = t; c < p.scale_cols; c += p.threads)
                    out_scales[static_cast<size_t>(row) * p.scale_cols + c] = scales[static_cast<size_t>(token) * p.scale_cols + c];
            if (weights != nullptr && t == 0) out_weights[row] = weights[route];
        }
    }
}

// ---- per-128 FP8 quantiser ------------------------------------------------------------------------
// One lane owns 16 consecutive BF16 values (two 16-byte loads), so 8 adjacent lanes own one
// 128-element block.  amax is reduced over those 8 lanes with DPP-free xor shuffles inside the wave.
struct Quant16 {
    u32x4 codes;  // 16 e4m3fn bytes
    float scale;  // amax / 448
};

// Largest of a value over the 8 lanes that share a 128-element block.
__device__ __forceinline__ uint32_t max8(uint32_t v)
{
    v = max(v, static_cast<uint32_t>(__shfl_xor(static_cast<int>(v), 1)));
    v = max(v, static_cast<uint32_t>(__shfl_xor(static_cast<int>(v), 2)));
    v = max(v, static_cast<uint32_t>(__shfl_xor(static_cast<int>(v), 4)));
    return v;
}

// fp32 -> e4m3fn byte pair, round-to-nearest-even, on the gfx950 converter (OCP FP8).
__device__ __forceinline__ uint32_t pack4_e4m3(float a, float b, float c, float d)
{
    int packed = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false);
    packed = __builtin_amdgcn_cvt_pk_fp8_f32(c, d, packed, true);
    return static_cast<uint32_t>(packed);
}

__device__ __forceinline__ Quant16 quantize16(u32x4 lo, u32x4 hi)
{
    float v[16];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v[2 * i] = bf16_to_f32(lo[i] & 0xffffu);
        v[2 * i + 1] = bf16_to_f32(lo[i] >> 16);
        v[8 + 2 * i] = bf16_to_f32(hi[i] & 0xffffu);
        v[8 + 2 * i + 1] = bf16_to_f32(hi[i] >> 16);
    }
    // amax as the largest magnitude BIT PATTERN (two BF16 magnitudes per word, v_pk_max_u16): for finite values that is
    // the largest magnitude, and a NaN, whose pattern lies above infinity's, wins over everything, as it does in the
    // reference's amax() and clamp() (torch propagates NaN through both, deep_ep/utils/math.py:52-53): a block that
    // holds a NaN gets a NaN scale and the NaN code 0x7F for every value, whatever the others are.
    typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
    u16x2 both = {0, 0};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        both = __builtin_elementwise_max(both, __builtin_bit_cast(u16x2, lo[i] & 0x7fff7fffu));
        both = __builtin_elementwise_max(both, __builtin_bit_cast(u16x2, hi[i] & 0x7fff7fffu));
    }
    const uint32_t mine = max(static_cast<uint32_t>(both[0]), static_cast<uint32_t>(both[1]));
    const uint32_t amax_bits = max(max8(mine) << 16, __float_as_uint(1e-4f));
    const float amax = __uint_as_float(amax_bits);
    const bool poisoned = amax_bits > 0x7f800000u;
    // The reference writes 448.0 / amax, which torch evaluates as reciprocal(amax) * 448:
    // two correctly rounded fp32 operations, reproduced here.
    const float inv = __fmul_rn(__fdiv_rn(1.0f, amax), 448.0f);
    Quant16 q;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t codes = pack4_e4m3(__fmul_rn(v[4 * i], inv), __fmul_rn(v[4 * i + 1], inv), __fmul_rn(v[4 * i + 2], inv),
                                          __fmul_rn(v[4 * i + 3], inv));
        q.codes[i] = poisoned ? 0x7f7f7f7fu : codes;
    }
    q.scale = __fdiv_rn(amax, 448.0f);
    return q;
}

// token-major; part_scales: LDS for the part's scales.
template <int kPolicy, typename Tokens>
__device__ __forceinline__ void quant_token(const u32x4* __restrict__ x, const float* __restrict__ weights, u32x4* __restrict__ out,
                                            float* __restrict__ out_scales, float* __restrict__ out_weights, const PayloadShape& p,
                                            const Tokens& tokens, unsigned block, int t, TokenLds& lds, float* part_scales)
{
    const int token = block / static_cast<unsigned>(p.parts), part = block % static_cast<unsigned>(p.parts);
    const int all = tokens.begin();
    const int u_begin = part * p.per_part, u_end = min(u_begin + p.per_part, p.units);
    const u32x4* src = x + static_cast<size_t>(token) * p.units * 2;
    // The token's first values are asked for before its routes are known: this grid is only used where most tokens own
    // rows, and the row lookup and the payload then travel together instead of one after the other.
    const int u_first = u_begin + t;
    constexpr int kEarly = 2;  // units per thread fetched up front (all of a 7168-wide row with 256 threads)
    u32x4 lo[kEarly], hi[kEarly];
#pragma unroll
    for (int j = 0; j < kEarly; ++j) {
        const int u = u_first + j * p.threads;
        if (u < u_end) {
            lo[j] = load16(src + 2 * u);
            hi[j] = load16(src + 2 * u + 1);
        }
    }
    if (!tokens.find_rows(p, all, token, t, lds)) return;
    const int scale_cols = p.units / 8;
    // per_part is a multiple of 8 and the threads of 64, so the 8 lanes of a block stay together.
    // Quantise first, then write row by row: at any moment the workgroup's stores run along ONE output row.
    u32x4 codes[kEarly];
#pragma unroll
    for (int j = 0; j < kEarly; ++j) {
        const int u = u_first + j * p.threads;
        if (u < u_end) {
            const Quant16 q = quantize16(lo[j], hi[j]);
            codes[j] = q.codes;
            if ((u & 7) == 0) part_scales[(u - u_begin) >> 3] = q.scale;
        }
    }
    for (int s = 0; s < p.num_topk; ++s) {
        const int row = lds.rows[s];
        if (row < 0) continue;
#pragma unroll
        for (int j = 0; j < kEarly; ++j) {
            const int u = u_first + j * p.threads;
            if (u < u_end) store16_as<kPolicy>(out + static_cast<size_t>(row) * p.units + u, codes[j]);
        }
    }
    for (int u = u_first + kEarly * p.threads; u < u_end; u += p.threads) {  // rows wider than that
        const Quant16 q = quantize16(load16(src + 2 * u), load16(src + 2 * u + 1));
        for (int s = 0; s < p.num_topk; ++s) {
            const int row = lds.rows[s];
            if (row >= 0) store16_as<kPolicy>(out + static_cast<size_t>(row) * p.units + u, q.codes);
        }
        if ((u & 7) == 0) part_scales[(u - u_begin) >> 3] = q.scale;
    }
    __syncthreads();
    // The part's scales leave as contiguous runs (consecutive lanes, consecutive floats) instead of one
    // 4-byte store per block of 128, which would turn every scale row into read-modify-write traffic.
    const int part_cols = (u_end - u_begin) >> 3, col0 = u_begin >> 3;
    for (int i = t; i < p.num_topk * part_cols; i += p.threads) {
        const int s = i / part_cols, c = i - s * part_cols;
        const int row = lds.rows[s];
        if (row >= 0) out_scales[static_cast<size_t>(row) * scale_cols + col0 + c] = part_scales[c];
    }
    if (part == 0 && weights != nullptr && t < p.num_topk && lds.rows[t] >= 0)
        out_weights[lds.rows[t]] = weights[static_cast<size_t>(token) * p.num_topk + t];
}

// row-major, in the layout's grid
template <int kPolicy, typename Rows>
__device__ __forceinline__ void quant_rows(const u32x4* __restrict__ x, const float* __restrict__ weights, u32x4* __restrict__ out,
                                           float* __restrict__ out_scales, float* __restrict__ out_weights, const PayloadShape& p,
                                           const Rows& source, unsigned block, int stride, int t)
{
    const int part = block % static_cast<unsigned>(p.parts);
    const int u_begin = part * p.per_part, u_end = min(u_begin + p.per_part, p.units);
    const int scale_cols = p.units / 8;
    int row = block / static_cast<unsigned>(p.parts);
    for (; row < source.rows; row += stride) {
        const int route = source.route_of(row);
        if (route < 0) return;
        const int token = route / p.num_topk;
        const u32x4* src = x + static_cast<size_t>(token) * p.units * 2;
        for (int u = u_begin + t; u < u_end; u += p.threads) {
            const Quant16 q = quantize16(load16(src + 2 * u), load16(src + 2 * u + 1));
            store16_as<kPolicy>(out + static_cast<size_t>(row) * p.units + u, q.codes);
            if ((u & 7) == 0) out_scales[static_cast<size_t>(row) * scale_cols + (u >> 3)] = q.scale;
        }
        if (part == 0 && weights != nullptr && t == 0) out_weights[row] = weights[route];
    }
}

// A payload that may ride in the layout's grid (host side).  blocks: tokens, or rows of the grid, times column parts.
struct LayoutPayload {
    const u32x4* x;
    const float* scales;
    const float* weights;
    u32x4* out;
    float* out_scales;
    float* out_weights;
    PayloadShape shape;
    bool quantize, staged, row_major;
    unsigned blocks;
    int rows, capacity, all_or_none;  // rows: row-major, the bound of R; the others: token-major
    int looks;                        // of a workgroup for a word of the layout's
};

}  // namespace dpep

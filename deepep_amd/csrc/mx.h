// MXFP8 activations (block 32 along the row): the quantiser's arithmetic, and the preparation of a MegaMoE forward's input rows.
//
// Numerics: experiments/megamoe/python/deep_ep_experimental/megamoe/reference.py:44-54.
#pragma once
#include "common.h"

#pragma clang fp contract(off)

namespace dpep {

// e8m0 byte of a block with maximum magnitude amax: biased_exponent(max(amax, 2^-119)) - 8.
__device__ __forceinline__ int mx_scale_byte(float amax)
{
    const float floored = fmaxf(amax, 0x1p-119f);
    return static_cast<int>(__float_as_uint(floored) >> 23) - 8;
}

// v * 2^(127 - byte), magnitude clamped to 448, rounded to e4m3fn (nearest even).
__device__ __forceinline__ float mx_scaled(float v, int byte)
{
    const float scaled = ldexpf(v, 127 - byte);
    return fminf(fmaxf(scaled, -448.0f), 448.0f);
}

__device__ __forceinline__ uint32_t mx_pack4(float a, float b, float c, float d)
{
    int packed = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false);
    packed = __builtin_amdgcn_cvt_pk_fp8_f32(c, d, packed, true);
    return static_cast<uint32_t>(packed);
}

// 16 consecutive BF16 values, half a block (the other half belongs to the neighbouring lane, which must be active) ->
// 16 codes and the block's scale byte.
__device__ __forceinline__ u32x4 mx_quantize16(u32x4 lo, u32x4 hi, int& byte)
{
    float v[16];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const uint32_t raw = i < 4 ? lo[i & 3] : hi[i & 3];
        v[2 * i] = bf16_to_f32(raw & 0xffffu);
        v[2 * i + 1] = bf16_to_f32(raw >> 16);
    }
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) amax = fmaxf(amax, fabsf(v[i]));
    amax = fmaxf(amax, __shfl_xor(amax, 1));
    byte = mx_scale_byte(amax);
    u32x4 out;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        out[i] = mx_pack4(mx_scaled(v[4 * i], byte), mx_scaled(v[4 * i + 1], byte), mx_scaled(v[4 * i + 2], byte), mx_scaled(v[4 * i + 3], byte));
    return out;
}

// What a MegaMoE forward's GEMMs need besides the routed layout; null / zero where there is nothing to do.
// Input rows: BF16 to be quantised, or (codes, scale bytes) to be copied behind which the padding columns lie; h columns in,
// hp out (hp a multiple of 256; zero codes and the scale byte of 1.0 behind column h).  The work is `units` pieces of 16
// output columns, one per thread of 256-thread workgroups.
// Shared experts: their rows follow the routed ones, expert-major, token order: offsets[num_local + 1 + s] = R + (s + 1) * B and
// row_to_route[R + s * B + t] = t * topk (so that the gather's route / topk is t).
struct MegaFront {
    const u32x4* bf16;
    const uint8_t* codes;
    const uint8_t* scales;
    int h, hp;
    unsigned units;
    u32x4* codes_out;
    uint8_t* scales_out;
    int num_shared, num_tokens, num_topk;
    // Not null: rows whose token has no route to experts expert_begin .. + num_local are left as they are (nobody reads them).
    const int32_t* topk_idx;
    int expert_begin, num_local;
};
constexpr int kFrontThreads = 256;
inline __host__ __device__ unsigned front_blocks(const MegaFront& f, int threads) { return (f.units + threads - 1) / threads; }

// Whether row `row` has a route to a local expert.  The rows of a wave's lanes follow one another, so their ids are one piece of memory: one
// load and a ballot.  (More than 64 ids, as with rows of 256 columns and 16 routes each: not looked at.)  Called by whole waves.
__device__ __forceinline__ bool row_is_served(const MegaFront& f, unsigned row)
{
    const unsigned lane = threadIdx.x & 63, last = f.num_tokens - 1, mine = row < last ? row : last;
    const unsigned first = __builtin_amdgcn_readfirstlane(mine), end = __builtin_amdgcn_readlane(mine, 63) + 1;
    const unsigned ids = (end - first) * f.num_topk;
    if (ids > 64) return true;
    const int id = lane < ids ? f.topk_idx[static_cast<size_t>(first) * f.num_topk + lane] - f.expert_begin : -1;
    const unsigned long long served = __ballot(id >= 0 && id < f.num_local) >> ((mine - first) * f.num_topk);
    return (served & (~0ull >> (64 - f.num_topk))) != 0ull;
}

// One workgroup's piece of the input rows.  staged: kThreads / 2 bytes of LDS, 16-byte aligned (the workgroup's scale bytes leave as
// 16-byte stores).  Called by all threads.
template <int kThreads>
__device__ __forceinline__ void prepare_rows(const MegaFront& f, unsigned block, uint8_t* staged)
{
    const unsigned unit = block * kThreads + threadIdx.x, per_row = f.hp / 16;
    const unsigned row = unit / per_row, at = unit - row * per_row;
    const bool wanted = f.topk_idx == nullptr || row_is_served(f, row), live = wanted && unit < f.units;
    const bool real = live && at * 16 < static_cast<unsigned>(f.h);  // (h is a multiple of 32: both lanes of a block agree)
    const u32x4 zero = {0u, 0u, 0u, 0u};
    u32x4 codes = zero;
    int byte = 127;
    if (f.bf16 != nullptr) {
        const u32x4* src = f.bf16 + (static_cast<size_t>(row) * (f.h / 16) + at) * 2;
        const u32x4 lo = real ? load16_nt(src) : zero, hi = real ? load16_nt(src + 1) : zero;
        int quantised;
        const u32x4 q = mx_quantize16(lo, hi, quantised);
        if (real) {
            codes = q;
            byte = quantised;
        }
    } else if (real) {
        codes = load16(f.codes + static_cast<size_t>(row) * f.h + at * 16);
        byte = f.scales[static_cast<size_t>(row) * (f.h / 32) + (at >> 1)];
    }
    if (live) f.codes_out[unit] = codes;  // (cached: the GEMM gathers these rows next)
    if ((threadIdx.x & 1) == 0) staged[threadIdx.x >> 1] = static_cast<uint8_t>(byte);
    __syncthreads();
    const unsigned first = block * (kThreads / 2), blocks = f.units >> 1;
    if (first + kThreads / 2 <= blocks) {
        if (threadIdx.x < kThreads / 32)
            *reinterpret_cast<u32x4*>(f.scales_out + first + threadIdx.x * 16) = *reinterpret_cast<const u32x4*>(staged + threadIdx.x * 16);
    } else if (threadIdx.x < blocks - first && threadIdx.x < kThreads / 2) {
        f.scales_out[first + threadIdx.x] = staged[threadIdx.x];
    }
}

// The shared experts' rows, by `threads` threads of which this is number `thread`; first = R.
__device__ __forceinline__ void shared_rows(const MegaFront& f, int first, int num_local, int* offsets, int* row_to_route, unsigned thread, unsigned threads)
{
    const unsigned total = static_cast<unsigned>(f.num_shared) * f.num_tokens;
    if (thread < static_cast<unsigned>(f.num_shared)) offsets[num_local + 1 + thread] = first + static_cast<int>(thread + 1) * f.num_tokens;
    for (unsigned i = thread; i < total; i += threads) row_to_route[first + i] = static_cast<int>(i % f.num_tokens) * f.num_topk;
}

}  // namespace dpep

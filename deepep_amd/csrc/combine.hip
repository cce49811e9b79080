// Combine: every token gathers its expert rows and reduces them in fp32, in slot order, with an
// optional per-row weight, then rounds once to BF16.  A token (column part) is owned by exactly one
// workgroup, so there are no atomics and the summation order is fixed.
//
// Operation order follows the reference's aggregate kernel
// (csrc/direct/kernels/aggregate/aggregate_impl.h:166-226): acc = +0; per valid slot
// tmp = float(y); tmp = tmp * w; acc = acc + tmp (separate multiply and add); final cast RNE.
// Unweighted form: tests/elastic/test_combine.py:504-515; weighted form:
// tests/elastic/test_ep_low_latency.py:449-463; weight-return channel: docs/elastic.md:71.
#include <algorithm>

#include "common.h"

#pragma clang fp contract(off)

namespace dpep {
namespace {

constexpr int kMaxThreads = 256;
constexpr int kSparseTargetBlocks = 2048;    // sparse shares: a workgroup per token while that fills the chip
constexpr int kBatch = 8;  // rows fetched per thread before the dependent adds start

// One vector of a token: the sum over its slots (rows[s] < 0: none), kBatch rows in flight.  Slots ascending, separate fp32 multiply and
// add, one rounding.
template <int kWeights, bool kHalf>
__device__ __forceinline__ u32x4 combined(const u32x4* __restrict__ y, const int* rows, const float* wts, int num_slots, int vec_per_row, int v)
{
    float acc[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = 0.0f;
    for (int s0 = 0; s0 < num_slots; s0 += kBatch) {
        u32x4 val[kBatch];
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            const int row = rows[s0 + j];
            if (row >= 0) val[j] = load16_nt(y + static_cast<size_t>(row) * vec_per_row + v);
        }
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            if (rows[s0 + j] < 0) continue;
            const float w = kWeights != 0 ? wts[s0 + j] : 1.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float lo = kHalf ? f16_to_f32(val[j][i] & 0xffffu) : bf16_to_f32(val[j][i] & 0xffffu);
                float hi = kHalf ? f16_to_f32(val[j][i] >> 16) : bf16_to_f32(val[j][i] >> 16);
                if (kWeights != 0) {
                    lo = __fmul_rn(lo, w);
                    hi = __fmul_rn(hi, w);
                }
                acc[2 * i] = __fadd_rn(acc[2 * i], lo);
                acc[2 * i + 1] = __fadd_rn(acc[2 * i + 1], hi);
            }
        }
    }
    u32x4 packed;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        packed[i] = kHalf ? pack_f16x2(acc[2 * i], acc[2 * i + 1]) : pack_bf16x2(acc[2 * i], acc[2 * i + 1]);
    return packed;
}

// kWeights: 0 = plain sum, 1 = weight per expert row (w[row]), 2 = weight per route (w[t*K + s]).
// kHalf: rows and output are IEEE half instead of BF16.
template <int kWeights, bool kHalf = false>
__global__ __launch_bounds__(kMaxThreads) void combine_kernel(
    const u32x4* __restrict__ y, const float* __restrict__ row_weights, const int* __restrict__ route_to_row,
    int num_topk, int vec_per_row, int vec_per_part, int parts, u32x4* __restrict__ out,
    const float* __restrict__ return_in, float* __restrict__ return_out, const int* __restrict__ shared_first_row,
    int num_shared, int num_tokens, const int* __restrict__ fill_state, int num_rows, int leave_unserved)
{
    __shared__ int rows[DPEP_MAX_TOPK + kBatch];
    __shared__ float wts[DPEP_MAX_TOPK + kBatch];
    const int token = blockIdx.x / parts, part = blockIdx.x % parts;
    if (threadIdx.x < DPEP_MAX_TOPK + kBatch) {
        int row = -1;
        if (threadIdx.x < num_topk) row = route_to_row[static_cast<size_t>(token) * num_topk + threadIdx.x];
        if (row >= num_rows) row = -1;  // a row the caller's y does not hold (capacity layouts drop surplus rows)
        rows[threadIdx.x] = row;
        if (kWeights == 1) wts[threadIdx.x] = row >= 0 ? row_weights[row] : 0.0f;
        if (kWeights == 2)
            wts[threadIdx.x] = row >= 0 ? row_weights[static_cast<size_t>(token) * num_topk + threadIdx.x] : 0.0f;
        if (part == 0 && return_out != nullptr && threadIdx.x < num_topk)
            return_out[static_cast<size_t>(token) * num_topk + threadIdx.x] = row >= 0 ? return_in[row] : 0.0f;
        // Shared experts (MegaMoE): slot K + j is row first + j * B + token with weight 1, summed after the routes.
        if (kWeights == 2 && threadIdx.x >= num_topk && threadIdx.x < num_topk + num_shared) {
            rows[threadIdx.x] = shared_first_row[0] + (threadIdx.x - num_topk) * num_tokens + token;
            wts[threadIdx.x] = 1.0f;
        }
    }
    const int num_slots = num_topk + (kWeights == 2 ? num_shared : 0);
    // Tokens without any row (the common case of a sparse receive share) are plain zero fill.  Streaming
    // stores: cached ones would push the rows read next, and the caller's other data, out of the caches.
    const bool any_row = __syncthreads_or(threadIdx.x < num_slots && rows[threadIdx.x] >= 0) != 0;
    const int v_begin = part * vec_per_part;
    const int v_end = min(v_begin + vec_per_part, vec_per_row);
    if (!any_row) {
        if (leave_unserved) return;  // the caller wants only the tokens that own a row written
        // (MegaMoE) rows that idle workgroups of the first GEMM have already zeroed: filler f of n took tokens
        // f, f + n, ... and got through fill_state[1 + f] of them
        if (kWeights == 2 && fill_state != nullptr) {
            const int fillers = fill_state[0];
            if (fillers > 0 && token / fillers < fill_state[1 + token % fillers]) return;
        }
        const u32x4 zero = {0u, 0u, 0u, 0u};
        for (int v = v_begin + threadIdx.x; v < v_end; v += blockDim.x)
            store16_nt(out + static_cast<size_t>(token) * vec_per_row + v, zero);
        return;
    }
    for (int v = v_begin + threadIdx.x; v < v_end; v += blockDim.x) {
        store16_through(out + static_cast<size_t>(token) * vec_per_row + v, combined<kWeights, kHalf>(y, rows, wts, num_slots, vec_per_row, v));
    }
}

// Dense routing, rows of more than 64 vectors that are no multiple of that: the output's vectors one after the other, 64 to a one-wave workgroup, which holds the slots
// of the two tokens that it may touch.  No wave has lanes behind a row's end, and every store is whole lines.
// Bound by HBM: rows read at 6 TB/s.  Against a workgroup for every started 64 vectors of a row (dispatch and combine, BF16): 6000 tokens x top-10 of 528
// columns 43.5 -> 38.1 us, 6249 x 7 of 1552 69.1 -> 65.3, 5000 x 6 of 832 29.4 -> 27.6.
template <int kWeights, bool kHalf = false>
__global__ __launch_bounds__(64) void combine_dense_kernel(
    const u32x4* __restrict__ y, const float* __restrict__ row_weights, const int* __restrict__ route_to_row,
    int num_topk, int vec_per_row, u32x4* __restrict__ out,
    const float* __restrict__ return_in, float* __restrict__ return_out, const int* __restrict__ shared_first_row,
    int num_shared, int num_tokens, const int* __restrict__ fill_state, int num_rows, int leave_unserved)
{
    __shared__ int rows[2][DPEP_MAX_TOPK + kBatch];
    __shared__ float wts[2][DPEP_MAX_TOPK + kBatch];
    static_assert(DPEP_MAX_TOPK == 32, "a half wave looks up a token's slots");
    const int lane = threadIdx.x, half = lane >> 5, slot = lane & 31;
    const unsigned first = blockIdx.x * 64u, vec = vec_per_row;
    const int token0 = static_cast<int>(first / vec), v0 = static_cast<int>(first - token0 * vec);
    const int looked_up = token0 + half;
    int row = -1;
    if (looked_up < num_tokens && slot < num_topk && (half == 0 || v0 + 64 > vec_per_row)) {
        const size_t route = static_cast<size_t>(looked_up) * num_topk + slot;
        row = route_to_row[route];
        if (row >= num_rows) row = -1;  // a row the caller's y does not hold (capacity layouts drop surplus rows)
        if (kWeights == 1) wts[half][slot] = row >= 0 ? row_weights[row] : 0.0f;
        if (kWeights == 2) wts[half][slot] = row >= 0 ? row_weights[route] : 0.0f;
        if (return_out != nullptr && (half == 1 || v0 == 0)) return_out[route] = row >= 0 ? return_in[row] : 0.0f;  // (where the token begins)
    }
    // Shared experts (MegaMoE): slot K + j is row first + j * B + token with weight 1, summed after the routes.
    if (kWeights == 2 && slot >= num_topk && slot < num_topk + num_shared) {
        row = shared_first_row[0] + (slot - num_topk) * num_tokens + looked_up;
        wts[half][slot] = 1.0f;
    }
    rows[half][slot] = row;
    if (slot < kBatch) rows[half][DPEP_MAX_TOPK + slot] = -1;
    const unsigned long long any = __ballot(row >= 0);
    __syncthreads();
    const int num_slots = num_topk + (kWeights == 2 ? num_shared : 0);
    const int mine = v0 + lane >= vec_per_row ? 1 : 0, token = token0 + mine, v = v0 + lane - (mine != 0 ? vec_per_row : 0);
    if (token >= num_tokens) return;
    if (static_cast<uint32_t>(any >> (32 * mine)) == 0u) {  // no row: zeros, unless
        if (leave_unserved) return;                          // the caller wants only the tokens that own a row written,
        if (kWeights == 2 && fill_state != nullptr) {        // or idle workgroups of the first GEMM have written them (see above)
            const int fillers = fill_state[0];
            if (fillers > 0 && token / fillers < fill_state[1 + token % fillers]) return;
        }
    }
    store16_through(out + first + lane, combined<kWeights, kHalf>(y, rows[mine], wts[mine], num_slots, vec_per_row, v));
}

// Sparse shares: most tokens own no row (one rank's part of an EP job).  A workgroup takes a few consecutive tokens, at most
// 64 / top-k: every wave loads their (at most 64) routes itself, one per lane, so that the tokens without a row (most of them)
// cost a lane of one load instead of a wave each, and nothing goes through LDS or a barrier.  The four waves share every row,
// a quarter of its vectors each, and walk the block's rows (set bits of the ballot, i.e. tokens ascending, slots ascending)
// with the loads of the next row in flight while the current one is accumulated: a workgroup with several rows pays one
// memory round trip, not one per row.  Tokens without a row are zeroed behind that (a wait for a load also waits for the
// stores in front of it), or left alone: kLeave (the rows of tokens this rank does not serve belong to other ranks), or rows
// that idle workgroups of the first GEMM have already zeroed (fill_state: filler f of n took tokens f, f + n, ... and got
// through fill_state[1 + f] of them).
// Same arithmetic as combine_kernel: slots ascending, separate fp32 multiply and add, one rounding.
// stream_out: the output is larger than the memory-side cache should take (kStreamBytes); below that, write-through stores: 6144
// tokens of 7168 columns of which 560 own a row 14.5 us against 22 with streaming ones, 2048 tokens 6.3 against 10.
// kCached: the rows were written by the kernel right before this one (the second GEMM) and are read through the caches.
constexpr int kShareWaves = 4;
constexpr int kShareBatch = 4;  // 16-byte vectors per lane and row in flight
constexpr int kShareBlocks = 1024;  // tokens are grouped while that leaves this many workgroups (four to a CU)
template <int kWeights, bool kCached, bool kHalf>
__global__ __launch_bounds__(64 * kShareWaves) void combine_share_kernel(
    const u32x4* __restrict__ y, const float* __restrict__ weights, const int* __restrict__ route_to_row, int num_topk,
    int tokens_per_block, int vec_per_row, u32x4* __restrict__ out, int num_tokens, const float* __restrict__ return_in,
    float* __restrict__ return_out, int num_rows, int leave_unserved, const int* __restrict__ fill_state, int stream_out)
{
    auto store = [&](u32x4* to, u32x4 v) {
        if (stream_out) store16_nt(to, v);
        else store16_through(to, v);
    };
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int token0 = blockIdx.x * tokens_per_block;
    const int tokens = min(tokens_per_block, num_tokens - token0);
    int row = -1;
    float weight = 0.0f;
    if (lane < tokens * num_topk) {
        const size_t route = static_cast<size_t>(token0) * num_topk + lane;
        row = route_to_row[route];
        if (row >= num_rows) row = -1;  // a row the caller's y does not hold
        if (kWeights == 1) weight = row >= 0 ? weights[row] : 0.0f;
        if (kWeights == 2) weight = weights[route];
        if (return_out != nullptr && wave == 0) return_out[route] = row >= 0 ? return_in[row] : 0.0f;
    }
    const uint64_t valid = __ballot(row >= 0);
    const int token_of_lane = lane / num_topk;
    const int quarter = (vec_per_row + kShareWaves - 1) / kShareWaves;
    const int vec_begin = wave * quarter, vec_end = min(vec_begin + quarter, vec_per_row);
    for (int v0 = valid != 0ull ? vec_begin : vec_end; v0 < vec_end; v0 += 64 * kShareBatch) {
        u32x4 buffer[2][kShareBatch];
        float acc[kShareBatch][8];
        auto clear = [&]() {
#pragma unroll
            for (int b = 0; b < kShareBatch; ++b)
#pragma unroll
                for (int i = 0; i < 8; ++i) acc[b][i] = 0.0f;
        };
        auto issue = [&](u32x4 (&into)[kShareBatch], int at) {
            const u32x4* src = y + static_cast<size_t>(__builtin_amdgcn_readlane(row, at)) * vec_per_row;
#pragma unroll
            for (int b = 0; b < kShareBatch; ++b) {
                const int v = v0 + b * 64 + lane;
                if (v < vec_end) into[b] = kCached ? load16(src + v) : load16_nt(src + v);
            }
        };
        // accumulates the row of lane `at`; stores the token when `next` (-1: none) belongs to another one
        auto consume = [&](const u32x4 (&from)[kShareBatch], int at, int next) {
            const float w = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, weight), at));
#pragma unroll
            for (int b = 0; b < kShareBatch; ++b) {
                if (v0 + b * 64 + lane >= vec_end) continue;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float lo = kHalf ? f16_to_f32(from[b][i] & 0xffffu) : bf16_to_f32(from[b][i] & 0xffffu);
                    float hi = kHalf ? f16_to_f32(from[b][i] >> 16) : bf16_to_f32(from[b][i] >> 16);
                    if (kWeights != 0) {
                        lo = __fmul_rn(lo, w);
                        hi = __fmul_rn(hi, w);
                    }
                    acc[b][2 * i] = __fadd_rn(acc[b][2 * i], lo);
                    acc[b][2 * i + 1] = __fadd_rn(acc[b][2 * i + 1], hi);
                }
            }
            const int token = __builtin_amdgcn_readlane(token_of_lane, at);
            if (next >= 0 && __builtin_amdgcn_readlane(token_of_lane, next) == token) return;
            u32x4* dst = out + static_cast<size_t>(token0 + token) * vec_per_row;
#pragma unroll
            for (int b = 0; b < kShareBatch; ++b) {
                const int v = v0 + b * 64 + lane;
                if (v >= vec_end) continue;
                u32x4 packed;
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    packed[i] = kHalf ? pack_f16x2(acc[b][2 * i], acc[b][2 * i + 1]) : pack_bf16x2(acc[b][2 * i], acc[b][2 * i + 1]);
                store(dst + v, packed);
            }
            clear();
        };
        clear();
        uint64_t rest = valid;
        int at = __builtin_ctzll(rest);
        rest &= rest - 1ull;
        issue(buffer[0], at);
        for (;;) {
            int next = rest != 0ull ? __builtin_ctzll(rest) : -1;
            rest &= rest - 1ull;
            if (next >= 0) issue(buffer[1], next);
            consume(buffer[0], at, next);
            if (next < 0) break;
            at = next;
            next = rest != 0ull ? __builtin_ctzll(rest) : -1;
            rest &= rest - 1ull;
            if (next >= 0) issue(buffer[0], next);
            consume(buffer[1], at, next);
            if (next < 0) break;
            at = next;
        }
    }
    if (leave_unserved) return;
    const u32x4 zero = {0u, 0u, 0u, 0u};
    const int fillers = fill_state != nullptr ? fill_state[0] : 0;
    for (int t = 0; t < tokens; ++t) {
        const uint64_t mine = num_topk < 64 ? ((1ull << num_topk) - 1ull) << (t * num_topk) : ~0ull;
        if ((valid & mine) != 0ull) continue;
        const int token = token0 + t;
        if (fillers > 0 && token / fillers < fill_state[1 + token % fillers]) continue;
        u32x4* dst = out + static_cast<size_t>(token) * vec_per_row;
        for (int v = vec_begin + lane; v < vec_end; v += 64) store(dst + v, zero);
    }
}

template <int kWeights, bool kCached, bool kHalf = false>
void launch_combine_share(hipStream_t stream, const void* y, const float* weights, const int32_t* route_to_row, int num_tokens,
                          int num_topk, int vec, void* out, const float* return_in, float* return_out, int num_rows,
                          int leave_unserved, const int32_t* fill_state = nullptr)
{
    // (tokens that are left alone cost nothing: as many to a workgroup as a wave has lanes for)
    int tokens_per_block = 64 / num_topk;  // top-k is at most 32
    if (!leave_unserved) tokens_per_block = std::max(1, std::min(tokens_per_block, num_tokens / kShareBlocks));
    hipLaunchKernelGGL((combine_share_kernel<kWeights, kCached, kHalf>), dim3((num_tokens + tokens_per_block - 1) / tokens_per_block),
                       dim3(64 * kShareWaves), 0, stream, static_cast<const u32x4*>(y), weights, route_to_row, num_topk,
                       tokens_per_block, vec, static_cast<u32x4*>(out), num_tokens, return_in, return_out, num_rows, leave_unserved,
                       fill_state, static_cast<size_t>(num_tokens) * vec * 16 > kStreamBytes);
}

// Dense routing (at least one row per token on average): a wave for every 64 vectors of the output, or of a token's row (at 4096 tokens x top-8 x 14 KiB rows parts of 1 KiB take
// 84 us, of 0.875 or 3.5 KiB 87, of 1.75 KiB on two waves 90 and of 0.5 KiB 125).  Sparse receive shares (most tokens own no row and only get
// zero-filled), and rows of less than 1 KiB: a workgroup per token while that still fills the chip.
template <int kWeights, bool kHalf = false>
void launch_combine(hipStream_t stream, const void* y, const float* weights, const int32_t* route_to_row, int num_tokens, int num_topk, int expected_rows,
                    int vec, void* out, const float* return_in, float* return_out, int num_rows, const int32_t* shared_first_row = nullptr,
                    int num_shared = 0, const int32_t* fill_state = nullptr, int leave_unserved = 0)
{
    const long long vectors = static_cast<long long>(num_tokens) * vec;
    // (Rows of whole kilobytes gain nothing from it: 4096 tokens x top-8 of 4096 columns there and back 220.4 and 220.1 us, with the communication
    // stream 256 against 252.)
    if (expected_rows >= num_tokens && vec >= 64 && vec % 64 != 0 && vectors < (1LL << 31)) {
        hipLaunchKernelGGL((combine_dense_kernel<kWeights, kHalf>), dim3(static_cast<unsigned>((vectors + 63) / 64)), dim3(64), 0, stream,
                           static_cast<const u32x4*>(y), weights, route_to_row, num_topk, vec, static_cast<u32x4*>(out), return_in, return_out,
                           shared_first_row, num_shared, num_tokens, fill_state, num_rows, leave_unserved);
        return;
    }
    int parts = 1;
    while (num_tokens * parts < kSparseTargetBlocks && vec / (parts * 2) >= 64 && parts < 16) parts *= 2;
    int per_part = (vec + parts - 1) / parts;
    if (expected_rows >= num_tokens && vec >= 64) per_part = 64;
    parts = (vec + per_part - 1) / per_part;
    const int threads = std::min(kMaxThreads, (per_part + 63) / 64 * 64);
    hipLaunchKernelGGL((combine_kernel<kWeights, kHalf>), dim3(num_tokens * parts), dim3(threads), 0, stream, static_cast<const u32x4*>(y),
                       weights, route_to_row, num_topk, vec, per_part, parts, static_cast<u32x4*>(out), return_in,
                       return_out, shared_first_row, num_shared, num_tokens, fill_state, num_rows, leave_unserved);
}

}  // namespace

// Route-weighted reduce used by the MegaMoE forward: out[t] = bf16( sum_s w[t,s] * float(y[row(t,s)]) ).
int combine_routes(const void* y, const float* route_weights, const int32_t* route_to_row, int num_tokens, int num_topk,
                   int num_rows_hint, int hidden, void* out, const int32_t* shared_first_row, int num_shared,
                   const int32_t* fill_state, int leave_unserved, hipStream_t stream)
{
    const int vec = hidden / 8;
    if (num_shared == 0 && 2LL * num_rows_hint < num_tokens) {  // a sparse share: most tokens own no row
        launch_combine_share<2, true>(stream, y, route_weights, route_to_row, num_tokens, num_topk, vec, out, nullptr, nullptr,
                                      0x7fffffff, leave_unserved, fill_state);
        return launch_status("combine_routes_share");
    }
    launch_combine<2>(stream, y, route_weights, route_to_row, num_tokens, num_topk, num_rows_hint, vec, out, nullptr, nullptr, 0x7fffffff,
                      shared_first_row, num_shared, fill_state, leave_unserved);
    return launch_status("combine_routes");
}

}  // namespace dpep

namespace dpep {
namespace {

template <bool kHalf>
int combine_entry(const char* what, const void* y, const float* row_weights, const int32_t* route_to_row, int num_tokens,
                  int num_topk, int num_rows, int hidden, void* out, const float* return_in, float* return_out, void* stream,
                  int leave_unserved = 0, int expected_rows = -1)
{
    DPEP_REQUIRE(num_tokens >= 0 && num_topk >= 1 && num_topk <= DPEP_MAX_TOPK, "%s: bad T=%d K=%d", what, num_tokens,
                 num_topk);
    // (num_rows may exceed T*K: a capacity layout holds more rows than the batch has routes; rows of route_to_row
    // at or beyond num_rows are treated as absent)
    DPEP_REQUIRE(num_rows >= 0, "%s: num_rows=%d is negative", what, num_rows);
    DPEP_REQUIRE(hidden > 0 && hidden % 8 == 0, "%s: hidden=%d must be a positive multiple of 8", what, hidden);
    // (with no rows at all the channel's input is an empty buffer, which may well be a null pointer)
    DPEP_REQUIRE(return_in == nullptr ? (return_out == nullptr || num_rows == 0) : return_out != nullptr,
                 "%s: return_in and return_out go together", what);
    if (num_tokens == 0) return DPEP_OK;
    DPEP_REQUIRE(route_to_row != nullptr && out != nullptr && aligned16(out), "%s: NULL or misaligned buffer", what);
    DPEP_REQUIRE(num_rows == 0 || (y != nullptr && aligned16(y)), "%s: y must be 16-byte aligned", what);
    const int vec = hidden / 8;
    hipStream_t s = static_cast<hipStream_t>(stream);
    // (of a capacity layout only the caller knows how many rows to expect)
    const int hint = expected_rows >= 0 ? expected_rows : num_rows;
    // (zero rows of more than kStreamBytes are written no faster by fewer, longer workgroups: 16384 tokens of 7168 columns of which
    // 1900 own a row 57 us against 53 with a workgroup per token)
    if (2LL * hint < num_tokens && (leave_unserved || static_cast<size_t>(num_tokens) * hidden * 2 <= kStreamBytes)) {
        if (row_weights != nullptr)
            launch_combine_share<1, false, kHalf>(s, y, row_weights, route_to_row, num_tokens, num_topk, vec, out, return_in, return_out,
                                                  num_rows, leave_unserved);
        else
            launch_combine_share<0, false, kHalf>(s, y, nullptr, route_to_row, num_tokens, num_topk, vec, out, return_in, return_out,
                                                  num_rows, leave_unserved);
        return launch_status(what);
    }
    if (row_weights != nullptr)
        launch_combine<1, kHalf>(s, y, row_weights, route_to_row, num_tokens, num_topk, hint, vec, out, return_in, return_out, num_rows, nullptr, 0,
                                 nullptr, leave_unserved);
    else
        launch_combine<0, kHalf>(s, y, nullptr, route_to_row, num_tokens, num_topk, hint, vec, out, return_in, return_out, num_rows, nullptr, 0,
                                 nullptr, leave_unserved);
    return launch_status(what);
}

}  // namespace
}  // namespace dpep

extern "C" {

int dpep_combine(const void* y, const float* row_weights, const int32_t* route_to_row, int num_tokens, int num_topk,
                 int num_rows, int hidden, void* out, const float* return_in, float* return_out, void* stream)
{
    return dpep::combine_entry<false>("combine", y, row_weights, route_to_row, num_tokens, num_topk, num_rows, hidden, out,
                                      return_in, return_out, stream);
}

int dpep_combine_expecting(const void* y, int half, const float* row_weights, const int32_t* route_to_row, int num_tokens, int num_topk,
                           int num_rows, int expected_rows, int hidden, void* out, const float* return_in, float* return_out,
                           void* stream)
{
    const auto entry = half ? dpep::combine_entry<true> : dpep::combine_entry<false>;
    return entry("combine", y, row_weights, route_to_row, num_tokens, num_topk, num_rows, hidden, out, return_in, return_out, stream,
                 /*leave_unserved=*/0, expected_rows < 0 ? 0 : expected_rows);
}

int dpep_combine_served(const void* y, const float* row_weights, const int32_t* route_to_row, int num_tokens, int num_topk,
                        int num_rows, int hidden, void* out, const float* return_in, float* return_out, void* stream)
{
    return dpep::combine_entry<false>("combine_served", y, row_weights, route_to_row, num_tokens, num_topk, num_rows, hidden,
                                      out, return_in, return_out, stream, /*leave_unserved=*/1);
}

int dpep_combine_fp16(const void* y, const float* row_weights, const int32_t* route_to_row, int num_tokens, int num_topk,
                      int num_rows, int hidden, void* out, const float* return_in, float* return_out, void* stream)
{
    return dpep::combine_entry<true>("combine_fp16", y, row_weights, route_to_row, num_tokens, num_topk, num_rows, hidden,
                                     out, return_in, return_out, stream);
}

}  // extern "C"

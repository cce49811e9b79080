// Expand-permute payload dispatch: out[row(t,s)] = x[t] for every route that owns a row, optionally
// fused with the per-128-element FP8 e4m3fn block quantiser.  HBM-bound: 16-byte coalesced loads,
// 16-byte stores, each input row read once and written to its K destinations.  How the token-major kernels store
// is a process-wide policy (dpep_dispatch_store_policy): streaming by default, write-through or cached on request.
//
// Observable contract: tests/elastic/test_dispatch.py:1391-1416 (payload, scales and weights arrive
// bit-exactly in row order), tests/clos/common.py:276-279; quantiser deep_ep/utils/math.py:45-61.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "payload.h"

#pragma clang fp contract(off)

namespace dpep {
namespace {

constexpr int kTargetBlocks = 8192;  // rows are split into column parts until a launch has about this many workgroups (4096 rows: two parts each measured 3-6 % faster than one, four no better)
constexpr int kRowMajorRatio = 1;  // row-major kernels when rows <= ratio * tokens

// Store policy of the payload rows.  Streaming (non-temporal, the default): the rows go to HBM past the caches at the
// streaming-write rate, and the kernel's time is the time of its traffic.  Write-through (device-scope `sc1`) and cached
// stores let the 256 MiB memory-side cache take the rows first: the kernel itself ends sooner when that cache holds clean
// lines at launch, but the rows still have to reach HBM, and whatever runs next pays for it (measured at T=4096, H=7168,
// top-8: the fused FP8 dispatch after a read-only sweep of 256 MiB takes 59.6 us streaming and 49.5 us write-through; with
// the sweep that follows charged to it, 60.9 against 85.9 us; inside a dispatch + combine loop 49.6 against 69.8 us, and the
// combine behind it 88.3 against 101.6 us).  A caller whose next kernel reads the rows while they are still in the
// memory-side cache may still prefer write-through, hence the knob.
int g_store_policy = DPEP_STORE_STREAMING;

// Calls launch(std::integral_constant<int, policy>) for the current policy.
template <typename Launch>
void with_store_policy(Launch&& launch)
{
    switch (__atomic_load_n(&g_store_policy, __ATOMIC_RELAXED)) {
    case DPEP_STORE_THROUGH: launch(std::integral_constant<int, DPEP_STORE_THROUGH>{}); break;
    case DPEP_STORE_CACHED: launch(std::integral_constant<int, DPEP_STORE_CACHED>{}); break;
    default: launch(std::integral_constant<int, DPEP_STORE_STREAMING>{}); break;
    }
}

template <int kPolicy, bool kStaged>
__global__ __launch_bounds__(kMaxThreads) void dispatch_copy_token_kernel(
    const u32x4* __restrict__ x, const float* __restrict__ scales, const float* __restrict__ weights, u32x4* __restrict__ out,
    float* __restrict__ out_scales, float* __restrict__ out_weights, PayloadShape p, MappedTokens tokens)
{
    __shared__ TokenLds lds;
    __shared__ u32x4 stage[kStaged ? kStagedVec : 1];
    copy_token<kPolicy, kStaged>(x, scales, weights, out, out_scales, out_weights, p, tokens, blockIdx.x, threadIdx.x, lds, stage);
}

// ---- row-major: one workgroup per (output row, column part); for sparse receive shares -------------
// Rows [0, rows): `rows` from the host, or, rows_on_device, the smaller of that bound and the count the layout left on the
// device (a payload queued before the host knows R); all_or_none, the outputs' capacity: no rows at all unless DPEP_ROWS_KEPT
// (0: the first rows in any case).  Such a launch has workgroups for about the expected number of rows;
// they walk on by the grid's rows until the real count is reached, and the first row's route is asked for together with
// the count (row_to_route has an entry for every row of the grid, so the load is in bounds whatever the count says).
struct RowRange {
    int rows;
    const int* rows_on_device;
    int all_or_none;
    __device__ __forceinline__ int count() const
    {
        if (rows_on_device == nullptr) return rows;
        const int all = *rows_on_device;
        return all_or_none == 0 || DPEP_ROWS_KEPT(all, all_or_none) ? min(all, rows) : 0;
    }
};

template <int kPolicy>
__global__ __launch_bounds__(kMaxThreads) void dispatch_copy_row_kernel(
    const u32x4* __restrict__ x, const float* __restrict__ scales, const float* __restrict__ weights,
    const int* __restrict__ row_to_route, RowRange range, int num_tokens, int num_topk, int vec_per_row, int vec_per_part,
    int parts, int scale_cols, u32x4* __restrict__ out, float* __restrict__ out_scales, float* __restrict__ out_weights)
{
    const int part = blockIdx.x % parts, stride = gridDim.x / parts;
    const int v_begin = part * vec_per_part;
    const int v_end = min(v_begin + vec_per_part, vec_per_row);
    int row = blockIdx.x / parts;
    int next_route = row_to_route[row];
    const int rows = range.count();
    for (; row < rows; row += stride) {
        // (clamped: a map left incomplete by a layout launch that reported a time-out must not become a wild address)
        const int route = min(max(next_route, 0), num_tokens * num_topk - 1);
        if (row + stride < rows) next_route = row_to_route[row + stride];
        const int token = route / num_topk;
        const u32x4* src = x + static_cast<size_t>(token) * vec_per_row;
        u32x4* dst = out + static_cast<size_t>(row) * vec_per_row;
        for (int v = v_begin + threadIdx.x; v < v_end; v += blockDim.x) store16_as<kPolicy>(dst + v, load16(src + v));
        if (part == 0) {
            if (scales != nullptr)
                for (int c = threadIdx.x; c < scale_cols; c += blockDim.x)
                    out_scales[static_cast<size_t>(row) * scale_cols + c] = scales[static_cast<size_t>(token) * scale_cols + c];
            if (weights != nullptr && threadIdx.x == 0) out_weights[row] = weights[route];
        }
    }
}

template <int kPolicy>
__global__ __launch_bounds__(kMaxThreads) void dispatch_quant_token_kernel(
    const u32x4* __restrict__ x, const float* __restrict__ weights, u32x4* __restrict__ out, float* __restrict__ out_scales,
    float* __restrict__ out_weights, PayloadShape p, MappedTokens tokens)
{
    __shared__ TokenLds lds;
    __shared__ float part_scales[kMaxScaleCols];
    quant_token<kPolicy>(x, weights, out, out_scales, out_weights, p, tokens, blockIdx.x, threadIdx.x, lds, part_scales);
}

// row-major: one workgroup per (output row, column part), rows as above; row_to_route == nullptr means identity
// (row == token), which is the stand-alone quantiser.
template <int kPolicy>
__global__ __launch_bounds__(kMaxThreads) void dispatch_quant_row_kernel(
    const u32x4* __restrict__ x, const float* __restrict__ weights, const int* __restrict__ row_to_route, RowRange range,
    int num_tokens, int num_topk, int units_per_row, int units_per_part, int parts, u32x4* __restrict__ out,
    float* __restrict__ out_scales, float* __restrict__ out_weights)
{
    const int part = blockIdx.x % parts, stride = gridDim.x / parts;
    const int u_begin = part * units_per_part;
    const int u_end = min(u_begin + units_per_part, units_per_row);
    const int scale_cols = units_per_row / 8;
    int row = blockIdx.x / parts;
    int next_route = row_to_route != nullptr ? row_to_route[row] : row;
    const int rows = range.count();
    for (; row < rows; row += stride) {
        const int route = row_to_route != nullptr ? min(max(next_route, 0), num_tokens * num_topk - 1) : row;
        if (row_to_route != nullptr && row + stride < rows) next_route = row_to_route[row + stride];
        const int token = row_to_route != nullptr ? route / num_topk : row;
        const u32x4* src = x + static_cast<size_t>(token) * units_per_row * 2;
        for (int u = u_begin + threadIdx.x; u < u_end; u += blockDim.x) {
            const Quant16 q = quantize16(load16(src + 2 * u), load16(src + 2 * u + 1));
            store16_as<kPolicy>(out + static_cast<size_t>(row) * units_per_row + u, q.codes);
            if ((u & 7) == 0) out_scales[static_cast<size_t>(row) * scale_cols + (u >> 3)] = q.scale;
        }
        if (part == 0 && weights != nullptr && threadIdx.x == 0) out_weights[row] = weights[route];
    }
}

// Stand-alone quantiser for rows whose width is not a multiple of 128: the last block of a row is short and is
// quantised as if padded with zeros (per_token_cast_to_fp8 pads, deep_ep/utils/math.py:52-53).  One thread per 16 values
// of the padded row, so the eight lanes of a block are always all present; padding units load and store nothing.
__global__ __launch_bounds__(256) void cast_to_fp8_short_block_kernel(const u32x4* __restrict__ x, int units_per_row,
                                                                      int blocks_per_row, long long padded_units,
                                                                      u32x4* __restrict__ out, float* __restrict__ out_scales)
{
    const long long id = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (id >= padded_units) return;  // padded_units is a multiple of 8: whole blocks leave together
    const long long row = id / (blocks_per_row * 8);
    const int unit = static_cast<int>(id % (blocks_per_row * 8));
    const bool real = unit < units_per_row;
    const u32x4 zero = {0u, 0u, 0u, 0u};
    const u32x4* src = x + (row * units_per_row + unit) * 2;
    const Quant16 q = quantize16(real ? load16(src) : zero, real ? load16(src + 1) : zero);
    if (real) store16_nt(out + row * units_per_row + unit, q.codes);
    if ((unit & 7) == 0) out_scales[row * blocks_per_row + (unit >> 3)] = q.scale;
}

// ---- dequantiser: bf16(fp32(code) * scale) per block of 128 columns ---------------------------------------------
// One thread per 8 codes (8 bytes in, 16 bytes out), so that consecutive lanes write consecutive 16-byte vectors: with 16
// codes per thread a lane's two output vectors sat 32 bytes apart and every store instruction filled only half of each
// 64 bytes it touched (187 us for 32768 x 7168 codes; this way 5 TB/s and more).  kByteScales: the scales are e8m0 bytes
// (four to an int32 in the caller's tensor), value 2^(byte - 127) built by moving the byte into the exponent field; else
// fp32.  The last block of a row may be short (hidden need only be a multiple of 16).
// kThrough: write-through stores (small outputs, which the memory-side cache takes), else streaming ones.
template <bool kByteScales, bool kThrough>
__global__ __launch_bounds__(256) void cast_back_kernel(const unsigned long long* __restrict__ codes, const void* __restrict__ scales,
                                                        int halves_per_row, int scales_per_row, long long total_halves,
                                                        u32x4* __restrict__ out)
{
    const long long id = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (id >= total_halves) return;
    long long row;
    int half;
    if (total_halves < (1ll << 31)) {  // 32-bit division where it suffices
        row = static_cast<unsigned>(id) / static_cast<unsigned>(halves_per_row);
        half = static_cast<int>(static_cast<unsigned>(id) - static_cast<unsigned>(row) * static_cast<unsigned>(halves_per_row));
    } else {
        row = id / halves_per_row;
        half = static_cast<int>(id - row * halves_per_row);
    }
    const long long at = row * scales_per_row + (half >> 4);
    const float scale = kByteScales ? __uint_as_float(static_cast<uint32_t>(static_cast<const uint8_t*>(scales)[at]) << 23)
                                    : static_cast<const float*>(scales)[at];
    const unsigned long long q = __builtin_nontemporal_load(codes + id);
    u32x4 value;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int word = static_cast<int>(static_cast<uint32_t>(q >> (32 * i)));
        const float a = __fmul_rn(__builtin_amdgcn_cvt_f32_fp8(word, 0), scale);
        const float b = __fmul_rn(__builtin_amdgcn_cvt_f32_fp8(word, 1), scale);
        const float c = __fmul_rn(__builtin_amdgcn_cvt_f32_fp8(word, 2), scale);
        const float d = __fmul_rn(__builtin_amdgcn_cvt_f32_fp8(word, 3), scale);
        value[2 * i] = pack_bf16x2(a, b);
        value[2 * i + 1] = pack_bf16x2(c, d);
    }
    if (kThrough) store16_through(out + id, value);
    else store16_nt(out + id, value);
}

// ---- small batches: routing layout and payload in ONE launch -------------------------------------------------
// With at most kSmallRoutes routes (a decode step) the whole routing table fits a workgroup's LDS, and a workgroup
// gets the rows of its own token faster by working them out itself than by waiting for a layout kernel: every
// workgroup (one per token and column part) reads all ids, histograms them (LDS atomics: a count does not depend on
// order), scans the histogram over the experts, and counts, for each of its token's routes, the earlier routes with
// the same expert.  row = first row of the expert + that count: the same stable permutation the layout kernels
// produce.  Nothing travels between workgroups.  Part 0 of each token writes the token's entries of route_to_row and
// row_to_route, workgroup 0 the per-expert outputs and the host mailbox.
constexpr int kSmallRoutes = 2048;

template <bool kQuant, int kSlots>  // kSlots: compile-time bound of top-k (8 or DPEP_MAX_TOPK)
__global__ __launch_bounds__(kMaxThreads) void layout_dispatch_small_kernel(
    const long long* __restrict__ idx, long long* __restrict__ idx_copy, int n_routes, int num_experts, int expert_begin,
    int num_local, int num_topk, const u32x4* __restrict__ x, const float* __restrict__ scales, const float* __restrict__ weights, int units_per_row,
    int units_per_part, int parts, int scale_cols, int capacity, SendCounts send, int* __restrict__ counts,
    int* __restrict__ psum, int* __restrict__ offsets, int* __restrict__ num_rows, int* __restrict__ route_to_row, int* __restrict__ row_to_route, u32x4* __restrict__ out,
    float* __restrict__ out_scales, float* __restrict__ out_weights, uint32_t* __restrict__ mailbox, uint32_t sequence)
{
    __shared__ short local_id[kSmallRoutes];
    __shared__ int first_row[DPEP_MAX_LOCAL_EXPERTS];  // per expert: count, then exclusive prefix
    __shared__ int before[DPEP_MAX_TOPK];
    __shared__ int rows[DPEP_MAX_TOPK];
    __shared__ int wave_sums[kMaxThreads / kWave];
    __shared__ float part_scales[kMaxScaleCols];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int token = blockIdx.x / parts, part = blockIdx.x % parts;
    // in units of 16 bytes of input (kQuant: 32 bytes = 16 BF16 values = 16 bytes of output)
    const int u_begin = part * units_per_part, u_end = min(u_begin + units_per_part, units_per_row);
    constexpr int kIn = kQuant ? 2 : 1;
    const u32x4* src = x + static_cast<size_t>(token) * units_per_row * kIn;
    // all ids at once (a route past the end reads the last id instead of branching around the load): one memory latency
    constexpr int kIds = kSmallRoutes / kMaxThreads;
    long long ids[kIds];
#pragma unroll
    for (int i = 0; i < kIds; ++i) ids[i] = idx[min(tid + i * kMaxThreads, n_routes - 1)];
    // the payload is asked for right behind them: it does not depend on the routing
    constexpr int kEarly = 2;
    u32x4 early[kEarly][kIn];
#pragma unroll
    for (int j = 0; j < kEarly; ++j) {
        const int u = u_begin + tid + j * kMaxThreads;
        if (u < u_end) {
#pragma unroll
            for (int h = 0; h < kIn; ++h) early[j][h] = load16(src + kIn * u + h);
        }
    }
    for (int e = tid; e < num_local; e += kMaxThreads) first_row[e] = 0;
    if (tid < DPEP_MAX_TOPK) before[tid] = 0;
    __syncthreads();
    const bool reporter = blockIdx.x == 0;
#pragma unroll
    for (int i = 0; i < kIds; ++i) {
        const int j = tid + i * kMaxThreads;
        if (j < n_routes) {
            if (reporter && idx_copy != nullptr) idx_copy[j] = ids[i];
            const int e = local_expert(ids[i], j, n_routes, num_experts, expert_begin, num_local);
            local_id[j] = static_cast<short>(e);
            if (e >= 0) atomicAdd(&first_row[e], 1);
        }
    }
    __syncthreads();
    // exclusive scan over the experts: four consecutive experts per thread, wave scan, then the waves' sums
    int mine[4], sum = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int e = tid * 4 + j;
        mine[j] = e < num_local ? first_row[e] : 0;
        sum += mine[j];
    }
    const int incl = wave_scan(sum);
    if (lane == kWave - 1) wave_sums[wave] = incl;
    __syncthreads();
    int offset = incl - sum;
    for (int w = 0; w < wave; ++w) offset += wave_sums[w];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int e = tid * 4 + j;
        if (e < num_local) {
            first_row[e] = offset;
            if (reporter) {
                counts[e] = mine[j];
                psum[e] = offset + mine[j];
                offsets[e + 1] = offset + mine[j];
                if (send.counts != nullptr) send.counts[send.expert_begin + e] = offset + mine[j];
            }
        }
        offset += mine[j];
    }
    if (reporter && tid == kMaxThreads - 1) {
        offsets[0] = 0;
        num_rows[0] = offset;  // the last thread's running offset is the total
    }
    if (reporter) send_counts_of_others(send, num_local, wave_sums[0] + wave_sums[1] + wave_sums[2] + wave_sums[3], tid, kMaxThreads);
    if (reporter && mailbox != nullptr) {
        if (tid * 4 < num_local) mailbox_store_counts(mailbox, tid * 4, mine, sequence, true);
        if (tid == kMaxThreads - 1) mailbox_store_rows(mailbox, offset, sequence);
    }
    __syncthreads();
    // earlier routes with the same expert, for each route of this token
    const int my_first = token * num_topk;
    int want[kSlots], seen[kSlots];
#pragma unroll
    for (int s = 0; s < kSlots; ++s) {
        want[s] = s < num_topk ? local_id[my_first + s] : -2;  // -2 matches nothing
        seen[s] = 0;
    }
    for (int j = tid; j < my_first + num_topk; j += kMaxThreads) {
        const int e = local_id[j];
#pragma unroll
        for (int s = 0; s < kSlots; ++s) seen[s] += (e == want[s] && j < my_first + s) ? 1 : 0;
    }
#pragma unroll
    for (int s = 0; s < kSlots; ++s)
        if (seen[s] != 0 && want[s] >= 0) atomicAdd(&before[s], seen[s]);
    __syncthreads();
    if (tid < num_topk) {
        const int e = local_id[my_first + tid];
        const int row = e >= 0 ? first_row[e] + before[tid] : -1;
        rows[tid] = row < capacity ? row : -1;
        if (part == 0) {
            route_to_row[my_first + tid] = row;
            if (row >= 0) {
                row_to_route[row] = my_first + tid;
                if (weights != nullptr && row < capacity) out_weights[row] = weights[my_first + tid];
            }
        }
    }
    __syncthreads();
    // payload: read once, write to every row of the token
    auto emit = [&](int u, const u32x4 (&in)[kIn]) {
        u32x4 value = in[0];
        if (kQuant) {
            const Quant16 q = quantize16(in[0], in[kIn - 1]);
            value = q.codes;
            if ((u & 7) == 0) part_scales[(u - u_begin) >> 3] = q.scale;
        }
        for (int s = 0; s < num_topk; ++s) {
            const int row = rows[s];
            if (row >= 0) store16_nt(out + static_cast<size_t>(row) * units_per_row + u, value);
        }
    };
#pragma unroll
    for (int j = 0; j < kEarly; ++j) {
        const int u = u_begin + tid + j * kMaxThreads;
        if (u < u_end) emit(u, early[j]);
    }
    for (int u = u_begin + tid + kEarly * kMaxThreads; u < u_end; u += kMaxThreads) {
        u32x4 in[kIn];
#pragma unroll
        for (int h = 0; h < kIn; ++h) in[h] = load16(src + kIn * u + h);
        emit(u, in);
    }
    if (kQuant) {
        __syncthreads();
        const int part_cols = (u_end - u_begin) >> 3, col0 = u_begin >> 3, out_cols = units_per_row / 8;
        for (int i = tid; i < num_topk * part_cols; i += kMaxThreads) {
            const int s = i / part_cols, c = i - s * part_cols;
            const int row = rows[s];
            if (row >= 0) out_scales[static_cast<size_t>(row) * out_cols + col0 + c] = part_scales[c];
        }
    } else if (part == 0 && scales != nullptr) {
        for (int c = tid; c < scale_cols; c += kMaxThreads) {
            const float value = scales[static_cast<size_t>(token) * scale_cols + c];
            for (int s = 0; s < num_topk; ++s) {
                const int row = rows[s];
                if (row >= 0) out_scales[static_cast<size_t>(row) * scale_cols + c] = value;
            }
        }
    }
}

// Split a row of `units` work items over `parts` workgroups so that a launch of `rows` rows has
// enough workgroups (target_blocks) to fill 256 CUs; each part is a multiple of `granule` units.
struct Split {
    int parts, per_part, threads;
};

Split choose_split(int rows, int units, int granule, int target_blocks = kTargetBlocks)
{
    Split s;
    int parts = 1;
    while (rows * parts < target_blocks && units / (parts * 2) >= 64 && parts < 16) parts *= 2;
    int per_part = (units + parts - 1) / parts;
    per_part = (per_part + granule - 1) / granule * granule;
    s.parts = (units + per_part - 1) / per_part;
    s.per_part = per_part;
    int threads = (per_part + 63) / 64 * 64;
    s.threads = threads > kMaxThreads ? kMaxThreads : threads;
    return s;
}

int check_common(const char* what, int num_tokens, int num_topk, int num_rows, const int32_t* route_to_row,
                 const int32_t* row_to_route)
{
    DPEP_REQUIRE(num_tokens >= 0 && num_topk >= 1 && num_topk <= DPEP_MAX_TOPK, "%s: bad T=%d K=%d", what, num_tokens,
                 num_topk);
    DPEP_REQUIRE(num_rows >= -1 && static_cast<long long>(num_rows) <= static_cast<long long>(num_tokens) * num_topk,
                 "%s: num_rows=%d outside [0, T*K] (or -1: not known yet)", what, num_rows);
    DPEP_REQUIRE(num_rows == 0 || route_to_row != nullptr, "%s: NULL routing maps", what);
    DPEP_REQUIRE(num_rows <= 0 || row_to_route != nullptr, "%s: NULL routing maps", what);
    return DPEP_OK;
}

// One payload launch.  units per row: 16-byte vectors (copy), or 16-value groups (quantise).
struct Payload {
    const u32x4* x;
    const float* scales;
    const float* weights;
    int num_tokens, num_topk, units, scale_cols;
    bool quantize;
    u32x4* out;
    float* out_scales;
    float* out_weights;
};

// The split of a payload launch over `lines` tokens or rows.  Parts end at multiples of 128 bytes.  Where the rows themselves do not,
// every part boundary is two partial lines to HBM in each of a token's rows, and a token-major launch with four and more rows per token has
// parts only while it would have fewer than 2048 workgroups (dispatch and combine, BF16: 6045 tokens x top-10 of 6064 columns 353 -> 335 us, 7421 x 7 of 2848 280 -> 264, 1874 x 7 of
// 2400 38.7 -> 36.3; rows of whole lines are better off with the finer split: 4096 x 8 of 4096 106.7 against 108.6, of 7168 to FP8 136.9 against 138.1).
// On both sides of the four rows, 2048 / 8192 workgroups: 3000 tokens of 5840 columns x top-2 43.0 / 42.3 us, 3 56.2 / 58.4, 4 68.1 / 71.9, 5 79.5 /
// 85.9; 4096 of 2832 32.7 / 32.1, 40.4 / 40.4, 50.4 / 52.9, 56.5 / 60.2; 6000 of 1552 28.5 / 28.3, 35.6 / 37.5, 42.5 / 45.9, 49.5 / 49.3.  Two rows per token
// are too few for it (2264 of 4464 too: 31.6 against 30.3), three are as good or better in these, four and more nearly always.
Split payload_split(const Payload& p, int lines, long long rows_to_write)
{
    const bool whole_lines = p.quantize || p.units % 8 == 0;
    return choose_split(lines, p.units, whole_lines ? 8 : 1, !whole_lines && rows_to_write >= 4LL * lines ? 2048 : kTargetBlocks);
}

// Whether a token-major copy goes through LDS (dispatch and combine, BF16: 6045 tokens x top-10 of 6064 columns 343.2 -> 321.6 us, 3054 x 9 of 3152 there
// and back 174.5 -> 166.7, 6249 x 7 of 1552 71.3 -> 69.8; 7782 x 5 of 1232, 154 vectors, 45.5 against 48.3).
bool payload_staged(const Payload& p, const Split& sp)
{
    return !p.quantize && p.units % 8 != 0 && sp.threads == kMaxThreads && sp.per_part <= kStagedVec;
}

PayloadShape payload_shape(const Payload& p, const Split& sp)
{
    return {p.num_tokens, p.num_topk, p.units, sp.per_part, sp.parts, sp.threads, p.scale_cols};
}

// token-major: the grid does not depend on R; rows at or beyond `capacity` are dropped; all_rows: all of them unless DPEP_ROWS_KEPT.  rows:
// their number, about.
int launch_token_major(const Payload& p, const int32_t* route_to_row, int capacity, const int32_t* all_rows, long long rows, hipStream_t s)
{
    const Split sp = payload_split(p, p.num_tokens, rows);
    const dim3 grid(p.num_tokens * sp.parts), block(sp.threads);
    // A launch that mostly writes is faster with twelve waves to a CU than with as many as there is room for (fewer rows open at a time;
    // 6045 tokens x top-10 of 6064 BF16 columns 335 -> 328 us, 6249 x 7 of 1552 145.7 -> 141.3; 1.25 rows per
    // token 39.6 -> 47.3; to FP8, whose reads are half of its rows' bytes, 146.6 -> 150.7): the LDS that it asks for keeps others out.  A quarter of
    // the CU's 160 KiB for 256 threads, beside the kernel's own 132 bytes: three workgroups fit (of 192 threads five, of 128 seven, of 64 fifteen).
    // On both sides of the five rows, so / without it, BF16, a cached dispatch and its combine: 4096 tokens of 4096 columns x top-2 34.9 / 33.2 us, 3
    // 43.4 / 43.5, 4 57.8 / 58.3, 5 62.8 / 64.0; 2000 of 5120 24.5 / 22.0, 29.7 / 28.1, 34.3 / 34.6, 40.1 / 41.1; 3000 of 5840 36.3 / 36.6, 51.4 / 52.8,
    // 59.9 / 62.1, 74.9 / 77.3.  Behind a layout four rows are too few: 65.8 / 64.6 and 42.4 / 40.2 for the first two, 66.4 / 68.1 for the third.
    const bool mostly_writes = !p.quantize && rows >= 5LL * p.num_tokens && rows * p.units * 16 >= (32LL << 20);
    const unsigned room = mostly_writes ? 40960 / kMaxThreads * sp.threads : 0;
    const MappedTokens tokens = {route_to_row, capacity, all_rows};
    with_store_policy([&](auto policy) {
        constexpr int kPolicy = decltype(policy)::value;
        if (p.quantize) hipLaunchKernelGGL(dispatch_quant_token_kernel<kPolicy>, grid, block, 0, s, p.x, p.weights, p.out, p.out_scales, p.out_weights, payload_shape(p, sp), tokens);
        else if (kPolicy == DPEP_STORE_STREAMING && payload_staged(p, sp))
            hipLaunchKernelGGL((dispatch_copy_token_kernel<kPolicy, true>), grid, block, room - std::min(room, kStagedVec * 16u), s, p.x, p.scales, p.weights,
                               p.out, p.out_scales, p.out_weights, payload_shape(p, sp), tokens);
        else
            hipLaunchKernelGGL((dispatch_copy_token_kernel<kPolicy, false>), grid, block, room, s, p.x, p.scales, p.weights, p.out, p.out_scales,
                               p.out_weights, payload_shape(p, sp), tokens);
    });
    return launch_status("dispatch_token");
}

// row-major: workgroups for `grid_rows` rows (row_to_route has at least as many entries), which walk on to the range's end.
int launch_row_major(const Payload& p, const int32_t* row_to_route, const RowRange& range, int grid_rows, hipStream_t s)
{
    const Split sp = payload_split(p, grid_rows, grid_rows);
    const dim3 grid(grid_rows * sp.parts), block(sp.threads);
    with_store_policy([&](auto policy) {
        constexpr int kPolicy = decltype(policy)::value;
        if (p.quantize)
            hipLaunchKernelGGL(dispatch_quant_row_kernel<kPolicy>, grid, block, 0, s, p.x, p.weights, row_to_route, range, p.num_tokens, p.num_topk,
                               p.units, sp.per_part, sp.parts, p.out, p.out_scales, p.out_weights);
        else
            hipLaunchKernelGGL(dispatch_copy_row_kernel<kPolicy>, grid, block, 0, s, p.x, p.scales, p.weights, row_to_route, range, p.num_tokens,
                               p.num_topk, p.units, sp.per_part, sp.parts, p.scale_cols, p.out, p.out_scales, p.out_weights);
    });
    return launch_status("dispatch_row");
}

// R known (num_rows >= 0), or not known and outputs of T*K rows (num_rows < 0: the token-major grid, which does not
// depend on R).
int launch_payload(const Payload& p, const int32_t* route_to_row, const int32_t* row_to_route, int num_rows, hipStream_t s)
{
    if (num_rows < 0 || static_cast<long long>(num_rows) > static_cast<long long>(kRowMajorRatio) * p.num_tokens)
        return launch_token_major(p, route_to_row, 0x7fffffff, nullptr, num_rows < 0 ? 0 : num_rows, s);
    return launch_row_major(p, row_to_route, RowRange{num_rows, nullptr, 0}, num_rows, s);
}

int launch_small(Workspace* w, const dpep_fresh_dispatch& c, int units, hipStream_t s)
{
    if (c.report_to_host) {
        w->sequence = w->sequence == 0xffffffffu ? 1u : w->sequence + 1u;  // never 0: that is "nothing launched"
        w->mailbox_local = c.num_local;
        w->mailbox_narrow = true;
    }
    const Split sp = choose_split(c.num_tokens, units, 8);
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(c.num_tokens * sp.parts), dim3(kMaxThreads), 0, s,
                           reinterpret_cast<const long long*>(c.topk_idx), reinterpret_cast<long long*>(c.topk_idx_copy),
                           c.num_tokens * c.num_topk, c.num_experts, c.expert_begin, c.num_local, c.num_topk,
                           static_cast<const u32x4*>(c.x), c.quantize ? nullptr : c.scales, c.topk_weights, units, sp.per_part,
                           sp.parts, c.quantize ? 0 : c.scale_cols, c.capacity_rows,
                           SendCounts{c.send_counts, c.expert_begin, c.num_experts}, c.counts, c.psum, c.offsets, c.num_rows,
                           c.route_to_row, c.row_to_route, static_cast<u32x4*>(c.out), c.out_scales, c.out_weights,
                           c.report_to_host ? w->mailbox_device : nullptr, w->sequence);
    };
    if (c.num_topk <= 8) {
        if (c.quantize) launch(layout_dispatch_small_kernel<true, 8>);
        else launch(layout_dispatch_small_kernel<false, 8>);
    } else {
        if (c.quantize) launch(layout_dispatch_small_kernel<true, DPEP_MAX_TOPK>);
        else launch(layout_dispatch_small_kernel<false, DPEP_MAX_TOPK>);
    }
    return launch_status("layout_dispatch_small");
}

// What the payload side of a fresh dispatch requires; *units: 16-byte vectors or 16-value groups per row.
int check_fresh_payload(const char* what, const dpep_fresh_dispatch& c, int* units)
{
    DPEP_REQUIRE(c.x && c.out && aligned16(c.x) && aligned16(c.out), "%s: x/out must be 16-byte aligned", what);
    DPEP_REQUIRE((c.topk_weights == nullptr) == (c.out_weights == nullptr), "%s: weights and out_weights go together", what);
    if (c.quantize) {
        DPEP_REQUIRE(c.row_bytes > 0 && c.row_bytes % 256 == 0 && c.row_bytes / 256 <= kMaxScaleCols,
                     "%s: a quantised row needs a BF16 width that is a multiple of 128 (row_bytes=%d)", what, c.row_bytes);
        DPEP_REQUIRE(c.scales == nullptr && c.out_scales != nullptr, "%s: the fused quantiser takes no input scales and needs out_scales", what);
        *units = c.row_bytes / 32;
    } else {
        DPEP_REQUIRE(c.row_bytes > 0 && c.row_bytes % 16 == 0, "%s: row_bytes=%d must be a positive multiple of 16", what, c.row_bytes);
        DPEP_REQUIRE((c.scales == nullptr) == (c.out_scales == nullptr), "%s: scales and out_scales go together", what);
        DPEP_REQUIRE(c.scales == nullptr || c.scale_cols > 0, "%s: scale_cols must be positive with scales", what);
        *units = c.row_bytes / 16;
    }
    return DPEP_OK;
}

int fresh_in_one_launch(Workspace* w, const dpep_fresh_dispatch& c, hipStream_t stream)
{
    DPEP_REQUIRE(c.num_tokens >= 1 && c.num_topk >= 1 && c.num_topk <= DPEP_MAX_TOPK &&
                     static_cast<long long>(c.num_tokens) * c.num_topk <= kSmallRoutes,
                 "layout_dispatch_small: T=%d K=%d: needs 1 <= T*K <= %d routes (larger batches take dpep_layout and a "
                 "dispatch call)", c.num_tokens, c.num_topk, kSmallRoutes);
    DPEP_REQUIRE(c.num_experts >= 1 && c.expert_begin >= 0 && c.num_local >= 1 && c.num_local <= DPEP_MAX_LOCAL_EXPERTS &&
                     c.expert_begin + c.num_local <= c.num_experts,
                 "layout_dispatch_small: bad expert range E=%d begin=%d L=%d", c.num_experts, c.expert_begin, c.num_local);
    DPEP_REQUIRE(c.topk_idx && c.counts && c.psum && c.offsets && c.route_to_row && c.row_to_route && c.num_rows,
                 "layout_dispatch_small: NULL routing buffer");
    int units = 0;
    if (int rc = check_fresh_payload("layout_dispatch_small", c, &units)) return rc;
    return launch_small(w, c, units, stream);
}

}  // namespace

// (layout.hip) *payload_launched: whether `payload` went along.
int layout_of_fresh(void* ws, const dpep_fresh_dispatch& c, const LayoutPayload* payload, bool* payload_launched, hipStream_t stream);

}  // namespace dpep

extern "C" {

int dpep_dispatch_store_policy(int policy)
{
    using namespace dpep;
    const int before = __atomic_load_n(&g_store_policy, __ATOMIC_RELAXED);
    if (policy == DPEP_STORE_QUERY) return before;
    DPEP_REQUIRE(policy == DPEP_STORE_THROUGH || policy == DPEP_STORE_STREAMING || policy == DPEP_STORE_CACHED,
                 "dispatch_store_policy: %d is not DPEP_STORE_THROUGH, _STREAMING, _CACHED or _QUERY", policy);
    __atomic_store_n(&g_store_policy, policy, __ATOMIC_RELAXED);
    return before;
}

int dpep_dispatch_copy(const void* x, const float* scales, const float* topk_weights, const int32_t* route_to_row,
                       const int32_t* row_to_route, int num_tokens, int num_topk, int num_rows, int row_bytes,
                       int scale_cols, void* out, float* out_scales, float* out_weights, void* stream)
{
    using namespace dpep;
    if (int rc = check_common("dispatch_copy", num_tokens, num_topk, num_rows, route_to_row, row_to_route)) return rc;
    DPEP_REQUIRE(row_bytes > 0 && row_bytes % 16 == 0, "dispatch_copy: row_bytes=%d must be a positive multiple of 16",
                 row_bytes);
    // (a share without rows or a batch without tokens: the outputs are empty buffers, which may well be null pointers)
    if (num_rows == 0 || num_tokens == 0) return DPEP_OK;
    DPEP_REQUIRE((scales == nullptr) == (out_scales == nullptr), "dispatch_copy: scales and out_scales go together");
    DPEP_REQUIRE(scales == nullptr || scale_cols > 0, "dispatch_copy: scale_cols must be positive with scales");
    DPEP_REQUIRE((topk_weights == nullptr) == (out_weights == nullptr), "dispatch_copy: weights and out_weights go together");
    DPEP_REQUIRE(x != nullptr && out != nullptr && aligned16(x) && aligned16(out), "dispatch_copy: x/out must be 16-byte aligned");
    const Payload p = {static_cast<const u32x4*>(x), scales, topk_weights, num_tokens, num_topk, row_bytes / 16, scale_cols, false, static_cast<u32x4*>(out),
                       out_scales, out_weights};
    return launch_payload(p, route_to_row, row_to_route, num_rows, static_cast<hipStream_t>(stream));
}

int dpep_dispatch_quant_fp8(const void* x, const float* topk_weights, const int32_t* route_to_row,
                            const int32_t* row_to_route, int num_tokens, int num_topk, int num_rows, int hidden,
                            void* out, float* out_scales, float* out_weights, void* stream)
{
    using namespace dpep;
    if (int rc = check_common("dispatch_quant_fp8", num_tokens, num_topk, num_rows, route_to_row, row_to_route)) return rc;
    DPEP_REQUIRE(hidden > 0 && hidden % 128 == 0 && hidden / 128 <= kMaxScaleCols,
                 "dispatch_quant_fp8: hidden=%d must be a positive multiple of 128, at most %d", hidden, 128 * kMaxScaleCols);
    if (num_rows == 0 || num_tokens == 0) return DPEP_OK;  // (empty outputs may be null pointers)
    DPEP_REQUIRE((topk_weights == nullptr) == (out_weights == nullptr), "dispatch_quant_fp8: weights and out_weights go together");
    DPEP_REQUIRE(x && out && out_scales && aligned16(x) && aligned16(out), "dispatch_quant_fp8: x/out must be 16-byte aligned");
    const Payload p = {static_cast<const u32x4*>(x), nullptr, topk_weights, num_tokens, num_topk, hidden / 16, 0, true, static_cast<u32x4*>(out),
                       out_scales, out_weights};
    return launch_payload(p, route_to_row, row_to_route, num_rows, static_cast<hipStream_t>(stream));
}

int dpep_dispatch_fresh(void* ws, const dpep_fresh_dispatch* call, void* stream)
{
    using namespace dpep;
    Workspace* w = as_workspace(ws);
    DPEP_REQUIRE(w != nullptr && call != nullptr, "dispatch_fresh: not a live workspace, or NULL call");
    const dpep_fresh_dispatch& c = *call;
    hipStream_t s = static_cast<hipStream_t>(stream);
    DPEP_REQUIRE(c.num_tokens >= 1 && c.num_topk >= 1 && c.num_topk <= DPEP_MAX_TOPK, "dispatch_fresh: bad T=%d K=%d", c.num_tokens,
                 c.num_topk);
    const long long n_routes = static_cast<long long>(c.num_tokens) * c.num_topk;
    if (n_routes > kSmallRoutes) {
        int units = 0;
        if (int rc = check_fresh_payload("dispatch_fresh", c, &units)) return rc;
        DPEP_REQUIRE(c.capacity_rows >= 0, "dispatch_fresh: capacity_rows=%d is negative", c.capacity_rows);
        const Payload p = {static_cast<const u32x4*>(c.x), c.scales, c.topk_weights, c.num_tokens, c.num_topk, units, c.quantize ? 0 : c.scale_cols,
                           c.quantize != 0, static_cast<u32x4*>(c.out), c.out_scales, c.out_weights};
        // Expected rows of this rank's share: what the caller made its outputs for, or the even share.  Many rows per token:
        // token-major, which reads every token once.  Otherwise row-major over the rows that the layout finds: a token-major
        // grid is mostly workgroups of tokens without a row (6144 tokens of which 560 own a row: 10.5 us).  16 384 BF16
        // tokens of 7168 columns, row-major / token-major: 0.5 rows per token 36.8 / 39.6 us, 1: 67.5 / 61.6, 1.5: 102 / 83, 4:
        // 268 / 175; FP8 20.3 / 24.7, 35.4 / 35.0, 53.3 / 45.2, 138 / 90.
        const bool all_or_none = c.report_to_host == DPEP_REPORT_ALL_OR_NONE;
        const long long expected =
            all_or_none ? (c.capacity_rows > 256 ? (c.capacity_rows - 256LL) * 8 / 9 : 0) : n_routes * c.num_local / c.num_experts;
        const bool token_major = expected > static_cast<long long>(kRowMajorRatio) * c.num_tokens;
        long long grid_rows = expected + expected / 8 + 64;
        if (grid_rows > c.capacity_rows) grid_rows = c.capacity_rows;
        if (grid_rows > n_routes) grid_rows = n_routes;
        const int bound = n_routes < c.capacity_rows ? static_cast<int>(n_routes) : c.capacity_rows;
        // In the layout's grid (launch_layout), where that is the better place.  A large token-major payload with several rows to a token ends
        // 1 to 15 us sooner there; beside a small one the GPU waits for the host, and the layout reports to it 0.5 to 3 us later with a
        // payload in its grid (dispatch and combine: 39 MB 33.0 -> 31.9 us, 43 MB 39.0 -> 34.6, 152 MB 91.8 -> 87.8, 18 MB 22.7 -> 23.5, 13 MB
        // 25.2 -> 28.1; 1.25 rows per token, 41 MB 39.8 -> 46.8, 142 MB 197.5 and 196.7.  On both sides of the five rows per token, one grid / two: BF16, 4096
        // tokens of 4096 columns x top-2 39.9 / 38.7, 3 48.2 / 49.8, 4 62.2 / 64.8, 5 68.4 / 70.8; 1500 of 7168 27.4 / 27.4, 34.8 / 35.0, 40.2 / 42.0, 47.4 /
        // 48.8; 6000 of 1552 29.6 / 28.4, 35.5 / 37.7, 42.0 / 42.6, 48.7 / 53.3; to FP8, 2500 of 5120 31.4 / 31.3, 35.9 / 37.1, 41.2 / 42.4, 47.0 / 48.3, 4096 of
        // 7168 62.6 / 57.8, 74.4 / 71.1, 89.6 / 88.7, 102.1 / 100.5 and, 6, 116.5 / 116.7.  The line lies where the largest quantised payloads stop losing;
        // 18 others of five to ten rows gain 1 to 4 %, 10 that are FP8 already 3 to 9 %.  BF16 gains 1 to 6 % with three and four rows too.)  Row-major workgroups wait for their row before they
        // can ask for its values, so it is only the launch that is saved, which counts where nothing is reported and the host is
        // the one to wait for: 0.4 to 2 MB 17 -> 14 us, 4 MB 28.3 and 28.4, 10 MB 60.5 -> 63.1, 117 MB 124 -> 156.
        LayoutPayload riding = {};
        const long long payload_bytes = expected * (c.quantize ? c.row_bytes / 2 : c.row_bytes);
        const bool worth_it = token_major ? payload_bytes >= (32LL << 20) && expected >= 5LL * c.num_tokens
                                          : c.report_to_host == 0 && payload_bytes <= (3LL << 20);
        const bool may_ride = worth_it && c.capacity_rows > 0 && dpep_dispatch_store_policy(DPEP_STORE_QUERY) == DPEP_STORE_STREAMING;
        if (may_ride) {
            const int lines = token_major ? c.num_tokens : static_cast<int>(grid_rows);
            Split sp = payload_split(p, lines, token_major ? expected : lines);
            // (A workgroup of the layout's has 256 threads; parts that leave a third of them idle are too fine: 3596 tokens x top-5 of 4608
            // columns to FP8, two parts of 144 units 56.8 us, one 54.3.)
            if (token_major && kMaxThreads / sp.threads * sp.per_part < 176) sp = choose_split(lines, units, p.quantize || units % 8 == 0 ? 8 : 1, 2048);
            riding = {p.x, p.scales, p.weights, p.out, p.out_scales, p.out_weights, payload_shape(p, sp), c.quantize != 0, payload_staged(p, sp), !token_major, static_cast<unsigned>(lines) * sp.parts, bound, c.capacity_rows,
                      all_or_none ? c.capacity_rows : 0, w->payload_looks};
        }
        bool launched = false;
        if (int rc = layout_of_fresh(ws, c, may_ride ? &riding : nullptr, &launched, s)) return rc;  // (checks the routing arguments)
        if (launched || c.capacity_rows == 0) return DPEP_OK;
        if (token_major) return launch_token_major(p, c.route_to_row, c.capacity_rows, all_or_none ? c.num_rows : nullptr, expected, s);
        return launch_row_major(p, c.row_to_route, RowRange{bound, c.num_rows, all_or_none ? c.capacity_rows : 0}, static_cast<int>(grid_rows), s);
    }
    return fresh_in_one_launch(w, c, s);
}

int dpep_layout_dispatch_small(void* ws, const int64_t* topk_idx, const void* x, const float* scales,
                               const float* topk_weights, int num_tokens, int num_topk, int num_experts, int expert_begin,
                               int num_local, int row_bytes, int scale_cols, int quantize, int32_t* counts, int32_t* psum,
                               int32_t* offsets, int32_t* route_to_row, int32_t* row_to_route, int32_t* num_rows, void* out,
                               float* out_scales, float* out_weights, void* stream)
{
    using namespace dpep;
    Workspace* w = as_workspace(ws);
    DPEP_REQUIRE(w != nullptr, "layout_dispatch_small: not a live workspace");
    const dpep_fresh_dispatch c = {topk_idx, nullptr, x, scales, topk_weights, counts, psum, offsets, route_to_row, row_to_route,
                                   num_rows, nullptr, out, out_scales, out_weights, num_tokens, num_topk, num_experts,
                                   expert_begin, num_local, row_bytes, scale_cols, quantize, /*capacity_rows=*/0x7fffffff,
                                   /*report_to_host=*/1};
    return fresh_in_one_launch(w, c, static_cast<hipStream_t>(stream));
}

int dpep_cast_to_fp8(const void* x, int num_tokens, int hidden, void* out, float* out_scales, void* stream)
{
    using namespace dpep;
    DPEP_REQUIRE(num_tokens >= 0, "cast_to_fp8: bad T=%d", num_tokens);
    DPEP_REQUIRE(hidden > 0 && hidden % 16 == 0, "cast_to_fp8: hidden=%d must be a positive multiple of 16", hidden);
    if (num_tokens == 0) return DPEP_OK;
    DPEP_REQUIRE(x && out && out_scales && aligned16(x) && aligned16(out), "cast_to_fp8: x/out must be 16-byte aligned");
    const int units = hidden / 16;
    if (hidden % 128 != 0) {
        const int blocks = (hidden + 127) / 128;
        const long long padded = static_cast<long long>(num_tokens) * blocks * 8;
        hipLaunchKernelGGL(cast_to_fp8_short_block_kernel, dim3(static_cast<unsigned>((padded + 255) / 256)), dim3(256), 0,
                           static_cast<hipStream_t>(stream), static_cast<const u32x4*>(x), units, blocks, padded,
                           static_cast<u32x4*>(out), out_scales);
        return launch_status("cast_to_fp8");
    }
    const Split sp = choose_split(num_tokens, units, 8);
    auto launch = [&](auto policy) {
        hipLaunchKernelGGL(dispatch_quant_row_kernel<decltype(policy)::value>, dim3(num_tokens * sp.parts),
                           dim3(sp.threads), 0, static_cast<hipStream_t>(stream), static_cast<const u32x4*>(x), nullptr,
                           nullptr, RowRange{num_tokens, nullptr, 0}, num_tokens, 1, units, sp.per_part, sp.parts,
                           static_cast<u32x4*>(out), out_scales, nullptr);
    };
    // (codes that the memory-side cache takes are written through, whatever the dispatch's policy: the quantiser's reader is next.
    // 10007 x 5120: quantise and dequantise 47.7 us instead of 53.2)
    if (static_cast<size_t>(num_tokens) * hidden <= kStreamBytes) launch(std::integral_constant<int, DPEP_STORE_THROUGH>{});
    else with_store_policy(launch);
    return launch_status("cast_to_fp8");
}

int dpep_cast_back(const void* codes, const void* scales, int scales_are_e8m0_bytes, int num_tokens, int hidden, void* out,
                   void* stream)
{
    using namespace dpep;
    DPEP_REQUIRE(num_tokens >= 0, "cast_back: bad T=%d", num_tokens);
    DPEP_REQUIRE(hidden > 0 && hidden % 16 == 0, "cast_back: hidden=%d must be a positive multiple of 16", hidden);
    if (num_tokens == 0) return DPEP_OK;
    DPEP_REQUIRE(codes && scales && out && aligned16(codes) && aligned16(out), "cast_back: codes/out must be 16-byte aligned");
    const int halves = hidden / 8, blocks_per_row = (hidden + 127) / 128;
    const long long total = static_cast<long long>(num_tokens) * halves;
    DPEP_REQUIRE((total + 255) / 256 < (1ll << 31), "cast_back: %d x %d codes are more than one launch takes", num_tokens, hidden);
    const unsigned grid = static_cast<unsigned>((total + 255) / 256);
    // (46 MB of BF16: 12.5 us write-through, 13.7 streaming; 61 MB behind the quantiser that made the codes: 32.1 and 30.7)
    const bool through = static_cast<size_t>(total) * 16 <= (48u << 20);
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), 0, static_cast<hipStream_t>(stream), static_cast<const unsigned long long*>(codes),
                           scales, halves, blocks_per_row, total, static_cast<u32x4*>(out));
    };
    if (scales_are_e8m0_bytes) through ? launch(cast_back_kernel<true, true>) : launch(cast_back_kernel<true, false>);
    else through ? launch(cast_back_kernel<false, true>) : launch(cast_back_kernel<false, false>);
    return launch_status("cast_back");
}

}  // extern "C"

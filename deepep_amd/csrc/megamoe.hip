// W4A8 expert FFN for one rank's local experts: MXFP8 (e4m3 + e8m0 per 32) activations times MXFP4
// (e2m1 + e8m0 per 32) weights on the gfx950 block-scaled MFMA, with a fused SwiGLU + MXFP8 requant
// epilogue after the first GEMM, grouped over ragged per-expert row counts.
//
// Numerics follow experiments/megamoe/python/deep_ep_experimental/megamoe/reference.py:44-100:
//   first = bf16(x @ w1^T); act = bf16(silu(gate) * up); qa = mx_quant(act); out = bf16(qa @ w2^T);
//   y[t] = bf16( sum_s w[t,s] * out[row(t,s)] )  (route weight applied after the second GEMM).
//
// Operand layout of v_mfma_scale_f32_32x32x64_f8f6f4 (fp8 A, fp4 B), as measured on gfx950:
//   A: lane l holds row l%32; VGPR 0-3 = k in [16g, 16g+16), VGPR 4-7 = k in [32+16g, 32+16g+16), g = l/32
//   B: lane l holds column l%32; 4 VGPRs = 32 nibbles k in [32g, 32g+32), low nibble first
//   scales: lane l supplies the e8m0 byte of (row or column l%32, 32-wide k block l/32)
//   D: acc[j] is row (j/4)*8 + (l/32)*4 + j%4, column l%32
#include <algorithm>
#include <atomic>
#include <type_traits>
#include <utility>

#include "common.h"
#include "gemm_schedule.h"
#include "mx.h"

#pragma clang fp contract(off)

namespace dpep {

int layout_i32(void* ws, const int32_t* idx, int num_tokens, int num_topk, int num_experts, int expert_begin,
               int num_local, int32_t* counts, int32_t* psum, int32_t* offsets, int32_t* route_to_row,
               int32_t* row_to_route, int32_t* num_rows, const MegaFront& front, hipStream_t stream);
int combine_routes(const void* y, const float* route_weights, const int32_t* route_to_row, int num_tokens, int num_topk,
                   int num_rows_hint, int hidden, void* out, const int32_t* shared_first_row, int num_shared,
                   const int32_t* fill_state, int leave_unserved, hipStream_t stream);

namespace {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>): a loop whose counter is a compile-time constant in
// the body (register arrays and instruction immediates are indexed by it).
template <typename F, int... I>
__device__ __forceinline__ void static_for_each(F&& f, std::integer_sequence<int, I...>)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f)
{
    static_for_each(f, std::make_integer_sequence<int, N>{});
}

// =====================================================================================================
// MXFP8 activation quantiser (block 32 along the row)
// =====================================================================================================
// One lane owns 16 consecutive BF16 values (32 bytes in, one 16-byte vector of codes out, consecutive lanes writing
// consecutive vectors); two adjacent lanes own one 32-element block.  The workgroup's 128 scale bytes are staged in LDS
// and leave as eight 16-byte stores instead of one byte-wide store per block, which turned every scale row into
// read-modify-write traffic.  The tensors are treated as flat arrays: hidden is a multiple of 32, so blocks never
// straddle rows.  Input and codes stream past the caches (the input is read once; with cached loads the kernel's time
// depended on what the caches held before: 48 us back to back, 89 us behind a 256 MiB fill, against 58-63 us this way
// under every protocol).  kVectorScales: the scale pointer is 16-byte aligned.
constexpr int kMxThreads = 256;

template <bool kVectorScales>
__global__ __launch_bounds__(kMxThreads) void mx_quant_kernel(const u32x4* __restrict__ x, long long num_units,
                                                              u32x4* __restrict__ codes, uint8_t* __restrict__ scales)
{
    __shared__ __attribute__((aligned(16))) uint8_t staged[kMxThreads / 2];
    const long long u = static_cast<long long>(blockIdx.x) * kMxThreads + threadIdx.x;
    const bool live = u < num_units;
    u32x4 raw[2] = {{0u, 0u, 0u, 0u}, {0u, 0u, 0u, 0u}};
    if (live) {
        raw[0] = load16_nt(x + 2 * u);
        raw[1] = load16_nt(x + 2 * u + 1);
    }
    int byte;
    const u32x4 out = mx_quantize16(raw[0], raw[1], byte);
    if (live) store16_nt(codes + u, out);
    if ((threadIdx.x & 1) == 0) staged[threadIdx.x >> 1] = static_cast<uint8_t>(byte);
    __syncthreads();
    // blocks (= scale bytes) of this workgroup: [first, first + 128) clipped to the end
    const long long first = static_cast<long long>(blockIdx.x) * (kMxThreads / 2);
    const long long num_blocks = num_units >> 1;
    const int present = static_cast<int>(min(static_cast<long long>(kMxThreads / 2), num_blocks - first));
    if (kVectorScales && present == kMxThreads / 2) {
        if (threadIdx.x < kMxThreads / 32)
            store16_through(scales + first + threadIdx.x * 16, *reinterpret_cast<const u32x4*>(staged + threadIdx.x * 16));
    } else if (static_cast<int>(threadIdx.x) < present) {
        scales[first + threadIdx.x] = staged[threadIdx.x];
    }
}

// =====================================================================================================
// Weight re-layout: raw [L][N][K/2] + [L][N][K/32]  ->  1 KiB blocks holding every lane's 16-byte B fragment of
// one (column tile of 32, k step of 64), ordered [expert][256 columns][k tile of 128][column tile][k step] so
// that a workgroup's 16 KiB per item are contiguous; scales as 2 bytes per lane per k=128.
// =====================================================================================================
__device__ __forceinline__ int source_row(int physical_col, int n, int gate_up)
{
    if (!gate_up) return physical_col;
    // column tiles alternate gate / up for the same 32 activation columns
    const int tile = physical_col >> 5, j = physical_col & 31;
    const int act_col = (tile >> 1) * 32 + j;
    return (tile & 1) * (n >> 1) + act_col;
}

// n, k: the raw matrix; np, kp: what the GEMM works on (padded_dim of each; for gate/up both halves are padded, so
// np = 2 * padded_dim(n / 2)).  Padding columns and k blocks get zero codes (FP4 0.0) and the scale byte of 1.0.
__global__ __launch_bounds__(256) void prepare_weights_kernel(const uint8_t* __restrict__ w,
                                                              const uint8_t* __restrict__ s, int n, int k, int np, int kp,
                                                              int gate_up, uint8_t* __restrict__ w_out,
                                                              uint8_t* __restrict__ s_out, long long packed_chunks,
                                                              long long scale_pairs)
{
    const long long id = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
    const int ktiles = kp / 128;
    // raw row of a physical (padded, interleaved) column, or -1 for a padding column
    auto raw_row = [&](int physical_col) {
        const int row = source_row(physical_col, np, gate_up);
        if (!gate_up) return row < n ? row : -1;
        const int half = np >> 1, in_half = row % half;
        return in_half < (n >> 1) ? (row / half) * (n >> 1) + in_half : -1;
    };
    if (id < packed_chunks) {
        // one 16-byte fragment; order [expert][block of 8 column tiles][k tile][column tile][k step][lane]: the
        // 16 KiB a workgroup copies per item are contiguous and its items follow each other in memory
        const int lane = id & 63, q = (id >> 6) & 15;
        long long rest = id >> 10;
        const int kt = rest % ktiles;
        rest /= ktiles;
        const int nb = rest % (np / 256);
        const long long e = rest / (np / 256);
        const int c = nb * 8 + (q >> 1), ks = kt * 2 + (q & 1);
        const int row = raw_row(c * 32 + (lane & 31));
        const int byte = ks * 32 + (lane >> 5) * 16;  // 16 bytes = 32 values of k, all inside the raw matrix or none
        u32x4 fragment = {0u, 0u, 0u, 0u};
        if (row >= 0 && byte * 2 < k) fragment = *reinterpret_cast<const u32x4*>(w + (e * n + row) * (k / 2) + byte);
        reinterpret_cast<u32x4*>(w_out)[id] = fragment;
    }
    if (id < scale_pairs) {
        // Scales: per (expert, block of 8 column tiles, span of 4 k tiles) one 4 KiB block
        // [column tile 8][lane 64][k tile 4][2 bytes = k blocks (2*kb + g) of that k tile]; a span is what
        // the GEMM copies in one go.  The last span is padded when kp % 512 != 0.
        const int spans = (ktiles + 3) / 4;
        const int kq = id & 3, lane = (id >> 2) & 63, c8 = (id >> 8) & 7;
        long long rest = id >> 11;
        const int span = rest % spans;
        rest /= spans;
        const int nb = rest % (np / 256);
        const long long e = rest / (np / 256);
        const int kt = span * 4 + kq;
        uint8_t lo = 127, hi = 127;
        const int row = raw_row((nb * 8 + c8) * 32 + (lane & 31));
        if (kt < ktiles && row >= 0) {
            const int block = kt * 4 + (lane >> 5);  // k blocks of 32: this lane half's two of the k tile
            const uint8_t* src = s + (e * n + row) * (k / 32);
            if (block < k / 32) lo = src[block];
            if (block + 2 < k / 32) hi = src[block + 2];
        }
        s_out[id * 2] = lo;
        s_out[id * 2 + 1] = hi;
    }
}

// =====================================================================================================
// Grouped GEMM
// =====================================================================================================
// Workgroup = 4 waves (2 row halves x 2 column halves), tile (64*RT) rows x 256 columns, k tile 128
// (two MFMA k steps) per LDS stage.  Workgroups are persistent (one per CU) and treat their tiles as ONE
// flat stream of (tile, k tile) items: asynchronous global->LDS copies run kAhead items ahead of the
// MFMAs and roll straight into the next tile, so a tile's epilogue overlaps the next tile's first copies.
// Per item there is one vmcnt wait + one barrier; the fragments of the next k step leave LDS while the
// MFMAs of the current one run.  A wave owns its SIMD alone and issues in order, so everything that is not
// an MFMA is placed in the shadow of one: the MFMAs are volatile asm statements (they keep source order;
// builtin MFMAs get gathered into bursts) and the item's copies are dealt out one after each MFMA.
// Scales and gather indices do not travel with every item (a 4-byte copy costs more per instruction than
// a 16-byte one): row scales (16 B per row = k 512), column scales (4 KiB per k 512) and
// the next tile's gather indices (once per tile) are fetched per span of four items.
// Rows are fetched 128 bytes at a time (full cache lines): the texture path handles about one line per
// cycle and CU, which a 64-byte k tile would saturate.
constexpr int kBK = 128;           // k per LDS stage = two MFMA k steps
constexpr int kCT = 4;             // 32-column MFMA tiles per wave
constexpr int kBN = 2 * kCT * 32;  // columns per workgroup tile
constexpr int kGemmThreads = 256;
constexpr int kGemmWaves = kGemmThreads / 64;
constexpr int kMaxMoeExperts = 128;
constexpr int kStagingRowStride = 80;  // 32 BF16 + 16 B pad: conflict-free 16-byte reads

template <int RT, bool kGather>
struct GemmCfg : GemmRing<RT> {
    using GemmRing<RT>::kStages;
    static constexpr int kBM = 64 * RT;
    static constexpr int kOffA = 0;                    // kBM rows x 128 B, 16-byte chunks XOR-swizzled
    static constexpr int kOffB = kBM * kBK;            // 8 column tiles x 2 k steps x 1 KiB fragments
    static constexpr int kStageBytes = kOffB + 16384;
    // Scales travel apart, once per span of four items, into three-slot rings: 16 bytes per row cover
    // k = 512 of row scales, and one 4 KiB block holds the column scales of the span.  (4-byte copies
    // are several times slower per instruction than 16-byte ones, and a 4-byte copy per row costs a
    // cache-line lookup per lane.)  Three slots, not two: a tile whose k is not a multiple of 512 ends with a span of
    // two items, and in a workgroup that goes on to another tile the copies, up to five items ahead, then reach the
    // span after next (two items + one: three items on) while the scales of the span before the short one are still
    // being read; with three slots the span that reuses a slot starts at least seven items behind the last read.
    static constexpr int kScaleSlots = 3;
    static constexpr int kRowScaleSlot = kBM * 16;
    static constexpr int kColScaleSlot = 4096;
    static constexpr int kOffRowScales = kStages * kStageBytes;
    static constexpr int kOffColScales = kOffRowScales + kScaleSlots * kRowScaleSlot;
    static constexpr int kStagingWave = 32 * kStagingRowStride;  // the epilogue handles one 32-row tile at a time
    static constexpr int kOffStaging = kOffColScales + kScaleSlots * kColScaleSlot;
    static constexpr int kLdsBytes = kOffStaging + 4 * kStagingWave;
};

struct GemmParams {
    const uint8_t* a_codes;    // [*, K] e4m3
    const uint8_t* a_scales;   // [*, K/32] e8m0
    const int* row_to_route;   // first GEMM: source row = row_to_route[r] / topk
    int topk;
    int a_rows;                // rows of a_codes (the gather clamps to them)
    const int* offsets;        // [L+1] exclusive row prefix per expert
    int num_local;
    const uint8_t* w;          // prepared fragments, expert stride N*K/2
    const uint8_t* ws;         // prepared scales, expert stride N*K/32
    int num_routed;            // experts >= num_routed are shared experts with weights of their own:
    const uint8_t* w_shared;   //   expert e reads w_shared / ws_shared at index e - num_routed
    const uint8_t* ws_shared;
    int n, k;                  // padded sizes: the strides of the operands (what is not padding of them: n_real, k_real)
    uint8_t* act_codes;        // first GEMM: [rows, N/2] e4m3
    uint8_t* act_scales;       //             [rows, N/64] e8m0
    uint16_t* out;             // second GEMM: [rows, out_cols] bf16
    int out_cols;              //   columns that exist (<= N, a multiple of 8; the padding columns of N are not stored)
    // Zero rows of the final output.  When a launch has fewer tiles than workgroups, the workgroups left
    // without a tile stream zeros into the output rows of the tokens that no local expert serves (most tokens of a
    // rank's share), which the weighted reduce would otherwise have to write after the GEMMs: the stores cost the
    // matrix pipes nothing.  kFillWaves waves of such a workgroup are fillers f and take tokens f, f + fillers, ...
    // until a workgroup with a tile reaches its epilogue and raises *fill_stop.  The word is a counter that only ever
    // grows (device memory of the workspace): a filler remembers the value it found when it started and stops when
    // the word differs, so nothing has to clear it, no value comes from the host, and every replay of a captured
    // launch stops its own fillers.  (Launches on a workspace run one after the other, so a filler's first read sees
    // every increment of the launches before it and none of its own launch: the first increment is a whole tile away.  One-wave launches
    // have few_rows_fillers workgroups more for it.)
    // fill_state[0] = number of fillers, fill_state[1 + f] = tokens filler f got through.  All of it is null / zero in
    // launches that do not fill.
    u32x4* fill_out;                // [fill_tokens, fill_vec] or nullptr
    const int* fill_route_to_row;   // [fill_tokens, fill_topk]
    int fill_tokens, fill_vec, fill_topk;
    int* fill_state;
    int* fill_stop;
    int forced;                     // 64 / 128 / 192: that tile height whatever the cost model says (tests), 128 | (1, 2) << 8: the paired kernel, its weights cached or streamed; 32: the
                                    //   few-rows kernel with (1, 4) << 8 waves per workgroup; 0: the model decides
    int column_waves;               // 1: the kernel whose waves split the tile's columns and load their weights straight into registers
    int n_real, k_real;             // what is not padding of n and k (first GEMM: n counts gate and up)
    int live_n_tiles;               // column tiles that the kernels that skip padding work on (first GEMM: all, unless the second reads none of it)
    int numbered_n_tiles;           // few-rows kernels: column tiles that a row tile's numbers are given to, those behind live_n_tiles in vain
    int few_rows_fillers;           // one-wave launches: workgroups in front of those with tiles that fill
};

// gate / (1 + exp(-gate)) * up with the hardware exponential and reciprocal (v_exp_f32, v_rcp_f32: about 1 ulp each; the
// result is rounded to BF16 right after).  The clamp keeps exp finite, like the reference's clip(+-80).  (The
// reciprocal is the instruction itself: a correctly rounded 1 / x is a ten-instruction sequence per value, a third of the
// first GEMM's epilogue, for a last bit that the rounding to BF16 drops.)
__device__ __forceinline__ float silu_mul(float gate, float up)
{
    const float clipped = fminf(fmaxf(-gate, -80.0f), 80.0f);
    return gate * __builtin_amdgcn_rcpf(1.0f + __expf(clipped)) * up;
}

// Asynchronous copy global -> LDS: lane l's bytes land at lds_base + l * size.  lds_base is wave-uniform.
// Written as assembly so that the compiler's own wait-count bookkeeping does not serialise the ring;
// completion is awaited explicitly with wait_copies_then_barrier<N>().
__device__ __forceinline__ void copy16_to_lds(const void* src, uint32_t lds_base)
{
    const uint32_t base = __builtin_amdgcn_readfirstlane(lds_base);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(base), "v"(src) : "memory");
}
// The same with the address split into a wave-uniform 64-bit base (SGPR pair) and a 32-bit lane offset.
__device__ __forceinline__ void copy16_to_lds(const void* uniform_base, uint32_t lane_offset, uint32_t lds_base)
{
    const uint32_t base = __builtin_amdgcn_readfirstlane(lds_base);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(base), "v"(lane_offset),
                 "s"(uniform_base)
                 : "memory");
}
// The weight copies carry a cache hint chosen by how often a launch reads a weight tile.  kStreamed (64-row tiles: few
// rows per expert, every weight byte is read once or twice): non-temporal, which measured 10 % faster for the first GEMM
// of a decode-like share (32 local experts x 16 rows: 98 -> 88 us) and costs large batches 1.6 % (their row tiles
// re-read the weights from the L2); otherwise device-scope (`sc1`): 2 % faster at an EP64 rank's share, neutral for
// large batches.
template <bool kStreamed>
__device__ __forceinline__ void copy16_weights_to_lds(const void* uniform_base, uint32_t lane_offset, uint32_t lds_base)
{
    const uint32_t base = __builtin_amdgcn_readfirstlane(lds_base);
    if (kStreamed)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(base), "v"(lane_offset),
                     "s"(uniform_base)
                     : "memory");
    else
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 sc1" ::"s"(base), "v"(lane_offset),
                     "s"(uniform_base)
                     : "memory");
}
__device__ __forceinline__ void copy4_to_lds(const void* uniform_base, uint32_t lane_offset, uint32_t lds_base)
{
    const uint32_t base = __builtin_amdgcn_readfirstlane(lds_base);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(base), "v"(lane_offset), "s"(uniform_base) : "memory");
}
__device__ __forceinline__ void copy4_to_lds(const void* src, uint32_t lds_base)
{
    const uint32_t base = __builtin_amdgcn_readfirstlane(lds_base);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" ::"s"(base), "v"(src) : "memory");
}
// The same 16-byte copy, skipped when the (wave-uniform) value skip is not zero.  The jump stays inside
// the asm statement so that the loop body around it remains straight-line code.
__device__ __forceinline__ void copy16_to_lds_unless(const void* src, uint32_t lds_base, int skip)
{
    const uint32_t base = __builtin_amdgcn_readfirstlane(lds_base);
    const int flag = __builtin_amdgcn_readfirstlane(skip);
    asm volatile(
        "s_mov_b32 m0, %0\n\ts_cmp_lg_u32 %2, 0\n\ts_cbranch_scc1 .Lskip_copy_%=\n\t"
        "global_load_lds_dwordx4 %1, off\n.Lskip_copy_%=:" ::"s"(base),
        "v"(src), "s"(flag)
        : "memory", "scc");
}
__device__ __forceinline__ void copy4_to_lds_unless(const void* uniform_base, uint32_t lane_offset, uint32_t lds_base, int skip)
{
    const uint32_t base = __builtin_amdgcn_readfirstlane(lds_base);
    const int flag = __builtin_amdgcn_readfirstlane(skip);
    asm volatile(
        "s_mov_b32 m0, %0\n\ts_cmp_lg_u32 %3, 0\n\ts_cbranch_scc1 .Lskip_copy_%=\n\t"
        "global_load_lds_dword %1, %2\n.Lskip_copy_%=:" ::"s"(base),
        "v"(lane_offset), "s"(uniform_base), "s"(flag)
        : "memory", "scc");
}
__device__ __forceinline__ void copy4_to_lds_unless(const void* src, uint32_t lds_base, int skip)
{
    const uint32_t base = __builtin_amdgcn_readfirstlane(lds_base);
    const int flag = __builtin_amdgcn_readfirstlane(skip);
    asm volatile(
        "s_mov_b32 m0, %0\n\ts_cmp_lg_u32 %2, 0\n\ts_cbranch_scc1 .Lskip_copy_%=\n\t"
        "global_load_lds_dword %1, off\n.Lskip_copy_%=:" ::"s"(base),
        "v"(src), "s"(flag)
        : "memory", "scc");
}
// Also waits for the wave's own LDS reads: past the barrier nothing reads the stage that is refilled next.
template <int kOutstanding>
__device__ __forceinline__ void wait_copies_then_barrier()
{
    // (Never weaken this for a timing experiment: the gather indices of the next tile travel through LDS too, so a
    // wave that runs ahead of a copy reads a stale index and fetches from a wild address.)
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kOutstanding) : "memory");
}

// One scaled MFMA (FP8 A, FP4 B) as a volatile asm statement: volatile statements keep their source order,
// which is what lets the copies and the barrier be placed between individual MFMAs (builtin MFMAs are pure
// and the compiler gathers them into bursts).  kSecond selects scale bytes 2|3 of A and byte 1 of B.
// The compiler cannot see an MFMA in here, so the code that reads an accumulator afterwards has to
// provide the wait states itself (settle_accumulators).  For the same reason these statements must stay in
// straight-line code: with a branch around one the register allocator splits the accumulator's live range
// and copies it out of the AGPRs right behind the instruction, before its last passes have written
// (measured: accumulator registers 10-15 of every tile stale).
template <bool kSecond>
__device__ __forceinline__ void mfma_fp8_fp4(v16f& acc, const v8i& a, const u32x4& b, int scale_a, int scale_b)
{
    if (!kSecond)
        asm volatile("v_mfma_scale_f32_32x32x64_f8f6f4 %0, %1, %2, %0, %3, %4 op_sel_hi:[0,0,0] blgp:4"
                     : "+a"(acc)
                     : "v"(a), "v"(b), "v"(scale_a), "v"(scale_b));
    else
        asm volatile("v_mfma_scale_f32_32x32x64_f8f6f4 %0, %1, %2, %0, %3, %4 op_sel:[0,1,0] op_sel_hi:[1,0,0] blgp:4"
                     : "+a"(acc)
                     : "v"(a), "v"(b), "v"(scale_a), "v"(scale_b));
}
// 16-pass MFMA results may be read by other instruction types 19 wait states after issue at the earliest.
__device__ __forceinline__ void settle_accumulators() { asm volatile("s_nop 15\n\ts_nop 7" ::: "memory"); }
// The same behind builtin MFMAs, for accumulators that other code may read or move from here on.  The compiler inserts wait
// states of its own, but counts an s_waitcnt as one of them, which it is not when nothing is left to wait for: a move of
// an accumulator at the end of a branch, 18 states and an s_waitcnt behind the MFMA, read the last two registers stale.
__device__ __forceinline__ void settle_accumulators(v16f (&acc)[2]) { asm volatile("s_nop 15\n\ts_nop 7" : "+v"(acc[0]), "+v"(acc[1])); }

// The lane's number, worked out on the spot (two instructions) instead of kept in a register: the code that runs once
// per tile or span (tile switches, scale requests, the epilogue) takes its lane-dependent addresses from this, so that the
// item loop does not have to carry them.
__device__ __forceinline__ int lane_now()
{
    int lane;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(lane));
    return lane;
}

// Tiles before each expert: tile_base[0 .. kMaxMoeExperts], the entries past the last expert hold the total.  One wave, two experts
// per lane: a walk over the experts, here and at every tile switch (where the matrix pipe waits for it), cost a dependent LDS
// read each.  Without the walks: 64 experts of 1024 x 512, 64 rows each, whole forward 47.9 -> 35.1 us, 100 of 2048 x 768,
// 330 rows each 291 -> 246, 32 of 7168 x 2048, 2048 rows each 2466 -> 2402.
template <int kBM>
__device__ __forceinline__ void number_tiles(const int* row_offsets, int num_local, int n_tiles, int lane, int* tile_base)
{
    static_assert(kMaxMoeExperts <= 128, "two experts per lane");
    int before = 0;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int e = lane + 64 * h;
        const int rows = e < num_local ? row_offsets[e + 1] - row_offsets[e] : 0;
        const int through = before + wave_scan((rows + kBM - 1) / kBM * n_tiles);
        tile_base[e + 1] = through;
        before = __builtin_amdgcn_readlane(through, 63);
    }
    if (lane == 0) tile_base[0] = 0;
}
// The expert that a tile (below the total) belongs to: how many experts end at or before it, asked of 64 at a time.
__device__ __forceinline__ int expert_of_tile(int tile, const int* tile_base, int num_local)
{
    const int lane = lane_now();
    int e = __popcll(__ballot(tile >= tile_base[lane + 1]));
    if (num_local > 64) e += __popcll(__ballot(tile >= tile_base[lane + 65]));
    return e;
}

// Wave number `filler` of `fillers`: zero rows of the output (see GemmParams).  Two waves of every workgroup without a tile: more of
// them fill faster, but what they take from the GEMM grows faster still, and the reduce writes what is left at 6 TB/s (one EP64
// rank's share of 16 384 tokens of 7168 columns, 64 idle workgroups, whole forward: four waves each 147.8 us, three 147.4, two 144.8, one
// 149, none 154).
constexpr int kFillWaves = 2;
__device__ __forceinline__ void fill_zero_rows(const GemmParams& p, int filler, int fillers, int lane)
{
    const u32x4 zero = {0u, 0u, 0u, 0u};
    int done = 0;
    const int stop_at_start = __hip_atomic_load(p.fill_stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (int token = filler; token < p.fill_tokens; token += fillers, ++done) {
        if (__hip_atomic_load(p.fill_stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != stop_at_start) break;
        const bool mine = lane < p.fill_topk && p.fill_route_to_row[static_cast<size_t>(token) * p.fill_topk + lane] >= 0;
        if (__ballot(mine) != 0ull) continue;  // some local expert serves the token: the reduce writes its row
        u32x4* row = p.fill_out + static_cast<size_t>(token) * p.fill_vec;
        for (int v = lane; v < p.fill_vec; v += 64) store16_nt(row + v, zero);
    }
    if (lane == 0) p.fill_state[1 + filler] = done;
}

struct TileInfo {
    int expert, nt, row0, valid;  // row0 = first row of the tile in the expanded layout; valid rows <= kBM
};

template <int RT, bool kGateUp>
__global__ __launch_bounds__(kGemmThreads, 1) void grouped_gemm_kernel(GemmParams p)
{
    constexpr bool kGather = kGateUp;
    using Cfg = GemmCfg<RT, kGather>;
    constexpr int kBM = Cfg::kBM, kStages = Cfg::kStages, kAhead = Cfg::kAhead, kStageBytes = Cfg::kStageBytes;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    __shared__ int tile_base[kMaxMoeExperts + 1];
    __shared__ int row_offsets[kMaxMoeExperts + 1];
    __shared__ int tile_index[2][kGemmThreads];  // row_to_route of a tile's rows; slots alternate per tile

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform: keeps LDS copy targets in SGPRs
    const int wm = wave >> 1, wn = wave & 1;
    const int g = lane >> 5, lr = lane & 31;
    const int n_tiles = p.n / kBN;
    const int ktiles = p.k / kBK;
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds));
    const uint32_t lds_index = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(&tile_index[0][0]));

    // Tiles per expert: ceil(rows/kBM) row tiles x n_tiles column tiles, expert-major, row tile fastest.
    // (The offsets are fetched by one thread each, in parallel; only the tiny scan is serial.)
    if (tid <= p.num_local) row_offsets[tid] = p.offsets[tid];
    __syncthreads();
    if (wave == 0) number_tiles<kBM>(row_offsets, p.num_local, n_tiles, lane, tile_base);
    __syncthreads();
    const int total_tiles = tile_base[p.num_local];

    // Consecutive tile ids share weights; give each XCD (workgroups are dealt round-robin over 8 XCDs)
    // a contiguous range of tiles so that its L2 sees each weight tile from one place.  With fewer tiles than
    // workgroups: a launch that fills keeps the ranges whole, so that the first XCDs are full and the workgroups
    // without a tile, the fillers, sit together on the XCDs left over (their stores then stay out of the L2s the
    // GEMM works from: fillers on every XCD fill faster but cost the GEMM three times as much); a launch that
    // does not fill shrinks the ranges evenly (about 4 % faster than leaving two XCDs idle).
    const bool one_round = total_tiles < static_cast<int>(gridDim.x);
    const int fillers = one_round && p.fill_out != nullptr ? (static_cast<int>(gridDim.x) - total_tiles) * kFillWaves : 0;
    const bool spread = one_round && fillers == 0 && (gridDim.x & 7) == 0;
    const int per_xcd = spread ? (total_tiles + 7) / 8 : (gridDim.x + 7) / 8;
    const int first = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    const int stride = one_round ? total_tiles + 1 : per_xcd * 8;  // one round: a single tile each
    const bool has_tile = first < total_tiles && (!spread || static_cast<int>(blockIdx.x >> 3) < per_xcd);
    if (blockIdx.x == 0 && tid == 0 && p.fill_state != nullptr) p.fill_state[0] = fillers;  // workgroup 0 always has tile 0
    if (!has_tile) {
        if (fillers != 0 && wave < kFillWaves) fill_zero_rows(p, (first - total_tiles) * kFillWaves + wave, fillers, lane);
        return;
    }
    const int my_tiles = one_round ? 1 : (total_tiles - first + stride - 1) / stride;

    auto decode = [&](int tile) {
        const int e = expert_of_tile(tile, tile_base, p.num_local);
        const int row_begin = __builtin_amdgcn_readfirstlane(row_offsets[e]), rows = __builtin_amdgcn_readfirstlane(row_offsets[e + 1]) - row_begin;
        const int m_tiles = (rows + kBM - 1) / kBM;
        const int local = tile - __builtin_amdgcn_readfirstlane(tile_base[e]);
        TileInfo info;
        info.expert = e;
        info.nt = local / m_tiles;
        const int m0 = (local % m_tiles) * kBM;
        info.row0 = row_begin + m0;
        info.valid = min(kBM, rows - m0);
        return info;
    };

    // ---- copy cursor -------------------------------------------------------------------------------
    // copy i of wave w fills LDS rows i*32 + w*8 + lane/8; chunk (lane%8) ^ ((row>>1)&7) of the 128-byte row
    const int a_chunk = ((lane & 7) ^ ((wave * 4 + (lane >> 4)) & 7)) * 16;
    uint32_t a_off[2 * RT];  // lane offsets from p.a_codes: source row * K + chunk
    const uint8_t* sa_src;
    uint32_t b_off[4];       // lane offsets from the tile's first weight fragment
    const uint8_t* b_base = p.w;
    const uint8_t* sb_src;
    const int* index_src = p.row_to_route;
    int copy_tile = first, copy_kt = 0, copy_stage = 0, copy_span = -1, copy_ordinal = 0;
    const int scale_bytes = p.k / 32;  // per row
    const int spans = (ktiles + 3) / 4;
    TileInfo next_info = decode(first);

    // Tile number j of this workgroup keeps its gather indices in tile_index[j & 1].
    auto point_at_tile = [&](const TileInfo& info) {
        const int* index = tile_index[copy_ordinal & 1];
        // rows past the tile's end repeat its last row
#pragma unroll
        for (int i = 0; i < 2 * RT; ++i) {
            const int r = min(i * 32 + wave * 8 + (lane >> 3), info.valid - 1);
            // (clamped: a map left incomplete by a layout launch that ran out of time must not become a wild address)
            const int src = kGather ? min(max(index[r] / p.topk, 0), p.a_rows - 1) : info.row0 + r;
            a_off[i] = static_cast<uint32_t>(src) * static_cast<uint32_t>(p.k) + a_chunk;
        }
        {
            // thread t serves row t % kBM (surplus waves repeat rows, which keeps every wave's copy count equal)
            const int r = min(tid % kBM, info.valid - 1);
            const int src = kGather ? min(max(index[r] / p.topk, 0), p.a_rows - 1) : info.row0 + r;
            sa_src = p.a_scales + static_cast<size_t>(src) * scale_bytes;
        }
        const bool shared = info.expert >= p.num_routed;
        const size_t weight_index = shared ? info.expert - p.num_routed : info.expert;
        b_base = (shared ? p.w_shared : p.w) + weight_index * p.n * (p.k / 2) +
                 static_cast<size_t>(info.nt) * ktiles * 16384;
        // fragment q = copy*4 + wave of the 16 (column tile, k step) fragments of one k tile
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int q = j * 4 + wave;
            b_off[j] = static_cast<uint32_t>(q * 1024 + lane * 16);
        }
        sb_src = (shared ? p.ws_shared : p.ws) + (weight_index * n_tiles + info.nt) * spans * Cfg::kColScaleSlot + tid * 16;
    };
    auto aim_index_prefetch = [&](const TileInfo& info) {
        if (kGather) index_src = p.row_to_route + info.row0 + min(tid, info.valid - 1);
    };

    // Copy number c (compile-time) of the item under the copy cursor; the pieces are issued between MFMAs.
    auto issue_copy = [&](int c) {
        const uint32_t stage = lds0 + copy_stage * kStageBytes;
        if (c < 2 * RT)
            copy16_to_lds(p.a_codes + static_cast<size_t>(copy_kt) * kBK, a_off[c], stage + Cfg::kOffA + c * 4096 + wave * 1024);
        else
            copy16_weights_to_lds<RT == 1>(b_base + static_cast<size_t>(copy_kt) * 16384, b_off[c - 2 * RT],
                          stage + Cfg::kOffB + ((c - 2 * RT) * 4 + wave) * 1024);
    };
    // Every fourth item starts a new span: a 16-byte window of row scales per row (clamped so that it never
    // leaves the row: k % 512 may be 256) and the span's 4 KiB of column scales.  A tile's first item also
    // fetches the gather indices of the workgroup's next tile.  These extra copies only make the counted
    // waits stricter.
    auto issue_span_copies = [&]() {
        if ((copy_kt & 3) == 0) copy_span = copy_span + 1 == Cfg::kScaleSlots ? 0 : copy_span + 1;
        const int window = min((copy_kt & ~3) * 4, scale_bytes - 16);
        const int slot = copy_span;
        copy16_to_lds_unless(sa_src + window, lds0 + Cfg::kOffRowScales + slot * Cfg::kRowScaleSlot + ((wave * 64) % kBM) * 16,
                             copy_kt & 3);
        copy16_to_lds_unless(sb_src + static_cast<size_t>(copy_kt >> 2) * Cfg::kColScaleSlot,
                             lds0 + Cfg::kOffColScales + slot * Cfg::kColScaleSlot + wave * 1024, copy_kt & 3);
        if (kGather) copy4_to_lds_unless(index_src, lds_index + ((copy_ordinal + 1) & 1) * (kGemmThreads * 4) + wave * 256, copy_kt);
    };
    // The cursor moves on after an item's copies: the next ring stage (advance_copy_stage), then the next k tile or tile.
    auto finish_copy_cursor = [&](bool in_prologue = false) {
        if (++copy_kt == ktiles) {
            if (copy_tile + stride < total_tiles) {
                // The next tile's indices were fetched with this tile's first item, so switching needs no global
                // load; they have landed unless the tile is too short for any counted wait to have covered that
                // fetch (gemm_schedule.h), in which case the cursor lets everything land first.
                if (kGather && switch_needs_drain(in_prologue, ktiles, kAhead)) wait_copies_then_barrier<0>();
                copy_tile += stride;
                copy_kt = 0;
                ++copy_ordinal;
                point_at_tile(next_info);
                if (copy_tile + stride < total_tiles) next_info = decode(copy_tile + stride);
                aim_index_prefetch(next_info);
            } else {
                copy_kt = ktiles - 1;  // past the last tile: keep re-copying its last item (never read)
            }
        }
    };
    auto advance_copy_cursor = [&](bool in_prologue) {
        copy_stage = copy_stage + 1 == kStages ? 0 : copy_stage + 1;
        finish_copy_cursor(in_prologue);
    };
    auto issue_item = [&]() {
#pragma unroll
        for (int c = 0; c < Cfg::kCopies; ++c) issue_copy(c);
        issue_span_copies();
        advance_copy_cursor(true);
    };

    // First tile: fetch its gather indices synchronously, then aim the prefetch at the second tile.
    if (kGather) {
        aim_index_prefetch(next_info);
        copy4_to_lds(index_src, lds_index + wave * 256);
        wait_copies_then_barrier<0>();
    }
    point_at_tile(next_info);
    if (first + stride < total_tiles) next_info = decode(first + stride);
    aim_index_prefetch(next_info);

    // ---- fragment addresses inside a stage ---------------------------------------------------------
    // Row tile i of a lane sits 32 rows = 4096 bytes below row tile 0 and has the same swizzle (32 rows is a multiple
    // of the swizzle period), so one set of lane addresses serves all row tiles with compile-time offsets.
    int a_addr[2][2];  // [k step][lo/hi 16 bytes] of row tile 0
    const int row_in_wave = wm * 32 * RT + lr;
    {
        const int sw = (row_in_wave >> 1) & 7;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            a_addr[kb][0] = Cfg::kOffA + row_in_wave * kBK + (((kb * 4 + g) ^ sw) << 4);
            a_addr[kb][1] = Cfg::kOffA + row_in_wave * kBK + (((kb * 4 + 2 + g) ^ sw) << 4);
        }
    }
    const int sa_addr = Cfg::kOffRowScales + row_in_wave * 16;  // row tile i: + i * 512
    const int b_addr = Cfg::kOffB + wn * kCT * 2048 + lane * 16;
    const int sb_addr = Cfg::kOffColScales + wn * kCT * 512 + lane * 8;

    v8i afrag[2][RT];     // [k step][row tile]
    u32x4 bfrag[2][kCT];  // [k step][column tile]
    int ascale[2][RT];    // [item parity][row tile]
    int bscale[2][kCT];
    // Fragment reads of one k step come in kGroups pieces (row tiles first, then column tiles) so that they can
    // be dealt out between MFMAs; the scale reads of an item likewise.
    constexpr int kGroups = RT + kCT;
    auto read_group = [&](int stage_index, int kb, int group) {
        const uint8_t* stage = lds + stage_index * kStageBytes;
        if (group < RT) {
            const int i = group;
            const u32x4 lo = *reinterpret_cast<const u32x4*>(stage + a_addr[kb][0] + i * (32 * kBK));
            const u32x4 hi = *reinterpret_cast<const u32x4*>(stage + a_addr[kb][1] + i * (32 * kBK));
            afrag[kb][i] = v8i{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
        } else {
            const int c = group - RT;
            bfrag[kb][c] = *reinterpret_cast<const u32x4*>(stage + b_addr + (c * 2 + kb) * 1024);
        }
    };
    // row_at / col_at = byte offsets of the item's scales: ring slot + position inside the span
    auto read_scale_group = [&](int slot, int row_at, int col_at, int group) {
        if (group < RT)
            ascale[slot][group] = static_cast<int>(*reinterpret_cast<const uint32_t*>(lds + sa_addr + group * 512 + row_at));
        else
            bscale[slot][group - RT] =
                static_cast<int>(*reinterpret_cast<const uint16_t*>(lds + sb_addr + (group - RT) * 512 + col_at));
    };

    v16f acc[RT][kCT];
    auto clear_acc = [&]() {
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int c = 0; c < kCT; ++c)
#pragma unroll
                for (int j = 0; j < 16; ++j) acc[i][c][j] = 0.0f;
    };
    // The row-scale word holds the four k blocks of the k tile; the upper lane half owns the odd ones
    // (shifted at use, not at the read, so that the read does not have to be waited for early).
    constexpr int kMfmas = RT * kCT;  // per k step
    int ashift[2][RT];  // row scale word moved so that this lane half's first k block is byte 0
    auto mfma_one = [&](int kb, int slot, int n) {
        const int c = n / RT, i = n % RT;
        if (kb == 0) mfma_fp8_fp4<false>(acc[i][c], afrag[0][i], bfrag[0][c], ashift[slot][i], bscale[slot][c]);
        else mfma_fp8_fp4<true>(acc[i][c], afrag[1][i], bfrag[1][c], ashift[slot][i], bscale[slot][c]);
    };
    auto shift_scales = [&](int slot) {
#pragma unroll
        for (int i = 0; i < RT; ++i) ashift[slot][i] = ascale[slot][i] >> (8 * g);
    };

    // ---- epilogue of one tile (per-wave staging region, no workgroup synchronisation) ----------------
    uint8_t* region = lds + Cfg::kOffStaging + wave * Cfg::kStagingWave;
    auto epilogue = [&](const TileInfo& info) {
        constexpr int kPasses = kGateUp ? kCT / 2 : kCT;
        // The staging region holds one 32 x 32 tile as BF16 rows.
#pragma unroll
        for (int i = 0; i < RT; ++i) {
            // The last row tile of the epilogue is about what a filler needs to finish the row it is on: tell them to
            // stop (the first workgroup to get here does; the others are at most a few microseconds behind).
            if (i == RT - 1 && fillers != 0 && tid == 0)
                __hip_atomic_fetch_add(p.fill_stop, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const int tile_rows = min(32, info.valid - wm * 32 * RT - 32 * i);  // may be <= 0
            const size_t out_row0 = static_cast<size_t>(info.row0) + wm * 32 * RT + 32 * i;
#pragma unroll
            for (int pass = 0; pass < kPasses; ++pass) {
#pragma unroll
                for (int j = 0; j < 16; j += 2) {
                    float value[2];
#pragma unroll
                    for (int d = 0; d < 2; ++d) {
                        if (kGateUp) {
                            // column tiles alternate gate / up for the same 32 activation columns
                            const uint32_t rounded = pack_bf16x2(acc[i][2 * pass][j + d], acc[i][2 * pass + 1][j + d]);
                            value[d] = silu_mul(__uint_as_float(rounded << 16), __uint_as_float(rounded & 0xffff0000u));
                        } else {
                            value[d] = acc[i][pass][j + d];
                        }
                    }
                    const uint32_t pair = pack_bf16x2(value[0], value[1]);  // rows r and r + 1 of this lane's column
                    const int r = (j >> 2) * 8 + g * 4 + (j & 3);
                    uint8_t* cell = region + r * kStagingRowStride + lr * 2;
                    *reinterpret_cast<uint16_t*>(cell) = static_cast<uint16_t>(pair);
                    *reinterpret_cast<uint16_t*>(cell + kStagingRowStride) = static_cast<uint16_t>(pair >> 16);
                }
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                if (kGateUp) {
                    // two lanes requantise one row: 2 x 16 BF16 -> e8m0 byte + 32 e4m3 codes
                    const int act_width = p.n / 2;
                    const int act_col = (info.nt * kCT + wn * (kCT / 2) + pass) * 32;
                    const int r = lane >> 1, half = lane & 1;
                    float v[16];
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        const u32x4 raw = *reinterpret_cast<const u32x4*>(region + r * kStagingRowStride + half * 32 + q * 16);
#pragma unroll
                        for (int t = 0; t < 4; ++t) {
                            v[q * 8 + 2 * t] = bf16_to_f32(raw[t] & 0xffffu);
                            v[q * 8 + 2 * t + 1] = bf16_to_f32(raw[t] >> 16);
                        }
                    }
                    float amax = 0.0f;
#pragma unroll
                    for (int t = 0; t < 16; ++t) amax = fmaxf(amax, fabsf(v[t]));
                    amax = fmaxf(amax, __shfl_xor(amax, 1));
                    const int byte = mx_scale_byte(amax);
                    u32x4 codes;
#pragma unroll
                    for (int t = 0; t < 4; ++t)
                        codes[t] = mx_pack4(mx_scaled(v[4 * t], byte), mx_scaled(v[4 * t + 1], byte),
                                              mx_scaled(v[4 * t + 2], byte), mx_scaled(v[4 * t + 3], byte));
                    if (r < tile_rows) {
                        *reinterpret_cast<u32x4*>(p.act_codes + (out_row0 + r) * act_width + act_col + half * 16) = codes;
                        if (half == 0)
                            p.act_scales[(out_row0 + r) * (act_width / 32) + (act_col >> 5)] = static_cast<uint8_t>(byte);
                    }
                } else {
                    // 4 lanes carry one 64-byte row segment
                    const int col = info.nt * kBN + (wn * kCT + pass) * 32 + (lane & 3) * 8;
#pragma unroll
                    for (int it = 0; it < 2; ++it) {
                        const int r = it * 16 + (lane >> 2);
                        if (r < tile_rows && col < p.out_cols) {
                            const u32x4 chunk = *reinterpret_cast<const u32x4*>(region + r * kStagingRowStride + (lane & 3) * 16);
                            // cached store: the weighted reduce that follows reads these rows back at once
                            *reinterpret_cast<u32x4*>(p.out + (out_row0 + r) * p.out_cols + col) = chunk;
                        }
                    }
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                __builtin_amdgcn_wave_barrier();
            }
        }
    };

    // ---- the flat item stream --------------------------------------------------------------------------
#pragma unroll
    for (int j = 0; j < kAhead; ++j) issue_item();
    wait_copies_then_barrier<(kAhead - 1) * Cfg::kCopies>();  // item 0 has landed
    // Scale bookkeeping of the item whose fragments are read next: span counter (ring slot) and k tile.
    int read_span = -1, read_kt = 0;
    int row_at = 0, col_at = 0;
    auto next_scale_offsets = [&]() {
        if ((read_kt & 3) == 0) read_span = read_span + 1 == Cfg::kScaleSlots ? 0 : read_span + 1;
        const int window = min((read_kt & ~3) * 4, scale_bytes - 16);
        const int ring = read_span;
        row_at = ring * Cfg::kRowScaleSlot + (read_kt * 4 - window);
        col_at = ring * Cfg::kColScaleSlot + (read_kt & 3) * 2;
        read_kt = read_kt + 1 == ktiles ? 0 : read_kt + 1;
    };
    next_scale_offsets();
#pragma unroll
    for (int group = 0; group < kGroups; ++group) {
        read_scale_group(0, row_at, col_at, group);
        read_group(0, 0, group);
    }
    clear_acc();
    asm volatile("s_nop 3");
    int stage_now = 0;  // stage of the item whose MFMAs run
    int tile = first, kt = 0;
    TileInfo info = decode(first);
    const long long total_items = static_cast<long long>(my_tiles) * ktiles;
    for (long long item = 0; item < total_items; item += 2) {
#pragma unroll
        for (int parity = 0; parity < 2; ++parity) {  // ktiles is even, so tiles start on even items
            const int stage_next = stage_now + 1 == kStages ? 0 : stage_now + 1;
            // A wave issues in order and owns its SIMD alone, so whatever is not an MFMA should sit in the
            // shadow of one.  First k step: its MFMAs are followed, one piece each, by the LDS reads of the
            // second k step's fragments and, once the barrier has passed, by the copies of the item kAhead
            // ahead.  Second k step: the remaining copies in its first half, then the item's scale / index copies and
            // the copy cursor's arithmetic, and all along the reads of the next item's scales and first fragments
            // (whose registers the first k step has released).
            shift_scales(parity);
            constexpr int kSlots = kMfmas;  // MFMAs behind the barrier that deal out the item's copies
            // enough read groups per MFMA that the second k step's fragments have all left LDS before the barrier
            constexpr int kReadsPerMfma = (kGroups + kMfmas / 2 - 1) / (kMfmas / 2);
#pragma unroll
            for (int n = 0; n < kMfmas; ++n) {
                mfma_one(0, parity, n);
#pragma unroll
                for (int group = kReadsPerMfma * n; group < kReadsPerMfma * (n + 1); ++group)
                    if (group < kGroups) read_group(stage_now, 1, group);
                if (n == kMfmas / 2 - 1) {
                    // item+1 has landed for every thread once each has at most kAhead-2 items of its own copies
                    // in flight; past the barrier every wave has also finished reading the stage refilled next.
                    wait_copies_then_barrier<Cfg::kWaitPlain>();
                }
                if (n >= kMfmas / 2) {
                    const int slot = n - kMfmas / 2;
#pragma unroll
                    for (int c = slot * Cfg::kCopies / kSlots; c < (slot + 1) * Cfg::kCopies / kSlots; ++c) issue_copy(c);
                }
            }
            next_scale_offsets();
#pragma unroll
            for (int n = 0; n < kMfmas; ++n) {
                mfma_one(1, parity, n);
                const int slot = n + kMfmas / 2;
                if (slot < kSlots) {
#pragma unroll
                    for (int c = slot * Cfg::kCopies / kSlots; c < (slot + 1) * Cfg::kCopies / kSlots; ++c) issue_copy(c);
                }
                // 2*kGroups read pieces for the next item: its scales first (they are shifted first), then fragments
#pragma unroll
                for (int piece = n * 2 * kGroups / kMfmas; piece < (n + 1) * 2 * kGroups / kMfmas; ++piece) {
                    if (piece < kGroups) read_scale_group(parity ^ 1, row_at, col_at, piece);
                    else read_group(stage_next, 0, piece - kGroups);
                }
                if (n == kMfmas / 2) {
                    // Every regular copy of the item is out: its scale / index copies and the cursor's stage arithmetic go
                    // under the remaining MFMAs instead of behind the last one, where the matrix pipe would drain
                    // meanwhile (45 scalar instructions used to sit there).  The counted waits only get stricter by it.
                    issue_span_copies();
                    copy_stage = copy_stage + 1 == kStages ? 0 : copy_stage + 1;
                    asm volatile("" : "+s"(copy_stage));  // computed here, not sunk to the end of the item
                }
            }
            finish_copy_cursor();
            stage_now = stage_next;
        }
        kt += 2;
        // (marked unlikely: the register allocator then keeps the loop's values in place and does its shuffling around the
        // epilogue, once per tile, instead of at the head of the item loop)
        if (__builtin_expect(kt == ktiles, 0)) {
                    settle_accumulators();
            // tie every accumulator to a statement behind the wait, so that no read of it can be moved above
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int c = 0; c < kCT; ++c) asm volatile("" : "+a"(acc[i][c]));
            epilogue(info);
                    clear_acc();
            asm volatile("s_nop 3");  // accumulator writes settle before the next MFMA reads them
            kt = 0;
            tile += stride;
            if (tile < total_tiles) info = decode(tile);
        }
    }
    // No copy may still be in flight into this workgroup's LDS when it retires.
    wait_copies_then_barrier<0>();
}

// =====================================================================================================
// Grouped GEMM, column-wave form: the weights go straight from memory to registers
// =====================================================================================================
// The prepared weight layout already is the per-lane B operand of the scaled MFMA, so a wave that owns whole
// 32-column tiles can load its weight fragments with plain 16-byte loads and never share them.  Here the four waves
// split the tile's 256 columns (64 each: two column tiles; for the first GEMM one gate / up pair) and every wave covers
// ALL the tile's rows (2 * RT row tiles of 32): the same RT * 4 accumulator tiles per wave as the 2 x 2 form, but the
// weights need no LDS write, no LDS read and no barrier, and the LDS ring holds activations only (8 KiB * RT per
// stage), which buys a fourth stage at 192 rows.  The ring has exactly as many stages as the item loop is unrolled
// (4): an item's stage, its weight registers and the selection of its scale bytes are all compile-time constants,
// the LDS target of a copy is one scalar add away from a per-wave base, and a tile ends only behind the fourth body
// (k is a multiple of 512 here).  Everything of item i + 4 is requested in the body of item i, so the one counted wait
// per item lets two whole items of copies and loads stay in flight.
// The weight fragments of the four items in flight live in the 64 accumulation registers behind the accumulators (a[192:255]
// at 192 rows), which the loads and the
// MFMAs name themselves: the compiler never sees them as values.  It could not be trusted with them: a register that
// an asynchronous load has been told to fill counts as defined right behind the load, and a register allocator that moves
// such a value (it parked weight fragments in spare registers when they were ordinary operands) copies what the register
// held BEFORE the load landed.  Every weight load declares all 64 clobbered, so nothing the compiler keeps alive in
// the loop can sit there (the accumulators end up below); that it also puts no short-lived value
// there is checked on the generated code by tests/test_gemm_registers.py.  Column scales travel through LDS like the row
// scales (each wave copies and reads only the 1 KiB of its own two column tiles).
template <int RT>
struct ColCfg : ColumnRing<RT> {
    using ColumnRing<RT>::kStages;                     // LDS stages = items the requests run ahead = unroll of the item loop
    static constexpr int kBM = 64 * RT;
    static constexpr int kRowTiles = 2 * RT;           // 32-row MFMA tiles per workgroup tile, all of them on every wave
    static constexpr int kColTiles = 2;                // 32-column MFMA tiles per wave
    static constexpr int kStageBytes = kBM * kBK;      // activations only
    static constexpr int kRowScaleSlot = kBM * 16;
    static constexpr int kOffRowScales = kStages * kStageBytes;
    static constexpr int kColScaleSlot = 4096;
    static constexpr int kOffColScales = kOffRowScales + 2 * kRowScaleSlot;
    static constexpr int kLdsBytes = kOffColScales + 2 * kColScaleSlot;
    static_assert(ColumnRing<RT>::kRequests == kRowTiles + 2 * kColTiles, "per thread and item: activation copies + weight loads");
    // 64-row tiles leave room (200 registers per lane, 53 KiB of LDS) for two workgroups on a CU: launches of that height are
    // bound by streaming their weights, and a second workgroup doubles the requests in flight
    static constexpr int kWorkgroupsPerCu = RT == 1 ? 2 : 1;
    static constexpr int kWeightRegs = 64 * RT;  // first of the 64 accumulation registers that hold weight fragments: right behind the accumulators
};

// Asynchronous 16-byte copy global -> LDS whose LDS address is a per-wave base (SGPR) plus a compile-time constant.
template <int kLdsConst>
__device__ __forceinline__ void copy16_to_lds_at(const void* uniform_base, uint32_t lane_offset, uint32_t wave_lds_base)
{
    asm volatile("s_add_u32 m0, %0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3" ::"s"(wave_lds_base), "n"(kLdsConst),
                 "v"(lane_offset), "s"(uniform_base)
                 : "memory", "scc");
}
// The 64 registers of the weight fragments, as clobber lists: they follow the accumulators (64 * RT registers), so that a
// kernel with few accumulators also needs few registers in all.
#define DPEP_WEIGHT_REGS_64 \
    "a64", "a65", "a66", "a67", "a68", "a69", "a70", "a71", "a72", "a73", "a74", "a75", "a76", "a77", "a78", "a79",    \
        "a80", "a81", "a82", "a83", "a84", "a85", "a86", "a87", "a88", "a89", "a90", "a91", "a92", "a93", "a94",       \
        "a95", "a96", "a97", "a98", "a99", "a100", "a101", "a102", "a103", "a104", "a105", "a106", "a107", "a108",     \
        "a109", "a110", "a111", "a112", "a113", "a114", "a115", "a116", "a117", "a118", "a119", "a120", "a121",        \
        "a122", "a123", "a124", "a125", "a126", "a127"
#define DPEP_WEIGHT_REGS_128 \
    "a128", "a129", "a130", "a131", "a132", "a133", "a134", "a135", "a136", "a137", "a138", "a139", "a140", "a141",    \
        "a142", "a143", "a144", "a145", "a146", "a147", "a148", "a149", "a150", "a151", "a152", "a153", "a154",        \
        "a155", "a156", "a157", "a158", "a159", "a160", "a161", "a162", "a163", "a164", "a165", "a166", "a167",        \
        "a168", "a169", "a170", "a171", "a172", "a173", "a174", "a175", "a176", "a177", "a178", "a179", "a180",        \
        "a181", "a182", "a183", "a184", "a185", "a186", "a187", "a188", "a189", "a190", "a191"
#define DPEP_WEIGHT_REGS_V192 \
    "v192", "v193", "v194", "v195", "v196", "v197", "v198", "v199", "v200", "v201", "v202", "v203", "v204", "v205",    \
        "v206", "v207", "v208", "v209", "v210", "v211", "v212", "v213", "v214", "v215", "v216", "v217", "v218",        \
        "v219", "v220", "v221", "v222", "v223", "v224", "v225", "v226", "v227", "v228", "v229", "v230", "v231",        \
        "v232", "v233", "v234", "v235", "v236", "v237", "v238", "v239", "v240", "v241", "v242", "v243", "v244",        \
        "v245", "v246", "v247", "v248", "v249", "v250", "v251", "v252", "v253", "v254", "v255"
// Asynchronous 16-byte load into the weight registers kReg .. kReg + 3.  Nothing is an output as far as the compiler knows.
// kFirst: the first of the kernel's 64 weight registers (all of them are declared clobbered, whichever four are loaded).
// At 64 and 128 rows they are accumulation registers right behind the accumulators (a64.. / a128..); at 192 rows, where the
// accumulators fill 192 of the 256 accumulation registers, they are the ordinary registers v192..v255 (the kernel's own
// values need fewer than 150, and with every accumulation register taken the register allocator started to put
// loop-carried values on the stack).
#define DPEP_WEIGHT_LOAD(file, hint, clobbers)                                                                                  \
    asm volatile("global_load_dwordx4 " file "[%3:%4], %0, %1 offset:%2 " hint ::"v"(lane_offset), "s"(uniform_base), "n"(kImm), \
                 "n"(kReg), "n"(kReg + 3)                                                                                       \
                 : "memory", clobbers)
template <int kFirst, int kReg, int kImm, bool kStreamed>
__device__ __forceinline__ void load16_to_weight_regs(const void* uniform_base, uint32_t lane_offset)
{
    static_assert(kFirst == 64 || kFirst == 128 || kFirst == 192, "weight registers start at a64, a128 or a192");
    static_assert(kReg >= kFirst && kReg + 3 < kFirst + 64, "not one of the kernel's weight registers");
    if constexpr (kFirst == 64) {
        if (kStreamed) DPEP_WEIGHT_LOAD("a", "nt", DPEP_WEIGHT_REGS_64);
        else DPEP_WEIGHT_LOAD("a", "sc1", DPEP_WEIGHT_REGS_64);
    } else if constexpr (kFirst == 128) {
        if (kStreamed) DPEP_WEIGHT_LOAD("a", "nt", DPEP_WEIGHT_REGS_128);
        else DPEP_WEIGHT_LOAD("a", "sc1", DPEP_WEIGHT_REGS_128);
    } else {
        if (kStreamed) DPEP_WEIGHT_LOAD("v", "nt", DPEP_WEIGHT_REGS_V192);
        else DPEP_WEIGHT_LOAD("v", "sc1", DPEP_WEIGHT_REGS_V192);
    }
}
// Scaled MFMA with the operands the other way round: the weights (FP4, a[kReg : kReg + 3]) are the instruction's A
// operand and the activations (FP8) its B operand, so the result comes out transposed: lane l holds activation row
// l % 32, and acc[j] is weight column (j/4)*8 + (l/32)*4 + j%4 of the tile: four consecutive columns per group of
// four registers.  A lane's results are then pieces of ONE output row, which the epilogue can store from registers (the
// other way round a lane holds sixteen rows of one column, and the tile has to be transposed through LDS).  The scale bytes
// are chosen at compile time: byte kByteW of scale_w, byte kByteX of scale_x.
template <int kReg, int kByteW, int kByteX>
__device__ __forceinline__ void mfma_fp4_fp8_regs(v16f& acc, const v8i& x, int scale_w, int scale_x)
{
    if constexpr (kReg >= 192)  // (192-row kernels keep their weights in v192..v255, the others behind their accumulators)
        asm volatile("v_mfma_scale_f32_32x32x64_f8f6f4 %0, v[%8:%9], %1, %0, %2, %3 op_sel:[%4,%5,0] op_sel_hi:[%6,%7,0] cbsz:4"
                     : "+a"(acc)
                     : "v"(x), "v"(scale_w), "v"(scale_x), "n"(kByteW & 1), "n"(kByteX & 1), "n"(kByteW >> 1), "n"(kByteX >> 1),
                       "n"(kReg), "n"(kReg + 3));
    else
        asm volatile("v_mfma_scale_f32_32x32x64_f8f6f4 %0, a[%8:%9], %1, %0, %2, %3 op_sel:[%4,%5,0] op_sel_hi:[%6,%7,0] cbsz:4"
                     : "+a"(acc)
                     : "v"(x), "v"(scale_w), "v"(scale_x), "n"(kByteW & 1), "n"(kByteX & 1), "n"(kByteW >> 1), "n"(kByteX >> 1),
                       "n"(kReg), "n"(kReg + 3));
}

// ---- epilogue pieces: a 32-row tile straight from the accumulators -------------------------------------------------------
// With the weights as the instruction's A operand a lane holds, for its row, columns q*8 + g*4 .. + 3 (q = 0..3) of a column
// tile, its partner lane (l ^ 32) the four columns in between.  Two register swaps between the lane halves give the lower lane
// columns 0..15 and the upper lane columns 16..31 of the row as consecutive bytes, which leave as 16-byte stores.
__device__ __forceinline__ void swap_halves(uint32_t lower_q, uint32_t upper_q, uint32_t (&out)[2])
{
    // lanes 0..31 get (their own lower_q, the partner's lower_q), lanes 32..63 (the partner's upper_q, their own upper_q)
    const auto swapped = __builtin_amdgcn_permlane32_swap(lower_q, upper_q, false, false);
    out[0] = swapped[0];
    out[1] = swapped[1];
}
// First GEMM: gate and up columns act_col .. act_col + 31 of one row -> SwiGLU -> one MXFP8 block.  pairs(j): columns j and j + 1 of
// both as BF16 pairs.
template <typename Pairs>
__device__ __forceinline__ void store_gate_up_pairs(const GemmParams& p, Pairs&& pairs, size_t row, bool row_exists, int act_col, int g)
{
    float v[16];
    float amax = 0.0f;
    static_for<8>([&](auto pair_constant) {
        constexpr int j = 2 * decltype(pair_constant)::value;
        const u32x2 both = pairs(std::integral_constant<int, j>{});
        const uint32_t gate = both[0], up = both[1];
        const uint32_t act = pack_bf16x2(silu_mul(__uint_as_float(gate << 16), __uint_as_float(up << 16)),
                                         silu_mul(__uint_as_float(gate & 0xffff0000u), __uint_as_float(up & 0xffff0000u)));
        v[j] = bf16_to_f32(act & 0xffffu);
        v[j + 1] = bf16_to_f32(act >> 16);
        amax = fmaxf(amax, fmaxf(fabsf(v[j]), fabsf(v[j + 1])));
    });
    amax = fmaxf(amax, __shfl_xor(amax, 32));  // the row's other sixteen columns
    const int byte = mx_scale_byte(amax);
    uint32_t code[4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
        code[q] = mx_pack4(mx_scaled(v[4 * q], byte), mx_scaled(v[4 * q + 1], byte), mx_scaled(v[4 * q + 2], byte), mx_scaled(v[4 * q + 3], byte));
    uint32_t first[2], second[2];
    swap_halves(code[0], code[2], first);
    swap_halves(code[1], code[3], second);
    const u32x4 codes = {first[0], first[1], second[0], second[1]};
    const int act_width = p.n / 2;
    if (row_exists) {
        *reinterpret_cast<u32x4*>(p.act_codes + row * act_width + act_col + g * 16) = codes;
        if (g == 0) p.act_scales[row * (act_width / 32) + (act_col >> 5)] = static_cast<uint8_t>(byte);
    }
}
__device__ __forceinline__ void store_gate_up(const GemmParams& p, const v16f& gates, const v16f& ups, size_t row, bool row_exists, int act_col, int g)
{
    store_gate_up_pairs(p, [&](auto at) {
        constexpr int j = decltype(at)::value;
        return u32x2{pack_bf16x2(gates[j], gates[j + 1]), pack_bf16x2(ups[j], ups[j + 1])};
    }, row, row_exists, act_col, g);
}
// Second GEMM: columns col0 .. col0 + 31 of one row as BF16.
__device__ __forceinline__ void store_output(const GemmParams& p, const v16f& acc, size_t row, bool row_exists, int col0, int g)
{
    uint32_t pairs[4][2];  // [q][columns +0,1 | +2,3]
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        pairs[q][0] = pack_bf16x2(acc[4 * q], acc[4 * q + 1]);
        pairs[q][1] = pack_bf16x2(acc[4 * q + 2], acc[4 * q + 3]);
    }
    uint32_t s00[2], s01[2], s10[2], s11[2];
    swap_halves(pairs[0][0], pairs[2][0], s00);
    swap_halves(pairs[0][1], pairs[2][1], s01);
    swap_halves(pairs[1][0], pairs[3][0], s10);
    swap_halves(pairs[1][1], pairs[3][1], s11);
    const u32x4 lower = {s00[0], s01[0], s00[1], s01[1]}, upper = {s10[0], s11[0], s10[1], s11[1]};
    const int col = col0 + g * 16;
    if (row_exists) {
        // cached stores: the weighted reduce that follows reads these rows back at once
        if (col < p.out_cols) *reinterpret_cast<u32x4*>(p.out + row * p.out_cols + col) = lower;
        if (col + 8 < p.out_cols) *reinterpret_cast<u32x4*>(p.out + row * p.out_cols + col + 8) = upper;
    }
}

// One-wave workgroups that fill stand in front of those with tiles: a filler has to start before a tile can end, or it would find the
// counter raised already.  (A multiple of 8 of them, so that the tiles keep their XCDs.)
__device__ __forceinline__ bool fill_of_few_rows(const GemmParams& p)
{
    if (blockIdx.x == 0 && threadIdx.x == 0 && p.fill_state != nullptr) p.fill_state[0] = p.few_rows_fillers;
    if (static_cast<int>(blockIdx.x) >= p.few_rows_fillers) return false;
    fill_zero_rows(p, static_cast<int>(blockIdx.x), p.few_rows_fillers, static_cast<int>(threadIdx.x));
    return true;
}

// The 32-row tiles of the few-rows kernels.  They are numbered through the experts, so that the grid does not depend on how the
// routes fell; every wave works the numbering out for itself (a lane has experts lane and lane + 64).
struct FewRowsTiles {
    static constexpr int kRows = 32;
    int through[2], first_row[2], rows[2];
    int total;
    __device__ __forceinline__ FewRowsTiles(const GemmParams& p, int lane)
    {
        static_assert(kMaxMoeExperts <= 128, "two experts per lane");
        total = 0;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int e = lane + 64 * h;
            through[h] = first_row[h] = rows[h] = 0;
            if (64 * h >= p.num_local) continue;
            if (e < p.num_local) {
                first_row[h] = p.offsets[e];
                rows[h] = p.offsets[e + 1] - first_row[h];
            }
            through[h] = total + wave_scan((rows[h] + kRows - 1) / kRows);
            total = __builtin_amdgcn_readlane(through[h], 63);
        }
    }
    // Expert, first row and number of rows of row tile `unit` (below the total), from the lane that has the expert: its offsets asked
    // for again were a memory trip in front of everything else.
    __device__ __forceinline__ void find(const GemmParams& p, int unit, int& expert, int& row0, int& valid) const
    {
        expert = __popcll(__ballot(through[0] <= unit));  // experts that end at or before this row tile
        int before = 0;
        if (expert == 64) {
            expert += __popcll(__ballot(through[1] <= unit));
            before = expert == 64 ? __builtin_amdgcn_readlane(through[0], 63) : __builtin_amdgcn_readlane(through[1], expert - 65);
        } else if (expert > 0) {
            before = __builtin_amdgcn_readlane(through[0], expert - 1);
        }
        expert = min(expert, p.num_local - 1);
        const int in_expert = (unit - before) * kRows;
        row0 = (expert < 64 ? __builtin_amdgcn_readlane(first_row[0], expert) : __builtin_amdgcn_readlane(first_row[1], expert - 64)) + in_expert;
        valid = min(kRows, (expert < 64 ? __builtin_amdgcn_readlane(rows[0], expert) : __builtin_amdgcn_readlane(rows[1], expert - 64)) - in_expert);
    }
};

// =====================================================================================================
// Grouped GEMM for few rows per expert
// =====================================================================================================
// With fewer rows per expert than one row tile (a decode step, a small batch) the GEMM is the streaming of its weights: every
// weight byte is read once and used for one 32-row MFMA tile, and what counts is how many requests are in flight and that
// nothing else gets in their way.  A wave owns 64 columns (two column tiles; for the first GEMM a gate / up pair) and holds the
// weight fragments of the next four k tiles in registers; the four waves of a workgroup share the activations, each fetching
// one k tile of a span of four, through 32 KiB of LDS and one barrier per span (fetched by every wave for itself they cost as
// many L1 requests as the weights: first GEMM below 82 us instead of 79).  Two workgroups fit on a CU, nothing is persistent
// beyond the routing being worse than expected, and the hardware hands out the next workgroup when one ends.  The sums are
// taken in the same order as in the other kernels, so the results are the same bits.
// Measured on an MI355X, 32 of 256 experts of 7168 x 2048, 16 rows each: first GEMM 82 -> 79 us, second 53 -> 44 us; the bare
// reads of the same bytes, by as many waves with as many requests in flight, take 78 and 43 us (6.4 and 5.8 TB/s, the launch
// included).  Whole forward: 0.5 rows per expert 92 -> 62 us, 2: 134 -> 106, 8: 144 -> 130, 16: 153 -> 137.
// (Tried and not kept: eight k tiles ahead at one workgroup per CU, 143 us; 64-row tiles, 154 us.)
// kWaves = 1 spreads a column tile over four workgroups of one wave each, for launches that would leave CUs idle (below).
// k tiles and column tiles of nothing but padding are left out.
typedef u32x4 u32x4_unaligned __attribute__((aligned(4)));
template <int kWaves, bool kGateUp>
__global__ __launch_bounds__(64 * kWaves, 2) void grouped_gemm_few_rows_kernel(GemmParams p)
{
    constexpr bool kGather = kGateUp;
    constexpr int kRows = 32;
    __shared__ __attribute__((aligned(16))) uint8_t lds[2][4][kRows * kBK];  // [span parity][k tile of the span][row][128 bytes]
    const int lane = threadIdx.x & 63, g = lane >> 5, lr = lane & 31;
    const int my_wave = kWaves == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    constexpr int kSplit = kGemmWaves / kWaves;  // workgroups per column tile
    const int n_tiles = p.n / kBN, stored_ktiles = p.k / kBK, stored_spans = (stored_ktiles + 3) / 4, scale_bytes = p.k / 32;
    // (k tiles and column tiles of nothing but padding are left out)
    const int ktiles = (p.k_real + kBK - 1) / kBK, spans = (ktiles + 3) / 4, numbered_n_tiles = p.numbered_n_tiles;

    if constexpr (kWaves == 1) {
        if (fill_of_few_rows(p)) return;
    } else if (blockIdx.x == 0 && threadIdx.x == 0 && p.fill_state != nullptr) {
        p.fill_state[0] = 0;
    }
    const FewRowsTiles tiles(p, lane);
    const int fillers = kWaves == 1 ? p.few_rows_fillers : 0;
    for (int tile_id = static_cast<int>(blockIdx.x) - fillers; tile_id < tiles.total * numbered_n_tiles * kSplit;
         tile_id += static_cast<int>(gridDim.x) - fillers) {
        const int unit = tile_id / (numbered_n_tiles * kSplit), piece = tile_id - unit * (numbered_n_tiles * kSplit);
        const int nt = piece / kSplit, wave = kWaves == 1 ? piece % kSplit : my_wave;  // the column tile, the quarter of it
        if (nt >= p.live_n_tiles) continue;
        int expert, row0, valid;
        tiles.find(p, unit, expert, row0, valid);
        const bool shared = expert >= p.num_routed;
        const size_t weight_index = shared ? expert - p.num_routed : expert;
        const uint8_t* const w = (shared ? p.w_shared : p.w) + weight_index * p.n * (p.k / 2) + static_cast<size_t>(nt) * stored_ktiles * 16384 +
                                 wave * 4096 + lane * 16;
        const uint8_t* const ws = (shared ? p.ws_shared : p.ws) + (weight_index * n_tiles + nt) * stored_spans * 4096 + wave * 1024 + lane * 8;

        v16f acc[2];
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int j = 0; j < 16; ++j) acc[c][j] = 0.0f;
        // (clamped: a map left incomplete by a layout launch that ran out of time must not become a wild address)
        const uint8_t* const codes = kGather ? p.a_codes : p.a_codes + static_cast<size_t>(row0) * p.k;
        const uint8_t* const row_scale_bytes = kGather ? p.a_scales : p.a_scales + static_cast<size_t>(row0) * scale_bytes;
        auto source = [&](int r) {
            r = min(r, valid - 1);
            return static_cast<uint32_t>(kGather ? min(max(p.row_to_route[row0 + r] / p.topk, 0), p.a_rows - 1) : r);
        };
        u32x4 wreg[4][4];  // [k tile of the span][column tile * 2 + k step]
        auto load_weights = [&](int slot, int kt) {
            const uint8_t* at = w + static_cast<size_t>(min(kt, ktiles - 1)) * 16384;  // (past the end: the last k tile again, never used)
#pragma unroll
            for (int f = 0; f < 4; ++f) wreg[slot][f] = load16_nt(at + f * 1024);
        };
        // Activations: wave q fetches k tile q of a span for the whole workgroup.  Copy f: lane l asks for 16-byte chunk l % 8 of
        // row 8 f + l / 8, so that eight lanes read a row's 128 bytes.  Rows past the end repeat the last one.
        uint32_t a_from[4];
#pragma unroll
        for (int f = 0; f < 4; ++f) a_from[f] = source(8 * f + (lane >> 3)) * static_cast<uint32_t>(p.k) + (lane & 7) * 16;
        const uint32_t s_from = source(lr) * static_cast<uint32_t>(scale_bytes);
        u32x4 areg[4 / kWaves][4];
        auto load_activations = [&](int span) {
#pragma unroll
            for (int t = 0; t < 4 / kWaves; ++t) {
                const uint8_t* at = codes + static_cast<size_t>(min(span * 4 + my_wave + t, ktiles - 1)) * kBK;
#pragma unroll
                for (int f = 0; f < 4; ++f) areg[t][f] = load16(at + a_from[f]);
            }
        };
        const int put = (lane >> 3) * kBK + (((lane & 7) ^ (lane >> 3)) << 4);  // (row 8 f + i: + f * 1024, the same swizzle)
        auto hand_over = [&](int parity) {
#pragma unroll
            for (int t = 0; t < 4 / kWaves; ++t)
#pragma unroll
                for (int f = 0; f < 4; ++f) *reinterpret_cast<u32x4*>(&lds[parity][my_wave + t][put + f * 1024]) = areg[t][f];
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        };
        u32x4 row_scales[2];
        u32x2 col_scales[2][2];  // [span parity][column tile]
        auto load_scales = [&](int parity, int span) {
            span = min(span, spans - 1);
            row_scales[parity] = *reinterpret_cast<const u32x4_unaligned*>(row_scale_bytes + s_from + min(span * 16, scale_bytes - 16));
#pragma unroll
            for (int c = 0; c < 2; ++c)
                col_scales[parity][c] = *reinterpret_cast<const u32x2*>(ws + static_cast<size_t>(span) * 4096 + c * 512);
        };
        load_activations(0);
        load_scales(0, 0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < 4; ++q) load_weights(q, q);
        hand_over(0);
        auto span_body = [&](auto parity_constant, auto more_constant, int span) {
            constexpr int kParity = decltype(parity_constant)::value;
            constexpr bool kMore = decltype(more_constant)::value;  // another span follows
            if constexpr (kMore) {
                load_activations(span + 1);
                load_scales(kParity ^ 1, span + 1);
            }
            __builtin_amdgcn_sched_barrier(0);
            const bool shifted_window = span * 16 > scale_bytes - 16;  // (k % 512 = 256: the last span's bytes sit two words up)
            static_for<4>([&](auto q_constant) {
                constexpr int q = decltype(q_constant)::value;
                if (q == 0 || kMore || span * 4 + q < ktiles) {
                    const uint32_t word = q < 2 && !kMore && shifted_window ? row_scales[kParity][(q + 2) & 3] : row_scales[kParity][q];
                    const int x_scale = static_cast<int>(word >> (8 * g));
                    const uint8_t* const tile = &lds[kParity][q][lr * kBK];
                    static_for<2>([&](auto step_constant) {
                        constexpr int step = decltype(step_constant)::value;
                        const u32x4 lo = *reinterpret_cast<const u32x4*>(tile + (((step * 4 + g) ^ (lr & 7)) << 4));
                        const u32x4 hi = *reinterpret_cast<const u32x4*>(tile + (((step * 4 + 2 + g) ^ (lr & 7)) << 4));
                        const v8i x = {(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
#pragma unroll
                        for (int c = 0; c < 2; ++c) {
                            const u32x4 f = wreg[q][2 * c + step];
                            const v8i m = {(int)f[0], (int)f[1], (int)f[2], (int)f[3], 0, 0, 0, 0};
                            acc[c] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(m, x, acc[c], 4, 0, 2 * (q & 1) + step,
                                                                                     static_cast<int>(col_scales[kParity][c][q >> 1]), 2 * step, x_scale);
                        }
                    });
                    if constexpr (q == 3 || !kMore) settle_accumulators(acc);
                }
                if constexpr (kMore) load_weights(q, (span + 1) * 4 + q);
                __builtin_amdgcn_sched_barrier(0);
            });
            if constexpr (kMore) hand_over(kParity ^ 1);
        };
        constexpr std::integral_constant<int, 0> even{};
        constexpr std::integral_constant<int, 1> odd{};
        constexpr std::integral_constant<bool, true> more{};
        constexpr std::integral_constant<bool, false> last{};
        // (The first and the last spans stand outside the loop on purpose: the first one's operands were asked for in
        // another order, and the compiler's counted waits have to suit every way into a body, so that a shared body waited
        // for everything in flight; the last asks for nothing more.)
        if (spans > 1) {
            span_body(even, more, 0);
            int span = 1;
            for (; span + 2 < spans; span += 2) {
                span_body(odd, more, span);
                span_body(even, more, span + 1);
            }
            if (span + 1 < spans) {
                span_body(odd, more, span);
                span_body(even, last, span + 1);
            } else {
                span_body(odd, last, span);
            }
        } else {
            span_body(even, last, 0);
        }
        // the next tile of this workgroup writes the LDS again
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (kWaves == 1 && fillers != 0 && tile_id == 0 && threadIdx.x == 0) __hip_atomic_fetch_add(p.fill_stop, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const bool row_exists = lr < valid;
        const size_t row = static_cast<size_t>(row0) + lr;
        if (kGateUp) {
            store_gate_up(p, acc[0], acc[1], row, row_exists, (nt * (kBN / 64) + wave) * 32, g);
        } else {
#pragma unroll
            for (int c = 0; c < 2; ++c) store_output(p, acc[c], row, row_exists, nt * kBN + (wave * 2 + c) * 32, g);
        }
    }
}

// The same with one wave per workgroup and no LDS, for launches that leave most SIMDs idle or whose tiles hold few rows.  Such a wave has
// its SIMD to itself (up to 512 registers): activations go straight to registers as well, in the layout that the MFMA takes,
// eight k tiles of everything are in flight, and no LDS, barrier or wait for either stands between the MFMAs, which then bound
// the loop (0.13 us a k tile).  First GEMM, us: 40 tokens over 5 experts of 4032 x 640 12.9 -> 10.0, 2 x top-5 over 44 of 4864 x 1152
// 18.9 -> 14.4, 1 x top-7 over 18 + 2 of 1216 x 1536 8.7 -> 7.3.  An activation load then touches one line per row instead of eight
// rows' lines: with full tiles and several waves to a CU that is what bounds it (66 rows for each of 6 experts of 1280 x 1536 9.9 -> 12.1).
template <bool kGateUp>
__global__ __launch_bounds__(64, 1) void grouped_gemm_one_wave_kernel(GemmParams p)
{
    constexpr bool kGather = kGateUp;
    const int lane = threadIdx.x, g = lane >> 5, lr = lane & 31;
    constexpr int kSplit = kGemmWaves;  // workgroups per column tile
    const int n_tiles = p.n / kBN, stored_ktiles = p.k / kBK, stored_spans = (stored_ktiles + 3) / 4, scale_bytes = p.k / 32;
    // (k tiles and column tiles of nothing but padding are left out)
    const int ktiles = (p.k_real + kBK - 1) / kBK, spans = (ktiles + 3) / 4, numbered_n_tiles = p.numbered_n_tiles;

    if (fill_of_few_rows(p)) return;
    const FewRowsTiles tiles(p, lane);
    const int fillers = p.few_rows_fillers;
    for (int tile_id = static_cast<int>(blockIdx.x) - fillers; tile_id < tiles.total * numbered_n_tiles * kSplit;
         tile_id += static_cast<int>(gridDim.x) - fillers) {
        const int unit = tile_id / (numbered_n_tiles * kSplit), piece = tile_id - unit * (numbered_n_tiles * kSplit);
        const int nt = piece / kSplit, wave = piece % kSplit;  // the column tile, the quarter of it
        if (nt >= p.live_n_tiles) continue;
        int expert, row0, valid;
        tiles.find(p, unit, expert, row0, valid);
        const bool shared = expert >= p.num_routed;
        const size_t weight_index = shared ? expert - p.num_routed : expert;
        const uint8_t* const w = (shared ? p.w_shared : p.w) + weight_index * p.n * (p.k / 2) + static_cast<size_t>(nt) * stored_ktiles * 16384 +
                                 wave * 4096 + lane * 16;
        const uint8_t* const ws = (shared ? p.ws_shared : p.ws) + (weight_index * n_tiles + nt) * stored_spans * 4096 + wave * 1024 + lane * 8;

        v16f acc[2];
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int j = 0; j < 16; ++j) acc[c][j] = 0.0f;
        // (clamped: a map left incomplete by a layout launch that ran out of time must not become a wild address)
        const uint8_t* const codes = kGather ? p.a_codes : p.a_codes + static_cast<size_t>(row0) * p.k;
        const uint8_t* const row_scale_bytes = kGather ? p.a_scales : p.a_scales + static_cast<size_t>(row0) * scale_bytes;
        // In the layout that the MFMA takes: lane l has row l % 32, two pieces of 16 bytes per k step.
        constexpr int kSlots = 8;
        u32x4 wreg[kSlots][4], areg[kSlots][4];  // [k tile % 8][column tile * 2 + k step], [k step * 2 + piece]
        // The row's route is asked for first and the first weights behind it: they travel together.
        const int my_row = min(lr, valid - 1);
        const int route = kGather ? p.row_to_route[row0 + my_row] : 0;
        __builtin_amdgcn_sched_barrier(0);
        auto load_weights = [&](int slot, int kt) {
            const uint8_t* const from = w + static_cast<size_t>(min(kt, ktiles - 1)) * 16384;  // (past the end: the last k tile again, never used)
#pragma unroll
            for (int f = 0; f < 4; ++f) wreg[slot][f] = load16_nt(from + f * 1024);
        };
        u32x4 row_scales[2];
        u32x2 col_scales[2][2];  // [span parity][column tile]
        auto load_col_scales = [&](int parity, int span) {
            span = min(span, spans - 1);
#pragma unroll
            for (int c = 0; c < 2; ++c)
                col_scales[parity][c] = *reinterpret_cast<const u32x2*>(ws + static_cast<size_t>(span) * 4096 + c * 512);
        };
        load_col_scales(0, 0);
#pragma unroll
        for (int q = 0; q < 4; ++q) load_weights(q, q);
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t from_row = static_cast<uint32_t>(kGather ? min(max(route / p.topk, 0), p.a_rows - 1) : my_row);
        const uint8_t* const my_codes = codes + from_row * static_cast<uint32_t>(p.k) + g * 16;
        const uint8_t* const my_scales = row_scale_bytes + from_row * static_cast<uint32_t>(scale_bytes);
        auto load_activations = [&](int slot, int kt) {
            const uint8_t* const row = my_codes + static_cast<size_t>(min(kt, ktiles - 1)) * kBK;
#pragma unroll
            for (int f = 0; f < 4; ++f) areg[slot][f] = load16(row + f * 32);
        };
        auto load_row_scales = [&](int parity, int span) {
            row_scales[parity] = *reinterpret_cast<const u32x4_unaligned*>(my_scales + min(min(span, spans - 1) * 16, scale_bytes - 16));
        };
        load_row_scales(0, 0);
#pragma unroll
        for (int q = 0; q < 4; ++q) load_activations(q, q);
        __builtin_amdgcn_sched_barrier(0);
        load_col_scales(1, 1);
        load_row_scales(1, 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 4; q < 8; ++q) {
            load_weights(q, q);
            load_activations(q, q);
        }
        __builtin_amdgcn_sched_barrier(0);
        auto span_body = [&](auto parity_constant, auto ask_constant, auto whole_constant, int span) {
            constexpr int kParity = decltype(parity_constant)::value;
            constexpr bool kAsk = decltype(ask_constant)::value;      // the span after the next one exists
            constexpr bool kWhole = decltype(whole_constant)::value;  // another span follows, so all four k tiles of this one are there
            u32x4 rows_now = row_scales[kParity];
            u32x2 cols_now[2] = {col_scales[kParity][0], col_scales[kParity][1]};
            // (moved out of the way: the next scales of this parity are asked for in front of the weights that they go with)
            asm volatile("" : "+v"(rows_now), "+v"(cols_now[0]), "+v"(cols_now[1]));
            if constexpr (kAsk) {
                load_col_scales(kParity, span + 2);
                load_row_scales(kParity, span + 2);
            }
            __builtin_amdgcn_sched_barrier(0);
            const bool shifted_window = span * 16 > scale_bytes - 16;  // (k % 512 = 256: the last span's bytes sit two words up)
            static_for<4>([&](auto q_constant) {
                constexpr int q = decltype(q_constant)::value, kSlot = 4 * kParity + q;
                if (q == 0 || kWhole || span * 4 + q < ktiles) {
                    const uint32_t word = q < 2 && !kWhole && shifted_window ? rows_now[(q + 2) & 3] : rows_now[q];
                    const int x_scale = static_cast<int>(word >> (8 * g));
                    static_for<2>([&](auto step_constant) {
                        constexpr int step = decltype(step_constant)::value;
                        const u32x4 lo = areg[kSlot][2 * step], hi = areg[kSlot][2 * step + 1];
                        const v8i x = {(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
#pragma unroll
                        for (int c = 0; c < 2; ++c) {
                            const u32x4 f = wreg[kSlot][2 * c + step];
                            const v8i m = {(int)f[0], (int)f[1], (int)f[2], (int)f[3], 0, 0, 0, 0};
                            acc[c] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(m, x, acc[c], 4, 0, 2 * (q & 1) + step,
                                                                                     static_cast<int>(cols_now[c][q >> 1]), 2 * step, x_scale);
                        }
                    });
                    if constexpr (q == 3 || !kWhole) asm volatile("s_nop 15\n\ts_nop 7" : "+a"(acc[0]), "+a"(acc[1]));  // (settle_accumulators, where they are)
                }
                if constexpr (kAsk) {
                    load_weights(kSlot, span * 4 + q + 8);
                    load_activations(kSlot, span * 4 + q + 8);
                }
                __builtin_amdgcn_sched_barrier(0);
            });
        };
        constexpr std::integral_constant<int, 0> even{};
        constexpr std::integral_constant<int, 1> odd{};
        constexpr std::integral_constant<bool, true> yes{};
        constexpr std::integral_constant<bool, false> no{};
        int span = 0;
        for (; span + 3 < spans; span += 2) {
            span_body(even, yes, yes, span);
            span_body(odd, yes, yes, span + 1);
        }
        if (spans - span == 3) {
            span_body(even, yes, yes, span);
            span_body(odd, no, yes, span + 1);
            span_body(even, no, no, span + 2);
        } else if (spans - span == 2) {
            span_body(even, no, yes, span);
            span_body(odd, no, no, span + 1);
        } else {
            span_body(even, no, no, span);
        }
        if (fillers != 0 && tile_id == 0 && threadIdx.x == 0) __hip_atomic_fetch_add(p.fill_stop, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const bool row_exists = lr < valid;
        const size_t row = static_cast<size_t>(row0) + lr;
        if (kGateUp) {
            store_gate_up(p, acc[0], acc[1], row, row_exists, (nt * (kBN / 64) + wave) * 32, g);
        } else {
#pragma unroll
            for (int c = 0; c < 2; ++c) store_output(p, acc[c], row, row_exists, nt * kBN + (wave * 2 + c) * 32, g);
        }
    }
}

template <int RT, bool kGateUp>
__global__ __launch_bounds__(kGemmThreads, ColCfg<RT>::kWorkgroupsPerCu) void grouped_gemm_colwave_kernel(GemmParams p)
{
    constexpr bool kGather = kGateUp;
    using Cfg = ColCfg<RT>;
    constexpr int kBM = Cfg::kBM, kStages = Cfg::kStages, kStageBytes = Cfg::kStageBytes, kRowTiles = Cfg::kRowTiles;
    constexpr int kCols = Cfg::kColTiles;
    constexpr bool kStreamed = RT == 1;  // few rows per expert: every weight byte is read once or twice
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    __shared__ int tile_base[kMaxMoeExperts + 1];
    __shared__ int row_offsets[kMaxMoeExperts + 1];
    __shared__ int tile_index[2][kGemmThreads];  // row_to_route of a tile's rows; slots alternate per tile
    // Where each thread's copies of the tile under the cursor start: [0 .. kRowTiles-1] byte offsets of its activation rows
    // from a_codes, [kRowTiles] of its row of scale bytes from a_scales.  Written at tile switches, read back right before
    // each copy: kept in registers instead, they are values that live across the whole item loop, and the register
    // allocator has put such values on the stack (every reload from there waits for all the copies in flight).
    __shared__ uint32_t copy_offsets[ColCfg<RT>::kRowTiles + 1][kGemmThreads];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 5, lr = lane & 31;
    const int n_tiles = p.n / kBN;
    const int ktiles = p.k / kBK;  // a multiple of 4
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds));
    const uint32_t lds_index = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(&tile_index[0][0]));
    const uint32_t wave_lds = __builtin_amdgcn_readfirstlane(lds0 + wave * 1024);

    if (tid <= p.num_local) row_offsets[tid] = p.offsets[tid];
    __syncthreads();
    if (wave == 0) number_tiles<kBM>(row_offsets, p.num_local, n_tiles, lane, tile_base);
    __syncthreads();
    const int total_tiles = tile_base[p.num_local];

    // Tiles to workgroups, and what the workgroups without a tile do: as in grouped_gemm_kernel.
    const bool one_round = total_tiles < static_cast<int>(gridDim.x);
    const int fillers = one_round && p.fill_out != nullptr ? (static_cast<int>(gridDim.x) - total_tiles) * kFillWaves : 0;
    const bool spread = one_round && fillers == 0 && (gridDim.x & 7) == 0;
    const int per_xcd = spread ? (total_tiles + 7) / 8 : (gridDim.x + 7) / 8;
    const int first = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    const int stride = one_round ? total_tiles + 1 : per_xcd * 8;
    const bool has_tile = first < total_tiles && (!spread || static_cast<int>(blockIdx.x >> 3) < per_xcd);
    if (blockIdx.x == 0 && tid == 0 && p.fill_state != nullptr) p.fill_state[0] = fillers;
    if (!has_tile) {
        if (fillers != 0 && wave < kFillWaves) fill_zero_rows(p, (first - total_tiles) * kFillWaves + wave, fillers, lane);
        return;
    }
    const int my_tiles = one_round ? 1 : (total_tiles - first + stride - 1) / stride;

    auto decode = [&](int tile) {
        const int e = expert_of_tile(tile, tile_base, p.num_local);
        const int row_begin = __builtin_amdgcn_readfirstlane(row_offsets[e]), rows = __builtin_amdgcn_readfirstlane(row_offsets[e + 1]) - row_begin;
        const int m_tiles = (rows + kBM - 1) / kBM;
        const int local = tile - __builtin_amdgcn_readfirstlane(tile_base[e]);
        // Inside an expert the tiles are numbered panel by panel: kPanel column tiles wide (the last panel may be
        // narrower), all row tiles high, row by row.  The 32 consecutive tiles an XCD works on at a time are then a block of
        // about 4 row tiles x 8 column tiles, whose activation rows and weight columns that XCD's L2 fetches once, instead
        // of every row tile of a few column tiles (which made each of the eight XCDs fetch all the rows of a large expert).
        constexpr int kPanel = 8;
        const int panel = local / (m_tiles * kPanel), in_panel = local - panel * (m_tiles * kPanel);
        const int width = min(kPanel, n_tiles - panel * kPanel);
        TileInfo info;
        info.expert = e;
        info.nt = panel * kPanel + in_panel % width;
        const int m0 = (in_panel / width) * kBM;
        info.row0 = row_begin + m0;
        info.valid = min(kBM, rows - m0);
        return info;
    };

    // ---- request cursor: what is asked for next (activation copies, weight loads, scales, gather indices) ----------
    // activation copy c of wave w fills LDS rows c*32 + w*8 + lane/8; chunk (lane%8) ^ ((row>>1)&7) of the 128-byte row
    auto a_chunk_of = [&](int l) { return ((l & 7) ^ ((wave * 4 + (l >> 4)) & 7)) * 16; };
    const uint32_t* my_offsets = &copy_offsets[0][tid];  // entry i: + i * kGemmThreads
    const uint32_t b_lane = static_cast<uint32_t>(wave * 4096 + lane * 16);  // this wave's four fragments of an item are contiguous
    const uint8_t* b_base = p.w;
    const uint8_t* sb_base = p.ws;  // column scales of the tile under the cursor (thread t copies bytes 16 t .. 16 t + 15 of a span)
    int index_row0 = 0, index_valid = 1;  // rows whose gather indices are fetched next
    int copy_tile = first, copy_kt = 0, copy_span = -1, copy_ordinal = 0;
    const int scale_bytes = p.k / 32;  // per row
    const int spans = ktiles / 4;
    TileInfo next_info = decode(first);

    auto point_at_tile = [&](const TileInfo& info) {
        const int* index = tile_index[copy_ordinal & 1];
        // (the lane's row numbers are worked out afresh at every tile switch: kept in registers across the item loop
        // they cost the loop a register each, or a place on the stack)
        const int lane_here = lane_now(), tid_here = wave * 64 + lane_here;
#pragma unroll
        for (int i = 0; i < kRowTiles; ++i) {
            const int r = min(i * 32 + wave * 8 + (lane_here >> 3), info.valid - 1);  // rows past the tile's end repeat its last row
            const int src = kGather ? min(max(index[r] / p.topk, 0), p.a_rows - 1) : info.row0 + r;
            copy_offsets[i][tid_here] = static_cast<uint32_t>(src) * static_cast<uint32_t>(p.k) + a_chunk_of(lane_here);
        }
        {
            const int r = min(tid_here % kBM, info.valid - 1);
            const int src = kGather ? min(max(index[r] / p.topk, 0), p.a_rows - 1) : info.row0 + r;
            copy_offsets[kRowTiles][tid_here] = static_cast<uint32_t>(src) * static_cast<uint32_t>(scale_bytes);
        }
        const bool shared = info.expert >= p.num_routed;
        const size_t weight_index = shared ? info.expert - p.num_routed : info.expert;
        b_base = (shared ? p.w_shared : p.w) + weight_index * p.n * (p.k / 2) + static_cast<size_t>(info.nt) * ktiles * 16384;
        sb_base = (shared ? p.ws_shared : p.ws) + (weight_index * n_tiles + info.nt) * spans * Cfg::kColScaleSlot;
    };
    auto aim_index_prefetch = [&](const TileInfo& info) {
        index_row0 = info.row0;
        index_valid = info.valid;
    };
    auto index_offset = [&]() {  // this thread's entry of row_to_route, in bytes
        return static_cast<uint32_t>(index_row0 + min(wave * 64 + lane_now(), index_valid - 1)) * 4u;
    };

    // Column scales of the current span and of the next one: [column tile] x 8 bytes = k tiles 0..3 x k steps 0..1.
    u32x2 bscale_now[kCols], bscale_next[kCols];

    // The requests of the item under the cursor, which goes to ring position kPos; issued in pieces between MFMAs.
    auto request_activations_at = [&](auto pos, auto piece, uint32_t offset) {
        constexpr int kPos = decltype(pos)::value, kPiece = decltype(piece)::value;
        copy16_to_lds_at<kPos * kStageBytes + kPiece * 4096>(p.a_codes + static_cast<size_t>(copy_kt) * kBK, offset, wave_lds);
    };
    auto request_activations = [&](auto pos, auto piece) {
        request_activations_at(pos, piece, my_offsets[decltype(piece)::value * kGemmThreads]);
    };
    auto request_weights = [&](auto pos, auto step) {
        constexpr int kPos = decltype(pos)::value, kStep = decltype(step)::value;
        const uint8_t* item = b_base + static_cast<size_t>(copy_kt) * 16384;
        // fragment (column tile c, k step) of the wave's four: 2048 c + 1024 step bytes in; registers 16 pos + 8 step + 4 c
        constexpr int kReg = Cfg::kWeightRegs + 16 * kPos + 8 * kStep;
        load16_to_weight_regs<Cfg::kWeightRegs, kReg, kStep * 1024, kStreamed>(item, b_lane);
        load16_to_weight_regs<Cfg::kWeightRegs, kReg + 4, 2048 + kStep * 1024, kStreamed>(item, b_lane);
    };
    // A span's first item (ring position 0) also asks for the span's scales, into the LDS slots of the span's parity: 16
    // bytes of row scales per row and the span's 4 KiB of column scales.  A tile's first item asks for the gather indices of
    // the workgroup's next tile.
    auto request_span = [&]() {
        ++copy_span;
        const int window = min(copy_kt * 4, scale_bytes - 16);
        copy16_to_lds(p.a_scales + window, my_offsets[kRowTiles * kGemmThreads], lds0 + Cfg::kOffRowScales + (copy_span & 1) * Cfg::kRowScaleSlot + ((wave * 64) % kBM) * 16);
        copy16_to_lds(sb_base + static_cast<size_t>(copy_kt >> 2) * Cfg::kColScaleSlot, static_cast<uint32_t>(wave * 1024 + lane_now() * 16),
                      lds0 + Cfg::kOffColScales + (copy_span & 1) * Cfg::kColScaleSlot + wave * 1024);
        if (kGather)
            copy4_to_lds_unless(p.row_to_route, index_offset(), lds_index + ((copy_ordinal + 1) & 1) * (kGemmThreads * 4) + wave * 256, copy_kt);
    };
    // (k tiles come in fours, so a tile can only end behind ring position 3)
    auto advance_cursor = [&](bool in_prologue, bool last_of_four) {
        ++copy_kt;
        if (last_of_four && copy_kt == ktiles) {
            if (copy_tile + stride < total_tiles) {
                // (a tile has at least four items, so only a switch inside the prologue can come before a counted wait
                // has covered the fetch of the next tile's indices)
                if (kGather && switch_needs_drain(in_prologue, ktiles, kStages)) wait_copies_then_barrier<0>();
                copy_tile += stride;
                copy_kt = 0;
                ++copy_ordinal;
                point_at_tile(next_info);
                if (copy_tile + stride < total_tiles) next_info = decode(copy_tile + stride);
                aim_index_prefetch(next_info);
            } else {
                copy_kt = ktiles - 4;  // past the last tile: keep asking for its last span (never used)
            }
        }
    };

    if (kGather) {
        aim_index_prefetch(next_info);
        copy4_to_lds(p.row_to_route, index_offset(), lds_index + wave * 256);
        wait_copies_then_barrier<0>();
    }
    point_at_tile(next_info);
    if (first + stride < total_tiles) next_info = decode(first + stride);
    aim_index_prefetch(next_info);

    // ---- fragment addresses inside a stage ---------------------------------------------------------
    int a_addr[2][2];  // [k step][lo/hi 16 bytes] of row tile 0; row tile i lies i * 4096 bytes further (same swizzle)
    {
        const int sw = (lr >> 1) & 7;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            a_addr[kb][0] = lr * kBK + (((kb * 4 + g) ^ sw) << 4);
            a_addr[kb][1] = lr * kBK + (((kb * 4 + 2 + g) ^ sw) << 4);
        }
    }
    // LDS address of this lane's row-scale entry in the slot of the span being read; row tile i lies i * 512 bytes further,
    // k tile q of the span 4 q bytes (one register and instruction offsets, not a register per row tile)
    int row_scale_at = Cfg::kOffRowScales + lr * 16;

    v8i afrag[2][kRowTiles];   // [k step][row tile]
    int ascale[2][kRowTiles];  // [item parity][row tile]: the row-scale word of the k tile, moved so that this lane half's
                               // first k block is byte 0 (its second is byte 2)
    auto read_fragment = [&](int stage, int kb, int i) {
        const uint8_t* at = lds + stage * kStageBytes + i * 4096;
        const u32x4 lo = *reinterpret_cast<const u32x4*>(at + a_addr[kb][0]);
        const u32x4 hi = *reinterpret_cast<const u32x4*>(at + a_addr[kb][1]);
        afrag[kb][i] = v8i{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
    };
    int col_scale_slot = 0;  // byte offset of the LDS slot whose span's column scales are read next
    auto read_row_scale = [&](int parity, int pos, int i) {
        ascale[parity][i] = static_cast<int>(*reinterpret_cast<const uint32_t*>(lds + row_scale_at + (i * 512 + pos * 4)));
    };
    auto read_col_scales = [&]() {
        const int sb_addr = Cfg::kOffColScales + wave * 1024 + lane_now() * 8;  // this wave's column tile c: + c * 512
#pragma unroll
        for (int c = 0; c < kCols; ++c) bscale_next[c] = *reinterpret_cast<const u32x2*>(lds + sb_addr + c * 512 + col_scale_slot);
    };

    v16f acc[kRowTiles][kCols];
    auto clear_acc = [&]() {
#pragma unroll
        for (int i = 0; i < kRowTiles; ++i)
#pragma unroll
            for (int c = 0; c < kCols; ++c)
#pragma unroll
                for (int j = 0; j < 16; ++j) acc[i][c][j] = 0.0f;
    };

    // ---- epilogue of one tile: straight from the accumulators (store_gate_up, store_output) ---------------------------------
    auto epilogue = [&](const TileInfo& info) {
        const int lane = lane_now(), g = lane >> 5, lr = lane & 31;  // (the epilogue's own copies: see lane_now)
#pragma unroll
        for (int i = 0; i < kRowTiles; ++i) {
            if (i == kRowTiles - 1 && fillers != 0 && wave == 0 && lane == 0)
                __hip_atomic_fetch_add(p.fill_stop, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const bool row_exists = lr < info.valid - 32 * i;
            const size_t row = static_cast<size_t>(info.row0) + 32 * i + lr;
            // (a row tile's accumulators leave their registers here, not earlier: read all at once at the head of the
            // epilogue, the twelve tiles would need 192 more registers than the loop's own state leaves free)
#pragma unroll
            for (int c = 0; c < kCols; ++c) asm volatile("" : "+a"(acc[i][c]));
            if (kGateUp) {
                store_gate_up(p, acc[i][0], acc[i][1], row, row_exists, (info.nt * (kBN / 64) + wave) * 32, g);
            } else {
#pragma unroll
                for (int c = 0; c < kCols; ++c) store_output(p, acc[i][c], row, row_exists, info.nt * kBN + (wave * kCols + c) * 32, g);
            }
        }
    };

    // ---- prologue: everything of items 0..3, then item 0's first fragments -------------------------------
    auto request_item = [&](auto pos) {
        if (decltype(pos)::value == 0) request_span();
        static_for<kRowTiles>([&](auto piece) { request_activations(pos, piece); });
        request_weights(pos, std::integral_constant<int, 0>{});
        request_weights(pos, std::integral_constant<int, 1>{});
        advance_cursor(true, decltype(pos)::value == 3);
    };
    request_item(std::integral_constant<int, 0>{});
    request_item(std::integral_constant<int, 1>{});
    request_item(std::integral_constant<int, 2>{});
    request_item(std::integral_constant<int, 3>{});
    wait_copies_then_barrier<Cfg::kPrologueWait>();  // item 0 and its span have arrived
    int read_span = 0;
    read_col_scales();
#pragma unroll
    for (int i = 0; i < kRowTiles; ++i) {
        read_row_scale(0, 0, i);
        read_fragment(0, 0, i);
    }
    clear_acc();
    asm volatile("s_nop 3");
    int tile = first, kt = 0;
    TileInfo info = decode(first);
    const long long total_items = static_cast<long long>(my_tiles) * ktiles;
    constexpr int kMfmas = kRowTiles * kCols;  // per k step; MFMA n works on row tile n % kRowTiles, column tile n / kRowTiles

    // One item at ring position kPos.  First k step: its MFMAs, with the LDS reads of the second k step's fragments dealt
    // out between them; then the wait + barrier, after which the item's own stage may be refilled.  Second k step: its
    // MFMAs, with the activation copies of the item four ahead, and the reads of the next item's row scales and first
    // fragments, dealt out between them.  Behind the last MFMA of a k step its weight registers are free: the weight loads
    // of the item four ahead follow.
    auto item_body = [&](auto pos) {
        constexpr int kPos = decltype(pos)::value;
        constexpr int kParity = kPos & 1, kNextPos = (kPos + 1) & 3;
        if (kPos == 0) {
            // the span's column scales were read from LDS under the previous item's last MFMAs
#pragma unroll
            for (int c = 0; c < kCols; ++c) bscale_now[c] = bscale_next[c];
        }
        const int scale_b0 = static_cast<int>(bscale_now[0][kPos >> 1]), scale_b1 = static_cast<int>(bscale_now[1][kPos >> 1]);
        int shifted[kRowTiles];
#pragma unroll
        for (int i = 0; i < kRowTiles; ++i) shifted[i] = ascale[kParity][i] >> (8 * g);
        // MFMA number n of a k step works on row tile n / kCols, column tile n % kCols.
        auto mfma = [&](auto step, auto number) {
            constexpr int kStep = decltype(step)::value, kN = decltype(number)::value;
            constexpr int kI = kN / kCols, kC = kN % kCols;
            mfma_fp4_fp8_regs<Cfg::kWeightRegs + 16 * kPos + 8 * kStep + 4 * kC, 2 * (kPos & 1) + kStep, 2 * kStep>(
                acc[kI][kC], afrag[kStep][kI], kC == 0 ? scale_b0 : scale_b1, shifted[kI]);
        };
        // First k step.  Behind MFMA kBarrierAt comes the wait + barrier: the second step's fragments were all asked for under
        // the first kRowTiles MFMAs and have had kBarrierAt - kRowTiles more to arrive.  The activation copies of the item four
        // ahead (into this item's own stage, free from the barrier on) are dealt out one per kCopyEvery MFMAs over what
        // is left of the item.
        constexpr int kBarrierAt = kRowTiles + 1;
        constexpr int kSlotsLeft = 2 * kMfmas - kBarrierAt - 1, kCopyEvery = kSlotsLeft / kRowTiles;
        // (the copies' offsets are read from LDS in one go right behind the barrier: read one by one in front of each copy,
        // every copy waited for its own read behind whatever fragment reads were queued before it)
        uint32_t copy_from[kRowTiles];
        auto copies_behind = [&](auto slot) {  // slot = MFMAs issued since the barrier, 1-based
            constexpr int kSlot = decltype(slot)::value;
            if constexpr (kSlot >= 1 && (kSlot - 1) % kCopyEvery == 0 && (kSlot - 1) / kCopyEvery < kRowTiles)
                request_activations_at(pos, std::integral_constant<int, (kSlot - 1) / kCopyEvery>{}, copy_from[(kSlot - 1) / kCopyEvery]);
        };
        static_for<kMfmas>([&](auto n) {
            constexpr int kN = decltype(n)::value;
            mfma(std::integral_constant<int, 0>{}, n);
            if constexpr (kN < kRowTiles) read_fragment(kPos, 1, kN);
            if constexpr (kN == kBarrierAt) {
                // The next item's operands have arrived once each thread has at most the requests of the two items after it
                // in flight; past the barrier every wave has also read the last fragment of this item's stage.
                wait_copies_then_barrier<Cfg::kWait>();
#pragma unroll
                for (int i = 0; i < kRowTiles; ++i) copy_from[i] = my_offsets[i * kGemmThreads];
                if (kPos == 0) request_span();
            }
            if constexpr (kN > kBarrierAt) copies_behind(std::integral_constant<int, kN - kBarrierAt>{});
        });
        request_weights(pos, std::integral_constant<int, 0>{});
        if (kPos == 3) {
            // the next item opens a span: its scales sit in the other LDS slots
            ++read_span;
            row_scale_at += (read_span & 1) ? Cfg::kRowScaleSlot : -Cfg::kRowScaleSlot;
            asm volatile("" : "+v"(row_scale_at));  // (kept as one value: see its declaration)
            col_scale_slot = (read_span & 1) * Cfg::kColScaleSlot;
            read_col_scales();
        }
        static_for<kMfmas>([&](auto n) {
            constexpr int kN = decltype(n)::value;
            mfma(std::integral_constant<int, 1>{}, n);
            copies_behind(std::integral_constant<int, kMfmas - 1 - kBarrierAt + kN + 1>{});
            // the next item's row scale and first fragment of the row tile just finished
            if constexpr (kN % kCols == kCols - 1) {
                read_row_scale(kParity ^ 1, kNextPos, kN / kCols);
                read_fragment(kNextPos, 0, kN / kCols);
            }
        });
        request_weights(pos, std::integral_constant<int, 1>{});
        advance_cursor(false, kPos == 3);
    };

    for (long long item = 0; item < total_items; item += 4) {
        item_body(std::integral_constant<int, 0>{});
        item_body(std::integral_constant<int, 1>{});
        item_body(std::integral_constant<int, 2>{});
        item_body(std::integral_constant<int, 3>{});
        kt += 4;
        if (__builtin_expect(kt == ktiles, 0)) {
            settle_accumulators();
#pragma unroll
            for (int i = 0; i < kRowTiles; ++i)
#pragma unroll
                for (int c = 0; c < kCols; ++c) asm volatile("" : "+a"(acc[i][c]));
            epilogue(info);
            clear_acc();
            asm volatile("s_nop 3");
            kt = 0;
            tile += stride;
            if (tile < total_tiles) info = decode(tile);
        }
    }
    // Nothing may still be in flight into this workgroup's LDS or registers when it retires.
    wait_copies_then_barrier<0>();
}

// =====================================================================================================
// Grouped GEMM, column-wave form with two workgroups to a CU: 128-row tiles that skip what is padding
// =====================================================================================================
// The column-wave kernel above owns its CU, so nothing runs on the matrix pipes while a tile starts or ends, and it works on whole
// tiles: 97 rows cost as much as 128, 2880 columns of k as much as 3072, and k must come in multiples of 512.  This one leaves
// room for a second workgroup on the CU (two waves per SIMD, 256 registers and half of the LDS each), whose MFMAs fill those gaps, and
// jumps over every MFMA of a row tile without rows, of a k step behind the end of k, and of a wave whose columns are only
// padding; column tiles of nothing but padding are not even numbered where the second GEMM does not read them.
// Bound by the matrix pipes (their clock falls with the work in flight: large batches take as long at 192 rows on one
// workgroup), by streaming the weights where an expert has about one row tile, and by a tile's start and end where a launch is
// a single round.  Measured on an MI355X against the best of the other heights, whole forwards, us: 4584 tokens over 29 + 2 experts of
// 1600 x 2944 243 -> 198, 8512 over 3 + 2 of 3264 x 3840 672 -> 565, 4560 x top-8 over 59 + 2 of 1088 x 384 77 -> 63, 777 x top-4 over
// 32 + 1 of 2880 x 1408 101 -> 94; 8192 x top-8 over 32 of 7168 x 2048: 2336 with 192 rows, 2408 with this.
//
// Accumulators and weight fragments live in registers that only the assembly statements name (a0..a127, v96..v127): with two
// workgroups to a CU the accumulators are all the accumulation registers there are, and the register allocator, which may not
// spill one, put all of them on the stack.  tests/test_gemm_registers.py checks that the compiler's own values stay out of them;
// the jumps are harmless to it for the same reason.
//
// Requests: the activation copies (and a span's scales, a tile's gather indices) run four items ahead, an LDS stage each, the
// weights two items ahead, 16 registers each (four ahead were 1 to 3 % slower).  Every item asks, in this order, for its first k step's weights of
// the item two ahead (2 loads, behind its own first step, whose registers are then free), its LDS stage's next
// activations (4 copies, behind the barrier), its second k step's weights (2 loads, behind its second step); a span's first
// item also for the scales of the span after this one, in front of the copies.  With that, an item's first weights have
// arrived when at most 6 + 8 later requests are in flight (kWaitFirst), its second ones when at most 8 + 2 are (kWaitSecond).  The wait
// for an item's second weights also covers everything that the items before the one two back asked for, which includes
// the next item's activations and scales, and, at a tile's last item, the gather indices asked for at its first; the barrier
// behind it makes them everybody's.  Requests of skipped work are issued all the same (for the last real k tile again), so the counts hold.
struct PairCfg : PairedRing {
    static constexpr int kBM = 128;
    static constexpr int kRowTiles = 4, kColTiles = 2;  // 32 x 32 MFMA tiles per wave
    static constexpr int kStageBytes = kBM * kBK;
    static constexpr int kRowScaleSlot = kBM * 16;
    static constexpr int kOffRowScales = kStages * kStageBytes;
    static constexpr int kColScaleSlot = 4096;
    static constexpr int kOffColScales = kOffRowScales + 2 * kRowScaleSlot;
    static constexpr int kLdsBytes = kOffColScales + 2 * kColScaleSlot;
    static constexpr int kWeightRegs = 96;  // first of the ordinary registers that hold weight fragments (v96..v127)
    static_assert(kActivations == kRowTiles && kWeights == kColTiles, "the waits count what the kernel asks for");
};
#define DPEP_PAIR_ACC_REGS \
    "a0", "a1", "a2", "a3", "a4", "a5", "a6", "a7", "a8", "a9", "a10", "a11", "a12", "a13", "a14", "a15", \
        "a16", "a17", "a18", "a19", "a20", "a21", "a22", "a23", "a24", "a25", "a26", "a27", "a28", "a29", "a30", "a31", \
        "a32", "a33", "a34", "a35", "a36", "a37", "a38", "a39", "a40", "a41", "a42", "a43", "a44", "a45", "a46", "a47", \
        "a48", "a49", "a50", "a51", "a52", "a53", "a54", "a55", "a56", "a57", "a58", "a59", "a60", "a61", "a62", "a63", \
        "a64", "a65", "a66", "a67", "a68", "a69", "a70", "a71", "a72", "a73", "a74", "a75", "a76", "a77", "a78", "a79", \
        "a80", "a81", "a82", "a83", "a84", "a85", "a86", "a87", "a88", "a89", "a90", "a91", "a92", "a93", "a94", "a95", \
        "a96", "a97", "a98", "a99", "a100", "a101", "a102", "a103", "a104", "a105", "a106", "a107", "a108", "a109", "a110", "a111", \
        "a112", "a113", "a114", "a115", "a116", "a117", "a118", "a119", "a120", "a121", "a122", "a123", "a124", "a125", "a126", "a127"
#define DPEP_PAIR_WEIGHT_REGS \
    "v96", "v97", "v98", "v99", "v100", "v101", "v102", "v103", "v104", "v105", "v106", "v107", "v108", "v109", "v110", "v111", \
        "v112", "v113", "v114", "v115", "v116", "v117", "v118", "v119", "v120", "v121", "v122", "v123", "v124", "v125", "v126", "v127"
// kStreamed: weights past the caches, where each is read by about one row tile and the memory-side cache does not hold them all (55
// experts of 57 rows, 409 MB: 106 -> 96.5 us; up to 250 MB it is 5 % slower on average, with several row tiles 10 to 20 %).
template <int kReg, int kImm, bool kStreamed>
__device__ __forceinline__ void load16_to_paired_weight_regs(const void* uniform_base, uint32_t lane_offset)
{
    static_assert(kReg >= PairCfg::kWeightRegs && kReg + 3 < 128, "not one of the kernel's weight registers");
    if constexpr (kStreamed)
        asm volatile("global_load_dwordx4 v[%3:%4], %0, %1 offset:%2 nt" ::"v"(lane_offset), "s"(uniform_base), "n"(kImm), "n"(kReg), "n"(kReg + 3)
                     : "memory", DPEP_PAIR_WEIGHT_REGS);
    else
        asm volatile("global_load_dwordx4 v[%3:%4], %0, %1 offset:%2 sc1" ::"v"(lane_offset), "s"(uniform_base), "n"(kImm), "n"(kReg), "n"(kReg + 3)
                     : "memory", DPEP_PAIR_WEIGHT_REGS);
}
// The MFMAs of row tile kI (both column tiles, accumulators a[32 kI : 32 kI + 31]; weights v[kReg : kReg + 3] and the four behind), jumped over
// unless kI < row_tiles.  Operands the other way round, as in mfma_fp4_fp8_regs.
template <int kI, int kReg, int kByteW, int kByteX>
__device__ __forceinline__ void mfma_row_tile(const v8i& x, int scale_w0, int scale_w1, int scale_x, int row_tiles)
{
    asm volatile("s_cmp_le_i32 %14, %15\n\ts_cbranch_scc1 .Lskip_mfma_%=\n\t"
                 "v_mfma_scale_f32_32x32x64_f8f6f4 a[%10:%11], v[%8:%9], %0, a[%10:%11], %1, %3 op_sel:[%4,%5,0] op_sel_hi:[%6,%7,0] cbsz:4\n\t"
                 "v_mfma_scale_f32_32x32x64_f8f6f4 a[%12:%13], v[%8+4:%9+4], %0, a[%12:%13], %2, %3 op_sel:[%4,%5,0] op_sel_hi:[%6,%7,0] cbsz:4\n"
                 ".Lskip_mfma_%=:" ::"v"(x),
                 "v"(scale_w0), "v"(scale_w1), "v"(scale_x), "n"(kByteW & 1), "n"(kByteX & 1), "n"(kByteW >> 1), "n"(kByteX >> 1), "n"(kReg), "n"(kReg + 3),
                 "n"(32 * kI), "n"(32 * kI + 15), "n"(32 * kI + 16), "n"(32 * kI + 31), "s"(row_tiles), "n"(kI)
                 : "scc", DPEP_PAIR_ACC_REGS);
}
template <int kAcc>
__device__ __forceinline__ void clear_acc_tile()
{
    asm volatile(".irp r, 0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15\n\tv_accvgpr_write_b32 a[%0+\\r], 0\n\t.endr" ::"n"(kAcc) : DPEP_PAIR_ACC_REGS);
}
template <int kAcc>
__device__ __forceinline__ float read_acc()
{
    float v;
    asm volatile("v_accvgpr_read_b32 %0, a[%1]" : "=v"(v) : "n"(kAcc) : "memory");
    return v;
}
template <int kAcc>
__device__ __forceinline__ v16f read_acc_tile()
{
    v16f v;
    static_for<16>([&](auto j) { v[decltype(j)::value] = read_acc<kAcc + decltype(j)::value>(); });
    return v;
}
template <int kOutstanding>
__device__ __forceinline__ void wait_requests()
{
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kOutstanding) : "memory");
}

template <bool kStreamed, bool kGateUp>
__global__ __launch_bounds__(kGemmThreads, 2) void grouped_gemm_paired_kernel(GemmParams p)
{
    constexpr bool kGather = kGateUp;
    using Cfg = PairCfg;
    constexpr int kBM = Cfg::kBM, kStageBytes = Cfg::kStageBytes, kRowTiles = Cfg::kRowTiles, kCols = Cfg::kColTiles;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    __shared__ int tile_base[kMaxMoeExperts + 1];
    __shared__ int row_offsets[kMaxMoeExperts + 1];
    __shared__ int tile_index[2][kBM];   // row_to_route of a tile's rows; slots alternate per tile
    __shared__ uint32_t row_from[2][kBM];  // byte offset from a_codes of each row of the tile under the request cursor; slots alternate per tile

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 5, lr = lane & 31;
    const int n_tiles = p.n / kBN;
    const int live_n_tiles = p.live_n_tiles;  // (column tiles of nothing but padding are left out)
    // The matrix is stored and addressed with its padded k (p.k); what is computed ends with the last k step that holds any of it.  An
    // item behind that keeps its place in the rings (the last real k tile is asked for again), without MFMAs.
    const int stored_ktiles = p.k / kBK, steps = (p.k_real + 63) / 64, last_kt = (steps - 1) / 2, ktiles = (last_kt + 4) & ~3;
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds));
    const uint32_t lds_index = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(&tile_index[0][0]));
    const uint32_t wave_lds = __builtin_amdgcn_readfirstlane(lds0 + wave * 1024);

    if (tid <= p.num_local) row_offsets[tid] = p.offsets[tid];
    __syncthreads();
    if (wave == 0) number_tiles<kBM>(row_offsets, p.num_local, live_n_tiles, lane, tile_base);
    __syncthreads();
    const int total_tiles = __builtin_amdgcn_readfirstlane(tile_base[p.num_local]);

    // Workgroups are dealt round-robin over the 8 XCDs.  A full round's tiles are dealt out in 8 contiguous ranges, one per XCD (consecutive
    // tiles share weights and rows: an XCD's L2 sees them from one place, and the ranges that share some are at work at the
    // same time).  So are those of the last round, which may not be full: it then leaves one tile, at full speed, to each of some
    // CUs on every XCD.
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3, grid = gridDim.x;
    const int full_rounds = total_tiles / grid, rest = total_tiles - full_rounds * grid, rest_first = rest * xcd / 8;
    const int my_tiles = full_rounds + (rest_first + slot < rest * (xcd + 1) / 8 ? 1 : 0);
    if (blockIdx.x == 0 && tid == 0 && p.fill_state != nullptr) p.fill_state[0] = 0;
    if (my_tiles == 0) return;
    auto tile_of = [&](int round) __attribute__((always_inline)) {
        return round * grid + slot + (round < full_rounds ? xcd * (grid >> 3) : rest_first);
    };

    auto decode = [&](int tile) __attribute__((always_inline)) {  // panels of eight column tiles: as in the column-wave kernel
        const int e = expert_of_tile(tile, tile_base, p.num_local);
        const int row_begin = __builtin_amdgcn_readfirstlane(row_offsets[e]), rows = __builtin_amdgcn_readfirstlane(row_offsets[e + 1]) - row_begin;
        const int m_tiles = (rows + kBM - 1) / kBM;
        const int local = tile - __builtin_amdgcn_readfirstlane(tile_base[e]);
        constexpr int kPanel = 8;
        const int panel = local / (m_tiles * kPanel), in_panel = local - panel * (m_tiles * kPanel);
        const int width = min(kPanel, live_n_tiles - panel * kPanel);
        TileInfo info;
        info.expert = e;
        info.nt = panel * kPanel + in_panel % width;
        const int m0 = (in_panel / width) * kBM;
        info.row0 = row_begin + m0;
        info.valid = min(kBM, rows - m0);
        return info;
    };

    // ---- request cursors ---------------------------------------------------------------------------------------------------
    const uint32_t b_lane = static_cast<uint32_t>(wave * 4096 + lane * 16);
    const uint8_t* b_next = p.w;   // first weight fragment of the tile under the activation cursor
    const uint8_t* b_at = p.w;     // of the item under the weight cursor
    int b_kt = 0;
    const uint8_t* sb_base = p.ws;
    int index_row0 = 0, index_valid = 1;
    int copy_kt = 0, copy_span = -1, copy_ordinal = 0;
    const int scale_bytes = p.k / 32, spans = (stored_ktiles + 3) / 4;
    TileInfo next_info = decode(tile_of(0));

    auto point_at_tile = [&](const TileInfo& info) __attribute__((always_inline)) {
        const int* index = tile_index[copy_ordinal & 1];
        const int r = min(wave * 64 + lane_now(), kBM - 1), from = min(r, info.valid - 1);  // rows past the tile's end repeat its last row
        const int src = kGather ? min(max(index[from] / p.topk, 0), p.a_rows - 1) : info.row0 + from;
        row_from[copy_ordinal & 1][r] = static_cast<uint32_t>(src) * static_cast<uint32_t>(p.k);
        const bool shared = info.expert >= p.num_routed;
        const size_t weight_index = shared ? info.expert - p.num_routed : info.expert;

        b_next = (shared ? p.w_shared : p.w) + weight_index * p.n * (p.k / 2) + static_cast<size_t>(info.nt) * stored_ktiles * 16384;
        sb_base = (shared ? p.ws_shared : p.ws) + (weight_index * n_tiles + info.nt) * spans * Cfg::kColScaleSlot;
    };
    auto aim_index_prefetch = [&](const TileInfo& info) __attribute__((always_inline)) {
        index_row0 = info.row0;
        index_valid = info.valid;
    };
    auto index_offset = [&]() __attribute__((always_inline)) { return static_cast<uint32_t>(index_row0 + min((wave & 1) * 64 + lane_now(), index_valid - 1)) * 4u; };

    u32x2 bscale_now[kCols], bscale_next[kCols];

    // activation copy c of wave w fills LDS rows c*32 + w*8 + lane/8; chunk (lane%8) ^ ((row>>1)&7) of the 128-byte row
    const uint32_t a_chunk = static_cast<uint32_t>(((lane & 7) ^ ((wave * 4 + (lane >> 4)) & 7)) * 16);
    const uint32_t* my_rows = &row_from[0][wave * 8 + (lane >> 3)];  // + kBM for the other slot
    auto request_activations_at = [&](auto pos, auto piece, uint32_t row_offset) __attribute__((always_inline)) {
        constexpr int kPos = decltype(pos)::value, kPiece = decltype(piece)::value;
        copy16_to_lds_at<kPos * kStageBytes + kPiece * 4096>(p.a_codes + static_cast<size_t>(min(copy_kt, last_kt)) * kBK, row_offset + a_chunk, wave_lds);
    };
    auto request_weights = [&](auto slot, auto step) __attribute__((always_inline)) {
        constexpr int kSlot = decltype(slot)::value, kStep = decltype(step)::value;
        constexpr int kReg = Cfg::kWeightRegs + 16 * kSlot + 8 * kStep;
        load16_to_paired_weight_regs<kReg, kStep * 1024, kStreamed>(b_at, b_lane);
        load16_to_paired_weight_regs<kReg + 4, 2048 + kStep * 1024, kStreamed>(b_at, b_lane);
    };
    auto request_span = [&]() __attribute__((always_inline)) {
        ++copy_span;
        const int window = min(copy_kt * 4, scale_bytes - 16);  // (a last span of two k tiles: its bytes sit two words up)
        const int t = wave * 64 + lane_now();
        copy16_to_lds(p.a_scales + window, row_from[copy_ordinal & 1][t % kBM] >> 5, lds0 + Cfg::kOffRowScales + (copy_span & 1) * Cfg::kRowScaleSlot + (wave & 1) * 1024);
        copy16_to_lds(sb_base + static_cast<size_t>(copy_kt >> 2) * Cfg::kColScaleSlot, static_cast<uint32_t>(t * 16),
                      lds0 + Cfg::kOffColScales + (copy_span & 1) * Cfg::kColScaleSlot + wave * 1024);
        if (kGather)
            copy4_to_lds_unless(p.row_to_route, index_offset(), lds_index + ((copy_ordinal + 1) & 1) * (kBM * 4) + (wave & 1) * 256, copy_kt);
    };
    auto advance_activations = [&](bool in_prologue, bool last_of_four) __attribute__((always_inline)) {
        ++copy_kt;
        if (last_of_four && copy_kt == ktiles) {
            if (copy_ordinal + 1 < my_tiles) {
                if (kGather && switch_needs_drain(in_prologue, ktiles, Cfg::kStages)) wait_copies_then_barrier<0>();
                copy_kt = 0;
                ++copy_ordinal;
                point_at_tile(next_info);
                if (copy_ordinal + 1 < my_tiles) next_info = decode(tile_of(copy_ordinal + 1));
                aim_index_prefetch(next_info);
            } else {
                copy_kt = ktiles - 4;  // past the last tile: keep asking for its last span (never used)
            }
        }
    };
    // The weight cursor enters a tile two items behind the activation cursor, which by then points at that tile and at no later one yet (a tile
    // has at least four items; past the last tile: at the same tile still, whose first items are asked for again and never used).
    auto advance_weights = [&](bool last_of_four) __attribute__((always_inline)) {
        if (b_kt < last_kt) b_at += 16384;
        ++b_kt;
        if (last_of_four && b_kt == ktiles) {
            b_kt = 0;
            b_at = b_next;
        }
    };

    if (kGather) {
        aim_index_prefetch(next_info);
        copy4_to_lds(p.row_to_route, index_offset(), lds_index + (wave & 1) * 256);
        wait_copies_then_barrier<0>();
    }
    point_at_tile(next_info);
    b_at = b_next;
    if (my_tiles > 1) next_info = decode(tile_of(1));
    aim_index_prefetch(next_info);
    __syncthreads();  // row_from

    int a_addr[2][2];  // [k step][lo/hi 16 bytes] of row tile 0; row tile i lies i * 4096 bytes further (same swizzle)
    {
        const int sw = (lr >> 1) & 7;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            a_addr[kb][0] = lr * kBK + (((kb * 4 + g) ^ sw) << 4);
            a_addr[kb][1] = lr * kBK + (((kb * 4 + 2 + g) ^ sw) << 4);
        }
    }
    // LDS address of this lane's row-scale entry in the slot of the span that begins with k tile `from`
    auto row_scales_of = [&](int slot, int from) __attribute__((always_inline)) {
        return Cfg::kOffRowScales + lr * 16 + slot * Cfg::kRowScaleSlot + (from * 4 > scale_bytes - 16 ? 8 : 0);
    };
    int row_scale_at = row_scales_of(0, 0);
    int col_scale_slot = 0;
    v8i afrag[kRowTiles];  // of the k step at work, overwritten row tile by row tile with the next one's
    int ascale[kRowTiles];
    auto read_fragment = [&](int stage, int kb, int i) __attribute__((always_inline)) {
        const uint8_t* at = lds + stage * kStageBytes + i * 4096;
        const u32x4 lo = *reinterpret_cast<const u32x4*>(at + a_addr[kb][0]);
        const u32x4 hi = *reinterpret_cast<const u32x4*>(at + a_addr[kb][1]);
        afrag[i] = v8i{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
    };
    auto read_row_scale = [&](int pos, int i) __attribute__((always_inline)) {
        ascale[i] = static_cast<int>(*reinterpret_cast<const uint32_t*>(lds + row_scale_at + (i * 512 + pos * 4)));
    };
    auto read_col_scales = [&]() __attribute__((always_inline)) {
        const int sb_addr = Cfg::kOffColScales + wave * 1024 + lane_now() * 8;
#pragma unroll
        for (int c = 0; c < kCols; ++c) bscale_next[c] = *reinterpret_cast<const u32x2*>(lds + sb_addr + c * 512 + col_scale_slot);
    };

    auto clear_acc = [&]() __attribute__((always_inline)) { static_for<kRowTiles * kCols>([&](auto n) __attribute__((always_inline)) { clear_acc_tile<16 * decltype(n)::value>(); }); };
    auto epilogue = [&](const TileInfo& info) __attribute__((always_inline)) {
        const int lane = lane_now(), g = lane >> 5, lr = lane & 31;
        static_for<kRowTiles>([&](auto i_constant) __attribute__((always_inline)) {
            constexpr int i = decltype(i_constant)::value;
            const bool row_exists = lr < info.valid - 32 * i;
            const size_t row = static_cast<size_t>(info.row0) + 32 * i + lr;
            if constexpr (kGateUp) {
                store_gate_up_pairs(p, [&](auto at) __attribute__((always_inline)) {
                    constexpr int gate = 32 * i + decltype(at)::value, up = gate + 16;
                    const uint32_t gates = pack_bf16x2(read_acc<gate>(), read_acc<gate + 1>());
                    return u32x2{gates, pack_bf16x2(read_acc<up>(), read_acc<up + 1>())};
                }, row, row_exists, (info.nt * (kBN / 64) + wave) * 32, g);
            } else {
                store_output(p, read_acc_tile<32 * i>(), row, row_exists, info.nt * kBN + wave * kCols * 32, g);
                store_output(p, read_acc_tile<32 * i + 16>(), row, row_exists, info.nt * kBN + (wave * kCols + 1) * 32, g);
            }
        });
    };

    // ---- prologue: activations and scales of items 0..3, weights of items 0 and 1; all of it arrives before item 0, which the counted waits build on -----------------------------------------
    static_for<4>([&](auto pos) __attribute__((always_inline)) {
        if (decltype(pos)::value == 0) request_span();
        static_for<kRowTiles>([&](auto piece) __attribute__((always_inline)) { request_activations_at(pos, piece, my_rows[(copy_ordinal & 1) * kBM + decltype(piece)::value * 32]); });
        advance_activations(true, decltype(pos)::value == 3);
    });
    static_for<Cfg::kRing>([&](auto slot) __attribute__((always_inline)) {
        request_weights(slot, std::integral_constant<int, 0>{});
        request_weights(slot, std::integral_constant<int, 1>{});
        advance_weights(false);
    });
    wait_copies_then_barrier<0>();
    int read_span = 0;
    read_col_scales();
#pragma unroll
    for (int i = 0; i < kRowTiles; ++i) {
        read_row_scale(0, i);
        read_fragment(0, 0, i);
    }
    clear_acc();
    asm volatile("s_nop 3");
    int ordinal = 0, kt = 0;
    // Row tiles that hold a row; none for a wave whose columns are only padding.
    auto live_row_tiles = [&](const TileInfo& tile_info) __attribute__((always_inline)) {
        return __builtin_amdgcn_readfirstlane(tile_info.nt * kBN + wave * 64 < p.n_real ? (tile_info.valid + 31) / 32 : 0);
    };
    TileInfo info = decode(tile_of(0));
    int row_tiles = live_row_tiles(info);
    long long items_left = static_cast<long long>(my_tiles) * ktiles;
    constexpr int kMfmas = kRowTiles * kCols;

    auto item_body = [&](auto pos) __attribute__((always_inline)) {
        constexpr int kPos = decltype(pos)::value, kSlot = kPos % Cfg::kRing;
        constexpr std::integral_constant<int, kSlot> slot{};
        if (kPos == 0) {
#pragma unroll
            for (int c = 0; c < kCols; ++c) bscale_now[c] = bscale_next[c];
        }
        const int scale_b0 = static_cast<int>(bscale_now[0][kPos >> 1]), scale_b1 = static_cast<int>(bscale_now[1][kPos >> 1]);
        int shifted[kRowTiles];
#pragma unroll
        for (int i = 0; i < kRowTiles; ++i) shifted[i] = ascale[i] >> (8 * g);
        const int first_step = 2 * (kt + kPos);
        const int live0 = first_step < steps ? row_tiles : 0, live1 = first_step + 1 < steps ? row_tiles : 0;
        auto mfma = [&](auto step, auto n) __attribute__((always_inline)) {
            constexpr int kStep = decltype(step)::value, kN = decltype(n)::value, kI = kN / kCols, kC = kN % kCols;
            if constexpr (kC == 0)
                mfma_row_tile<kI, Cfg::kWeightRegs + 16 * kSlot + 8 * kStep, 2 * (kPos & 1) + kStep, 2 * kStep>(
                    afrag[kI], scale_b0, scale_b1, shifted[kI], kStep == 0 ? live0 : live1);
        };
        wait_requests<Cfg::kWaitFirst>();
        static_for<kMfmas>([&](auto n) __attribute__((always_inline)) {
            constexpr int kN = decltype(n)::value;
            mfma(std::integral_constant<int, 0>{}, n);
            if constexpr (kN % kCols == kCols - 1) read_fragment(kPos, 1, kN / kCols);
        });
        request_weights(slot, std::integral_constant<int, 0>{});
        wait_requests<Cfg::kWaitSecond>();
        if (kPos == 3) {
            ++read_span;
            row_scale_at = row_scales_of(read_span & 1, kt + 4 == ktiles ? 0 : kt + 4);
            col_scale_slot = (read_span & 1) * Cfg::kColScaleSlot;
            read_col_scales();
        }
        uint32_t copy_from[kRowTiles];
        static_for<kMfmas>([&](auto n) __attribute__((always_inline)) {
            constexpr int kN = decltype(n)::value;
            mfma(std::integral_constant<int, 1>{}, n);
            if constexpr (kN == kCols - 1) {
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
                for (int i = 0; i < kRowTiles; ++i) copy_from[i] = my_rows[(copy_ordinal & 1) * kBM + i * 32];
                if (kPos == 0) request_span();
            }
            if constexpr (kN >= 3 && kN < 3 + kRowTiles) request_activations_at(pos, std::integral_constant<int, kN - 3>{}, copy_from[kN - 3]);
            if constexpr (kN % kCols == kCols - 1) {
                read_row_scale((kPos + 1) & 3, kN / kCols);
                read_fragment((kPos + 1) & 3, 0, kN / kCols);
            }
        });
        request_weights(slot, std::integral_constant<int, 1>{});
        advance_activations(false, kPos == 3);
        advance_weights(((kPos + Cfg::kRing) & 3) == 3);
    };

    for (; items_left > 0; items_left -= 4) {
        static_for<4>(item_body);
        kt += 4;
        if (__builtin_expect(kt == ktiles, 0)) {
            settle_accumulators();
            epilogue(info);
            clear_acc();
            // (read once more: kept across the epilogue, the next item's fragments and row scales would cost it 36 registers)
#pragma unroll
            for (int i = 0; i < kRowTiles; ++i) {
                read_row_scale(0, i);
                read_fragment(0, 0, i);
            }
            asm volatile("s_nop 3");
            kt = 0;
            if (++ordinal < my_tiles) {
                info = decode(tile_of(ordinal));
                row_tiles = live_row_tiles(info);
            }
        }
    }
    // Nothing may still be in flight into this workgroup's LDS or registers when it retires.
    wait_copies_then_barrier<0>();
}

// What the GEMM works on for a logical dimension (hidden or intermediate): whole 256-column tiles and whole spans of
// scales, at least 512 (a row's scale bytes fill one 16-byte copy).  Weights are padded when they are prepared,
// activations by a copy of their own before the first GEMM; padding multiplies zero codes.
int padded_dim(int dim) { return dim <= 512 ? 512 : (dim + 255) / 256 * 256; }

int check_gemm(const char* what, int n, int k, int num_local)
{
    DPEP_REQUIRE(num_local >= 1 && num_local <= kMaxMoeExperts, "%s: number of local experts %d outside [1, %d]", what,
                 num_local, kMaxMoeExperts);
    DPEP_REQUIRE(k >= 512 && k % 256 == 0, "%s: K=%d must be a multiple of 256, at least 512", what, k);
    DPEP_REQUIRE(n > 0 && n % kBN == 0, "%s: N=%d must be a positive multiple of %d", what, n, kBN);
    return DPEP_OK;
}

int gemm_grid()
{
    int device = 0, cus = 256;
    if (hipGetDevice(&device) == hipSuccess) {
        int value = 0;
        if (hipDeviceGetAttribute(&value, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess && value > 0) cus = value;
    }
    return cus / 8 * 8;  // one resident workgroup per CU (the LDS ring takes most of the 160 KiB)
}

// Raising the dynamic LDS limit is a setting per function and per device (each device holds its own copy of the code
// object).  One flag per device; two threads that both find it clear both make the (idempotent) call.
template <typename Kernel>
int allow_lds(Kernel kernel, int bytes, std::atomic<bool>* configured, int max_devices)
{
    int device = 0;
    DPEP_HIP(hipGetDevice(&device));
    const bool tracked = device >= 0 && device < max_devices;
    if (!tracked || !configured[device].load(std::memory_order_acquire)) {
        DPEP_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
        if (tracked) configured[device].store(true, std::memory_order_release);
    }
    return DPEP_OK;
}

// Two workgroups on a CU each run at about half speed: worth it where that does not add rounds (512 tiles on 256 CUs: one
// round of 512 instead of two of 256, with twice the requests in flight; 700 tiles: two slow rounds would replace three
// fast ones).
bool two_workgroups_pay(double tiles, int cus) { return 2.0 * ceil(tiles / (2.0 * cus)) <= ceil(tiles / cus); }

template <bool kStreamed, bool kGateUp>
int launch_paired(const GemmParams& p, hipStream_t stream, const char* what)
{
    constexpr int kMaxDevices = 64;
    static std::atomic<bool> configured[kMaxDevices];
    if (int rc = allow_lds(&grouped_gemm_paired_kernel<kStreamed, kGateUp>, PairCfg::kLdsBytes, configured, kMaxDevices)) return rc;
    hipLaunchKernelGGL((grouped_gemm_paired_kernel<kStreamed, kGateUp>), dim3(2 * gemm_grid()), dim3(kGemmThreads), PairCfg::kLdsBytes, stream, p);
    return launch_status(what);
}

bool column_waves(const GemmParams& p) { return p.column_waves && p.k % 512 == 0; }

template <int RT, bool kGateUp>
int launch_gemm_rt(const GemmParams& p, double expected_tiles, hipStream_t stream, const char* what)
{
    constexpr int kMaxDevices = 64;
    if (column_waves(p)) {
        constexpr int kLds = ColCfg<RT>::kLdsBytes;
        static std::atomic<bool> configured[kMaxDevices];
        if (int rc = allow_lds(&grouped_gemm_colwave_kernel<RT, kGateUp>, kLds, configured, kMaxDevices)) return rc;
        const int cus = gemm_grid();
        const int per_cu = ColCfg<RT>::kWorkgroupsPerCu == 2 && two_workgroups_pay(expected_tiles, cus) ? 2 : 1;
        hipLaunchKernelGGL((grouped_gemm_colwave_kernel<RT, kGateUp>), dim3(cus * per_cu), dim3(kGemmThreads), kLds, stream, p);
        return launch_status(what);
    }
    constexpr int kLds = GemmCfg<RT, kGateUp>::kLdsBytes;
    static std::atomic<bool> configured[kMaxDevices];
    if (int rc = allow_lds(&grouped_gemm_kernel<RT, kGateUp>, kLds, configured, kMaxDevices)) return rc;
    hipLaunchKernelGGL((grouped_gemm_kernel<RT, kGateUp>), dim3(gemm_grid()), dim3(kGemmThreads), kLds, stream, p);
    return launch_status(what);
}

// How many rows an expert is expected to have (the true counts stay on the device).
struct ExpectedRows {
    double routed;  // of a routed expert
    double spread;  // standard deviation of that: a token goes to a given expert or not
    int shared;     // of a shared expert: every token
};

// Kernel and row-tile height, by a small cost model: 64, 128 or 192 rows, or the few-rows kernel's 32 with one or four waves per
// workgroup.  Judged from the expected rows per expert (the true counts stay on the device).  Routing scatters the counts
// around that mean, and one expert a few rows over a multiple of the tile height costs a whole extra row tile each: the tile
// count is therefore the expectation of ceil(rows / height) under a normal spread, not ceil(mean / height); an expert
// without rows has no tile.  (Mean 256 over 8 experts: 128-row tiles need 2.5 row tiles per expert on average = 320 tiles = two
// rounds on 256 CUs, 192-row tiles need 2 = one round; measured 94 vs 67 us.)
// Times are in microseconds, fitted to kernel traces of both GEMMs on an MI355X at 263 shapes (2 to 100 experts, k from 512 to
// 8192): once per launch; per round of one tile per CU its epilogue and switch, and per k tile the main loop and the weights'
// way from memory, which the row tiles of an expert share; nothing below the time to read the weights once.  What it picks is 1.3 %
// slower than the best on average.  How to refit: force each height with the workspace setting "gemm_tile_rows" and
// take a kernel trace.
// The few-rows kernel is the better one for small launches whatever the rows: a CU draws no more than about 50 GB/s from
// memory, and with up to 64 tiles one-wave workgroups spread the columns over four times as many CUs (2 experts of
// 7168 x 2048, 24 rows each: first GEMM 27 us with 64-row tiles, 24 with four waves, 17.5 with one; 192 rows: 35, 23, 34; 16 of
// 1024 x 512, 24 rows: 12.7, 7.7, 6.6).  Large ones it streams as well as the 64-row kernel up to about 20 rows, where a
// tile of 32 still holds nearly all experts (64 of 7168 x 2048, 20 rows: 148 against 154 us; 28 rows: 168 against 159).
struct GemmChoice {
    int rows;      // row-tile height: 64, 128, 192; 32: the few-rows kernel
    int waves;     // per workgroup (4 but for the few-rows kernel's small launches)
    double tiles;  // expected, of that height
    bool paired, streamed;  // 128 rows: the kernel with two workgroups to a CU; its weights past the caches
    bool direct;            // 32 rows, one wave: the kernel without LDS
    double row_tiles_per_expert;  // 32 rows: of the experts that have any
};
template <bool kGateUp>
GemmChoice choose_gemm(const GemmParams& p, const ExpectedRows& expected, int cus)
{
    const int n_tiles = p.n / kBN, ktiles = p.k / kBK;
    const int num_shared = p.num_local - p.num_routed;
    const double mean = expected.routed;
    const double routed_with_rows = 1.0 - exp(-mean);
    auto expected_row_tiles = [&](int bm) {
        // E[ceil(X / bm)] = sum over j >= 0 of P(X > j * bm), which is 1 up to six deviations below the mean
        const int sure = std::max(0, static_cast<int>((mean - 6.0 * expected.spread) / bm));
        double m_tiles = routed_with_rows + sure;
        for (int j = sure + 1; j * bm < mean + 6.0 * expected.spread; ++j)
            m_tiles += 0.5 * erfc((j * bm + 0.5 - mean) / (expected.spread * 1.4142135623730951));
        return p.num_routed * m_tiles + static_cast<double>(num_shared) * ((expected.shared + bm - 1) / bm);
    };
    // Rounds of `unit` workgroups; a stray tile in one launch out of a hundred does not count.
    auto rounds_of = [](double tiles, double unit) { return std::max(1.0, ceil(tiles / unit - 0.01)); };
    const double weight_bytes = (p.num_routed * routed_with_rows + num_shared) * n_tiles * ktiles * 16896.0;
    // Nothing ends before the weights are read; where that decides, the one that would be done first otherwise is still better.
    auto bounded = [&](double t) { return std::max(2.0 + weight_bytes / 6.3e6, t) + 0.05 * t; };
    const int kind = column_waves(p) ? 0 : 1;  // the kernel that launch_gemm_rt takes: column waves, 2 x 2
    double paired_row_tiles = 0.0;
    int best = 2;
    double best_cost = 1e30, tiles_of[4] = {0.0, 0.0, 0.0, 0.0};
    for (int rt = 1; rt <= 3; ++rt) {
        const double row_tiles = expected_row_tiles(64 * rt);
        if (rt == 2) paired_row_tiles = row_tiles;
        const double tiles = row_tiles * n_tiles;
        tiles_of[rt] = tiles;
        const bool in_pairs = rt == 1 && kind == 0 && two_workgroups_pay(tiles, cus);
        const double rounds = in_pairs ? 2.0 * rounds_of(tiles, 2.0 * cus) : rounds_of(tiles, cus);
        constexpr double kFirst[2][3] = {{1.7, 0.4, 0.3}, {5.3, 3.1, 1.2}}, kPerTile[2][3] = {{3.7, 4.4, 8.7}, {3.2, 4.5, 6.5}};
        constexpr double kPerItem[2][3] = {{0.61, 0.77, 0.99}, {0.52, 0.85, 1.10}}, kWeights[2][3] = {{0.0, 0.01, 0.10}, {0.02, 0.03, 0.06}};
        const double per_item = kPerItem[kind][rt - 1] + kWeights[kind][rt - 1] * p.num_local / std::max(row_tiles, 1e-3);
        const double cost = bounded(kFirst[kind][rt - 1] + rounds * (kPerTile[kind][rt - 1] + ktiles * per_item));
        if (cost < best_cost - 1e-9) {
            best_cost = cost;
            best = rt;
        }
    }
    // The 128-row paired kernel: full rounds of two tiles per CU, then a last one that is a pair or, with at most one tile per CU, a
    // single tile; per tile its start and end, per item a part that grows with the 32-row tiles that hold rows and one for weights that
    // few row tiles share.  It counts only what is not padding.  Fitted to kernel traces of both GEMMs at 240 shapes (8 to 10 000 rows for
    // each of 2 to 64 experts), three sets of inputs in turn: 7 % off on average; with it among the candidates the chosen kernels
    // are 5.6 % faster on average (1.2 % slower than the best ones, 6.8 % without it).
    double paired = 1e30;
    bool streamed = false;
    const double experts_with_rows = p.num_routed * routed_with_rows + num_shared, live_row_tiles = expected_row_tiles(32);
    if (p.column_waves) {
        const int steps = (p.k_real + 63) / 64, items = ((steps - 1) / 2 + 4) / 4 * 4, slots = 2 * cus;
        const double live = live_row_tiles / std::max(paired_row_tiles, 1e-3);
        const double share = experts_with_rows / std::max(paired_row_tiles, 1e-3);
        const double tiles = paired_row_tiles * p.live_n_tiles, full = floor(std::max(0.0, tiles / slots - 0.01)), rest = (tiles - full * slots) / cus;
        const double pair = 5.0 + items * (0.652 + 0.147 * live + 0.269 * share), single = 3.37 + items * (0.236 + 0.112 * live + 0.135 * share);
        const double t = 2.94 + full * pair + (rest > 1.01 ? pair : rest > 0.0 ? single : 0.0);
        const double live_bytes = experts_with_rows * p.live_n_tiles * ((steps + 1) / 2) * 16896.0;
        // A long launch pulls its own clock down (1.8 to 1.9 GHz where a reduce has 2.3), and where it has nothing to jump over, 192-row tiles win by moving a third fewer
        // weights: of nine launches of 8 and more rounds with less than 6 % of padding in those tiles they were 1.6 % faster on average
        // (8192 x top-8 over 32 experts of 7168 x 2048: first GEMM 1343 us against 1375, second 803 against 840).
        const double tall_work = tiles_of[3] * 6.0 * ktiles * 2.0, live_work = live_row_tiles * p.live_n_tiles * steps;
        const bool power_limited = kind == 0 && best == 3 && full >= 8.0 && tall_work < 1.06 * live_work;
        // (the factor: a kernel as good by the model is the safer choice. It halves the launches that get slower, 28 of 920, at the same mean)
        if (!power_limited) paired = 1.05 * (std::max(2.0 + live_bytes / 5.32e6, t) + 0.05 * t);
        // Weights that the memory-side cache does not hold, each read by about one row tile: past the caches.
        streamed = live_bytes > 256e6 && paired_row_tiles < 1.3 * experts_with_rows;
    }
    const GemmChoice pair_choice = {128, kGemmWaves, paired_row_tiles * p.live_n_tiles, true, streamed, false, 0.0};
    // Source rows are addressed with 32 bits in the few-rows kernel.
    const double tiles = live_row_tiles * p.live_n_tiles, row_tiles_per_expert = live_row_tiles / std::max(experts_with_rows, 1e-3);
    // One-wave workgroups without LDS while there is at most one to a CU (16 % faster than with it over 167 launches, a tenth where tiles are
    // full), or two with about half a dozen rows per tile (4 % over 67); with more of either they are 1 to 20 % slower.
    const double waves = kGemmWaves * tiles, rows_per_tile = (p.num_routed * mean + static_cast<double>(num_shared) * expected.shared) * p.live_n_tiles / std::max(tiles, 1e-3);
    // And while k is long enough for its requests to run ahead: up to four k tiles (one span) it is no faster, up to eight 6 % slower with more waves
    // than CUs (42 launches with more than eight there: 9 % faster; 9 tokens over 38 experts of 1216 x 512, second GEMM 4.4 us with LDS, 5.6).
    const bool direct = (waves <= cus && p.k_real > 4 * kBK) || (waves <= 2.0 * cus && rows_per_tile <= 6.0 && p.k_real > 8 * kBK);
    if (p.column_waves && p.forced == 0) {
        // (by the padded sizes, as fitted: by the real ones these kernels look too good where little of a tile is real)
        const double all_tiles = live_row_tiles * n_tiles;
        const bool few_allowed = !kGateUp || static_cast<long long>(p.a_rows) * p.k < (1LL << 32);
        const double one = few_allowed ? bounded(3.0 + 0.30 * ktiles + (rounds_of(kGemmWaves * all_tiles, cus) - 1.0) * (1.1 + 0.17 * ktiles)) : 1e30;
        const double four = few_allowed ? bounded(1.5 + rounds_of(all_tiles, cus) * (2.7 + 0.50 * ktiles)) : 1e30;
        // Zero rows of the output that another kernel's idle workgroups write meanwhile (at about 30 GB/s each): the paired kernel leaves
        // them to the reduce, which writes them at 8 TB/s. (Not held against the few-rows kernels: where the model prefers them they win by
        // far more; 4300 zero rows of 6272 columns beside 3 experts of 6272 x 768, 95 rows each: 48 us with 64-row tiles and fillers, 36 without.)
        double unfilled = 0.0;
        if (p.fill_tokens > 0 && tiles_of[best] < cus) {
            const double zeros = p.fill_tokens * exp(-mean * p.num_routed / p.fill_tokens) * p.fill_vec * 16.0;
            unfilled = std::min(zeros, (cus - tiles_of[best]) * 30e3 * best_cost) / 11e6;
        }
        const double few = std::min(one, four);
        // (Against 64-row tiles, whose model is the worst of these where an expert has one of them, the paired kernel has to be a tenth ahead, but for
        // the shortest k: whole forwards 336 tokens x top-1 of 8000 x 2688 over 14 experts and a shared one 159.3 -> 147.0 us, 888 x 4 of 5312 x 512 over 40
        // 77.8 -> 67.7, 1000 x 2 of 7168 x 1024 over 48 146.2 -> 135.3; with k of 256, 1424 x 6 of 4224 x 256 over 26 46.9 and 56.5.)
        const double margin = best == 1 && p.k_real > 384 ? 1.1 : 1.0;
        if (paired + unfilled < few && (paired + unfilled) * margin < best_cost) return pair_choice;
        if (few < best_cost) return {32, one < four ? 1 : kGemmWaves, tiles, false, false, one < four && direct, row_tiles_per_expert};
    }
    if ((p.forced & 0xff) == 32) return {32, p.forced >> 8, tiles, false, false, (p.forced >> 8) == 1 && direct, row_tiles_per_expert};
    if ((p.forced & 0xff) == 128 && p.forced >> 8 != 0) return {128, kGemmWaves, paired_row_tiles * p.live_n_tiles, true, p.forced >> 8 == 2, false, 0.0};
    if (p.forced != 0) best = p.forced / 64;
    return {64 * best, kGemmWaves, tiles_of[best], false, false, false, 0.0};
}

// A one-wave launch of a share with more than 64 rows per expert fills with this many waves: 16 to 60 MB of zeros beside 4 to 12 experts
// cost the forward between 1 % more and 2.5 % less than in the reduce, nearly the same with 32 or 128 of them. With fewer rows, and beside
// four-wave workgroups, whose CUs the fillers take, it costs more than it gives (3584 tokens of 2176 columns, 4 experts: first GEMM 15.7 us
// alone, 16.9 with fillers, the reduce 4.5 either way).
constexpr int kFewRowsFillers = 64;

template <bool kGateUp>
int launch_gemm(const GemmParams& p, const GemmChoice& choice, const ExpectedRows& expected, hipStream_t stream, const char* what)
{
    if (choice.rows == 32) {
        DPEP_REQUIRE(!kGateUp || static_cast<long long>(p.a_rows) * p.k < (1LL << 32), "%s: 32-row tiles address at most 4 GiB of input rows", what);
        // Workgroups for more rows than expected (those without a tile end at once, while one with two doubles the time).
        const int num_shared = p.num_local - p.num_routed;
        const long long row_tiles =
            static_cast<long long>(p.num_routed) * static_cast<long long>(ceil(std::max(1.0, expected.routed + 3.0 * expected.spread) / 32.0)) +
            static_cast<long long>(num_shared) * ((expected.shared + 31) / 32);
        // One-wave workgroups whose expert has several row tiles: an even number of column tiles, so that a quarter of a column tile
        // lands on the same XCD for every row tile (workgroups are dealt round-robin over the 8) and its weights are in that XCD's
        // L2 (38 rows for each of 5 experts of 3904 x 1152, nine column tiles: 29.3 us, numbered as ten 27.8).
        GemmParams numbered = p;
        numbered.numbered_n_tiles = p.live_n_tiles + (choice.waves == 1 && choice.row_tiles_per_expert > 1.25 ? p.live_n_tiles & 1 : 0);
        const unsigned grid = static_cast<unsigned>(row_tiles * numbered.numbered_n_tiles);
        if (choice.waves == 1 && p.fill_out != nullptr && expected.routed > 64.0) numbered.few_rows_fillers = kFewRowsFillers;
        if (choice.direct)
            hipLaunchKernelGGL(grouped_gemm_one_wave_kernel<kGateUp>, dim3(kGemmWaves * grid + numbered.few_rows_fillers), dim3(64), 0, stream, numbered);
        else if (choice.waves == 1)
            hipLaunchKernelGGL((grouped_gemm_few_rows_kernel<1, kGateUp>), dim3(kGemmWaves * grid + numbered.few_rows_fillers), dim3(64), 0, stream, numbered);
        else
            hipLaunchKernelGGL((grouped_gemm_few_rows_kernel<kGemmWaves, kGateUp>), dim3(grid), dim3(kGemmThreads), 0, stream, numbered);
        return launch_status(what);
    }
    if (choice.paired) return choice.streamed ? launch_paired<true, kGateUp>(p, stream, what) : launch_paired<false, kGateUp>(p, stream, what);
    if (choice.rows == 64) return launch_gemm_rt<1, kGateUp>(p, choice.tiles, stream, what);
    if (choice.rows == 128) return launch_gemm_rt<2, kGateUp>(p, choice.tiles, stream, what);
    return launch_gemm_rt<3, kGateUp>(p, choice.tiles, stream, what);
}

// The sizes of one of the two GEMMs of a forward, and the workspace's settings for it (ws == nullptr: the defaults).
struct MegaSizes {
    int num_tokens, hidden, intermediate, num_topk, num_experts, num_local, num_shared;
};
GemmParams gemm_of(const MegaSizes& m, const Workspace* w, bool second)
{
    const int hp = padded_dim(m.hidden), ip = padded_dim(m.intermediate);
    GemmParams p{};
    p.topk = second ? 1 : m.num_topk;
    p.a_rows = second ? 0 : m.num_tokens;
    p.num_local = m.num_local + m.num_shared;
    p.num_routed = m.num_local;
    p.n = second ? hp : 2 * ip;
    p.k = second ? ip : hp;
    p.n_real = second ? m.hidden : 2 * m.intermediate;
    p.k_real = second ? m.intermediate : m.hidden;
    p.live_n_tiles = second ? (m.hidden + kBN - 1) / kBN : p.n / kBN;
    const int forced = w == nullptr ? 0 : w->gemm_tile_rows;
    p.forced = forced == 32 ? 32 | w->gemm_few_rows_waves << 8 : forced == 128 ? 128 | w->gemm_paired << 8 : forced;
    p.column_waves = w != nullptr ? w->gemm_column_waves : 1;
    // Without shared experts most tokens of a share have no row: workgroups of the first GEMM that get no tile
    // zero those rows of y meanwhile, and the weighted reduce skips what they got through.  (Served-only: rows of y whose
    // token no local expert serves are nobody's business, neither the fillers' nor the reduce's; with shared experts every
    // token is served.)
    if (!second && m.num_shared == 0 && m.num_local < m.num_experts && (w == nullptr || (w->gemm_zero_fill && !w->megamoe_served_only))) {
        p.fill_tokens = m.num_tokens;
        p.fill_vec = m.hidden / 8;
        p.fill_topk = m.num_topk;
    }
    return p;
}
// Expected rows (the true counts stay on the device): tokens * topk / experts per routed expert, every token for a shared one.
ExpectedRows expected_rows_of(const MegaSizes& m)
{
    const double routed = static_cast<double>(m.num_tokens) * m.num_topk / m.num_experts;
    return {routed, sqrt(routed * std::max(0.0, 1.0 - static_cast<double>(m.num_topk) / m.num_experts)) + 1e-3, m.num_tokens};
}
// Kernels of both GEMMs.  The second one first: the paired and the few-rows kernel read no padding of the activations, so that the first
// GEMM, if it is one of these too, leaves out the column tiles that would only write some.
struct GemmChoices {
    GemmChoice first, second;
};
GemmChoices choose_gemms(const MegaSizes& m, GemmParams& g1, const GemmParams& g2)
{
    const ExpectedRows expected = expected_rows_of(m);
    GemmChoices c;
    c.second = choose_gemm<false>(g2, expected, gemm_grid());
    if (c.second.paired || c.second.rows == 32) g1.live_n_tiles = (g1.n_real + kBN - 1) / kBN;
    c.first = choose_gemm<true>(g1, expected, gemm_grid());
    return c;
}

}  // namespace

// ---- host replay of one workgroup's schedule ---------------------------------------------------------------
// Vector-memory operations complete in issue order, and a wait for "at most N in flight" guarantees no more than
// that all but the newest N have completed.  The replay issues what the kernel issues, in the kernel's order (the
// prologue's kAhead items; per item: the counted wait, the copies of the item kAhead ahead with their scale and index
// copies, the cursor's tile switch; epilogue stores at tile ends), lets nothing complete that a wait has not
// forced, and checks that every item's copies have completed when its fragments are read and that the gather
// indices of a tile have when the cursor reads them.
struct ScheduleFault {
    int item, what;  // what: 1 = an item's operands, 2 = gather indices, 3 = scale slots, 4 = weights of another item
};

// The rings of scale slots: a span's scales (the scales of item x are read during the body of item x - 1) must all have
// been read when the copies of a later span go into the same slot; the copies are issued behind the barrier of the body
// that is running (-1: the prologue, before anything is read).
struct ScaleSlots {
    long long last_item[4] = {-1, -1, -1, -1};  // of the span each slot holds
    int slots, next = 0;
    explicit ScaleSlots(int n) : slots(n) {}
    bool take(long long span_last_item, long long body)  // false: the slot's present span is still being read
    {
        const long long held = last_item[next];
        last_item[next] = span_last_item;
        next = next + 1 == slots ? 0 : next + 1;
        return held < 0 || held <= body;
    }
};

template <int RT>
bool replay_workgroup(int my_tiles, int ktiles, int epilogue_stores, bool drain_at_switches, int scale_slots, ScheduleFault* fault)
{
    using Ring = GemmRing<RT>;
    constexpr int kAhead = Ring::kAhead, kCopies = Ring::kCopies;
    ScaleSlots scales(scale_slots);
    long long body = -1;
    const long long n_items = static_cast<long long>(my_tiles) * ktiles;
    if (n_items == 0) return true;
    long long issued = 0, done = 0;  // operations [0, done) have certainly completed
    auto wait = [&](long long in_flight) {
        if (issued - in_flight > done) done = issued - in_flight;
    };
    int copy_kt = 0, copy_tile = 0;
    long long copy_item = 0;   // ordinal of the item under the cursor
    long long index_op = -1;   // operation that fetches the indices of the cursor's next tile
    static thread_local long long item_last_op[1 << 16];
    if (n_items >= (1 << 16)) return true;  // not replayed (far beyond any real workgroup's share)
    bool ok = true, past_end = false;
    auto issue_copies = [&]() {
        issued += kCopies;
        if ((copy_kt & 3) == 0) {
            issued += 2;  // row and column scales of the span
            if (!scales.take(copy_item + (ktiles - 1 - copy_kt < 3 ? ktiles - 1 - copy_kt : 3), body) && ok) {
                ok = false;
                *fault = {static_cast<int>(body), 3};
            }
        }
        if (copy_kt == 0) index_op = issued++;    // (re-copies past the end sit on the last k tile, never 0)
        if (!past_end) item_last_op[copy_item] = issued - 1;
    };
    auto advance = [&](bool in_prologue, int item) {
        if (++copy_kt == ktiles) {
            if (copy_tile + 1 < my_tiles) {
                if (drain_at_switches && switch_needs_drain(in_prologue, ktiles, kAhead)) wait(0);
                if (index_op >= done && ok) {
                    ok = false;
                    *fault = {item, 2};
                }
                ++copy_tile;
                copy_kt = 0;
                ++copy_item;
            } else {
                copy_kt = ktiles - 1;  // past the last tile: keep re-copying its last item (never read)
                past_end = true;
            }
        } else if (!past_end) {
            ++copy_item;
        }
    };
    auto check_item = [&](long long item) {
        if (item < n_items && item_last_op[item] >= done && ok) {
            ok = false;
            *fault = {static_cast<int>(item), 1};
        }
    };
    ++issued;  // the first tile's own indices, fetched synchronously
    wait(0);
    for (int j = 0; j < kAhead; ++j) {
        issue_copies();
        advance(true, -1);
    }
    wait((kAhead - 1) * kCopies);
    check_item(0);
    int kt = 0;
    for (long long item = 0; item < n_items; ++item) {
        wait(Ring::kWaitPlain);
        check_item(item + 1);  // its first fragments leave LDS during this item's second k step
        body = item;
        issue_copies();
        advance(false, static_cast<int>(item));
        if (++kt == ktiles) {
            issued += epilogue_stores;
            kt = 0;
        }
    }
    return ok;
}

// The same replay for the column-wave kernel: the prologue requests items 0..3 (each: its span's scales and the next tile's
// gather indices where it opens a span / a tile, its activation copies, its weight loads), then waits; every item's body
// waits (kWait + slack in flight), then requests the item four ahead in the same order; tiles end behind every ktiles-th
// item with the epilogue's stores.  slack > 0 replays a kernel whose wait is laxer than the real one.
template <int RT>
bool replay_column_waves(int my_tiles, int ktiles, int epilogue_stores, int slack, ScheduleFault* fault)
{
    using Ring = ColumnRing<RT>;
    const long long n_items = static_cast<long long>(my_tiles) * ktiles;
    if (n_items == 0) return true;
    static thread_local long long item_last_op[1 << 16];
    if (n_items >= (1 << 16)) return true;  // not replayed (far beyond any real workgroup's share)
    long long issued = 0, done = 0;
    auto wait = [&](long long in_flight) {
        if (issued - in_flight > done) done = issued - in_flight;
    };
    int copy_kt = 0, copy_tile = 0;
    long long copy_item = 0, index_op = -1;
    bool ok = true, past_end = false;
    ScaleSlots scales(2);
    long long body = -1;
    auto request_item = [&]() {
        if ((copy_kt & 3) == 0) {
            issued += 2;                            // row and column scales of the span
            if (!past_end && !scales.take(copy_item + 3, body) && ok) {
                ok = false;
                *fault = {static_cast<int>(body), 3};
            }
            if (copy_kt == 0) index_op = issued++;  // gather indices of the tile after the cursor's
        }
        issued += Ring::kRequests;
        if (!past_end) item_last_op[copy_item] = issued - 1;
    };
    auto advance = [&](bool in_prologue, int item) {
        ++copy_kt;
        if (!past_end) ++copy_item;
        if (copy_kt == ktiles) {
            if (copy_tile + 1 < my_tiles) {
                if (switch_needs_drain(in_prologue, ktiles, Ring::kStages)) wait(0);
                if (index_op >= done && ok) {
                    ok = false;
                    *fault = {item, 2};
                }
                ++copy_tile;
                copy_kt = 0;
            } else {
                copy_kt = ktiles - 4;  // past the last tile: its last span again (never used)
                if (!past_end) --copy_item;
                past_end = true;
            }
        }
    };
    auto check_item = [&](long long item) {
        if (item < n_items && item_last_op[item] >= done && ok) {
            ok = false;
            *fault = {static_cast<int>(item), 1};
        }
    };
    ++issued;  // the first tile's own indices, fetched synchronously
    wait(0);
    for (int j = 0; j < Ring::kStages; ++j) {
        request_item();
        advance(true, -1);
    }
    wait(Ring::kPrologueWait);
    check_item(0);
    int kt = 0;
    for (long long item = 0; item < n_items; ++item) {
        wait(Ring::kWait + slack);
        check_item(item + 1);  // its first fragments leave LDS during this item's second k step, its weights right after
        body = item;
        request_item();
        advance(false, static_cast<int>(item));
        if (++kt == ktiles) {
            issued += epilogue_stores;
            kt = 0;
        }
    }
    return ok;
}

// The same for the paired kernel, whose weights have a cursor of their own: the prologue asks for items 0..3 (weights: 0 and 1) and waits for all of it;
// an item's body waits for its first weights, asks for the first weights of the item two ahead, waits for its second weights and
// the next item's activations and scales, and asks for the activations of the item four ahead (their span's scales in front) and the rest
// of the weights.  `first_slack`, `second_slack`: a kernel whose waits are laxer by that much.
bool replay_paired(int my_tiles, int ktiles, int epilogue_stores, int first_slack, int second_slack, ScheduleFault* fault)
{
    using Ring = PairedRing;
    const long long n_items = static_cast<long long>(my_tiles) * ktiles;
    constexpr int kMost = 1 << 16;
    if (n_items == 0) return true;
    static thread_local long long activations_op[kMost], scales_op[kMost], weights_op[2][kMost];
    if (n_items >= kMost) return true;  // not replayed (far beyond any real workgroup's share)
    long long issued = 0, done = 0, body = -1;
    bool ok = true;
    auto broken = [&](long long item, int what) {
        if (ok) *fault = {static_cast<int>(item), what};
        ok = false;
    };
    auto wait = [&](long long in_flight) { done = issued - in_flight > done ? issued - in_flight : done; };
    int copy_kt = 0, copy_tile = 0, weight_kt = 0, weight_tile = 0;  // k tile and tile under the two cursors
    long long copy_item = 0, weight_item = 0, index_op = -1;
    bool past_end = false;
    ScaleSlots scales(2);
    auto request_activations = [&](int pos) {
        if (pos == 0) {
            issued += 2;
            if (!scales.take(past_end ? -1 : copy_item + 3, body)) broken(body, 3);
            for (int i = 0; i < 4 && !past_end; ++i) scales_op[copy_item + i] = issued - 1;
            if (copy_kt == 0) index_op = issued++;
        }
        issued += Ring::kActivations;
        if (!past_end) activations_op[copy_item] = issued - 1;
    };
    auto request_weights = [&](int step) {
        issued += Ring::kWeights;
        if (weight_item < n_items) {
            weights_op[step][weight_item] = issued - 1;
            if (weight_item != static_cast<long long>(weight_tile) * ktiles + weight_kt) broken(weight_item, 4);
        }
    };
    auto advance_activations = [&](bool in_prologue, bool last_of_four) {
        ++copy_kt;
        ++copy_item;
        if (!last_of_four || copy_kt != ktiles) return;
        if (copy_tile + 1 < my_tiles) {
            if (switch_needs_drain(in_prologue, ktiles, Ring::kStages)) wait(0);
            if (index_op >= done) broken(body, 2);
            copy_kt = 0;
            ++copy_tile;
        } else {
            copy_kt = ktiles - 4;
            past_end = true;
        }
    };
    auto advance_weights = [&](bool last_of_four) {
        ++weight_kt;
        ++weight_item;
        if (last_of_four && weight_kt == ktiles) {
            weight_kt = 0;
            weight_tile = copy_tile;
        }
    };
    ++issued;  // the first tile's own indices
    wait(0);
    for (int pos = 0; pos < Ring::kStages; ++pos) {
        request_activations(pos);
        advance_activations(true, pos == 3);
    }
    for (int item = 0; item < Ring::kRing; ++item) {
        request_weights(0);
        request_weights(1);
        advance_weights(false);
    }
    wait(0);
    int kt = 0;
    for (long long item = 0; item < n_items; ++item) {
        const int pos = static_cast<int>(item & 3);
        body = item;
        wait(Ring::kWaitFirst + first_slack);
        if (weights_op[0][item] >= done || activations_op[item] >= done) broken(item, 1);
        request_weights(0);
        wait(Ring::kWaitSecond + second_slack);
        if (weights_op[1][item] >= done) broken(item, 1);
        if (item + 1 < n_items && (activations_op[item + 1] >= done || scales_op[item + 1] >= done)) broken(item + 1, 1);
        request_activations(pos);
        request_weights(1);
        advance_activations(false, pos == 3);
        advance_weights(((pos + Ring::kRing) & 3) == 3);
        if (++kt == ktiles) {
            issued += epilogue_stores;
            kt = 0;
        }
    }
    return ok;
}

int launch_gemm1(const GemmParams& p, const GemmChoice& choice, const ExpectedRows& expected, hipStream_t stream)
{
    if (int rc = check_gemm("gemm1", p.n, p.k, p.num_local)) return rc;
    DPEP_REQUIRE(p.row_to_route != nullptr && p.topk >= 1, "gemm1: needs the row -> route map");
    return launch_gemm<true>(p, choice, expected, stream, "grouped_gemm1");
}

int launch_gemm2(const GemmParams& p, const GemmChoice& choice, const ExpectedRows& expected, hipStream_t stream)
{
    if (int rc = check_gemm("gemm2", p.n, p.k, p.num_local)) return rc;
    return launch_gemm<false>(p, choice, expected, stream, "grouped_gemm2");
}

}  // namespace dpep

extern "C" {

int dpep_mx_quant(const void* x, int rows, int hidden, void* codes, uint8_t* scales, void* stream)
{
    using namespace dpep;
    DPEP_REQUIRE(rows >= 0, "mx_quant: bad row count %d", rows);
    DPEP_REQUIRE(hidden > 0 && hidden % 32 == 0, "mx_quant: hidden=%d must be a positive multiple of 32", hidden);
    if (rows == 0) return DPEP_OK;
    DPEP_REQUIRE(x && codes && scales && aligned16(x) && aligned16(codes), "mx_quant: NULL or misaligned buffer");
    const long long units = static_cast<long long>(rows) * (hidden / 16);
    DPEP_REQUIRE((units + kMxThreads - 1) / kMxThreads < (1ll << 31), "mx_quant: %d x %d values are more than one launch takes",
                 rows, hidden);
    const unsigned blocks = static_cast<unsigned>((units + kMxThreads - 1) / kMxThreads);
    if (aligned16(scales))
        hipLaunchKernelGGL(mx_quant_kernel<true>, dim3(blocks), dim3(kMxThreads), 0, static_cast<hipStream_t>(stream),
                           static_cast<const u32x4*>(x), units, static_cast<u32x4*>(codes), scales);
    else
        hipLaunchKernelGGL(mx_quant_kernel<false>, dim3(blocks), dim3(kMxThreads), 0, static_cast<hipStream_t>(stream),
                           static_cast<const u32x4*>(x), units, static_cast<u32x4*>(codes), scales);
    return launch_status("mx_quant");
}

int dpep_megamoe_schedule_check(int tile_rows, int tiles_per_workgroup, int ktiles, int epilogue_stores, int without_drain)
{
    using namespace dpep;
    DPEP_REQUIRE(tile_rows == 64 || tile_rows == 128 || tile_rows == 192, "schedule_check: tile_rows is 64, 128 or 192");
    DPEP_REQUIRE(tiles_per_workgroup >= 0 && ktiles >= 2 && ktiles % 2 == 0 && epilogue_stores >= 0,
                 "schedule_check: bad arguments");
    ScheduleFault fault = {0, 0};
    const bool drain = (without_drain & 1) == 0;
    const int slots = (without_drain & 2) != 0 ? 2 : GemmCfg<1, false>::kScaleSlots;  // (bit 1: the rings as they were, two slots)
    const bool ok = tile_rows == 64    ? replay_workgroup<1>(tiles_per_workgroup, ktiles, epilogue_stores, drain, slots, &fault)
                    : tile_rows == 128 ? replay_workgroup<2>(tiles_per_workgroup, ktiles, epilogue_stores, drain, slots, &fault)
                                       : replay_workgroup<3>(tiles_per_workgroup, ktiles, epilogue_stores, drain, slots, &fault);
    if (!ok && fault.what == 3)
        return fail(DPEP_EINVAL, "schedule_check: a span's scales are overwritten while they are still being read (behind item %d)",
                    fault.item);
    if (!ok)
        return fail(DPEP_EINVAL, "schedule_check: %s read before any wait covers them (item %d)",
                    fault.what == 1 ? "an item's copies are" : "the next tile's gather indices are", fault.item);
    return DPEP_OK;
}

int dpep_megamoe_schedule_check_column_waves(int tile_rows, int tiles_per_workgroup, int ktiles, int epilogue_stores, int slack)
{
    using namespace dpep;
    DPEP_REQUIRE(tile_rows == 64 || tile_rows == 128 || tile_rows == 192, "schedule_check: tile_rows is 64, 128 or 192");
    DPEP_REQUIRE(tiles_per_workgroup >= 0 && ktiles >= 4 && ktiles % 4 == 0 && epilogue_stores >= 0 && slack >= 0,
                 "schedule_check: bad arguments (the column-wave kernel takes k tiles in fours)");
    ScheduleFault fault = {0, 0};
    const bool ok = tile_rows == 64    ? replay_column_waves<1>(tiles_per_workgroup, ktiles, epilogue_stores, slack, &fault)
                    : tile_rows == 128 ? replay_column_waves<2>(tiles_per_workgroup, ktiles, epilogue_stores, slack, &fault)
                                       : replay_column_waves<3>(tiles_per_workgroup, ktiles, epilogue_stores, slack, &fault);
    if (!ok && fault.what == 3)
        return fail(DPEP_EINVAL, "schedule_check: a span's scales are overwritten while they are still being read (behind item %d)",
                    fault.item);
    if (!ok)
        return fail(DPEP_EINVAL, "schedule_check: %s read before any wait covers them (item %d)",
                    fault.what == 1 ? "an item's operands are" : "the next tile's gather indices are", fault.item);
    return DPEP_OK;
}

int dpep_megamoe_schedule_check_paired(int tiles_per_workgroup, int ktiles, int epilogue_stores, int first_slack, int second_slack)
{
    using namespace dpep;
    DPEP_REQUIRE(tiles_per_workgroup >= 0 && ktiles >= 4 && ktiles % 4 == 0 && epilogue_stores >= 0 && first_slack >= 0 && second_slack >= 0,
                 "schedule_check: bad arguments (the paired kernel takes k tiles in fours)");
    ScheduleFault fault = {0, 0};
    if (replay_paired(tiles_per_workgroup, ktiles, epilogue_stores, first_slack, second_slack, &fault)) return DPEP_OK;
    if (fault.what == 3)
        return fail(DPEP_EINVAL, "schedule_check: a span's scales are overwritten while they are still being read (behind item %d)", fault.item);
    if (fault.what == 4) return fail(DPEP_EINVAL, "schedule_check: the weights asked for item %d are another item's", fault.item);
    return fail(DPEP_EINVAL, "schedule_check: %s read before any wait covers them (item %d)", fault.what == 1 ? "operands" : "gather indices", fault.item);
}

int dpep_megamoe_padded_dim(int dim) { return dim < 1 ? 0 : dpep::padded_dim(dim); }

int dpep_megamoe_prepared_shape(int n, int k, int gate_up, int* padded_n, int* padded_k, int* scale_cols)
{
    using namespace dpep;
    DPEP_REQUIRE(padded_n && padded_k && scale_cols, "prepared_shape: NULL output");
    DPEP_REQUIRE(k > 0 && k % 64 == 0, "prepared_shape: K=%d must be a positive multiple of 64", k);
    DPEP_REQUIRE(n > 0 && n % (gate_up ? 256 : 64) == 0, "prepared_shape: N=%d must be a positive multiple of %d", n,
                 gate_up ? 256 : 64);
    *padded_n = gate_up ? 2 * padded_dim(n / 2) : padded_dim(n);
    *padded_k = padded_dim(k);
    *scale_cols = (*padded_k / 128 + 3) / 4 * 16;  // groups of four k tiles, the last one padded
    return DPEP_OK;
}

int dpep_megamoe_prepare_weights(const uint8_t* w_packed, const uint8_t* w_scales, int num_local, int n, int k,
                                 int gate_up, uint8_t* out_packed, uint8_t* out_scales, void* stream)
{
    using namespace dpep;
    DPEP_REQUIRE(num_local >= 1, "prepare_weights: bad expert count %d", num_local);
    int np = 0, kp = 0, scale_cols = 0;
    if (int rc = dpep_megamoe_prepared_shape(n, k, gate_up, &np, &kp, &scale_cols)) return rc;
    DPEP_REQUIRE(w_packed && w_scales && out_packed && out_scales && aligned16(w_packed) && aligned16(out_packed),
                 "prepare_weights: NULL or misaligned buffer");
    DPEP_REQUIRE(w_packed != out_packed && w_scales != out_scales, "prepare_weights: cannot run in place");
    const long long chunks = static_cast<long long>(num_local) * np * (kp / 2) / 16;
    const long long pairs = static_cast<long long>(num_local) * np * scale_cols / 2;
    const long long threads = chunks > pairs ? chunks : pairs;
    const unsigned blocks = static_cast<unsigned>((threads + 255) / 256);
    hipLaunchKernelGGL(prepare_weights_kernel, dim3(blocks), dim3(256), 0, static_cast<hipStream_t>(stream), w_packed,
                       w_scales, n, k, np, kp, gate_up, out_packed, out_scales, chunks, pairs);
    return launch_status("prepare_weights");
}

// Workspace carve-up shared by workspace_bytes and forward.
struct MegaLayout {
    size_t hist, meta, fill_state, route_to_row, row_to_route, x_codes, x_scales, act_codes, act_scales, out2, total;
};

static MegaLayout mega_layout(int num_tokens, int num_topk, int hidden, int intermediate, int num_local, int num_shared)
{
    auto up = [](size_t v) { return (v + 255) / 256 * 256; };
    const size_t routes = static_cast<size_t>(num_tokens) * num_topk;
    const size_t shared_rows = static_cast<size_t>(num_tokens) * num_shared;
    const size_t max_rows = static_cast<size_t>(num_tokens) * (num_topk < num_local ? num_topk : num_local) + shared_rows;
    MegaLayout l;
    size_t at = 0;
    l.hist = at;         at += up(dpep_layout_workspace_bytes(num_tokens, num_topk, num_local));
    l.meta = at;         at += up((3 * static_cast<size_t>(num_local) + num_shared + 2) * 4);
    l.fill_state = at;   at += up((1 + 4096) * 4);  // fillers of the first GEMM: count + progress of each (<= 1024 CUs x 4 waves)
    l.route_to_row = at; at += up(routes * 4);
    l.row_to_route = at; at += up((routes + shared_rows) * 4);
    const size_t hp = dpep::padded_dim(hidden), ip = dpep::padded_dim(intermediate);
    // padded copy of the input rows, only when hidden is not already what the GEMM works on
    l.x_codes = at;      at += hp != static_cast<size_t>(hidden) ? up(static_cast<size_t>(num_tokens) * hp) : 0;
    l.x_scales = at;     at += hp != static_cast<size_t>(hidden) ? up(static_cast<size_t>(num_tokens) * (hp / 32)) : 0;
    l.act_codes = at;    at += up(max_rows * ip);
    l.act_scales = at;   at += up(max_rows * (ip / 32));
    l.out2 = at;         at += up(max_rows * hidden * 2);
    l.total = at;
    return l;
}

size_t dpep_megamoe_workspace_bytes(int num_tokens, int num_topk, int hidden, int intermediate, int num_local,
                                    int num_shared)
{
    if (num_tokens < 1 || num_topk < 1 || hidden < 1 || intermediate < 1 || num_local < 1 || num_shared < 0) return 0;
    return mega_layout(num_tokens, num_topk, hidden, intermediate, num_local, num_shared).total;
}

// What a forward of these sizes takes for its first or second GEMM: the choice, and whether the kernels of every height split the columns.
static int choice_of(const char* what, void* ws, const dpep::MegaSizes& m, bool second, dpep::GemmChoice* choice, bool* by_columns)
{
    using namespace dpep;
    const Workspace* w = as_workspace(ws);
    DPEP_REQUIRE(ws == nullptr || w != nullptr, "%s: not a live workspace", what);
    DPEP_REQUIRE(m.num_tokens >= 1 && m.hidden >= 1 && m.intermediate >= 1 && m.num_topk >= 1 && m.num_experts >= m.num_local && m.num_local >= 1 && m.num_shared >= 0,
                 "%s: bad sizes", what);
    GemmParams g1 = gemm_of(m, w, false), g2 = gemm_of(m, w, true);
    const GemmChoices choices = choose_gemms(m, g1, g2);
    *choice = second ? choices.second : choices.first;
    *by_columns = column_waves(second ? g2 : g1);
    return DPEP_OK;
}

int dpep_megamoe_gemm_choice(void* ws, int num_tokens, int hidden, int intermediate, int num_topk, int num_experts, int num_local,
                             int num_shared, int second, int32_t* tile_rows, int32_t* waves)
{
    DPEP_REQUIRE(tile_rows != nullptr && waves != nullptr, "megamoe_gemm_choice: NULL output");
    dpep::GemmChoice choice;
    bool by_columns;
    if (int rc = choice_of("megamoe_gemm_choice", ws, {num_tokens, hidden, intermediate, num_topk, num_experts, num_local, num_shared}, second != 0, &choice, &by_columns))
        return rc;
    *tile_rows = choice.rows;
    *waves = choice.waves;
    return DPEP_OK;
}

int dpep_megamoe_gemm_kernel(void* ws, int num_tokens, int hidden, int intermediate, int num_topk, int num_experts, int num_local,
                             int num_shared, int second, int32_t* kernel)
{
    DPEP_REQUIRE(kernel != nullptr, "megamoe_gemm_kernel: NULL output");
    dpep::GemmChoice choice;
    bool by_columns;
    if (int rc = choice_of("megamoe_gemm_kernel", ws, {num_tokens, hidden, intermediate, num_topk, num_experts, num_local, num_shared}, second != 0, &choice, &by_columns))
        return rc;
    if (choice.rows == 32) *kernel = choice.direct ? DPEP_GEMM_ONE_WAVE : DPEP_GEMM_FEW_ROWS;
    else if (choice.paired) *kernel = choice.streamed ? DPEP_GEMM_PAIRED_STREAMED : DPEP_GEMM_PAIRED;
    else *kernel = by_columns ? DPEP_GEMM_COLUMN_WAVES : DPEP_GEMM_TWO_BY_TWO;
    return DPEP_OK;
}

int dpep_megamoe_fill_report(void* ws, int num_tokens, int num_topk, int hidden, int intermediate, int num_local,
                             int num_shared, int32_t* fillers_host, int64_t* tokens_filled_host, void* stream)
{
    using namespace dpep;
    Workspace* w = as_workspace(ws);
    DPEP_REQUIRE(w != nullptr && fillers_host != nullptr && tokens_filled_host != nullptr,
                 "megamoe_fill_report: not a live workspace, or NULL output");
    DPEP_REQUIRE(num_tokens >= 1 && num_topk >= 1 && hidden >= 1 && intermediate >= 1 && num_local >= 1 && num_shared >= 0,
                 "megamoe_fill_report: bad sizes");
    const MegaLayout l = mega_layout(num_tokens, num_topk, hidden, intermediate, num_local, num_shared);
    DPEP_REQUIRE(l.total <= w->bytes, "megamoe_fill_report: these are not the sizes of a forward on this workspace");
    static thread_local int32_t state[1 + 4096];
    DPEP_HIP(hipStreamSynchronize(static_cast<hipStream_t>(stream)));
    DPEP_HIP(hipMemcpy(state, static_cast<uint8_t*>(w->base) + l.fill_state, sizeof(state), hipMemcpyDeviceToHost));
    const int fillers = state[0] < 0 ? 0 : state[0] > 4096 ? 4096 : state[0];
    int64_t filled = 0;
    for (int f = 0; f < fillers; ++f) filled += state[1 + f];
    *fillers_host = fillers;
    *tokens_filled_host = filled;
    return DPEP_OK;
}

int dpep_megamoe_forward(void* ws, const void* x_codes, const uint8_t* x_scales, const int32_t* topk_idx,
                         const float* topk_weights, const uint8_t* w1, const uint8_t* s1, const uint8_t* w2,
                         const uint8_t* s2, const uint8_t* shared_w1, const uint8_t* shared_s1,
                         const uint8_t* shared_w2, const uint8_t* shared_s2, int num_shared, int num_tokens, int hidden,
                         int intermediate, int num_topk, int num_experts, int expert_begin, int num_local, void* y,
                         int32_t* expert_token_nums, void* stream)
{
    const dpep_megamoe_call call = {x_codes, x_scales, nullptr, nullptr, nullptr, topk_idx, topk_weights, w1, s1, w2, s2, shared_w1,
                                    shared_s1, shared_w2, shared_s2, y, expert_token_nums, num_shared, num_tokens, hidden,
                                    intermediate, num_topk, num_experts, expert_begin, num_local};
    return dpep_megamoe_run(ws, &call, stream);
}

int dpep_megamoe_run(void* ws, const dpep_megamoe_call* call, void* stream)
{
    using namespace dpep;
    Workspace* w = as_workspace(ws);
    DPEP_REQUIRE(w != nullptr && call != nullptr, "megamoe_forward: not a live workspace, or NULL call");
    const dpep_megamoe_call& c = *call;
    const int num_shared = c.num_shared, num_tokens = c.num_tokens, hidden = c.hidden, intermediate = c.intermediate,
              num_topk = c.num_topk, num_experts = c.num_experts, expert_begin = c.expert_begin, num_local = c.num_local;
    const int32_t* topk_idx = c.topk_idx;
    const float* topk_weights = c.topk_weights;
    const uint8_t *w1 = c.w1, *s1 = c.s1, *w2 = c.w2, *s2 = c.s2;
    const uint8_t *shared_w1 = c.shared_w1, *shared_s1 = c.shared_s1, *shared_w2 = c.shared_w2, *shared_s2 = c.shared_s2;
    void* y = c.y;
    int32_t* expert_token_nums = c.expert_token_nums;
    DPEP_REQUIRE(num_tokens >= 1 && num_topk >= 1 && num_topk <= DPEP_MAX_TOPK, "megamoe_forward: bad B=%d K=%d",
                 num_tokens, num_topk);
    DPEP_REQUIRE(hidden >= 64 && hidden % 64 == 0 && intermediate >= 128 && intermediate % 128 == 0,
                 "megamoe_forward: hidden=%d must be a positive multiple of 64, intermediate=%d of 128", hidden,
                 intermediate);
    const int hp = padded_dim(hidden), ip = padded_dim(intermediate);
    DPEP_REQUIRE(num_local >= 1 && num_local <= kMaxMoeExperts && expert_begin >= 0 &&
                     expert_begin + num_local <= num_experts,
                 "megamoe_forward: bad expert range E=%d begin=%d L=%d (at most %d local experts)", num_experts,
                 expert_begin, num_local, kMaxMoeExperts);
    DPEP_REQUIRE(num_shared >= 0 && num_shared <= 8 && num_topk + num_shared <= DPEP_MAX_TOPK &&
                     num_local + num_shared <= kMaxMoeExperts,
                 "megamoe_forward: %d shared experts with K=%d, L=%d (at most 8, K+S <= %d, L+S <= %d)", num_shared,
                 num_topk, num_local, DPEP_MAX_TOPK, kMaxMoeExperts);
    DPEP_REQUIRE(topk_idx && topk_weights && w1 && s1 && w2 && s2 && y && expert_token_nums, "megamoe_forward: NULL buffer");
    DPEP_REQUIRE(c.x_bf16 == nullptr ? c.x_codes != nullptr && c.x_scales != nullptr && aligned16(c.x_codes)
                                     : c.x_codes_scratch != nullptr && c.x_scales_scratch != nullptr && aligned16(c.x_bf16) &&
                                           aligned16(c.x_codes_scratch) && aligned16(c.x_scales_scratch),
                 "megamoe_forward: NULL or misaligned input rows");
    DPEP_REQUIRE(num_shared == 0 || (shared_w1 && shared_s1 && shared_w2 && shared_s2 && aligned16(shared_w1) &&
                                     aligned16(shared_w2) && aligned16(shared_s1) && aligned16(shared_s2)),
                 "megamoe_forward: shared experts need their four prepared weight buffers, 16-byte aligned");
    DPEP_REQUIRE(aligned16(w1) && aligned16(w2) && aligned16(s1) && aligned16(s2) && aligned16(y),
                 "megamoe_forward: misaligned buffer");
    // the GEMM's copies address activation rows with 32-bit byte offsets
    const long long max_rows = static_cast<long long>(num_tokens) * ((num_topk < num_local ? num_topk : num_local) + num_shared);
    DPEP_REQUIRE(static_cast<long long>(num_tokens) * hp < (1LL << 32) && max_rows * ip < (1LL << 32),
                 "megamoe_forward: activation tensors of B=%d tokens exceed 4 GiB", num_tokens);
    const MegaLayout l = mega_layout(num_tokens, num_topk, hidden, intermediate, num_local, num_shared);
    DPEP_REQUIRE(l.total <= w->bytes, "megamoe_forward: workspace too small (%zu needed, %zu available)", l.total, w->bytes);
    hipStream_t s = static_cast<hipStream_t>(stream);
    uint8_t* base = static_cast<uint8_t*>(w->base);
    int32_t* meta = reinterpret_cast<int32_t*>(base + l.meta);
    int32_t* psum = meta;
    int32_t* offsets = meta + num_local;                          // [L + S + 1]
    int32_t* num_rows = meta + 2 * num_local + num_shared + 1;    // rows of the routed experts
    int32_t* route_to_row = reinterpret_cast<int32_t*>(base + l.route_to_row);
    int32_t* row_to_route = reinterpret_cast<int32_t*>(base + l.row_to_route);
    // Rows that are not what the GEMM works on (BF16, or sizes that are no whole tiles) are prepared by the layout's launch.
    MegaFront front{};
    front.num_shared = num_shared;
    front.num_tokens = num_tokens;
    front.num_topk = num_topk;
    const bool from_bf16 = c.x_bf16 != nullptr;
    const uint8_t* codes = static_cast<const uint8_t*>(c.x_codes);
    const uint8_t* scales = c.x_scales;
    if (from_bf16 || hp != hidden) {
        front.bf16 = static_cast<const u32x4*>(c.x_bf16);
        front.codes = codes;
        front.scales = scales;
        front.h = hidden;
        front.hp = hp;
        front.units = static_cast<unsigned>(static_cast<long long>(num_tokens) * (hp / 16));
        uint8_t* const codes_out = from_bf16 ? c.x_codes_scratch : base + l.x_codes;
        front.scales_out = from_bf16 ? c.x_scales_scratch : base + l.x_scales;
        front.codes_out = reinterpret_cast<u32x4*>(codes_out);
        codes = codes_out;
        scales = front.scales_out;
        // Where most tokens are expected to have no row here, only those that have one are prepared: for 6976 tokens of 4160 columns
        // that go to one of 64 ranks the forward took 80.6 us and takes 56.6, for 15 424 of 3456 (16 ranks, top-4) 105.0 and 97.4, and
        // none of 29 shares from 8 to 16 192 tokens got slower.  (The look at the ids delays a row that is wanted.)
        if (num_shared == 0 && pow(1.0 - static_cast<double>(num_local) / num_experts, num_topk) > 0.5) {
            front.topk_idx = topk_idx;
            front.expert_begin = expert_begin;
            front.num_local = num_local;
        }
    }
    if (int rc = layout_i32(ws, topk_idx, num_tokens, num_topk, num_experts, expert_begin, num_local, expert_token_nums,
                            psum, offsets, route_to_row, row_to_route, num_rows, front, s))
        return rc;
    const MegaSizes sizes = {num_tokens, hidden, intermediate, num_topk, num_experts, num_local, num_shared};
    GemmParams g1 = gemm_of(sizes, w, false), g2 = gemm_of(sizes, w, true);
    const GemmChoices choices = choose_gemms(sizes, g1, g2);
    g1.a_codes = codes;
    g1.a_scales = scales;
    g1.row_to_route = row_to_route;
    g1.offsets = offsets;
    g1.w = w1;
    g1.ws = s1;
    g1.w_shared = shared_w1;
    g1.ws_shared = shared_s1;
    g1.act_codes = base + l.act_codes;
    g1.act_scales = base + l.act_scales;
    const long long expected_routed = static_cast<long long>(num_tokens) * num_topk * num_local / num_experts;
    const long long expected_rows = expected_routed + static_cast<long long>(num_tokens) * num_shared;
    const ExpectedRows expected = expected_rows_of(sizes);
    int* fill_state = reinterpret_cast<int*>(base + l.fill_state);
    int* fill_stop = reinterpret_cast<int*>(static_cast<char*>(w->sync) + kSyncFillStop);
    const bool served_only = num_shared == 0 && w->megamoe_served_only;
    const bool fill = g1.fill_tokens > 0;
    if (fill) {
        g1.fill_out = static_cast<u32x4*>(y);
        g1.fill_route_to_row = route_to_row;
        g1.fill_stop = fill_stop;
    }
    g1.fill_state = fill_state;  // written even when nothing fills (then as "no fillers")
    if (int rc = launch_gemm1(g1, choices.first, expected, s)) return rc;
    g2.a_codes = base + l.act_codes;
    g2.a_scales = base + l.act_scales;
    g2.row_to_route = nullptr;
    g2.offsets = offsets;
    g2.w = w2;
    g2.ws = s2;
    g2.w_shared = shared_w2;
    g2.ws_shared = shared_s2;
    g2.out = reinterpret_cast<uint16_t*>(base + l.out2);
    g2.out_cols = hidden;
    if (int rc = launch_gemm2(g2, choices.second, expected, s)) return rc;
    return combine_routes(base + l.out2, topk_weights, route_to_row, num_tokens, num_topk,
                          static_cast<int>(expected_rows),
                          hidden, y, num_shared > 0 ? num_rows : nullptr, num_shared, fill ? fill_state : nullptr,
                          served_only ? 1 : 0, s);
}

}  // extern "C"

// Routing layout for one rank: per-expert counts, prefix sums and the stable expert-major
// permutation of the T*K routes (a stable counting sort); no atomic decides the order of rows.
//
// Observable contract (reference: tests/utils/reference.py:39-73, tests/clos/common.py:248-287,
// tests/elastic/test_dispatch.py:538-548): rows are ordered (local expert, token, slot); every valid
// slot gets its own row (duplicates included); invalid ids produce no row.
//
// Decomposition: the flat route stream is cut into chunks, one wavefront each, four per workgroup.
//   count  : each wave histograms its chunk in LDS (atomic adds: a count does not depend on order)
//            -> wave_hist[chunk][expert] and the workgroup's sum block_hist[workgroup][expert]
//   assign : each workgroup sums block_hist over the workgroups (expert totals and their exclusive scan; the
//            workgroups before it -> its own base) and adds its waves' rows, then every wave replays its chunk in
//            order.  Inside a 64-route step the lanes with the same expert find each other through a 64-bit
//            mask per expert in LDS (each lane ORs its bit in, then all read the mask back): a route's row is
//            its expert's next free row plus the number of lower lanes in the mask.  The carry between steps
//            lives in LDS.  There is no separate scan launch.
// The smallest inputs take one workgroup, which holds everything (see "one workgroup" below).
// Inputs whose chunks fit a wave's registers (at most kKeep steps of 64 routes) take ONE launch: the workgroups
// (at most 129, 17 to an XCD with room for 64 of the largest; whatever else runs ends by itself, so all become resident together unless four
// such launches are at work at once, and then the wait has its bound) count, publish their histograms as
// self-validating words (count + the launch's tag in one 64-bit store), read each other's as soon as they appear, and
// assign from the ids they still hold: no barrier, no counter that anybody has to reset.  The wait for the others'
// words is bounded; a launch whose wait runs out assigns nothing (a histogram is missing): it reports no rows, marks
// every route as having none, and leaves its number in the workspace's mailbox, where the host finds it; later layouts
// on that workspace take two launches.  Larger inputs take two launches anyway.
#include <algorithm>
#include <mutex>
#include <type_traits>

#include "common.h"
#include "mx.h"
#include "payload.h"

namespace dpep {
namespace {

constexpr int kWaves = 4;             // wavefronts (= chunks) per workgroup
constexpr int kThreads = kWaves * kWave;
constexpr int kHistInts = 16384;      // chunks * padded experts never exceeds this
constexpr int kBlockHistInts = kHistInts / kWaves + DPEP_MAX_LOCAL_EXPERTS;  // workgroups * experts, rounded up
constexpr int kLargeHistInts = 65536;  // the two-launch form of large inputs, where the workspace has the room
constexpr int kLargeBlockHistInts = kLargeHistInts / kWaves + DPEP_MAX_LOCAL_EXPERTS;
constexpr int kMinChunk = 256;        // routes per wavefront, lower bound (multiple of 64)
constexpr int kPrefetch = 8;          // 64-route steps whose ids are fetched at once
constexpr int kKeep = 16;             // 64-route steps of a chunk that the one-launch kernel holds in registers
constexpr int kMegaExperts = 128;     // local experts of a MegaMoE forward, at most
constexpr int kColumnBatch = 16;      // histogram loads in flight per thread
constexpr int kTaggedInts = 32768;    // chunks * padded experts of the one-launch form
static_assert(kSyncTaggedWords >= static_cast<size_t>(kTaggedInts / kWaves + DPEP_MAX_LOCAL_EXPERTS), "the tagged histograms need a word per (workgroup, expert)");

__device__ __forceinline__ uint64_t lanes_below()
{
    return (1ull << (threadIdx.x & 63)) - 1ull;
}

// Orders this wave's LDS accesses before the call against those after it, for all its lanes.
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Local experts of kSteps consecutive 64-route steps from `base` on.  All loads are issued before the first is
// used (a route past the end reads the last id instead of branching around the load), so that the wave pays
// one memory latency for the batch, not one per step.  Needs n_routes > 0.  idx_copy: where the ids are copied to
// (a handle's own routing tensor; the copy rides on ids that are read anyway), or nullptr.
template <int kSteps, typename IdxT>
__device__ __forceinline__ void fetch_experts(int (&experts)[kSteps], const IdxT* __restrict__ idx, int base, int end,
                                              int n_routes, int num_experts, int expert_begin, int num_local,
                                              IdxT* __restrict__ idx_copy = nullptr)
{
    const int lane = threadIdx.x & 63;
    IdxT raw[kSteps];
#pragma unroll
    for (int i = 0; i < kSteps; ++i) raw[i] = idx[min(base + i * kWave + lane, n_routes - 1)];
#pragma unroll
    for (int i = 0; i < kSteps; ++i)
        experts[i] = local_expert(static_cast<long long>(raw[i]), base + i * kWave + lane, end, num_experts, expert_begin,
                                  num_local);
    if (idx_copy != nullptr) {
#pragma unroll
        for (int i = 0; i < kSteps; ++i)
            if (base + i * kWave + lane < end) idx_copy[base + i * kWave + lane] = raw[i];
    }
}

// LDS of one workgroup.  running[w][e]: wave w's histogram, later its next free row of expert e; match[w][e]: bit
// per lane of wave w whose route in the current step goes to expert e (all zero between steps); totals[e]: rows
// of expert e.
template <int kMaxLocal, bool kOneLaunch>
struct LayoutLds {
    int totals[kMaxLocal];
    int running[kWaves][kMaxLocal];
    unsigned long long match[kWaves][kMaxLocal];
    int seen[kOneLaunch ? kWaves : 1][kOneLaunch ? kMaxLocal : 1];  // one-launch kernel: routes of expert e that wave w has ranked
    int partial[kThreads * 2];
    int wave_sums[kWaves];
    int timed_out;  // one-launch kernel: some thread's wait for another workgroup's histogram ran out
    unsigned long long tag;  // one-launch kernel: the tag of this launch, read once per workgroup
};

template <typename Lds>
__device__ __forceinline__ void clear_wave_lds(Lds& lds, int num_local)
{
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int e = lane; e < num_local; e += kWave) {
        lds.running[wave][e] = 0;
        lds.match[wave][e] = 0ull;
    }
    wave_sync();
}

__device__ __forceinline__ void count_step(int e, int* __restrict__ mine)
{
    if (e >= 0) __hip_atomic_fetch_add(mine + e, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}

// The waves' histograms (lds.running) out to wave_hist, and their sum to block_hist.  Called by all threads.
template <typename Lds>
__device__ __forceinline__ void publish_histograms(Lds& lds, int num_local, int num_chunks,
                                                   int* __restrict__ wave_hist, int* __restrict__ block_hist)
{
    __syncthreads();
    for (int e = threadIdx.x; e < num_local; e += kThreads) {
        int sum = 0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            const int g = blockIdx.x * kWaves + w;
            const int count = lds.running[w][e];
            sum += count;
            if (g < num_chunks) wave_hist[static_cast<size_t>(g) * num_local + e] = count;
        }
        block_hist[static_cast<size_t>(blockIdx.x) * num_local + e] = sum;
    }
}

// One 64-route step of the ordered replay.
__device__ __forceinline__ void assign_step(int e, int route, int end, unsigned long long* __restrict__ match,
                                            int* __restrict__ next_row, int* __restrict__ route_to_row,
                                            int* __restrict__ row_to_route)
{
    if (e >= 0)
        __hip_atomic_fetch_or(match + e, 1ull << (threadIdx.x & 63), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    wave_sync();
    int row = -1, ahead = 0, group = 0;
    if (e >= 0) {
        const unsigned long long mask = match[e];
        ahead = __popcll(mask & lanes_below());
        group = __popcll(mask);
        row = next_row[e] + ahead;
    }
    wave_sync();  // every lane has read its expert's mask and next row before the first lane of the group moves them
    if (e >= 0 && ahead == 0) {
        next_row[e] = row + group;
        match[e] = 0ull;
    }
    wave_sync();
    if (route < end) {
        route_to_row[route] = row;
        if (row >= 0) row_to_route[row] = route;
    }
}

// One 64-route step of the ranking: the number of routes of this wave, so far, with this lane's expert.
__device__ __forceinline__ int rank_step(int e, unsigned long long* __restrict__ match, int* __restrict__ seen)
{
    if (e >= 0)
        __hip_atomic_fetch_or(match + e, 1ull << (threadIdx.x & 63), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    wave_sync();
    int rank = 0, ahead = 0, group = 0;
    if (e >= 0) {
        const unsigned long long mask = match[e];
        ahead = __popcll(mask & lanes_below());
        group = __popcll(mask);
        rank = seen[e] + ahead;
    }
    wave_sync();  // every lane has read its expert's mask and count before the first lane of the group moves them
    if (e >= 0 && ahead == 0) {
        seen[e] = rank + group;
        match[e] = 0ull;
    }
    wave_sync();
    return rank;
}

template <typename IdxT>
__global__ __launch_bounds__(kThreads) void layout_count_kernel(const IdxT* __restrict__ idx, int n_routes,
                                                                int num_experts, int expert_begin, int num_local,
                                                                int chunk, int num_chunks, int* __restrict__ wave_hist,
                                                                int* __restrict__ block_hist, IdxT* __restrict__ idx_copy)
{
    __shared__ LayoutLds<DPEP_MAX_LOCAL_EXPERTS, false> lds;
    const int wave = threadIdx.x >> 6;
    const int g = blockIdx.x * kWaves + wave;
    const int begin = g < num_chunks ? g * chunk : 0;
    const int end = g < num_chunks ? min(begin + chunk, n_routes) : 0;
    clear_wave_lds(lds, num_local);
    for (int base = begin; base < end; base += kPrefetch * kWave) {
        int experts[kPrefetch];
        fetch_experts(experts, idx, base, end, n_routes, num_experts, expert_begin, num_local, idx_copy);
#pragma unroll
        for (int i = 0; i < kPrefetch; ++i) count_step(experts[i], lds.running[wave]);
    }
    publish_histograms(lds, num_local, num_chunks, wave_hist, block_hist);
}

// For one expert, over the workgroups {first, first+stride, ...}: the sum of all block_hist rows and of those
// of workgroups before this one.
struct ColumnSums {
    int total;
    int before;
};

__device__ __forceinline__ ColumnSums column_sums(const int* __restrict__ block_hist, int num_local, int e, int first,
                                                  int stride, int num_blocks)
{
    ColumnSums sums = {0, 0};
    for (int b0 = first; b0 < num_blocks; b0 += kColumnBatch * stride) {
        int v[kColumnBatch];
#pragma unroll
        for (int j = 0; j < kColumnBatch; ++j) {
            const int b = b0 + j * stride;
            v[j] = b < num_blocks ? block_hist[static_cast<size_t>(b) * num_local + e] : 0;
        }
#pragma unroll
        for (int j = 0; j < kColumnBatch; ++j) {
            sums.total += v[j];
            sums.before += b0 + j * stride < static_cast<int>(blockIdx.x) ? v[j] : 0;
        }
    }
    return sums;
}

// Words of the one-launch kernel's exchange (see "one launch" below): tag above kCountBits, count below.
constexpr int kCountBits = 24;
constexpr unsigned long long kCountMask = (1ull << kCountBits) - 1ull;

__device__ __forceinline__ unsigned long long load_word(const unsigned long long* src)
{
    return __hip_atomic_load(src, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void store_word(unsigned long long* dst, unsigned long long word)
{
    __hip_atomic_store(dst, word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The workgroup's histogram (sum of its waves') out to its row of `tagged`.  Called by all threads, after a workgroup
// barrier behind the counting.
template <typename Lds>
__device__ __forceinline__ void publish_tagged(Lds& lds, int num_local, unsigned long long* __restrict__ tagged,
                                               unsigned long long tag)
{
    for (int e = threadIdx.x; e < num_local; e += kThreads) {
        int sum = 0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) sum += lds.running[w][e];
        __hip_atomic_store(tagged + static_cast<size_t>(blockIdx.x) * num_local + e,
                           (tag << kCountBits) | static_cast<unsigned long long>(sum), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    }
}

// column_sums over tagged rows {first, first+stride, ...} below `rows`: every word is re-read until it carries `tag`.
// Sets lds_timed_out and gives up when that takes longer than limit_ticks.
__device__ __forceinline__ ColumnSums tagged_column_sums(const unsigned long long* __restrict__ tagged, int num_local, int e,
                                                         int first, int stride, int rows, unsigned long long tag,
                                                         long long limit_ticks, int* lds_timed_out)
{
    ColumnSums sums = {0, 0};
    long long start = 0;
    for (int b0 = first; b0 < rows; b0 += kColumnBatch * stride) {
        unsigned long long v[kColumnBatch];
        for (int spins = 0;; ++spins) {
            bool all = true;
#pragma unroll
            for (int j = 0; j < kColumnBatch; ++j) {
                const int b = b0 + j * stride;
                v[j] = b < rows ? load_word(tagged + static_cast<size_t>(b) * num_local + e) : tag << kCountBits;
            }
#pragma unroll
            for (int j = 0; j < kColumnBatch; ++j) all = all && (v[j] >> kCountBits) == tag;
            if (all) break;
            if ((spins & 15) == 15) {
                const long long now = wall_clock64();
                if (start == 0) start = now;
                if (now - start > limit_ticks) {
                    *lds_timed_out = 1;
                    return sums;
                }
            }
            __builtin_amdgcn_s_sleep(1);
        }
#pragma unroll
        for (int j = 0; j < kColumnBatch; ++j) {
            const int count = static_cast<int>(v[j] & kCountMask);
            sums.total += count;
            sums.before += b0 + j * stride < static_cast<int>(blockIdx.x) ? count : 0;
        }
    }
    return sums;
}

// Where the one-launch kernel's workgroups find each other's histograms.
struct TaggedSource {
    const unsigned long long* tagged;
    unsigned long long tag;
    int rows;
    long long limit_ticks;
    uint32_t* timeouts;  // host mailbox word that receives launch_id when the wait runs out
    uint32_t launch_id;
};

// From the histograms to every wave's first row per expert (lds.running).  The launch's last workgroup owns no
// chunk: it is the reporter, which writes the per-expert outputs and reports to the host, so that the wait for the
// host stores (a PCIe round trip) delays no workgroup that still has routes to assign.  Called by all threads.
// num_blocks = workgroups that own chunks.  kTagged: the one-launch kernel (the workgroup's own wave histograms are
// still in lds.running, the others' arrive as tagged words from `source`); else the count launch left everything in
// wave_hist / block_hist.  Returns false if the wait for the tagged words ran out: every count is then reported as zero.
template <bool kTagged, typename Lds>
__device__ __forceinline__ bool expert_bases(Lds& lds, const int* __restrict__ wave_hist,
                                             const int* __restrict__ block_hist, int n_routes, int num_local, int padded_local,
                                             int num_chunks, int num_blocks, int* __restrict__ counts,
                                             int* __restrict__ psum, int* __restrict__ offsets, int* __restrict__ num_rows,
                                             const SendCounts& send, uint32_t* __restrict__ mailbox, uint32_t sequence,
                                             const TaggedSource* source = nullptr)
{
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const bool reporter = static_cast<int>(blockIdx.x) == num_blocks;
    // This workgroup's own rows are asked for before the column sums, so that all loads are in flight together.
    auto own_rows = [&](int e, int (&own)[kWaves]) {
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            const int g = blockIdx.x * kWaves + w;
            if (kTagged) own[w] = lds.running[w][e];  // (the reporter's are zero: it counted nothing)
            else own[w] = g < num_chunks ? wave_hist[static_cast<size_t>(g) * num_local + e] : 0;
        }
    };
    auto sums_of = [&](int e, int first, int stride) {
        if (kTagged)
            return tagged_column_sums(source->tagged, num_local, e, first, stride, source->rows, source->tag,
                                      source->limit_ticks, &lds.timed_out);
        return column_sums(block_hist, num_local, e, first, stride, num_blocks);
    };
    auto finish = [&](int e, int total, int before, const int (&own)[kWaves]) {  // the waves one after the other
        lds.totals[e] = total;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            lds.running[w][e] = before;
            before += own[w];
        }
    };
    if (padded_local >= kThreads) {
        for (int e = tid; e < num_local; e += kThreads) {
            int own[kWaves];
            own_rows(e, own);
            const ColumnSums sums = sums_of(e, 0, 1);
            finish(e, sums.total, sums.before, own);
        }
    } else {
        // Few experts: split the workgroups' rows over `parts` thread groups (at most 16), then reduce through LDS.
        int parts = kThreads / padded_local;
        if (parts > 16) parts = 16;
        const int p = tid / padded_local, e = tid % padded_local;
        int own[kWaves] = {0, 0, 0, 0};
        if (tid < num_local) own_rows(tid, own);
        if (p < parts && e < num_local) {
            const ColumnSums sums = sums_of(e, p, parts);
            lds.partial[tid * 2] = sums.total;
            lds.partial[tid * 2 + 1] = sums.before;
        }
        __syncthreads();
        if (tid < num_local) {
            int total = 0, before = 0;
            for (int q = 0; q < parts; ++q) {
                total += lds.partial[(q * padded_local + tid) * 2];
                before += lds.partial[(q * padded_local + tid) * 2 + 1];
            }
            finish(tid, total, before, own);
        }
    }
    __syncthreads();
    const bool valid = !kTagged || lds.timed_out == 0;
    if (!valid) {
        // A histogram is missing: every count is reported as zero, and the host is told.  (The reporter's own store is
        // acknowledged before it reports to the mailbox below, so the host never sees a reporter's
        // time-out later than its report; another workgroup's time-out may reach the host after the report, and is
        // then found by the next call on the workspace.)
        if (tid == 0) {
            __hip_atomic_store(source->timeouts, source->launch_id, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        for (int e = tid; e < num_local; e += kThreads) {
            lds.totals[e] = 0;
#pragma unroll
            for (int w = 0; w < kWaves; ++w) lds.running[w][e] = 0;
        }
        __syncthreads();
    }

    // Exclusive scan of totals over experts: four consecutive experts per thread, then a workgroup scan.
    int mine[4], local_sum = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int e = tid * 4 + j;
        mine[j] = e < num_local ? lds.totals[e] : 0;
        local_sum += mine[j];
    }
    const int incl = wave_scan(local_sum);
    if (lane == kWave - 1) lds.wave_sums[wave] = incl;
    __syncthreads();
    int offset = incl - local_sum;
    for (int w = 0; w < wave; ++w) offset += lds.wave_sums[w];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int e = tid * 4 + j;
        if (e < num_local) {
#pragma unroll
            for (int w = 0; w < kWaves; ++w) lds.running[w][e] += offset;
            if (reporter) {
                counts[e] = mine[j];
                psum[e] = offset + mine[j];
                offsets[e + 1] = offset + mine[j];
                if (send.counts != nullptr) send.counts[send.expert_begin + e] = offset + mine[j];
            }
        }
        offset += mine[j];
    }
    if (reporter && tid == kThreads - 1) {
        offsets[0] = 0;
        num_rows[0] = offset;
    }
    if (reporter) send_counts_of_others(send, num_local, lds.wave_sums[0] + lds.wave_sums[1] + lds.wave_sums[2] + lds.wave_sums[3], tid, kThreads);
    if (reporter && mailbox != nullptr) {
        if (tid * 4 < num_local) mailbox_store_counts(mailbox, tid * 4, mine, sequence, mailbox_narrow(n_routes));
        if (tid == kThreads - 1) mailbox_store_rows(mailbox, offset, sequence);
    }
    __syncthreads();
    return valid;
}

template <typename IdxT>
__global__ __launch_bounds__(kThreads) void layout_assign_kernel(
    const IdxT* __restrict__ idx, int n_routes, int num_experts, int expert_begin, int num_local, int padded_local,
    int chunk, int num_chunks, const int* __restrict__ wave_hist, const int* __restrict__ block_hist,
    int* __restrict__ counts, int* __restrict__ psum, int* __restrict__ offsets, int* __restrict__ num_rows,
    int* __restrict__ route_to_row, int* __restrict__ row_to_route, SendCounts send, uint32_t* __restrict__ mailbox,
    uint32_t sequence)
{
    __shared__ LayoutLds<DPEP_MAX_LOCAL_EXPERTS, false> lds;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int g = blockIdx.x * kWaves + wave;
    const int begin = g < num_chunks ? g * chunk : 0;
    const int end = g < num_chunks ? min(begin + chunk, n_routes) : 0;
    int experts[kPrefetch];  // the first ids travel while the histograms are summed
    if (begin < end) fetch_experts(experts, idx, begin, end, n_routes, num_experts, expert_begin, num_local);
    clear_wave_lds(lds, num_local);
    __syncthreads();  // expert_bases writes the rows of all waves
    expert_bases<false>(lds, wave_hist, block_hist, n_routes, num_local, padded_local, num_chunks, gridDim.x - 1, counts, psum,
                        offsets, num_rows, send, mailbox, sequence);
    for (int base = begin; base < end; base += kPrefetch * kWave) {
        if (base != begin) fetch_experts(experts, idx, base, end, n_routes, num_experts, expert_begin, num_local);
#pragma unroll
        for (int i = 0; i < kPrefetch; ++i)
            assign_step(experts[i], base + i * kWave + lane, end, lds.match[wave], lds.running[wave], route_to_row,
                        row_to_route);
    }
}

// ---- one launch: histograms exchanged as tagged words -------------------------------------------------------------
// A published histogram entry is one 64-bit word: the launch's tag in the upper kTagBits, the count below.  A reader
// knows from the word itself whether it belongs to this launch, so there is nothing to wait for but the data, and
// nothing to clear afterwards.  Tags only grow: a launch uses epoch + 1, where the epoch (device memory) is the highest
// tag any launch on this workspace has used, read by every workgroup before it publishes and raised with an atomic max
// when the workgroup ends.  No workgroup can end before every workgroup has read the epoch: it ends only after it has
// seen the words of everybody who owns a chunk, which are published after that read, and the tag of the reporter, which
// owns none, in a word of its own (the reporter stores it right after its read; the others look for it as the last
// thing they do, when it has long been there).  So all workgroups of a launch agree on the tag; a launch that ran
// out of time may use two tags, and the atomic max still leaves the epoch above both.  Replays of a captured launch
// therefore get fresh tags without any host involvement.  40 tag bits last 10^12 launches.
// Count, exchange, assign in one launch; every wave keeps the ids of its chunk (at most kSteps steps) in registers, and ranks
// them within (wave, expert) while the words travel.  kSteps is the smallest of 2, 4, 8 and kKeep that holds the chunk: the code is
// straight-line, every launch finds the instruction caches cold, and steps that do nothing still had to be fetched (65 536
// routes, 256 per wave, launches back to back: 6.8 us with sixteen steps that assigned behind the exchange, 6.3 with four
// ranked ahead of it; with sixteen ranked ahead of it 7.7).
// `rows` = histogram rows to wait for (the workgroups that own chunks; one more in a test that wants the wait to run out),
// `limit_ticks` the bound of that wait (100 MHz ticks).
// kMega: a MegaMoE forward's layout (at most 128 local experts).  Workgroups behind the reporter prepare the input rows
// (quantise or pad them), which does not depend on the routing, and every workgroup of the layout writes a piece of the shared
// experts' rows once it knows R: up to three launches fewer (777 tokens of 2880 BF16 columns with a shared expert: layout 8.3 +
// quantise 4.1 + pad 3.3 + shared rows 1.9 us as launches of their own).
// What the layout's workgroups do.  kWords: a payload in the same grid waits for the rows of the routes (1) or the routes of the rows (2).
template <typename IdxT, bool kMega, int kSteps, int kWords, typename Lds>
__device__ __forceinline__ void fused_layout(
    Lds& lds, const IdxT* __restrict__ idx, int n_routes, int num_experts, int expert_begin, int num_local, int padded_local,
    int chunk, int num_chunks, int* __restrict__ counts, int* __restrict__ psum, int* __restrict__ offsets,
    int* __restrict__ num_rows, int* __restrict__ route_to_row, int* __restrict__ row_to_route, IdxT* __restrict__ idx_copy,
    SendCounts send, uint32_t* __restrict__ mailbox, uint32_t sequence, unsigned long long* __restrict__ epoch,
    unsigned long long* __restrict__ tagged, int num_blocks, int rows, long long limit_ticks, uint32_t* __restrict__ timeouts,
    uint32_t launch_id, const MegaFront& front,
    unsigned long long* __restrict__ total_word = nullptr, unsigned long long* __restrict__ row_words = nullptr)
{
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int g = blockIdx.x * kWaves + wave;
    const int begin = g < num_chunks ? g * chunk : 0;
    const int end = g < num_chunks ? min(begin + chunk, n_routes) : 0;
    // One thread reads the epoch for the whole workgroup (asked for together with the ids): every thread must use the
    // same tag, and the tag must be final before anything this workgroup publishes can be seen.
    unsigned long long* reporter_tag = epoch + kSyncReporterTag / sizeof(unsigned long long);
    const bool reporter = static_cast<int>(blockIdx.x) == num_blocks;
    if (threadIdx.x == 0) {
        lds.tag = load_word(epoch) + 1ull;
        lds.timed_out = 0;
        if (reporter) __hip_atomic_store(reporter_tag, lds.tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    int experts[kSteps];
    fetch_experts(experts, idx, begin, end, n_routes, num_experts, expert_begin, num_local, idx_copy);
    clear_wave_lds(lds, num_local);
    for (int e = lane; e < num_local; e += kWave) lds.seen[wave][e] = 0;
#pragma unroll
    for (int i = 0; i < kSteps; ++i) count_step(experts[i], lds.running[wave]);
    __syncthreads();
    const unsigned long long tag = lds.tag;
    // (the reporter owns no chunk and publishes nothing: row num_blocks is only ever waited for by a test that wants
    // the wait to run out)
    if (!reporter) publish_tagged(lds, num_local, tagged, tag);
    // Ranked while the words travel: behind the exchange a route's row is one LDS read away.
    int rank[kSteps];
#pragma unroll
    for (int i = 0; i < kSteps; ++i)
        if (begin + i * kWave < end) rank[i] = rank_step(experts[i], lds.match[wave], lds.seen[wave]);
    // The reporter gives up first (the others wait twice as long): a launch that the reporter passes as valid is then
    // one in which every histogram arrived within the reporter's bound, so another workgroup can only have run out of
    // time if its own wait began more than a whole bound before the reporter's.  What remains of that window is closed
    // on the consumers' side: such a workgroup marks its routes as having no row, and the kernels that read
    // row_to_route clamp what they find there.
    const TaggedSource source = {tagged, tag, rows, reporter ? limit_ticks : 2 * limit_ticks, timeouts, launch_id};
    const bool in_time = expert_bases<true>(lds, nullptr, nullptr, n_routes, num_local, padded_local, num_chunks, num_blocks, counts, psum,
                                            offsets, num_rows, send, mailbox, sequence, &source);
    if (kWords != 0 && reporter && threadIdx.x == 0)  // (0 where the exchange ran out of time)
        store_word(total_word, row_word(launch_id, lds.wave_sums[0] + lds.wave_sums[1] + lds.wave_sums[2] + lds.wave_sums[3]));
    // (asked for here, needed only at the very end: the load travels while the routes are assigned)
    unsigned long long reporter_seen = threadIdx.x == 0 && !reporter ? load_word(reporter_tag) : 0ull;
    if (in_time) {
#pragma unroll
        for (int i = 0; i < kSteps; ++i) {
            const int route = begin + i * kWave + lane;
            if (route < end) {
                const int row = experts[i] >= 0 ? lds.running[wave][experts[i]] + rank[i] : -1;
                route_to_row[route] = row;
                if (row >= 0) row_to_route[row] = route;
                if (kWords == 1) store_word(row_words + route, row_word(launch_id, row));
                if (kWords == 2 && row >= 0) store_word(row_words + row, row_word(launch_id, route));
            }
        }
    } else {
        // Some workgroup's histogram is missing: rows computed without it could lie anywhere.  No route gets a row
        // (and the counts above are all zero).
        for (int route = begin + lane; route < end; route += kWave) {
            route_to_row[route] = -1;
            if (kWords == 1) store_word(row_words + route, row_word(launch_id, -1));
        }
    }
    if (kMega && front.num_shared > 0)  // (R = 0 where the exchange ran out of time)
        shared_rows(front, lds.wave_sums[0] + lds.wave_sums[1] + lds.wave_sums[2] + lds.wave_sums[3], num_local, offsets, row_to_route,
                    blockIdx.x * kThreads + threadIdx.x, (num_blocks + 1) * kThreads);
    if (threadIdx.x == 0) {
        // The epoch may only move once the reporter has read it (a reporter that read the raised epoch would wait for
        // words nobody publishes).  Tags only grow, so any value from this launch's tag on means that it has; the wait
        // is bounded like the others, and a reporter that comes later still reports the launch as failed.
        if (!reporter) {
            long long start = 0;
            for (int spins = 0; reporter_seen < tag; ++spins) {
                if ((spins & 15) == 15) {
                    const long long now = wall_clock64();
                    if (start == 0) start = now;
                    if (now - start > limit_ticks) break;
                }
                __builtin_amdgcn_s_sleep(1);
                reporter_seen = load_word(reporter_tag);
            }
        }
        __hip_atomic_fetch_max(epoch, tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

template <typename IdxT, bool kMega, int kSteps>
__global__ __launch_bounds__(kThreads) void layout_fused_kernel(
    const IdxT* __restrict__ idx, int n_routes, int num_experts, int expert_begin, int num_local, int padded_local,
    int chunk, int num_chunks, int* __restrict__ counts, int* __restrict__ psum, int* __restrict__ offsets,
    int* __restrict__ num_rows, int* __restrict__ route_to_row, int* __restrict__ row_to_route, IdxT* __restrict__ idx_copy,
    SendCounts send, uint32_t* __restrict__ mailbox, uint32_t sequence, unsigned long long* __restrict__ epoch,
    unsigned long long* __restrict__ tagged, int num_blocks, int rows, long long limit_ticks, uint32_t* __restrict__ timeouts,
    uint32_t launch_id, MegaFront front)
{
    __shared__ LayoutLds<kMega ? kMegaExperts : DPEP_MAX_LOCAL_EXPERTS, true> lds;
    if (kMega && static_cast<int>(blockIdx.x) > num_blocks) {
        __shared__ __attribute__((aligned(16))) uint8_t staged[kFrontThreads / 2];
        prepare_rows<kFrontThreads>(front, blockIdx.x - num_blocks - 1, staged);
        return;
    }
    fused_layout<IdxT, kMega, kSteps, 0>(lds, idx, n_routes, num_experts, expert_begin, num_local, padded_local, chunk, num_chunks, counts, psum, offsets, num_rows, route_to_row, row_to_route, idx_copy, send, mailbox, sequence, epoch, tagged, num_blocks, rows, limit_ticks, timeouts, launch_id, front);
}

// ---- layout and payload in one grid ------------------------------------------------------------------------------------
// The payload's workgroups, behind the layout's in the same grid, ask for their tokens at once and look for the words that say where
// these go: between the routes' ids and the first payload store there is no second launch, whose ramp and first loads would follow
// the layout's last store.  A payload workgroup looks for a while only (kPayloadLooks); where the words do not come it works its rows out
// from the ids itself and waits for nobody.  It must not wait without such a bound: a grid is dealt over eight XCDs, each of which starts
// its share by itself, the layout's workgroups need each other across them, and two such grids at once could each hold an
// XCD that the other's layout has yet to enter.  The words carry the number of the launch, which comes from the host, so a
// captured launch (whose replays would repeat it) takes two.  128 registers, as the layout wants: four workgroups to a CU carry the payload
// as fast as eight (with 64 the layout spills, and the kernel takes 7 us longer).
// Bound by HBM once the words are there.  Dispatch and combine, launches back to back, one grid / two: 1000 tokens x top-6 of 5120 BF16 30.5 / 31.7 us,
// 618 x 7 of 5824 28.8 / 32.7, 3407 x 6 of 1584 37.5 / 42.5, 4372 x 7 of 5840 169.5 / 177.2.  Up to kSingleRoutes routes the layout's
// workgroup of its own is the better one (710 x 4 of 2672 20.1 / 18.7).
// Chunks of at most four steps: with eight (32 768 routes over 256 experts, skewed popularity, 235 MB) one grid took 149.9 us, two 146.6.
constexpr int kRidingExperts = 256, kRidingSteps = 4;

// What the rows follow from.
struct Routing {
    const int64_t* idx;
    int n_routes, num_experts, expert_begin, num_local;
    // Calls visit(local expert or -1, route) for all routes in order, 64 at a time.  Called by whole waves.
    template <typename Visit>
    __device__ __forceinline__ void scan(Visit&& visit) const
    {
        for (int base = 0; base < n_routes; base += kPrefetch * kWave) {
            int experts[kPrefetch];
            fetch_experts(experts, idx, base, n_routes, n_routes, num_experts, expert_begin, num_local);
#pragma unroll
            for (int i = 0; i < kPrefetch; ++i) visit(experts[i], base + i * kWave + (static_cast<int>(threadIdx.x) & 63));
        }
    }
};

// One look: whether the word is this launch's, and its value.
__device__ __forceinline__ bool look(const unsigned long long* word, uint32_t launch, int& value)
{
    const unsigned long long v = load_word(word);
    value = static_cast<int>(static_cast<uint32_t>(v));
    return static_cast<uint32_t>(v >> 32) == launch;
}

// Looks past the caches, by a thousand workgroups, delay the layout that they wait for: kNaps of 256 cycles lie between two (1000 tokens x top-6
// 31.0 us with one look per microsecond, 32.3 with one per two; a few hundred rows of 6144 tokens 28.6 with one per two, 28.8 with
// one, 29.7 with three).
template <int kNaps>
__device__ __forceinline__ void nap()
{
    for (int i = 0; i < kNaps; ++i) __builtin_amdgcn_s_sleep(4);
}

// Where a token's rows come from.
struct AwaitedTokens {
    static constexpr int kGaveUp = -2;
    Routing routing;
    const unsigned long long* words;
    const unsigned long long* total;
    uint32_t launch;
    int looks;
    int capacity, all_or_none;
    int (*rows_of)[kRidingExperts];  // LDS of this wave: rows of every expert, and those of them from tokens before
    __device__ __forceinline__ int begin() const { return 0; }
    __device__ __forceinline__ int await(const unsigned long long* word) const
    {
        for (int i = 0; i < looks; ++i, nap<8>()) {
            int value;
            if (look(word, launch, value)) return value;
        }
        return kGaveUp;
    }
    __device__ __forceinline__ int kept(int row, int all) const
    {
        return row < capacity && (all_or_none == 0 || DPEP_ROWS_KEPT(all, capacity)) ? row : -1;
    }
    // The token's rows into lds.rows; whether there is any.  Called by all threads of the workgroup.
    __device__ __forceinline__ bool find_rows(const PayloadShape& p, int, int token, int t, TokenLds& lds) const
    {
        if (t < p.num_topk) {
            int row = await(words + static_cast<size_t>(token) * p.num_topk + t);
            if (row >= 0 && all_or_none != 0) {
                const int all = await(total);
                row = all == kGaveUp ? kGaveUp : kept(row, all);
            }
            lds.rows[t] = row < capacity ? row : -1;
        }
        __syncthreads();
        const int lane = threadIdx.x & 63;
        int row = lane < p.num_topk ? lds.rows[lane] : -1;
        if (__ballot(row == kGaveUp) != 0) row = work_out(p, token, lds.rows);
        return __ballot(row >= 0) != 0;
    }
    // The same rows without the words: row = rows of the experts before + earlier routes to the same expert.  Each of the token's waves works
    // all of them out for itself (they write the same values, and one that finds nothing missing any more finds these).
    __device__ __forceinline__ int work_out(const PayloadShape& p, int token, int* rows) const
    {
        const int lane = threadIdx.x & 63, first = token * p.num_topk;
        for (int e = lane; e < routing.num_local; e += kWave) rows_of[0][e] = rows_of[1][e] = 0;
        wave_sync();
        routing.scan([&](int e, int route) {
            count_step(e, rows_of[0]);
            count_step(route < first ? e : -1, rows_of[1]);
        });
        wave_sync();
        int row = -1;
        if (lane < p.num_topk) {
            auto expert_of = [&](int s) {
                return local_expert(routing.idx[first + s], first + s, routing.n_routes, routing.num_experts, routing.expert_begin, routing.num_local);
            };
            const int mine = expert_of(lane);
            int all = 0;
            row = mine < 0 ? -1 : rows_of[1][mine];
            for (int e = 0; e < routing.num_local; ++e) {
                if (e < mine) row += rows_of[0][e];
                all += rows_of[0][e];
            }
            for (int s = 0; s < lane && mine >= 0; ++s) row += expert_of(s) == mine ? 1 : 0;
            row = row < 0 ? -1 : kept(row, all);
            rows[lane] = row;
        }
        wave_sync();
        return row;
    }
};

// Where a row's route comes from; every wave looks by itself.
struct AwaitedRows {
    Routing routing;
    const unsigned long long* words;
    const unsigned long long* total;
    uint32_t launch;
    int looks;
    int rows;      // bound of R
    int* rows_of;  // LDS of this wave: rows of every expert
    // The route of row `row` below the bound; -1: there is no such row.  Called by whole waves.
    __device__ __forceinline__ int route_of(int row) const
    {
        for (int i = 0; i < looks; ++i, nap<16>()) {
            int route, all;
            const bool has_route = look(words + row, launch, route), has_total = look(total, launch, all);
            if (__builtin_amdgcn_readfirstlane(has_route ? 1 : 0)) return __builtin_amdgcn_readfirstlane(route);
            if (__builtin_amdgcn_readfirstlane(has_total && row >= all ? 1 : 0)) return -1;
        }
        return work_out(row);
    }
    // The same without the words: the expert whose rows hold `row`, then that expert's route by its rank.
    __device__ __forceinline__ int work_out(int row) const
    {
        for (int e = threadIdx.x & 63; e < routing.num_local; e += kWave) rows_of[e] = 0;
        wave_sync();
        routing.scan([&](int e, int) { count_step(e, rows_of); });
        wave_sync();
        int expert = 0, rank = row, route = -1;
        while (expert < routing.num_local && rank >= rows_of[expert]) rank -= rows_of[expert++];
        wave_sync();  // (the next row's counts go to the same place)
        if (expert == routing.num_local) return -1;
        routing.scan([&](int e, int at) {
            const unsigned long long same = __ballot(e == expert);
            const unsigned long long it = __ballot(e == expert && __popcll(same & lanes_below()) == rank);
            if (it != 0) route = at - (static_cast<int>(threadIdx.x) & 63) + __ffsll(it) - 1;  // (once: the rank falls below zero)
            rank -= __popcll(same);
        });
        return __builtin_amdgcn_readfirstlane(route);
    }
};

template <bool kQuant, bool kRowMajor, bool kStaged>
__global__ __launch_bounds__(kThreads, 4) void layout_payload_kernel(
    const int64_t* __restrict__ idx, int n_routes, int num_experts, int expert_begin, int num_local, int padded_local,
    int chunk, int num_chunks, int* __restrict__ counts, int* __restrict__ psum, int* __restrict__ offsets,
    int* __restrict__ num_rows, int* __restrict__ route_to_row, int* __restrict__ row_to_route, int64_t* __restrict__ idx_copy,
    SendCounts send, uint32_t* __restrict__ mailbox, uint32_t sequence, unsigned long long* __restrict__ epoch,
    unsigned long long* __restrict__ tagged, int num_blocks, int rows, long long limit_ticks, uint32_t* __restrict__ timeouts,
    uint32_t launch_id,
    unsigned long long* __restrict__ total_word, unsigned long long* __restrict__ row_words, LayoutPayload payload)
{
    using Lds = LayoutLds<kRidingExperts, true>;
    struct Riding {
        TokenLds tokens[kWaves];
        float scales[kQuant && !kRowMajor ? kMaxScaleCols : 1];
        u32x4 stage[kStaged ? kStagedVec : 1];
        int rows_of[kWaves][2][kRidingExperts];
    };
    __shared__ union Both {
        Lds layout;
        Riding riding;
        __device__ Both() {}
    } lds;
    if (static_cast<int>(blockIdx.x) <= num_blocks) {
        fused_layout<int64_t, false, kRidingSteps, kRowMajor ? 2 : 1>(lds.layout, idx, n_routes, num_experts, expert_begin, num_local, padded_local, chunk, num_chunks, counts, psum, offsets, num_rows, route_to_row, row_to_route, idx_copy, send, mailbox, sequence, epoch, tagged, num_blocks, rows, limit_ticks, timeouts, launch_id, MegaFront{}, total_word, row_words);
        return;
    }
    // Payload workgroups of fewer threads share one of these: `per` of them, each of whole waves.
    const PayloadShape& p = payload.shape;
    const int per = kThreads / p.threads, sub = threadIdx.x / p.threads, t = threadIdx.x - sub * p.threads;
    const unsigned block = (blockIdx.x - num_blocks - 1) * per + sub;
    if (sub >= per || block >= payload.blocks) return;  // (whole waves)
    const Routing routing = {idx, n_routes, num_experts, expert_begin, num_local};
    if (kRowMajor) {
        const AwaitedRows rows = {routing, row_words, total_word, launch_id, payload.looks, payload.rows, lds.riding.rows_of[threadIdx.x >> 6][0]};
        if (kQuant) quant_rows<DPEP_STORE_STREAMING>(payload.x, payload.weights, payload.out, payload.out_scales, payload.out_weights, p, rows, block, payload.blocks / p.parts, t);
        else copy_rows<DPEP_STORE_STREAMING>(payload.x, payload.scales, payload.weights, payload.out, payload.out_scales, payload.out_weights, p, rows, block, payload.blocks / p.parts, t);
    } else {
        const AwaitedTokens tokens = {routing, row_words, total_word, launch_id, payload.looks, payload.capacity, payload.all_or_none, lds.riding.rows_of[threadIdx.x >> 6]};
        if (kQuant) quant_token<DPEP_STORE_STREAMING>(payload.x, payload.weights, payload.out, payload.out_scales, payload.out_weights, p, tokens, block, t, lds.riding.tokens[sub], lds.riding.scales + sub * (p.threads / 8));
        else copy_token<DPEP_STORE_STREAMING, kStaged>(payload.x, payload.scales, payload.weights, payload.out, payload.out_scales, payload.out_weights, p, tokens, block, t,
                                                       lds.riding.tokens[sub], lds.riding.stage);
    }
}

// ---- one workgroup ---------------------------------------------------------------------------------------------------
// Up to kSingleRoutes routes over up to kSingleExperts local experts: sixteen waves of ONE workgroup hold them all, and
// nothing travels between workgroups (the exchange of the kernel above takes 2 us, whatever the size).  Every wave ranks
// its routes within (wave, expert) as it counts them; after one scan over waves and experts a route's row is one LDS read away.
// Bound by latencies (the ids 1 us, the scans, the stores) and by what one CU's LDS and store path take: 0.13 us per 256 routes.
// row_to_route is scattered in LDS and leaves as whole lines: scattered stores cost a cycle per lane, 1.3 us at 4096 routes.
// Measured on an MI355X, launches back to back, against the kernel above: 2400 routes over 256 experts 5.7 -> 3.8 us, 4096:
// 5.9 -> 4.5, 4096 of which one in eight is local 5.5 -> 3.9; at 6144 routes both take 5.9 us, at 16 384 10.7 against 6.4.
constexpr int kSingleWaves = 16;
constexpr int kSingleThreads = kSingleWaves * kWave;
constexpr int kSingleExperts = 256;
constexpr int kSingleSteps = 4;  // 64-route steps per wave
constexpr int kSingleRoutes = kSingleThreads * kSingleSteps;

// kMega: as above; the workgroups behind the first prepare rows.
template <typename IdxT, bool kMega>
__global__ __launch_bounds__(kSingleThreads) void layout_single_kernel(
    const IdxT* __restrict__ idx, int n_routes, int num_experts, int expert_begin, int num_local, int* __restrict__ counts,
    int* __restrict__ psum, int* __restrict__ offsets, int* __restrict__ num_rows, int* __restrict__ route_to_row,
    int* __restrict__ row_to_route, IdxT* __restrict__ idx_copy, SendCounts send, uint32_t* __restrict__ mailbox, uint32_t sequence,
    MegaFront front)
{
    __shared__ int rows_of[kSingleWaves][kSingleExperts];  // routes per wave and expert, later the wave's first row
    __shared__ unsigned long long match[kSingleWaves][kSingleExperts];
    __shared__ int totals[kSingleExperts];
    __shared__ int wave_sums[kSingleWaves];
    __shared__ int route_of[kSingleSteps * kSingleThreads];  // row_to_route: scattered here, copied out in order
    if (kMega && blockIdx.x > 0) {
        prepare_rows<kSingleThreads>(front, blockIdx.x - 1, reinterpret_cast<uint8_t*>(match));
        return;
    }
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int steps = (n_routes + kSingleThreads - 1) / kSingleThreads;  // the routes are dealt out evenly
    const int begin = min(wave * steps * kWave, n_routes), end = min(begin + steps * kWave, n_routes);
    int experts[kSingleSteps], rank[kSingleSteps];
    fetch_experts(experts, idx, begin, end, n_routes, num_experts, expert_begin, num_local, idx_copy);
    for (int e = lane; e < num_local; e += kWave) {
        rows_of[wave][e] = 0;
        match[wave][e] = 0ull;
    }
    wave_sync();
#pragma unroll
    for (int i = 0; i < kSingleSteps; ++i)
        if (begin + i * kWave < end) rank[i] = rank_step(experts[i], match[wave], rows_of[wave]);
    __syncthreads();
    int own[kSingleWaves], total = 0;
    if (tid < num_local) {
#pragma unroll
        for (int w = 0; w < kSingleWaves; ++w) {
            own[w] = rows_of[w][tid];
            total += own[w];
        }
    }
    const int incl = wave_scan(total);
    if (lane == kWave - 1) wave_sums[wave] = incl;
    if (tid < kSingleExperts) totals[tid] = total;
    __syncthreads();
    int sums[kSingleExperts / kWave], all = 0, offset = incl - total;
#pragma unroll
    for (int w = 0; w < kSingleExperts / kWave; ++w) {
        sums[w] = wave_sums[w];
        if (w < wave) offset += sums[w];
        all += sums[w];
    }
    if (tid < num_local) {
        int next = offset;
#pragma unroll
        for (int w = 0; w < kSingleWaves; ++w) {
            rows_of[w][tid] = next;
            next += own[w];
        }
        counts[tid] = total;
        psum[tid] = next;
        offsets[tid + 1] = next;
        if (send.counts != nullptr) send.counts[send.expert_begin + tid] = next;
    }
    if (tid == 0) {
        offsets[0] = 0;
        num_rows[0] = all;
    }
    if (mailbox != nullptr) {
        if (tid * 4 < num_local) {
            const int four[4] = {totals[tid * 4], totals[tid * 4 + 1], totals[tid * 4 + 2], totals[tid * 4 + 3]};
            mailbox_store_counts(mailbox, tid * 4, four, sequence, mailbox_narrow(n_routes));
        }
        if (tid == 0) mailbox_store_rows(mailbox, all, sequence);
    }
    send_counts_of_others(send, num_local, all, tid, kSingleThreads);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kSingleSteps; ++i) {
        const int route = begin + i * kWave + lane;
        if (route < end) {
            const int row = experts[i] >= 0 ? rows_of[wave][experts[i]] + rank[i] : -1;
            route_to_row[route] = row;
            if (row >= 0) route_of[row] = route;
        }
    }
    __syncthreads();
    for (int row = tid; row < all; row += kSingleThreads) row_to_route[row] = route_of[row];
    if (kMega && front.num_shared > 0) shared_rows(front, all, num_local, offsets, row_to_route, tid, kSingleThreads);
}

// The same preparation behind a layout that took two launches.
__global__ __launch_bounds__(kFrontThreads) void mega_front_kernel(MegaFront front, const int* __restrict__ num_rows, int num_local,
                                                                   int* __restrict__ offsets, int* __restrict__ row_to_route)
{
    __shared__ __attribute__((aligned(16))) uint8_t staged[kFrontThreads / 2];
    const unsigned blocks = front_blocks(front, kFrontThreads);
    if (blockIdx.x < blocks) prepare_rows<kFrontThreads>(front, blockIdx.x, staged);
    else shared_rows(front, num_rows[0], num_local, offsets, row_to_route, (blockIdx.x - blocks) * kFrontThreads + threadIdx.x,
                     (gridDim.x - blocks) * kFrontThreads);
}

int padded_experts(int num_local)
{
    int padded = 1;
    while (padded < num_local) padded <<= 1;
    return padded;
}

// Chunk length: as many chunks as the histogram budget allows (16..256), at least kMinChunk routes each.
int chunk_routes(int n_routes, int padded_local, int hist_ints = kHistInts)
{
    int max_chunks = hist_ints / padded_local;
    max_chunks = max_chunks > 256 ? 256 : (max_chunks < 16 ? 16 : max_chunks);
    int chunk = (n_routes + max_chunks - 1) / max_chunks;
    chunk = (chunk + kWave - 1) / kWave * kWave;
    return chunk < kMinChunk ? kMinChunk : chunk;
}

// The one-launch form's: 128 to 256 routes a wave, so that 128 waves share what there is; then 256, as long as that is at most 512 waves and the
// histograms have room; then longer ones.  Shorter chunks than two-launch ones, because a wave's steps are a serial chain and the exchange costs
// the same for 16 and for 128 workgroups (whole passes: 98 304 routes over 6 experts 144.5 -> 143.0 us, 32 768 over 256 147.9 -> 146.2, 36 864 over 6
// 28.4 -> 28.2, 6000 over 160 30.8 -> 30.2; with 128 everywhere 32 768 over 128 experts 255.3 against 253.2).
int one_launch_chunk(int n_routes, int padded_local)
{
    const int max_chunks = std::clamp(kTaggedInts / padded_local, 16, 512);
    const int even = std::clamp((n_routes + 127) / 128, kMinChunk / 2, kMinChunk);
    return (std::max(even, (n_routes + max_chunks - 1) / max_chunks) + kWave - 1) / kWave * kWave;
}

int check_layout_arguments(const void* idx, int num_tokens, int num_topk, int num_experts, int expert_begin, int num_local,
                           const int32_t* counts, const int32_t* psum, const int32_t* offsets, const int32_t* route_to_row,
                           const int32_t* row_to_route, const int32_t* num_rows)
{
    DPEP_REQUIRE(num_tokens >= 0 && num_topk >= 1 && num_topk <= DPEP_MAX_TOPK, "layout: bad T=%d K=%d", num_tokens,
                 num_topk);
    DPEP_REQUIRE(num_experts >= 1 && expert_begin >= 0 && num_local >= 1 && num_local <= DPEP_MAX_LOCAL_EXPERTS &&
                     expert_begin + num_local <= num_experts,
                 "layout: bad expert range E=%d begin=%d L=%d (at most %d local experts)", num_experts, expert_begin, num_local,
                 DPEP_MAX_LOCAL_EXPERTS);
    DPEP_REQUIRE(static_cast<long long>(num_tokens) * num_topk < (1ll << 31), "layout: T*K must fit int32");
    DPEP_REQUIRE(counts && psum && offsets && num_rows, "layout: NULL output");
    DPEP_REQUIRE(static_cast<long long>(num_tokens) * num_topk == 0 || (idx && route_to_row && row_to_route),
                 "layout: NULL routing buffer");
    return DPEP_OK;
}

// The two-launch form: count, then assign.  The count launch writes every histogram entry the assign launch reads, so
// the scratch needs no clearing and holds nothing between calls.
template <typename IdxT>
int enqueue_count_and_assign(const IdxT* idx, int n_routes, int num_experts, int expert_begin, int num_local, int padded, int chunk,
                             int num_chunks, int* wave_hist, int* block_hist, int32_t* counts, int32_t* psum, int32_t* offsets,
                             int32_t* num_rows, int32_t* route_to_row, int32_t* row_to_route, IdxT* idx_copy, const SendCounts& send,
                             uint32_t* mailbox, uint32_t sequence, hipStream_t stream)
{
    const int blocks = (num_chunks + kWaves - 1) / kWaves;
    if (blocks > 0) {
        hipLaunchKernelGGL(layout_count_kernel<IdxT>, dim3(blocks), dim3(kThreads), 0, stream, idx, n_routes, num_experts,
                           expert_begin, num_local, chunk, num_chunks, wave_hist, block_hist, idx_copy);
        if (int rc = launch_status("layout_count")) return rc;
    }
    // One workgroup more than there are chunks to assign: the reporter (with no routes, it alone publishes the
    // all-zero counts and prefix sums).
    hipLaunchKernelGGL(layout_assign_kernel<IdxT>, dim3(blocks + 1), dim3(kThreads), 0, stream, idx,
                       n_routes, num_experts, expert_begin, num_local, padded, chunk, num_chunks, wave_hist, block_hist, counts,
                       psum, offsets, num_rows, route_to_row, row_to_route, send, mailbox, sequence);
    return launch_status("layout_assign");
}

bool is_capturing(hipStream_t s)
{
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(s, &status) != hipSuccess || status != hipStreamCaptureStatusNone;
}

template <typename IdxT>
int launch_layout(void* ws, const IdxT* idx, int num_tokens, int num_topk, int num_experts, int expert_begin,
                  int num_local, int32_t* counts, int32_t* psum, int32_t* offsets, int32_t* route_to_row,
                  int32_t* row_to_route, int32_t* num_rows, IdxT* idx_copy, const SendCounts& send, bool report_to_host,
                  const MegaFront* front, const LayoutPayload* payload, bool* payload_launched, hipStream_t stream)
{
    Workspace* w = as_workspace(ws);
    DPEP_REQUIRE(w != nullptr, "layout: not a live workspace");
    if (int rc = check_layout_arguments(idx, num_tokens, num_topk, num_experts, expert_begin, num_local, counts, psum, offsets,
                                        route_to_row, row_to_route, num_rows))
        return rc;
    const int n_routes = num_tokens * num_topk;
    const size_t need = dpep_layout_workspace_bytes(num_tokens, num_topk, num_local);
    DPEP_REQUIRE(need <= w->bytes, "layout: workspace too small (%zu needed, %zu available)", need, w->bytes);
    // A one-launch layout whose wait for the other workgroups' histograms ran out left its number in the mailbox.  If nobody has been told yet
    // (the launch reported to no host wait: MegaMoE's internal layout), this call is; either way the workspace
    // takes two launches from then on.
    if (const uint32_t timed_out = w->mailbox_host[kMailboxTimeout]; timed_out != w->timeout_seen) {
        w->timeout_seen = timed_out;
        w->layout_one_launch = 0;
        return fail(DPEP_ERUNTIME, "layout: an earlier layout kernel on this workspace ran out of time waiting for the "
                                   "other workgroups' histograms and reported no rows; layouts on this workspace take two launches from now on");
    }
    w->layout_launches = w->layout_launches == 0xffffffffu ? 1u : w->layout_launches + 1u;  // never 0
    const int padded = padded_experts(num_local);
    int chunk = one_launch_chunk(n_routes, padded);
    const bool one_launch = n_routes > 0 && chunk_routes(n_routes, padded) <= kKeep * kWave && w->layout_one_launch;
    // Inputs that take two launches anyway get shorter chunks (more waves at work), with the larger histograms the
    // workspace has room for: 131 072 routes over 256 local experts 16 -> 64 workgroups.
    int hist_ints = kHistInts;
    if (!one_launch) {
        hist_ints = kLargeHistInts;
        chunk = chunk_routes(n_routes, padded, kLargeHistInts);
    }
    const int num_chunks = (n_routes + chunk - 1) / chunk;
    int* wave_hist = static_cast<int*>(w->base);
    int* block_hist = wave_hist + hist_ints;
    const int blocks = (num_chunks + kWaves - 1) / kWaves;
    if (report_to_host) {
        w->sequence = w->sequence == 0xffffffffu ? 1u : w->sequence + 1u;  // never 0: that is "nothing launched"
        w->mailbox_local = num_local;
        w->mailbox_narrow = mailbox_narrow(n_routes);
    }
    uint32_t* mailbox = report_to_host ? w->mailbox_device : nullptr;
    // (a test that wants the exchange to run out of time gets the kernel that has one)
    if (one_launch && n_routes <= kSingleRoutes && num_local <= kSingleExperts && w->exchange_extra_rows == 0) {
        auto launch = [&](auto kernel, unsigned more, const MegaFront& f) {
            hipLaunchKernelGGL(kernel, dim3(1 + more), dim3(kSingleThreads), 0, stream, idx, n_routes, num_experts, expert_begin,
                               num_local, counts, psum, offsets, num_rows, route_to_row, row_to_route, idx_copy, send, mailbox,
                               w->sequence, f);
        };
        if (front != nullptr) launch(layout_single_kernel<IdxT, true>, front_blocks(*front, kSingleThreads), *front);
        else launch(layout_single_kernel<IdxT, false>, 0u, MegaFront{});
        return launch_status("layout_single");
    }
    if (one_launch) {
        char* sync = static_cast<char*>(w->sync);
        auto launch = [&](auto kernel, unsigned more, const MegaFront& f) {
            hipLaunchKernelGGL(kernel, dim3(blocks + 1 + more), dim3(kThreads), 0, stream, idx, n_routes, num_experts, expert_begin,
                               num_local, padded, chunk, num_chunks, counts, psum, offsets, num_rows, route_to_row, row_to_route,
                               idx_copy, send, mailbox, w->sequence, reinterpret_cast<unsigned long long*>(sync),
                               reinterpret_cast<unsigned long long*>(sync + kSyncTagged), blocks, blocks + w->exchange_extra_rows,
                               w->exchange_ticks, w->mailbox_device + kMailboxTimeout, w->layout_launches, f);
        };
        // The payload rides along where the words have room for every route and the launch is not captured.
        if (payload != nullptr && chunk <= kRidingSteps * kWave && num_local <= kRidingExperts && n_routes <= kSyncRowWords && !is_capturing(stream)) {
            if constexpr (std::is_same_v<IdxT, int64_t>) {
                const unsigned per = kThreads / payload->shape.threads, more = (payload->blocks + per - 1) / per;
                auto ride = [&](auto kernel) {
                    hipLaunchKernelGGL(kernel, dim3(blocks + 1 + more), dim3(kThreads), 0, stream, idx, n_routes, num_experts, expert_begin,
                                       num_local, padded, chunk, num_chunks, counts, psum, offsets, num_rows, route_to_row, row_to_route,
                                       idx_copy, send, mailbox, w->sequence, reinterpret_cast<unsigned long long*>(sync),
                                       reinterpret_cast<unsigned long long*>(sync + kSyncTagged), blocks, blocks + w->exchange_extra_rows,
                                       w->exchange_ticks, w->mailbox_device + kMailboxTimeout, w->layout_launches,
                                       reinterpret_cast<unsigned long long*>(sync + kSyncTotal), reinterpret_cast<unsigned long long*>(sync + kSyncRows),
                                       *payload);
                };
                if (payload->row_major) payload->quantize ? ride(layout_payload_kernel<true, true, false>) : ride(layout_payload_kernel<false, true, false>);
                else if (payload->quantize) ride(layout_payload_kernel<true, false, false>);
                else payload->staged ? ride(layout_payload_kernel<false, false, true>) : ride(layout_payload_kernel<false, false, false>);
                *payload_launched = true;
                return launch_status("layout_payload");
            }
        }
        auto launch_steps = [&](auto steps_constant) {
            constexpr int kSteps = decltype(steps_constant)::value;
            if (front != nullptr) launch(layout_fused_kernel<IdxT, true, kSteps>, front_blocks(*front, kFrontThreads), *front);
            else launch(layout_fused_kernel<IdxT, false, kSteps>, 0u, MegaFront{});
        };
        if (chunk <= 2 * kWave) launch_steps(std::integral_constant<int, 2>{});
        else if (chunk <= 4 * kWave) launch_steps(std::integral_constant<int, 4>{});
        else if (chunk <= 8 * kWave) launch_steps(std::integral_constant<int, 8>{});
        else launch_steps(std::integral_constant<int, kKeep>{});
        return launch_status("layout_fused");
    }
    if (int rc = enqueue_count_and_assign<IdxT>(idx, n_routes, num_experts, expert_begin, num_local, padded, chunk, num_chunks,
                                                wave_hist, block_hist, counts, psum, offsets, num_rows, route_to_row, row_to_route,
                                                idx_copy, send, mailbox, w->sequence, stream))
        return rc;
    if (front != nullptr && (front->units > 0 || front->num_shared > 0)) {
        const unsigned rows_blocks = (static_cast<unsigned>(front->num_shared) * front->num_tokens + kFrontThreads - 1) / kFrontThreads;
        hipLaunchKernelGGL(mega_front_kernel, dim3(front_blocks(*front, kFrontThreads) + rows_blocks), dim3(kFrontThreads), 0, stream, *front, num_rows,
                           num_local, offsets, row_to_route);
        return launch_status("mega_front");
    }
    return DPEP_OK;
}

}  // namespace

// Shared with the MegaMoE forward, which routes on int32 ids; front: what else is prepared in front of its GEMMs.
int layout_i32(void* ws, const int32_t* idx, int num_tokens, int num_topk, int num_experts, int expert_begin,
               int num_local, int32_t* counts, int32_t* psum, int32_t* offsets, int32_t* route_to_row,
               int32_t* row_to_route, int32_t* num_rows, const MegaFront& front, hipStream_t stream)
{
    DPEP_REQUIRE(num_local <= kMegaExperts, "layout: %d local experts, at most %d", num_local, kMegaExperts);
    return launch_layout<int32_t>(ws, idx, num_tokens, num_topk, num_experts, expert_begin, num_local, counts, psum,
                                  offsets, route_to_row, row_to_route, num_rows, nullptr, SendCounts{}, /*report_to_host=*/false, &front, nullptr, nullptr, stream);
}

// The layout of a fresh dispatch (dpep_dispatch_fresh), and its payload, if it may ride along.
int layout_of_fresh(void* ws, const dpep_fresh_dispatch& c, const LayoutPayload* payload, bool* payload_launched, hipStream_t stream)
{
    return launch_layout<int64_t>(ws, c.topk_idx, c.num_tokens, c.num_topk, c.num_experts, c.expert_begin, c.num_local, c.counts,
                                  c.psum, c.offsets, c.route_to_row, c.row_to_route, c.num_rows, c.topk_idx_copy,
                                  SendCounts{c.send_counts, c.expert_begin, c.num_experts}, c.report_to_host != 0, nullptr, payload, payload_launched, stream);
}

}  // namespace dpep

// ---- the layout for callers that cannot allocate -------------------------------------------------------------
// Scratch of dpep_layout_static: the histograms a workspace would hold, in a device array of this library instead.
// Every GPU the library runs on has its own copy, at its own address, for the life of the process.
namespace dpep {
namespace {
constexpr size_t kStaticScratchInts = kHistInts + kBlockHistInts;  // 21 504 ints = 84 KiB
}
}
static __device__ __align__(256) int scratch[dpep::kStaticScratchInts];

namespace dpep {
namespace {

constexpr int kMaxDevices = 64;
int* g_scratch_of_device[kMaxDevices];  // device address of `scratch` on each GPU, looked up on first use
std::mutex g_scratch_mutex;

// The address of this GPU's copy of `scratch` (the current device's).  In host code the array's name is only a
// handle for the runtime, not a device address: kernels and memory calls get the looked-up pointer, never the name.
int scratch_of_current_device(int** out)
{
    int device = -1;
    DPEP_HIP(hipGetDevice(&device));
    DPEP_REQUIRE(device >= 0 && device < kMaxDevices, "layout_static: device %d outside [0, %d)", device, kMaxDevices);
    std::lock_guard<std::mutex> guard(g_scratch_mutex);
    if (g_scratch_of_device[device] == nullptr) {
        int* ptr = nullptr;
        DPEP_HIP(hipGetSymbolAddress(reinterpret_cast<void**>(&ptr), HIP_SYMBOL(scratch)));
        DPEP_REQUIRE(ptr != nullptr, "layout_static: the scratch array has no address on device %d", device);
        g_scratch_of_device[device] = ptr;
    }
    *out = g_scratch_of_device[device];
    return DPEP_OK;
}

}  // namespace
}  // namespace dpep

extern "C" {

size_t dpep_layout_workspace_bytes(int num_tokens, int num_topk, int num_local_experts)
{
    if (num_tokens < 0 || num_topk < 1 || num_local_experts < 1) return 0;
    return static_cast<size_t>(dpep::kLargeHistInts + dpep::kLargeBlockHistInts) * sizeof(int);
}

int dpep_layout(void* ws, const int64_t* topk_idx, int num_tokens, int num_topk, int num_experts, int expert_begin,
                int num_local, int32_t* counts, int32_t* psum, int32_t* offsets, int32_t* route_to_row,
                int32_t* row_to_route, int32_t* num_rows, void* stream)
{
    return dpep::launch_layout<int64_t>(ws, topk_idx, num_tokens, num_topk, num_experts, expert_begin, num_local,
                                        counts, psum, offsets, route_to_row, row_to_route, num_rows, nullptr, dpep::SendCounts{},
                                        /*report_to_host=*/true, nullptr, nullptr, nullptr, static_cast<hipStream_t>(stream));
}

int dpep_layout_static(const int64_t* topk_idx, int num_tokens, int num_topk, int num_experts, int expert_begin,
                       int num_local, int32_t* counts, int32_t* psum, int32_t* offsets, int32_t* route_to_row,
                       int32_t* row_to_route, int32_t* num_rows, void* stream)
{
    using namespace dpep;
    if (int rc = check_layout_arguments(topk_idx, num_tokens, num_topk, num_experts, expert_begin, num_local, counts, psum,
                                        offsets, route_to_row, row_to_route, num_rows))
        return rc;
    const int n_routes = num_tokens * num_topk;
    const int padded = padded_experts(num_local);
    const int chunk = chunk_routes(n_routes, padded);
    const int num_chunks = (n_routes + chunk - 1) / chunk;
    const int blocks = (num_chunks + kWaves - 1) / kWaves;
    // what the two launches address: num_chunks rows of wave histograms, blocks rows of workgroup histograms
    DPEP_REQUIRE(static_cast<size_t>(num_chunks) * num_local <= static_cast<size_t>(kHistInts) &&
                     static_cast<size_t>(blocks) * num_local <= static_cast<size_t>(kBlockHistInts),
                 "layout_static: %d chunks x %d local experts exceed the static scratch of %zu bytes", num_chunks, num_local,
                 kStaticScratchInts * sizeof(int));
    int* base = nullptr;
    if (int rc = scratch_of_current_device(&base)) return rc;
    return enqueue_count_and_assign<int64_t>(topk_idx, n_routes, num_experts, expert_begin, num_local, padded, chunk, num_chunks,
                                             base, base + kHistInts, counts, psum, offsets, num_rows, route_to_row, row_to_route,
                                             /*idx_copy=*/nullptr, SendCounts{}, /*mailbox=*/nullptr, 0u, static_cast<hipStream_t>(stream));
}

}  // extern "C"

// Shared host/device helpers for the gfx950 kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>

#include "../../include/deepep_amd.h"

namespace dpep {

int fail(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));

#define DPEP_REQUIRE(cond, ...)                              \
    do {                                                     \
        if (!(cond)) return ::dpep::fail(DPEP_EINVAL, __VA_ARGS__); \
    } while (0)

#define DPEP_HIP(expr)                                                                          \
    do {                                                                                        \
        hipError_t err_ = (expr);                                                               \
        if (err_ != hipSuccess)                                                                 \
            return ::dpep::fail(DPEP_ERUNTIME, "%s failed: %s", #expr, hipGetErrorString(err_)); \
    } while (0)

inline int launch_status(const char* what)
{
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) return fail(DPEP_ERUNTIME, "launch of %s failed: %s", what, hipGetErrorString(err));
    return DPEP_OK;
}

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

struct Workspace {
    uint32_t magic;
    void* base;
    size_t bytes;
    // Host mailbox of the routing layout: pinned host memory the layout kernel writes straight into, so that
    // the host learns the output sizes by polling instead of a device-to-host copy plus a stream wait (its words: see
    // kMailboxCounts below).
    uint32_t* mailbox_host;
    uint32_t* mailbox_device;  // the same memory as the kernels address it
    uint32_t sequence;         // of the most recent layout launch
    int mailbox_local;         // its number of local experts
    bool mailbox_narrow;       // and the form of its counts
    // One-launch layout: the memory its workgroups exchange histograms through, the bound of a workgroup's wait for the
    // others' histograms in 100 MHz ticks, and two switches for tests (take two launches instead; expect more
    // histogram rows than there are workgroups, so that the wait runs out).
    void* sync;  // kSyncBytes of device memory behind the caller's bytes, see below
    long long exchange_ticks;
    int exchange_extra_rows;
    int layout_one_launch;
    int payload_looks;         // of a payload in the layout's grid for a word of the layout's, before it works its rows out itself
    uint32_t layout_launches;  // number of the most recent layout launch (never 0)
    uint32_t timeout_seen;     // number of the last timed-out launch the host has been told about
    int gemm_zero_fill;        // 1 (default): idle workgroups of the first GEMM zero rows of unserved tokens; 0: the reduce does
    int megamoe_served_only;   // 1: rows of y whose token no local expert serves are left untouched; 0 (default): zeroed
    int gemm_tile_rows;  // 0: the grouped GEMM chooses its tile height; 64 / 128 / 192, or 32 (the few-rows kernel): forced (tests)
    int gemm_few_rows_waves;  // waves per workgroup of a forced few-rows kernel: 4 (default) or 1
    int gemm_paired;          // forced 128 rows: 0 (default) one of the kernels of every height, 1 the paired kernel, 2 that with streamed weights
    int gemm_column_waves;  // which grouped GEMM kernel runs: 1 = waves split the columns, weights straight to registers; 0 = 2 x 2 waves, weights through LDS
};
// Device memory the kernels synchronise through, behind the caller's bytes, zero when the workspace is created:
// at offset 0 the one-launch layout's epoch (64 bits: the highest tag any launch has used; a launch tags what it
// publishes with epoch + 1 and raises the epoch when it ends, so a replayed HIP graph gets a fresh tag too); at
// kSyncFillStop the word through which the MegaMoE fillers are told to stop (a counter that only grows: a filler stops when
// it differs from what the filler found at its start, so it needs no clearing and no value from the host); at kSyncReporterTag the tag the one-launch layout's reporter workgroup has settled on
// (64 bits; it publishes no histogram, so this is how the others know that it has read the epoch); from kSyncTagged on the
// tagged per-workgroup histograms of the one-launch layout; at kSyncTotal and from kSyncRows on the number of rows and the rows of the
// routes (or the routes of the rows), for a payload in the layout's grid, tagged with the number of the launch.
constexpr size_t kSyncFillStop = 64;
constexpr size_t kSyncReporterTag = 128;
constexpr size_t kSyncTagged = 256;
constexpr size_t kSyncTaggedWords = 8192 + DPEP_MAX_LOCAL_EXPERTS;  // (workgroups + 1) * experts never exceeds this
constexpr size_t kSyncTotal = kSyncTagged + kSyncTaggedWords * 8;
constexpr size_t kSyncRows = kSyncTotal + 256;
constexpr int kSyncRowWords = 65536;
constexpr size_t kSyncBytes = kSyncRows + static_cast<size_t>(kSyncRowWords) * 8;
// The host mailbox (pinned memory, 32-bit words): word 0 = number of rows and word 1 = sequence number of the layout
// that reported last (one 8-byte store); word kMailboxTimeout = launch number of a layout kernel whose wait for the
// other workgroups' histograms ran out; from word kMailboxCounts on the per-expert counts, 16 bytes for experts 4i .. 4i + 3:
// (counts of two experts, sequence number, counts of the other two, sequence number) where every count fits 16 bits;
// else (count, sequence number) of the first two there and of the other two in a second block of the same size.
// Every 8 bytes say themselves which launch they belong to, so the device sends everything at once and the host waits
// for what it reads (with one sequence number behind all counts the device had to wait for the counts' acknowledgement
// first, a trip across PCIe and back).  Lanes write consecutive 16-byte pieces: the same words at a stride of 32 bytes
// took 5 us longer for 256 experts.
constexpr int kMailboxTimeout = 2;
constexpr int kMailboxCounts = 4;
constexpr int kMailboxBlock = DPEP_MAX_LOCAL_EXPERTS;  // words of one block of counts
constexpr int kMailboxWords = kMailboxCounts + 2 * kMailboxBlock;
inline __host__ __device__ bool mailbox_narrow(int n_routes) { return n_routes < 65536; }
constexpr long long kLayoutExchangeTicks = 200000000;  // 2 s
constexpr int kPayloadLooks = 64;  // one or two microseconds apart; the words are there after about six
constexpr uint32_t kWorkspaceMagic = 0x44504550u;  // "DPEP"
Workspace* as_workspace(void* ws);

constexpr int kWave = 64;

// ---- device helpers -------------------------------------------------------------------------
__device__ __forceinline__ float bf16_to_f32(uint32_t bits16) { return __uint_as_float(bits16 << 16); }

// Inclusive sum over the wave's lanes, by row shifts and row broadcasts (an LDS permute per step costs 50 ns and more).
__device__ __forceinline__ int wave_scan(int v)
{
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);  // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);  // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);  // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1 and 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2 and 3
    return v;
}

// Round-to-nearest-even fp32 -> bf16 bits, two at a time: lo in bits 0-15, hi in bits 16-31
// (v_cvt_pk_bf16_f32; NaN stays a quiet NaN).
typedef float dpep_f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 dpep_bf16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi)
{
    const dpep_f32x2 v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, dpep_bf16x2));
}
__device__ __forceinline__ uint32_t f32_to_bf16(float v) { return pack_bf16x2(v, 0.0f) & 0xffffu; }

// The same pair of helpers for IEEE half (low-latency payloads): exact widening, round-to-nearest-even narrowing.
typedef _Float16 dpep_f16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float f16_to_f32(uint32_t bits16)
{
    return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(bits16)));
}
__device__ __forceinline__ uint32_t pack_f16x2(float lo, float hi)
{
    const dpep_f32x2 v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, dpep_f16x2));
}

// Local expert of a raw id, -1 if the route is past `end` or its expert is not one of this rank's.
__device__ __forceinline__ int local_expert(long long e, int route, int end, int num_experts, int expert_begin,
                                            int num_local)
{
    const long long local = e - expert_begin;
    const bool valid = route < end && e >= 0 && e < num_experts && local >= 0 && local < num_local;
    return valid ? static_cast<int>(local) : -1;
}

// Rows of experts 0..e on this rank for EVERY expert e of the job (a low-latency handle's send_counts): zero in front of the
// local experts, their inclusive prefix, the total behind them.  counts == nullptr: not wanted.
struct SendCounts {
    int* counts;
    int expert_begin, num_experts;
};
// The entries of experts that are not local, by `threads` threads that know the total.
__device__ __forceinline__ void send_counts_of_others(const SendCounts& send, int num_local, int total, int tid, int threads)
{
    if (send.counts == nullptr) return;
    for (int e = tid; e < send.num_experts; e += threads)
        if (e < send.expert_begin || e >= send.expert_begin + num_local) send.counts[e] = e < send.expert_begin ? 0 : total;
}

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ u32x4 load16(const void* p) { return *reinterpret_cast<const u32x4*>(p); }
// Streaming (non-temporal) 16-byte accesses: the byte movers write rows nobody reads again soon, and combine reads
// rows once.
__device__ __forceinline__ void store16_nt(void* p, u32x4 v) { __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(p)); }
// Write-through 16-byte store (device scope): the line goes to memory without waiting in the L2 for an eviction.  For
// the combine's output, which shares HBM with eight times as many reads, this measured 1 % faster than the streaming store.
__device__ __forceinline__ void store16_through(void* p, u32x4 v)
{
    asm volatile("global_store_dwordx4 %0, %1, off sc1" ::"v"(p), "v"(v) : "memory");
}
// Outputs beyond this go to HBM past the caches; smaller ones are written through, which the 256 MiB memory-side cache takes at
// up to 7.9 TB/s (88 MB zeroed: 11.2 us write-through, 14.7 us streaming; 235 MB: 40.8 and 39.3 us).
constexpr size_t kStreamBytes = 128u << 20;
__device__ __forceinline__ u32x4 load16_nt(const void* p) { return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p)); }

// Counts of four consecutive local experts, first of them `first` (a multiple of 4), into the host mailbox as 16-byte
// stores that go through every cache (system scope).
__device__ __forceinline__ void mailbox_store_counts(uint32_t* mailbox, int first, const int (&four)[4], uint32_t sequence, bool narrow)
{
    const uint32_t c[4] = {static_cast<uint32_t>(four[0]), static_cast<uint32_t>(four[1]), static_cast<uint32_t>(four[2]), static_cast<uint32_t>(four[3])};
    uint32_t* const to = mailbox + kMailboxCounts + first;
    const u32x4 a = {narrow ? c[0] | (c[1] << 16) : c[0], sequence, narrow ? c[2] | (c[3] << 16) : c[1], sequence};
    asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1" ::"v"(to), "v"(a) : "memory");
    if (!narrow) {
        const u32x4 b = {c[2], sequence, c[3], sequence};
        asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1" ::"v"(to + kMailboxBlock), "v"(b) : "memory");
    }
}
// The row count, with the sequence number the host polls for.
__device__ __forceinline__ void mailbox_store_rows(uint32_t* mailbox, int rows, uint32_t sequence)
{
    const unsigned long long word = (static_cast<unsigned long long>(sequence) << 32) | static_cast<uint32_t>(rows);
    __hip_atomic_store(reinterpret_cast<unsigned long long*>(mailbox), word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace dpep

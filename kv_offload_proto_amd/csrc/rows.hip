// Row movers for gfx950: decode miss import (host segments -> HBM hot buffer)
// and prefill export (HBM -> host segments).
//
// Semantics follow kvops/kernel/kvc_gather_rows.cpp:12-96 and
// kvc_scatter_rows_alllayer.cpp:11-67 of the reference, with the row
// ownership of kv_layout.h.  The reference moves each row with one HCOMM
// ReadNbi/WriteNbi; here the host segments are pinned host memory mapped
// into the device address space.  The import is one launch: each workgroup
// finds the winners (the last miss position per destination row) among its own
// positions, lists their rows in LDS with the reference's queued counts, and
// moves them as 16-byte chunks, 8 chunks in flight per lane.  Calls whose
// requests share rows over more than 8192 positions, and larger ones on
// striped segments, take two launches: winners in memory, then the listing and
// the copy, where 64 workgroups claim 256 positions at a time.
//
// Completion: the last workgroup to finish (atomicInc ticket) stores the
// status words with a system-scope release, after every workgroup fenced its
// own row stores, or waited for stores that go through the caches.  The
// reference's per-block Commit/Drain + MTE3 flush has the same meaning: all
// rows of the launch have landed.
#include <cstddef>

#include "kvx_internal.h"

namespace kvx {
namespace {

constexpr int kWaves = 4;          // waves per workgroup
constexpr int kUnroll = 8;         // 16-byte chunks in flight per lane

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
// 16-byte chunk of device or host memory, addressed in the global address
// space (global_* instructions: flat ones also count against the LDS wait
// counter, and the copy loops read their row addresses from LDS)
typedef __attribute__((address_space(1))) u32x4 GVec;
// device and host memory read through global-space pointers, for the same reason
#define KVX_G __attribute__((address_space(1)))

// winner tags (the scratch table): relaxed device-scope max and load
__device__ __forceinline__ void win_max(unsigned long long *p, unsigned long long v)
{
    __hip_atomic_fetch_max((KVX_G unsigned long long *)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long win_load(const unsigned long long *p)
{
    return __hip_atomic_load((const KVX_G unsigned long long *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

struct GatherExtra {
    uint64_t segBases[64];
    unsigned long long *win;
    uint64_t winEntries;
    uint32_t *chunkNext;   // next position chunk of the current import
    uint32_t *counters;
    uint32_t *errs;
    uint32_t *tickets;
    uint32_t *epoch;       // winner-tag epoch of the current call (device counter)
    uint32_t fused;
    uint32_t spanRows;
    uint32_t statusWords;
};

struct GatherParams {
    KvxLaunch<KvcGatherArgs> l;  // the reference launch block comes first
    GatherExtra x;
};

struct ExportExtra {
    uint32_t *tickets;
    uint64_t q0;          // first stripe owned by myNode
    uint64_t nStripes;    // stripes owned by myNode inside [rowLo, rowLo+rowCnt)
    uint64_t ownedRows;   // rows owned by myNode inside the range (reference queued / layer)
    uint32_t S;           // stripe rows used for item math (S == 0 mapped to 1)
    uint32_t N;           // node count used for item math (S == 0 mapped to 1)
};

struct ExportParams {
    KvxLaunch<KvcScatterAllArgs> l;
    ExportExtra x;
};

__device__ __forceinline__ int lane_id() { return __lane_id(); }

__device__ __forceinline__ void wave_sync_lds()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ void store_status(uint64_t addr, uint64_t word)
{
    __hip_atomic_store(reinterpret_cast<uint64_t *>(addr), word, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// A 16-byte store that goes through the caches to memory.  Once a workgroup's
// stores of this kind are done (wait_stores) its rows are visible everywhere,
// and it can report them without a fence: a device-scope release writes back
// the whole L2 of its XCD, and one per workgroup, while others still copy,
// took a fifth of the import (131072 positions from 1024 workgroups 859 -> 671
// us without it, 1665 positions from 105 27 -> 19).  The data registers of a
// store of more than 8 bytes may not be rewritten for two wait states, and the
// compiler, which does not see the store, does not keep them: they are part
// of the asm.
__device__ __forceinline__ void store_through(uint64_t addr, u32x4 v)
{
    asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1 nt\n\ts_nop 1" : : "v"(addr), "v"(v) : "memory");
}
__device__ __forceinline__ void wait_stores() { asm volatile("s_waitcnt vmcnt(0)" : : : "memory"); }

// Waits for N predicated loads at one point: each value passes through the
// asm, so the compiler waits for all of them before it and for none after it.
// Without it, every use under a condition of its own waits for everything in
// flight (vmcnt(0)), stores included: a copy's stores then go one round trip
// after another, and where a load's registers are reused for its address, its
// loads too (an export of 4000 rows 203 us, 98 so; 64 rows' append 7.3, 6.8).
template <int N>
__device__ __forceinline__ void wait_loads(u32x4 *v)
{
#pragma unroll
    for (int j = 0; j < N; ++j) asm volatile("" : "+v"(v[j]));
}

// The counters and error words of a call are zero between calls: the kernel
// that stores the status words zeroes them, and a first pass whose second one
// never ran leaves them zero too.  An error word holds ~p, max-reduced, of the
// lowest failing position or entry p (below 2^32 - 1), 0 for none.
__device__ __forceinline__ uint32_t error_word(uint32_t e) { return e == 0u ? 0u : row_error_code(~e); }

// A status word cleared at the start of a launch: the last workgroup's word
// follows it (its ticket comes after the clearing workgroup's wait).
__device__ __forceinline__ void clear_status(uint64_t addr)
{
    __hip_atomic_store(reinterpret_cast<uint64_t *>(addr), 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Copy `n` rows whose byte addresses sit in src[0..n), dst[0..n) (LDS or
// global) with the whole wave: chunk c covers bytes [16*(c%cpr), +16) of row
// c/cpr.  kUnroll loads are issued before their stores.  (kThrough false, the
// two-launch import: its stores wait for one another; in flight together they
// make it slower by 1 % at 32768 positions.)
template <bool kThrough = false>
__device__ __forceinline__ void wave_copy_rows(const uint64_t *src, const uint64_t *dst, uint32_t n, uint32_t cpr)
{
    const uint32_t total = n * cpr;
    const uint32_t lane = static_cast<uint32_t>(lane_id());
    for (uint32_t base = 0; base < total; base += 64u * kUnroll) {
        u32x4 v[kUnroll];
        uint64_t d[kUnroll];
#pragma unroll
        for (int j = 0; j < kUnroll; ++j) {
            const uint32_t c = base + static_cast<uint32_t>(j) * 64u + lane;
            d[j] = 0;
            if (c < total) {
                const uint32_t r = c / cpr;
                const uint32_t o = (c - r * cpr) * 16u;
                v[j] = __builtin_nontemporal_load(reinterpret_cast<const GVec *>(src[r] + o));
                d[j] = dst[r] + o;
            }
        }
        if constexpr (kThrough) wait_loads<kUnroll>(v);
#pragma unroll
        for (int j = 0; j < kUnroll; ++j) {
            if (d[j] == 0) continue;
            if constexpr (kThrough) store_through(d[j], v[j]);
            else __builtin_nontemporal_store(v[j], reinterpret_cast<GVec *>(d[j]));
        }
    }
}

__device__ __forceinline__ int32_t clamp_num_real(uint64_t numRealAddr, uint32_t maxNumReqs)
{
    int32_t n = *reinterpret_cast<const int32_t *>(numRealAddr);
    if (n > static_cast<int32_t>(maxNumReqs)) n = static_cast<int32_t>(maxNumReqs);  // kvc_gather_rows.cpp:17-21
    return n < 0 ? 0 : n;
}

__device__ __forceinline__ uint64_t win_index(int64_t bid, int32_t slot, uint32_t spanRows)
{
    return static_cast<uint64_t>(bid) * spanRows + static_cast<uint64_t>(slot);
}

// Pass 1: per destination row, the last valid miss position (tagged with the
// call's epoch so the scratch never needs clearing; the epoch lives in device
// memory and the last copy workgroup advances it, so a captured graph replays
// correctly).  Block 0 also zeroes the chunk counter, the queued counters
// and the status words of the nodes this call reports.
__global__ __launch_bounds__(256) void kvx_gather_prep(GatherParams P)
{
    const KvcGatherArgs &a = P.l.a;
    const GatherExtra &x = P.x;
    const int32_t numReal = clamp_num_real(a.numReal, a.maxNumReqs);
    const int64_t total = static_cast<int64_t>(numReal) * a.topK;
    if (blockIdx.x == 0) {
        const uint32_t n0 = x.fused ? 0u : a.myNode;
        const uint32_t n1 = x.fused ? a.nodeNum : a.myNode + 1u;
        if (threadIdx.x == 0) *x.chunkNext = 0u;
        for (uint32_t i = threadIdx.x; i < (n1 - n0) * 8u; i += blockDim.x) {
            x.counters[n0 * 8u + i] = 0u;
            x.errs[n0 * 8u + i] = 0u;
        }
        if (a.status != 0) {
            for (uint32_t i = threadIdx.x; i < (n1 - n0) * x.statusWords; i += blockDim.x) {
                const uint32_t node = n0 + i / x.statusWords, b = i % x.statusWords;
                store_status(a.status + node * 64ull + b * 8ull, 0ull);
            }
        }
    }
    const KVX_G int32_t *topk = reinterpret_cast<const KVX_G int32_t *>(a.topkIndices);
    const KVX_G int32_t *slots = reinterpret_cast<const KVX_G int32_t *>(a.topKDeviceSlots);
    const KVX_G int8_t *miss = reinterpret_cast<const KVX_G int8_t *>(a.isMiss);
    const KVX_G int64_t *pool = reinterpret_cast<const KVX_G int64_t *>(a.reqPoolIndices);
    const unsigned long long tagHi = static_cast<unsigned long long>(*x.epoch) << 32;
    for (int64_t p = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; p < total;
         p += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        if (miss[p] == 0) continue;
        const int32_t t = topk[p], s = slots[p];
        if (t < 0 || s < 0 || s >= 65536) continue;
        const int64_t bid = p / a.topK;
        if (pool[bid] < 0) continue;
        const uint64_t d = win_index(bid, s, x.spanRows);
        if (d < x.winEntries) win_max(x.win + d, tagHi | static_cast<unsigned long long>(p));
    }
}

// Pass 2: each workgroup claims kSpan consecutive positions at a time (a
// counter the first pass zeroes), lists the winners owned by the node(s) of
// this call in LDS while counting the queued rows per (node, status word),
// and moves them with its four waves; no row list passes through HBM.
// kSpanBlocks workgroups: fewer concurrent readers of host memory move more
// bytes per second over the link than one workgroup per chunk, and claiming
// chunks keeps them evenly loaded.  The last workgroup (ticket) advances the
// epoch and stores the status words.
constexpr uint32_t kSpan = 256;
constexpr uint32_t kSpanBlocks = 64;

__global__ __launch_bounds__(256) void kvx_gather_span(GatherParams P)
{
    __shared__ uint32_t sCnt[64 * 8];
    __shared__ uint64_t sSrc[kSpan], sDst[kSpan];
    __shared__ uint32_t sN, sEpoch, sChunk;
    __shared__ int sLast;
    const KvcGatherArgs &a = P.l.a;
    const GatherExtra &x = P.x;
    const uint32_t tid = threadIdx.x;
    const uint32_t wave = tid / 64u;
    const uint32_t lane = static_cast<uint32_t>(lane_id());
    const uint32_t cpr = a.rowBytes / 16u;
    const int32_t numReal = clamp_num_real(a.numReal, a.maxNumReqs);
    const int64_t total = static_cast<int64_t>(numReal) * a.topK;
    const int64_t chunks = (total + kSpan - 1) / kSpan;
    const uint64_t ppc = a.positionsPerCore == 0 ? 1ull : a.positionsPerCore;
    const KVX_G int32_t *topk = reinterpret_cast<const KVX_G int32_t *>(a.topkIndices);
    const KVX_G int32_t *slots = reinterpret_cast<const KVX_G int32_t *>(a.topKDeviceSlots);
    const KVX_G int8_t *miss = reinterpret_cast<const KVX_G int8_t *>(a.isMiss);
    const KVX_G int64_t *pool = reinterpret_cast<const KVX_G int64_t *>(a.reqPoolIndices);
    const KVX_G int64_t *hostBase = reinterpret_cast<const KVX_G int64_t *>(a.reqHostBase);
    for (uint32_t i = tid; i < 64u * 8u; i += blockDim.x) sCnt[i] = 0u;
    if (tid == 0) sEpoch = *x.epoch;
    __syncthreads();
    const unsigned long long tagHi = static_cast<unsigned long long>(sEpoch) << 32;
    for (;;) {
        if (tid == 0) {
            sN = 0u;
            sChunk = atomicAdd(x.chunkNext, 1u);
        }
        __syncthreads();
        const int64_t chunk = sChunk;
        if (chunk >= chunks) break;
#pragma unroll
        for (uint32_t q = 0; q < kSpan / 256u; ++q) {
            const int64_t p = chunk * kSpan + q * 256u + tid;
            bool copy = false;
            uint64_t src = 0, dst = 0;
            if (p < total && miss[p] != 0) {
                const int32_t t = topk[p], s = slots[p];
                const int64_t bid = p / a.topK;
                if (t >= 0 && s >= 0 && pool[bid] >= 0) {
                    const uint32_t row = static_cast<uint32_t>(hostBase[bid] + t);  // kvc_gather_rows.cpp:69-73
                    const uint32_t node = kvx_node_of(row, a.stripeRows, a.nodeNum);
                    const bool owned = x.fused ? (node < a.nodeNum) : (node == a.myNode);
                    if (owned) {
                        const uint32_t key = node * 8u + static_cast<uint32_t>(static_cast<uint64_t>(p) / ppc);
                        atomicAdd(&sCnt[key], 1u);
                        bool winner = true;
                        if (s < 65536) {
                            const uint64_t d = win_index(bid, s, x.spanRows);
                            if (d < x.winEntries) winner = (win_load(x.win + d) == (tagHi | static_cast<unsigned long long>(p)));
                        }
                        const uint64_t segRow = kvx_seg_row_of(row, a.stripeRows, a.nodeNum);
                        if (segRow >= a.perLayerSegRows) {  // row outside the segment: report, do not read
                            atomicMax(&x.errs[key], ~static_cast<uint32_t>(p));
                            winner = false;
                        }
                        copy = winner;
                        const uint64_t segBase = x.fused ? x.segBases[node] : a.segBase;
                        src = segBase + (static_cast<uint64_t>(a.layerOffsetRows) + segRow) * a.rowBytes;
                        dst = a.hotRowBase +
                              (static_cast<uint64_t>(s) + static_cast<uint64_t>(bid) * a.hotReqStrideRows) * a.rowBytes;
                    }
                }
            }
            const uint64_t cm = __ballot(copy);
            uint32_t base = 0;
            if (lane == 0 && cm != 0ull) base = atomicAdd(&sN, static_cast<uint32_t>(__popcll(cm)));
            base = static_cast<uint32_t>(__shfl(static_cast<int>(base), 0));
            if (copy) {
                const uint32_t at = base + static_cast<uint32_t>(__popcll(cm & ((1ull << lane) - 1ull)));
                sSrc[at] = src;
                sDst[at] = dst;
            }
        }
        __syncthreads();
        const uint32_t n = sN, share = (n + kWaves - 1u) / kWaves, r0 = wave * share;
        if (r0 < n) wave_copy_rows(sSrc + r0, sDst + r0, (n - r0 < share) ? n - r0 : share, cpr);
        __syncthreads();  // the list and the chunk are rewritten by the next round
    }
    for (uint32_t i = tid; i < 64u * 8u; i += blockDim.x) {
        if (sCnt[i] != 0u) atomicAdd(&x.counters[i], sCnt[i]);
    }

    __threadfence();
    __syncthreads();
    if (tid == 0) {
        const unsigned int ticket = atomicInc(&x.tickets[0], gridDim.x - 1u);
        sLast = (ticket == gridDim.x - 1u) ? 1 : 0;
    }
    __syncthreads();
    if (!sLast) return;
    // the next call's epoch; at the wrap to 0 the tags of 2^32 calls ago
    // could alias, so the table is cleared (once in 2^32 calls)
    if (sEpoch + 1u == 0u) {
        for (uint64_t i = tid; i < x.winEntries; i += blockDim.x) x.win[i] = 0ull;
    }
    if (tid == 0) *x.epoch = sEpoch + 1u;
    __threadfence();
    const uint32_t n0 = x.fused ? 0u : a.myNode;
    const uint32_t n1 = x.fused ? a.nodeNum : a.myNode + 1u;
    for (uint32_t i = tid; i < (n1 - n0) * 8u; i += blockDim.x) {
        const uint32_t node = n0 + i / 8u, b = i % 8u;
        const uint32_t q = __hip_atomic_load(&x.counters[node * 8u + b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const uint32_t e = __hip_atomic_load(&x.errs[node * 8u + b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        x.counters[node * 8u + b] = 0u;
        x.errs[node * 8u + b] = 0u;
        if (a.status == 0 || b >= x.statusWords) continue;
        uint64_t word = 1ull << 32;  // kvc_gather_rows.cpp:29-33, :93
        if (static_cast<int64_t>(b * ppc) < total) {
            word |= (static_cast<uint64_t>(q) << 40) | error_word(e);
        }
        store_status(a.status + node * 64ull + b * 8ull, word);
    }
}

// The import in one launch, where a group -- the positions that can share a
// destination row -- is short: a request (rows of request b start at
// b * spanRows), or the whole call where every request has the same rows
// (spanRows 0).  A winner is the last miss on its destination row.  Each
// workgroup takes `span` consecutive positions of one group and marks the
// slots of the group's later positions in a bitmap; an own position wins when
// its slot is neither there nor at a later own position.  A slot at or past
// spanRows also reaches rows of later requests: such positions (none in a
// buffer of spanRows slots a request) are looked for in those requests one by
// one.  The workgroup counts its own queued rows and errors, adds them to the
// call's counters and moves its rows; the last one (ticket) stores the status
// words and leaves the counters zeroed for the next call.
//
// The bound is the host link.  The reads of many CUs fill it (1638 rows of
// 1152 bytes alone: 72 us from 16 workgroups, 46 from 32, 40 from 128 and
// more), so the spans are short: 16 positions up to 1024 spans, so that a
// workgroup's next span is listed while others copy (50 requests of 300
// positions: 182 us in spans of 64, 172 of 32, 159 of 16), then up to 64, taken
// in turn by 256 workgroups, which keeps the rows in flight near each other
// (64 requests of 2048 positions: 64 workgroups 674 us, 128 639, 256 633, 512
// 651, 1024 662; spans of 128: 654 from 256).  Against a launch that marked
// the winners in memory and one that listed and moved the rows: 8192 positions
// 56 -> 47 us, 1665 positions in the earlier one-launch form, where every
// workgroup counted all positions, 29 -> 19; 131072 positions 639 -> 633 (0.2
// misses: the link).  The spans are those of the positions in use: a call, or a captured
// graph's replay, with fewer requests than it was made for does nothing for
// the others (256 requests of 1024 positions with 16 in use 102 us when every
// span of the largest batch was walked, 77 so; with none 20 and 7).
constexpr uint32_t kOneMinSpan = 16, kOneMaxSpan = 64;
constexpr uint32_t kOneMaxGroup = 8192;  // positions of a group (each workgroup reads the later ones)
constexpr uint32_t kOneMaxBlocks = 256;  // workgroups; more spans are taken in turn
// Rows of a stripe share one segment row, whose repeats an XCD's L2 serves
// when neighbouring positions meet there: larger calls of that kind keep the
// two launches, whose 64 workgroups take 256 positions each.  The line lies
// where no stripe loses (0.3 misses, us in two launches and in one): 4096
// positions 41.7 and 38.3 at stripes of 2, 38.6 and 38.3 at 64; 8192 66.7 and
// 59.5 at 2, 61.3 and 58.9 at 16, 49.9 and 57.3 at 64; 32768 221 and 211 at 2,
// 193 and 205 at 16, 142 and 185 at 64.
constexpr uint32_t kOneMaxStriped = 4096;
constexpr int kOneThreads = 256;

struct GatherSpans {
    uint32_t span, parts, count;  // positions of a span, spans of a group and in all
};

// The spans of `positions` positions in groups of `group` (a divisor).
__host__ __device__ __forceinline__ GatherSpans gather_spans(uint32_t positions, uint32_t group)
{
    GatherSpans g{kOneMinSpan, 0u, 0u};
    if (positions == 0u) return g;
    while (g.span < kOneMaxSpan && positions / g.span > 4u * kOneMaxBlocks) g.span *= 2u;
    g.parts = (group + g.span - 1u) / g.span;
    g.count = positions / group * g.parts;
    return g;
}

__global__ __launch_bounds__(kOneThreads) void kvx_gather_one(GatherParams P)
{
    __shared__ uint32_t sLater[65536 / 32];
    __shared__ uint32_t sCnt[64 * 8], sErr[64 * 8];
    __shared__ uint64_t sSrc[kOneMaxSpan], sDst[kOneMaxSpan];
    __shared__ int32_t sKey[kOneMaxSpan];   // slot of an own position in the winner rule, else -1
    __shared__ uint32_t sLose[kOneMaxSpan / 32];
    __shared__ uint32_t sN;
    __shared__ int sLast;
    const KvcGatherArgs &a = P.l.a;
    const GatherExtra &x = P.x;
    const uint32_t tid = threadIdx.x, lane = static_cast<uint32_t>(lane_id());
    const uint32_t n0 = x.fused ? 0u : a.myNode;
    const uint32_t n1 = x.fused ? a.nodeNum : a.myNode + 1u;
    const uint32_t ppc = a.positionsPerCore == 0 ? 1u : a.positionsPerCore;
    const KVX_G int32_t *topk = reinterpret_cast<const KVX_G int32_t *>(a.topkIndices);
    const KVX_G int32_t *slots = reinterpret_cast<const KVX_G int32_t *>(a.topKDeviceSlots);
    const KVX_G int8_t *miss = reinterpret_cast<const KVX_G int8_t *>(a.isMiss);
    const KVX_G int64_t *pool = reinterpret_cast<const KVX_G int64_t *>(a.reqPoolIndices);
    const KVX_G int64_t *hostBase = reinterpret_cast<const KVX_G int64_t *>(a.reqHostBase);
    const int32_t numReal = __builtin_amdgcn_readfirstlane(clamp_num_real(a.numReal, a.maxNumReqs));
    const uint32_t total = static_cast<uint32_t>(numReal) * a.topK;  // (host: below 2^31)
    const uint32_t groupSize = x.spanRows == 0u ? total : a.topK;
    const GatherSpans sp = gather_spans(total, groupSize);
    const uint32_t span = sp.span;
    if (blockIdx.x == 0 && a.status != 0) {  // the call's status words read 0 until its rows have landed
        for (uint32_t i = tid; i < (n1 - n0) * x.statusWords; i += kOneThreads) {
            clear_status(a.status + (n0 + i / x.statusWords) * 64ull + (i % x.statusWords) * 8ull);
        }
    }
    for (uint32_t i = n0 * 8u + tid; i < n1 * 8u; i += kOneThreads) {
        sCnt[i] = 0u;
        sErr[i] = 0u;
    }
    for (uint32_t blk = blockIdx.x; blk < sp.count; blk += gridDim.x) {
        const uint32_t group = blk / sp.parts, part = blk - group * sp.parts;
        const uint32_t g0 = group * groupSize, lo = g0 + part * span, p = lo + tid, bid = p / a.topK;
        for (uint32_t i = tid; i < 65536u / 32u / 4u; i += kOneThreads) reinterpret_cast<uint4 *>(sLater)[i] = make_uint4(0, 0, 0, 0);
        if (tid < kOneMaxSpan / 32u) sLose[tid] = 0u;
        if (tid == 0) sN = 0u;
        const uint32_t gEnd = min(g0 + groupSize, total);
        const uint32_t hi = min(lo + span, gEnd);
        int8_t m = 0;
        int32_t t = -1, s = -1;
        int64_t pl = -1, hb = 0;
        if (tid < span && p < gEnd) {  // the own position's five reads, issued together
            m = miss[p];
            t = topk[p];
            s = slots[p];
            pl = pool[bid];
            hb = hostBase[bid];
        }
        // a position in the winner rule: a miss with a token and a slot (16 bits)
        const bool valid = m != 0 && t >= 0 && s >= 0 && pl >= 0;
        const bool rule = valid && s < 65536;
        if (tid < span) sKey[tid] = rule ? s : -1;
        __syncthreads();
        for (uint32_t q0 = hi + tid; q0 < gEnd; q0 += 4u * kOneThreads) {
            int8_t mq[4];
            int32_t tq[4], sq[4];
            int64_t pq[4];
#pragma unroll
            for (uint32_t j = 0; j < 4u; ++j) {  // issued together
                const uint32_t q = q0 + j * kOneThreads, c = q < gEnd ? q : gEnd - 1u;
                mq[j] = q < gEnd ? miss[c] : static_cast<int8_t>(0);
                tq[j] = topk[c];
                sq[j] = slots[c];
                pq[j] = pool[c / a.topK];
            }
#pragma unroll
            for (uint32_t j = 0; j < 4u; ++j) {
                if (mq[j] != 0 && tq[j] >= 0 && sq[j] >= 0 && sq[j] < 65536 && pq[j] >= 0) {
                    atomicOr(&sLater[sq[j] >> 5], 1u << (sq[j] & 31));
                }
            }
        }
        // own positions against the later own ones, kOneThreads / span lanes each
        {
            const uint32_t per = kOneThreads / span, i = tid / per;  // span: a power of two
            const int32_t k = sKey[i];
            bool later = false;
            if (k >= 0) {
                for (uint32_t j = i + 1u + (tid & (per - 1u)); j < span; j += per) later |= sKey[j] == k;
            }
            if (later) atomicOr(&sLose[i >> 5], 1u << (i & 31u));
        }
        const bool far = rule && x.spanRows != 0u && static_cast<uint32_t>(s) >= x.spanRows;
        if (__syncthreads_or(far ? 1 : 0)) {
            for (uint32_t i = 0; i < span; ++i) {
                const int32_t k = sKey[i];
                if (k < 0 || static_cast<uint32_t>(k) < x.spanRows) continue;
                const uint32_t b0 = (lo + i) / a.topK;
                const uint32_t b1 = min(static_cast<uint32_t>(numReal) - 1u, b0 + static_cast<uint32_t>(k) / x.spanRows);
                bool later = false;
                for (uint32_t q = (b0 + 1u) * a.topK + tid; q < (b1 + 1u) * a.topK; q += kOneThreads) {
                    const uint32_t bq = q / a.topK;
                    later |= miss[q] != 0 && topk[q] >= 0 && pool[bq] >= 0 &&
                             slots[q] == k - static_cast<int32_t>((bq - b0) * x.spanRows);
                }
                if (later) atomicOr(&sLose[i >> 5], 1u << (i & 31u));
            }
            __syncthreads();
        }
        bool copy = false;
        uint64_t src = 0, dst = 0;
        if (valid) {
            const uint32_t row = static_cast<uint32_t>(hb + t);  // kvc_gather_rows.cpp:69-73
            const uint32_t node = kvx_node_of(row, a.stripeRows, a.nodeNum);
            if (x.fused ? (node < a.nodeNum) : (node == a.myNode)) {
                const uint32_t key = node * 8u + p / ppc;
                atomicAdd(&sCnt[key], 1u);
                const uint64_t segRow = kvx_seg_row_of(row, a.stripeRows, a.nodeNum);
                if (segRow >= a.perLayerSegRows) {  // row outside the segment: report the lowest, do not read
                    atomicMax(&sErr[key], ~p);
                } else {
                    copy = !rule || (((sLater[s >> 5] >> (s & 31)) | (sLose[tid >> 5] >> (tid & 31u))) & 1u) == 0u;
                    src = (x.fused ? x.segBases[node] : a.segBase) +
                          (static_cast<uint64_t>(a.layerOffsetRows) + segRow) * a.rowBytes;
                    dst = a.hotRowBase + (static_cast<uint64_t>(s) + static_cast<uint64_t>(bid) * a.hotReqStrideRows) * a.rowBytes;
                }
            }
        }
        const uint64_t cm = __ballot(copy);
        uint32_t at = 0;
        if (lane == 0 && cm != 0ull) at = atomicAdd(&sN, static_cast<uint32_t>(__popcll(cm)));
        at = static_cast<uint32_t>(__shfl(static_cast<int>(at), 0));
        if (copy) {
            at += static_cast<uint32_t>(__popcll(cm & ((1ull << lane) - 1ull)));
            sSrc[at] = src;
            sDst[at] = dst;
        }
        __syncthreads();
        // the rows' chunks over all lanes
        const uint32_t cpr = a.rowBytes / 16u, chunks = sN * cpr;
        for (uint32_t c0 = tid; c0 < chunks; c0 += kOneThreads * kUnroll) {
            u32x4 v[kUnroll];
            uint64_t d[kUnroll];
#pragma unroll
            for (int j = 0; j < kUnroll; ++j) {
                const uint32_t c = c0 + static_cast<uint32_t>(j) * kOneThreads;
                d[j] = 0;
                if (c < chunks) {
                    const uint32_t r = c / cpr, o = (c - r * cpr) * 16u;
                    v[j] = __builtin_nontemporal_load(reinterpret_cast<const GVec *>(sSrc[r] + o));
                    d[j] = sDst[r] + o;
                }
            }
            wait_loads<kUnroll>(v);
#pragma unroll
            for (int j = 0; j < kUnroll; ++j) {
                if (d[j] != 0) store_through(d[j], v[j]);
            }
        }
        __syncthreads();  // the lists are rewritten by the next span
    }
    // the call's counts
    for (uint32_t i = n0 * 8u + tid; i < n1 * 8u; i += kOneThreads) {
        if (sCnt[i] != 0u) atomicAdd(&x.counters[i], sCnt[i]);
        if (sErr[i] != 0u) atomicMax(&x.errs[i], sErr[i]);
    }
    wait_stores();
    __syncthreads();
    if (tid == 0) {
        const unsigned int ticket = atomicInc(&x.tickets[3], gridDim.x - 1u);
        sLast = (ticket == gridDim.x - 1u) ? 1 : 0;
    }
    __syncthreads();
    if (!sLast) return;
    __threadfence();
    for (uint32_t i = tid; i < (n1 - n0) * 8u; i += kOneThreads) {
        const uint32_t node = n0 + i / 8u, b = i % 8u;
        const uint32_t q = __hip_atomic_load(&x.counters[node * 8u + b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const uint32_t e = __hip_atomic_load(&x.errs[node * 8u + b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (q != 0u) __hip_atomic_store(&x.counters[node * 8u + b], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (e != 0u) __hip_atomic_store(&x.errs[node * 8u + b], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (a.status == 0 || b >= x.statusWords) continue;
        uint64_t word = 1ull << 32;  // kvc_gather_rows.cpp:29-33, :93
        if (static_cast<uint64_t>(b) * ppc < total) word |= (static_cast<uint64_t>(q) << 40) | error_word(e);
        store_status(a.status + node * 64ull + b * 8ull, word);
    }
}

// Prefill export: item (layer l, owned stripe i) copies the stripe's winning
// row (its highest row inside the range) to segment row q/N of layer l.  Rows
// are stored through the caches: with a system-scope fence per workgroup, each
// a write-back of an XCD's L2, 144 MB took 2751 us, now 2534 (56.9 GB/s of the
// link's 57.0).  Up to 64 workgroups: with their chunks in flight they fill
// the link, and 128 or more get less from it (131072 rows, 2671 us from 48 or
// 64, 2681 from 96, 2690 from 128 to 512).
constexpr uint32_t kExportBlocks = 64;

__global__ __launch_bounds__(256) void kvx_export_alllayer(ExportParams P)
{
    __shared__ uint64_t sSrc[kWaves][64];
    __shared__ uint64_t sDst[kWaves][64];
    __shared__ int sLast;
    const KvcScatterAllArgs &a = P.l.a;
    const ExportExtra &x = P.x;
    const int wave = threadIdx.x / 64;
    const uint32_t lane = static_cast<uint32_t>(lane_id());
    const uint64_t items = x.nStripes * a.layerNum;
    const uint64_t rowHi = static_cast<uint64_t>(a.rowLo) + a.rowCnt;
    const uint32_t cpr = a.rowBytes / 16u;

    for (uint64_t base = (static_cast<uint64_t>(blockIdx.x) * kWaves + wave) * 64ull; base < items;
         base += static_cast<uint64_t>(gridDim.x) * kWaves * 64ull) {
        const uint64_t it = base + lane;
        if (it < items) {
            const uint64_t l = it / x.nStripes, i = it - l * x.nStripes;
            const uint64_t q = x.q0 + i * x.N;
            uint64_t w = q * x.S + x.S - 1ull;
            if (w > rowHi - 1ull) w = rowHi - 1ull;
            const uint64_t segRow = q / x.N;
            sSrc[wave][lane] = a.srcLayer0Base + l * a.srcLayerStride + w * a.rowBytes;
            sDst[wave][lane] = a.segBase + (l * a.perLayerSegRows + segRow) * a.rowBytes;
        }
        wave_sync_lds();
        const uint64_t left = items - base;
        wave_copy_rows<true>(sSrc[wave], sDst[wave], static_cast<uint32_t>(left < 64ull ? left : 64ull), cpr);
        wave_sync_lds();
    }

    wait_stores();
    __syncthreads();
    if (threadIdx.x == 0) {
        const unsigned int ticket = atomicInc(&x.tickets[1], gridDim.x - 1u);
        sLast = (ticket == gridDim.x - 1u) ? 1 : 0;
    }
    __syncthreads();
    if (!sLast || a.status == 0) return;
    const uint32_t words = a.blockDim == 0 ? 1u : a.blockDim;
    for (uint32_t b = threadIdx.x; b < words; b += blockDim.x) {
        uint64_t word = 1ull << 32;  // kvc_scatter_rows_alllayer.cpp:59-61
        if (b == 0) word |= (x.ownedRows * a.layerNum) << 40;
        store_status(a.status + a.myNode * 64ull + b * 8ull, word);
    }
}

// Decode-incremental export of one layer (the reference design's
// export_rows / kvc_scatter_rows, doc/kv_offload_design.md:322-327,394-396:
// the import's shape with the direction reversed).  Entry i < num_real names
// host row indices[i]; the row owned by myNode is copied from
// srcLayerBase + i*rowBytes to its segment row of layer layerId.  Entries
// naming one segment row resolve as a sequential walk would: the last wins.
struct ExportRowsParams {
    ExportRowsArgs a;
    uint64_t segBases[64];   // fused form: every node's segment base
    unsigned long long *win;
    uint64_t winEntries;
    uint32_t *counters;
    uint32_t *errs;
    uint32_t *tickets;
    uint32_t *epoch;
};

// Segment base of `node` from the kernel's argument block, read in place
// (the kernels' only argument starts at offset 0 of the argument segment):
// indexing the by-value argument at run time would copy the whole block to
// private memory.
__device__ __forceinline__ uint64_t export_seg_base(uint32_t node)
{
    typedef __attribute__((address_space(4))) const uint64_t KU64;
    typedef __attribute__((address_space(4))) const char KChar;
    const KChar *k = (KChar *)__builtin_amdgcn_kernarg_segment_ptr();
    return reinterpret_cast<KU64 *>(k + offsetof(ExportRowsParams, segBases))[node];
}

__device__ __forceinline__ bool export_row_target(const ExportRowsArgs &a, int64_t row, uint32_t &node,
                                                  uint32_t &segRow)
{
    if (row < 0) return false;
    const uint32_t r = static_cast<uint32_t>(row);  // the mapping is u32 math (kvc_common.h:81-89)
    node = kvx_node_of(r, a.stripeRows, a.nodeNum);
    if (a.fused ? node >= a.nodeNum : node != a.myNode) return false;
    segRow = kvx_seg_row_of(r, a.stripeRows, a.nodeNum);
    return true;
}

// Pass 1: the last entry per segment row (winner tags, as in the import);
// block 0 resets this node's counters and status words.
__global__ __launch_bounds__(256) void kvx_export_rows_prep(ExportRowsParams P)
{
    const ExportRowsArgs &a = P.a;
    const int32_t n = clamp_num_real(a.numReal, a.maxRows);
    const uint32_t n0 = a.fused ? 0u : a.myNode, n1 = a.fused ? a.nodeNum : a.myNode + 1u;
    if (blockIdx.x == 0) {
        for (uint32_t k = threadIdx.x; k < (n1 - n0) * a.statusWords; k += blockDim.x) {
            const uint32_t node = n0 + k / a.statusWords, b = k % a.statusWords;
            P.counters[node * 8u + b] = 0u;
            P.errs[node * 8u + b] = 0u;
            if (a.status != 0) store_status(a.status + node * 64ull + b * 8ull, 0ull);
        }
    }
    const KVX_G int64_t *idx = reinterpret_cast<const KVX_G int64_t *>(a.indicesHost);
    const unsigned long long tagHi = static_cast<unsigned long long>(*P.epoch) << 32;
    for (int32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        uint32_t node, segRow;
        if (!export_row_target(a, idx[i], node, segRow) || segRow >= a.perLayerSegRows) continue;
        const uint64_t w = (a.fused ? static_cast<uint64_t>(node) * a.perLayerSegRows : 0ull) + segRow;
        if (w < P.winEntries) win_max(P.win + w, tagHi | static_cast<unsigned long long>(i));
    }
}

// Pass 2: each wave takes kExportRowsPerWave entries (a decode step exports
// a few rows per layer: spread over many waves they move in one round trip),
// counts the owned ones per status word, records out-of-segment rows and
// copies its winners; the last workgroup advances the epoch and writes the
// status words.
constexpr int kExportRowsPerWave = 8;
__global__ __launch_bounds__(256) void kvx_export_rows_copy(ExportRowsParams P)
{
    __shared__ uint64_t sSrc[kWaves][64];
    __shared__ uint64_t sDst[kWaves][64];
    __shared__ int sLast;
    __shared__ uint32_t sEpoch;
    const ExportRowsArgs &a = P.a;
    const int wave = threadIdx.x / 64;
    const uint32_t lane = static_cast<uint32_t>(lane_id());
    const int32_t n = clamp_num_real(a.numReal, a.maxRows);
    const KVX_G int64_t *idx = reinterpret_cast<const KVX_G int64_t *>(a.indicesHost);
    const unsigned long long tagHi = static_cast<unsigned long long>(*P.epoch) << 32;
    const uint32_t cpr = a.rowBytes / 16u;
    const uint32_t words = a.statusWords;
    const uint32_t ppc = (a.maxRows + words - 1u) / words;  // entries per status word
    constexpr int32_t R = kExportRowsPerWave;
    for (int32_t base = (blockIdx.x * kWaves + wave) * R; base < n; base += gridDim.x * kWaves * R) {
        const int32_t i = base + static_cast<int32_t>(lane);
        bool copy = false;
        uint64_t src = 0, dst = 0;
        uint32_t node, segRow;
        if (static_cast<int32_t>(lane) < R && i < n && export_row_target(a, idx[i], node, segRow)) {
            const uint32_t key = node * 8u + static_cast<uint32_t>(i) / ppc;
            atomicAdd(&P.counters[key], 1u);
            if (segRow >= a.perLayerSegRows) {  // outside the segment's layer region: report, do not write
                atomicMax(&P.errs[key], ~static_cast<uint32_t>(i));
            } else {
                const uint64_t w = (a.fused ? static_cast<uint64_t>(node) * a.perLayerSegRows : 0ull) + segRow;
                copy = w >= P.winEntries || win_load(P.win + w) == (tagHi | static_cast<unsigned long long>(i));
                src = a.srcLayerBase + static_cast<uint64_t>(i) * a.rowBytes;
                dst = (a.fused ? export_seg_base(node) : a.segBase) +
                      (static_cast<uint64_t>(a.layerId) * a.perLayerSegRows + segRow) * a.rowBytes;
            }
        }
        const uint64_t cm = __ballot(copy);
        if (copy) {
            const uint32_t at = static_cast<uint32_t>(__popcll(cm & ((1ull << lane) - 1ull)));
            sSrc[wave][at] = src;
            sDst[wave][at] = dst;
        }
        wave_sync_lds();
        wave_copy_rows<true>(sSrc[wave], sDst[wave], static_cast<uint32_t>(__popcll(cm)), cpr);
        wave_sync_lds();
    }

    wait_stores();
    __syncthreads();
    if (threadIdx.x == 0) {
        const unsigned int ticket = atomicInc(&P.tickets[2], gridDim.x - 1u);
        sLast = (ticket == gridDim.x - 1u) ? 1 : 0;
    }
    __syncthreads();
    if (!sLast) return;
    if (threadIdx.x == 0) sEpoch = *P.epoch + 1u;
    __syncthreads();
    if (sEpoch == 0u) {
        for (uint64_t k = threadIdx.x; k < P.winEntries; k += blockDim.x) P.win[k] = 0ull;
    }
    if (threadIdx.x == 0) *P.epoch = sEpoch;
    __threadfence_system();
    const uint32_t n0 = a.fused ? 0u : a.myNode, n1 = a.fused ? a.nodeNum : a.myNode + 1u;
    for (uint32_t k = threadIdx.x; k < (n1 - n0) * words; k += blockDim.x) {
        const uint32_t node = n0 + k / words, b = k % words;
        const uint32_t q = __hip_atomic_load(&P.counters[node * 8u + b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const uint32_t e = __hip_atomic_load(&P.errs[node * 8u + b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        P.counters[node * 8u + b] = 0u;
        P.errs[node * 8u + b] = 0u;
        if (a.status == 0) continue;
        uint64_t word = 1ull << 32;
        if (static_cast<int64_t>(b) * ppc < n) {
            word |= (static_cast<uint64_t>(q) << 40) | error_word(e);
        }
        store_status(a.status + node * 64ull + b * 8ull, word);
    }
}

// Short exports (max_rows <= kExportSmallMax, the rows a decode step
// appends): both passes in one launch.  Rows share a destination iff they lie
// in one stripe, and the last entry wins: each workgroup takes a few entries
// and looks for a later entry in the same stripe among all of them, counts its
// own owned and out-of-region entries, and copies its winners with all lanes;
// the last workgroup (ticket) stores the status words and leaves the call's
// counters zeroed.  The bound is latency: three dependent reads, a row's way
// over the link and back.  Entries go to many workgroups (4 each up to 1024:
// 64 rows, one layer: 9.7 us from 2 workgroups ending in system-scope fences,
// 6.8 now).
constexpr uint32_t kExportSmallMax = 4096;
constexpr uint32_t kExportSpanRows = 1024;  // up to here 4 entries a workgroup, else 16
constexpr uint32_t kExportMaxSpan = 16;

__global__ __launch_bounds__(256) void kvx_export_rows_small(ExportRowsParams P)
{
    __shared__ uint64_t sSrc[kExportMaxSpan], sDst[kExportMaxSpan];
    __shared__ uint64_t sKey[kExportMaxSpan];  // stripe of an own entry in the winner rule, else ~0
    __shared__ uint32_t sLose, sN;             // sLose bit e: own entry e is not a winner
    __shared__ int sLast;
    const ExportRowsArgs &a = P.a;
    const uint32_t tid = threadIdx.x;
    const int32_t n = clamp_num_real(a.numReal, a.maxRows);  // <= kExportSmallMax (host)
    const KVX_G int64_t *idx = reinterpret_cast<const KVX_G int64_t *>(a.indicesHost);
    const uint32_t cpr = a.rowBytes / 16u;
    const uint32_t words = a.statusWords;
    const uint32_t ppc = (a.maxRows + words - 1u) / words;  // entries per status word
    const uint32_t n0 = a.fused ? 0u : a.myNode, n1 = a.fused ? a.nodeNum : a.myNode + 1u;
    const int32_t span = a.maxRows <= kExportSpanRows ? 4 : static_cast<int32_t>(kExportMaxSpan);
    const int32_t lo = static_cast<int32_t>(blockIdx.x) * span;
    auto stripe = [&](int64_t row) {  // (the mapping is u32 math; a stripe of 0 rows is the identity)
        const uint32_t r = static_cast<uint32_t>(row);
        return static_cast<uint64_t>(a.stripeRows == 0u ? r : r / a.stripeRows);
    };
    if (blockIdx.x == 0 && a.status != 0) {  // the call's status words read 0 until its rows have landed
        for (uint32_t k = tid; k < (n1 - n0) * words; k += blockDim.x) {
            clear_status(a.status + (n0 + k / words) * 64ull + (k % words) * 8ull);
        }
    }
    if (tid == 0) sLose = sN = 0u;
    uint32_t node = 0, segRow = 0;
    bool owned = false, rule = false;
    if (static_cast<int32_t>(tid) < span) {
        const int32_t i = lo + static_cast<int32_t>(tid);
        const int64_t row = i < n ? idx[i] : -1;
        owned = export_row_target(a, row, node, segRow);
        rule = owned && segRow < a.perLayerSegRows;
        sKey[tid] = rule ? stripe(row) : ~0ull;
    }
    __syncthreads();
    uint32_t lose = 0u;
    for (int32_t i0 = lo + static_cast<int32_t>(tid); i0 < n; i0 += 4 * 256) {
        int64_t row[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) row[j] = idx[min(i0 + j * 256, n - 1)];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int32_t i = i0 + j * 256;
            if (i >= n || row[j] < 0) continue;
            const uint64_t q = stripe(row[j]);
            for (int32_t e = 0; e < span && lo + e < i; ++e) lose |= sKey[e] == q ? 1u << e : 0u;
        }
    }
    if (lose != 0u) atomicOr(&sLose, lose);
    __syncthreads();
    if (owned) {
        const uint32_t i = static_cast<uint32_t>(lo) + tid, key = node * 8u + i / ppc;
        atomicAdd(&P.counters[key], 1u);
        if (!rule) {
            atomicMax(&P.errs[key], ~i);  // the lowest failing entry
        } else if (((sLose >> tid) & 1u) == 0u) {
            const uint32_t at = atomicAdd(&sN, 1u);
            sSrc[at] = a.srcLayerBase + static_cast<uint64_t>(i) * a.rowBytes;
            sDst[at] = (a.fused ? export_seg_base(node) : a.segBase) +
                       (static_cast<uint64_t>(a.layerId) * a.perLayerSegRows + segRow) * a.rowBytes;
        }
    }
    __syncthreads();
    const uint32_t chunks = sN * cpr;
    for (uint32_t c0 = tid; c0 < chunks; c0 += 256u * 4u) {
        u32x4 v[4];
        uint64_t d[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t c = c0 + static_cast<uint32_t>(j) * 256u;
            d[j] = 0;
            if (c < chunks) {
                const uint32_t r = c / cpr, o = (c - r * cpr) * 16u;
                v[j] = __builtin_nontemporal_load(reinterpret_cast<const GVec *>(sSrc[r] + o));
                d[j] = sDst[r] + o;
            }
        }
        wait_loads<4>(v);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (d[j] != 0) store_through(d[j], v[j]);
        }
    }
    wait_stores();
    __syncthreads();
    if (tid == 0) {
        const unsigned int ticket = atomicInc(&P.tickets[4], gridDim.x - 1u);
        sLast = (ticket == gridDim.x - 1u) ? 1 : 0;
    }
    __syncthreads();
    if (!sLast) return;
    for (uint32_t k = tid; k < (n1 - n0) * 8u; k += blockDim.x) {
        const uint32_t nd = n0 + k / 8u, b = k % 8u;
        const uint32_t q = __hip_atomic_load(&P.counters[nd * 8u + b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const uint32_t e = __hip_atomic_load(&P.errs[nd * 8u + b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (q != 0u) __hip_atomic_store(&P.counters[nd * 8u + b], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (e != 0u) __hip_atomic_store(&P.errs[nd * 8u + b], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (a.status == 0 || b >= words) continue;
        uint64_t word = 1ull << 32;
        if (static_cast<int64_t>(b) * ppc < n) word |= (static_cast<uint64_t>(q) << 40) | error_word(e);
        store_status(a.status + nd * 64ull + b * 8ull, word);
    }
}

// Plain streaming copy, 16 B per lane, kUnroll chunks in flight per lane.
__global__ __launch_bounds__(256) void kvx_stream_copy(u32x4 *dst, const u32x4 *src, uint64_t n16)
{
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
    uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    for (; i + (kUnroll - 1) * stride < n16; i += kUnroll * stride) {
        u32x4 v[kUnroll];
#pragma unroll
        for (int j = 0; j < kUnroll; ++j) v[j] = __builtin_nontemporal_load(src + i + j * stride);
#pragma unroll
        for (int j = 0; j < kUnroll; ++j) __builtin_nontemporal_store(v[j], dst + i + j * stride);
    }
    for (; i < n16; i += stride) __builtin_nontemporal_store(__builtin_nontemporal_load(src + i), dst + i);
}

}  // namespace

hipError_t launch_stream_copy(uint64_t dst, uint64_t src, uint64_t bytes, hipStream_t stream)
{
    const uint64_t n16 = bytes / 16;
    uint64_t blocks = (n16 + 255) / 256;
    if (blocks < 1) blocks = 1;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(kvx_stream_copy, dim3(static_cast<uint32_t>(blocks)), dim3(256), 0, stream,
                       reinterpret_cast<u32x4 *>(dst), reinterpret_cast<const u32x4 *>(src), n16);
    return hipGetLastError();
}

hipError_t launch_gather(const GatherPlan &plan, const RowScratch &scr, uint64_t overflowSlot, hipStream_t stream)
{
    GatherParams P{};
    P.l.a = plan.a;
    P.l.overflowSlot = overflowSlot;
    if (plan.fused) {
        for (uint32_t s = 0; s < plan.a.nodeNum && s < 64u; ++s) P.x.segBases[s] = plan.segBases[s];
    }
    P.x.win = scr.win;
    P.x.winEntries = scr.winEntries;
    P.x.chunkNext = scr.chunkNext;
    P.x.counters = scr.counters;
    P.x.errs = scr.errs;
    P.x.tickets = scr.tickets;
    P.x.fused = plan.fused;
    P.x.epoch = scr.epoch;
    P.x.spanRows = plan.spanRows;
    P.x.statusWords = plan.statusWords;
    const uint64_t positions = static_cast<uint64_t>(plan.a.maxNumReqs) * plan.a.topK;
    // the positions that can share a destination row
    const uint64_t group = plan.spanRows == 0 ? positions : plan.a.topK;
    const bool striped = plan.a.stripeRows > 1u && positions > kOneMaxStriped;
    if (positions != 0 && group <= kOneMaxGroup && positions < (1ull << 31) && !striped) {
        // (spans of the largest batch; the kernel takes those of the real one)
        const uint32_t count = gather_spans(static_cast<uint32_t>(positions), static_cast<uint32_t>(group)).count;
        hipLaunchKernelGGL(kvx_gather_one, dim3(count < kOneMaxBlocks ? count : kOneMaxBlocks), dim3(kOneThreads), 0, stream, P);
        return hipGetLastError();
    }
    uint64_t prepBlocks = (positions + 255ull) / 256ull;
    if (prepBlocks < 1) prepBlocks = 1;
    if (prepBlocks > 2048) prepBlocks = 2048;
    hipLaunchKernelGGL(kvx_gather_prep, dim3(static_cast<uint32_t>(prepBlocks)), dim3(256), 0, stream, P);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    uint64_t spanBlocks = (positions + kSpan - 1ull) / kSpan;
    if (spanBlocks > kSpanBlocks) spanBlocks = kSpanBlocks;
    hipLaunchKernelGGL(kvx_gather_span, dim3(static_cast<uint32_t>(spanBlocks)), dim3(256), 0, stream, P);
    return hipGetLastError();
}

hipError_t launch_export(const KvcScatterAllArgs &a, const RowScratch &scr, uint64_t overflowSlot,
                         hipStream_t stream)
{
    ExportParams P{};
    P.l.a = a;
    P.l.overflowSlot = overflowSlot;
    P.x.tickets = scr.tickets;
    const ExportGeometry geo = export_geometry(a);
    P.x.q0 = geo.q0;
    P.x.nStripes = geo.nStripes;
    P.x.ownedRows = geo.ownedRows;
    P.x.S = geo.S;
    P.x.N = geo.N;
    const uint64_t items = P.x.nStripes * a.layerNum;
    uint64_t blocks = (items + 64ull * kWaves - 1ull) / (64ull * kWaves);
    if (blocks < 1) blocks = 1;
    if (blocks > kExportBlocks) blocks = kExportBlocks;
    hipLaunchKernelGGL(kvx_export_alllayer, dim3(static_cast<uint32_t>(blocks)), dim3(256), 0, stream, P);
    return hipGetLastError();
}

hipError_t launch_export_rows(const ExportRowsArgs &a, const uint64_t *segBases, const RowScratch &scr,
                              hipStream_t stream)
{
    ExportRowsParams P{};
    P.a = a;
    if (a.fused) {
        for (uint32_t s = 0; s < a.nodeNum && s < 64u; ++s) P.segBases[s] = segBases[s];
    }
    P.win = scr.win;
    P.winEntries = scr.winEntries;
    P.counters = scr.counters;
    P.errs = scr.errs;
    P.tickets = scr.tickets;
    P.epoch = scr.epoch;
    if (a.maxRows <= kExportSmallMax) {
        const uint32_t span = a.maxRows <= kExportSpanRows ? 4u : kExportMaxSpan;
        const uint32_t blocks = (a.maxRows + span - 1u) / span;
        hipLaunchKernelGGL(kvx_export_rows_small, dim3(blocks), dim3(256), 0, stream, P);
        return hipGetLastError();
    }
    uint64_t prep = (static_cast<uint64_t>(a.maxRows) + 255ull) / 256ull;
    prep = prep < 1 ? 1 : (prep > 1024 ? 1024 : prep);
    hipLaunchKernelGGL(kvx_export_rows_prep, dim3(static_cast<uint32_t>(prep)), dim3(256), 0, stream, P);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    uint64_t copy = (static_cast<uint64_t>(a.maxRows) + kExportRowsPerWave * kWaves - 1ull) / (kExportRowsPerWave * kWaves);
    copy = copy < 1 ? 1 : (copy > 256 ? 256 : copy);
    hipLaunchKernelGGL(kvx_export_rows_copy, dim3(static_cast<uint32_t>(copy)), dim3(256), 0, stream, P);
    return hipGetLastError();
}

}  // namespace kvx

// SIEVE (ring CLOCK) miss detector and hash-table build for gfx950.
//
// Semantics follow kvops/kernel/hisp_sieve_update.cpp:17-176 and
// hisp_sieve_ht_init.cpp:14-60 of the reference; the state format is that of
// hisp_kernel_common.h (uint16 entries = slot+1, Knuth hash, linear probing,
// backward-shift deletion, visited bitmap 8 slots per byte).
//
// Layout on the device: one workgroup per batch row.  The request's state row
// (tokens padded*4 B, hash table htSize*2 B, visited visStrideB B) is staged
// in LDS when it fits the per-workgroup LDS limit (160 KiB on gfx950) and
// written back at the end; otherwise the kernel works on the HBM-resident row
// in place.  Within the row, positions are processed in order -- the exact
// sequential recurrence of the reference -- by one wave whose probes, sweeps
// and shifts take 64 cells or slots per step (LDS-staged), or by one lane
// (HBM-resident).
#include "kvx_internal.h"
#include "sieve_common.h"

namespace kvx {
namespace {

using namespace sieve;

template <bool kLds>
__global__ __launch_bounds__(256) void kvx_sieve_update(KvxLaunch<HispSieveUpdateArgs> L)
{
    extern __shared__ __align__(16) uint8_t smem[];
    __shared__ int32_t s_dirty;
    const HispSieveUpdateArgs &a = L.a;
    const int32_t topK = static_cast<int32_t>(a.topK);
    const int32_t dbs = static_cast<int32_t>(a.deviceBufferSize);
    const int32_t padded = static_cast<int32_t>(a.paddedBufferSize);
    const int32_t visStrideB = static_cast<int32_t>(a.visitedStrideB);
    const int32_t maxNumReqs = static_cast<int32_t>(a.maxNumReqs);
    const int32_t htSize = static_cast<int32_t>(a.htSize);
    const int32_t poolSize = static_cast<int32_t>(a.poolSize);
    const int32_t bid = blockIdx.x;
    if (bid >= maxNumReqs) return;

    int32_t numReal = *reinterpret_cast<const int32_t *>(a.numReal);
    if (numReal > maxNumReqs) numReal = maxNumReqs;  // hisp_sieve_update.cpp:31-34

    int32_t *rs = reinterpret_cast<int32_t *>(a.topKDeviceSlots) + static_cast<int64_t>(bid) * topK;
    int8_t *rm = reinterpret_cast<int8_t *>(a.isMiss) + static_cast<int64_t>(bid) * topK;
    if (bid >= numReal) {  // padding rows (:72-78)
        write_dummy_row(rs, rm, topK);
        return;
    }
    const int64_t reqIdx = reinterpret_cast<const int64_t *>(a.reqPoolIndices)[bid];
    if (reqIdx < 0 || reqIdx >= poolSize) {  // (:80-88)
        write_dummy_row(rs, rm, topK);
        return;
    }
    const int32_t seqLen = reinterpret_cast<const int32_t *>(a.seqLens)[bid];
    const int32_t prefill = reinterpret_cast<const int32_t *>(a.prefillLens)[reqIdx];
    const int32_t *rt = reinterpret_cast<const int32_t *>(a.topkIndices) + static_cast<int64_t>(bid) * topK;
    int32_t *gTok = reinterpret_cast<int32_t *>(a.deviceBufferTokens) + reqIdx * padded;
    uint8_t *gVis = reinterpret_cast<uint8_t *>(a.deviceBufferVisited) + reqIdx * visStrideB;
    uint16_t *gHt = reinterpret_cast<uint16_t *>(a.deviceBufferHt) + reqIdx * htSize;
    int32_t *gHand = reinterpret_cast<int32_t *>(a.sieveHand) + reqIdx * kHandStride;

    int32_t *tok = gTok;
    uint8_t *vis = gVis;
    uint16_t *ht = gHt;
    if constexpr (kLds) {
        tok = reinterpret_cast<int32_t *>(smem);
        ht = reinterpret_cast<uint16_t *>(smem + static_cast<size_t>(padded) * 4);
        vis = smem + static_cast<size_t>(padded) * 4 + static_cast<size_t>(htSize) * 2;
        block_copy16(tok, gTok, static_cast<uint32_t>(padded) * 4u);
        block_copy16(ht, gHt, static_cast<uint32_t>(htSize) * 2u);
        block_copy16(vis, gVis, static_cast<uint32_t>(visStrideB));
        __syncthreads();
    }

    if (kLds && htSize > kSmallTable) {
        if (threadIdx.x < 64) {  // one wave: 64 cells/slots per probe, sweep and shift step
            int32_t hand = *gHand;
            if (hand < 0 || hand >= dbs) hand = 0;  // (:108-111)
            Guard g;
            const bool dirty =
                sieve_row_wave(rt, rs, rm, topK, seqLen, prefill, dbs, padded, htSize - 1, tok, vis, ht, hand, g);
            if (threadIdx.x == 0) {
                *gHand = hand;
                s_dirty = dirty ? 1 : 0;
                report_overflow(L.overflowSlot, g.code);
            }
        }
    } else if (threadIdx.x == 0) {
        int32_t hand = *gHand;
        if (hand < 0 || hand >= dbs) hand = 0;  // (:108-111)
        Guard g;
        const bool dirty =
            sieve_row_sequential(rt, rs, rm, topK, seqLen, prefill, dbs, padded, htSize - 1, tok, vis, ht, hand, g);
        *gHand = hand;
        s_dirty = dirty ? 1 : 0;
        report_overflow(L.overflowSlot, g.code);
    }
    if constexpr (kLds) {
        __syncthreads();
        block_copy16(gVis, vis, static_cast<uint32_t>(visStrideB));
        if (s_dirty) {  // (:165-172)
            block_copy16(gTok, tok, static_cast<uint32_t>(padded) * 4u);
            block_copy16(gHt, ht, static_cast<uint32_t>(htSize) * 2u);
        }
    }
}

// hisp_sieve_ht_init.cpp:14-60: block b -> (layer b/numReqs, pool row
// reqStart + b%numReqs); clear the row's table, insert tokens[s] >= 0 for
// s < dbs in increasing s, comparing through the HBM tokens row.
template <bool kLds>
__global__ __launch_bounds__(256) void kvx_sieve_ht_init(KvxLaunch<HispSieveHtInitArgs> L)
{
    extern __shared__ __align__(16) uint8_t smem[];
    const HispSieveHtInitArgs &a = L.a;
    const int32_t numReqs = static_cast<int32_t>(a.numReqs);
    const int32_t layerNum = static_cast<int32_t>(a.layerNum);
    const int32_t poolSize = static_cast<int32_t>(a.poolSize);
    const int32_t dbs = static_cast<int32_t>(a.deviceBufferSize);
    const int32_t padded = static_cast<int32_t>(a.paddedBufferSize);
    const int32_t htSize = static_cast<int32_t>(a.htSize);
    const int32_t b = blockIdx.x;
    if (b >= layerNum * numReqs) return;
    const int32_t layer = b / numReqs;
    const int64_t reqIdx = static_cast<int64_t>(a.reqStart) + b % numReqs;
    if (reqIdx < 0 || reqIdx >= poolSize) return;

    const int32_t *tok = reinterpret_cast<const int32_t *>(a.deviceBufferTokens) +
                         (static_cast<int64_t>(layer) * poolSize + reqIdx) * padded;
    uint16_t *gHt = reinterpret_cast<uint16_t *>(a.deviceBufferHt) +
                    (static_cast<int64_t>(layer) * poolSize + reqIdx) * htSize;
    uint16_t *ht = kLds ? reinterpret_cast<uint16_t *>(smem) : gHt;
    uint4 *ht16 = reinterpret_cast<uint4 *>(ht);
    for (int32_t i = threadIdx.x; i < htSize / 8; i += blockDim.x) ht16[i] = make_uint4(0, 0, 0, 0);
    __syncthreads();
    if (threadIdx.x == 0) {
        Guard g;
        for (int32_t s = 0; s < dbs && g.code == 0; ++s) {
            const int32_t t = tok[s];
            if (t >= 0) ht_insert(ht, tok, padded, t, s, htSize - 1, g);
        }
        report_overflow(L.overflowSlot, g.code);
    }
    if constexpr (kLds) {
        __syncthreads();
        block_copy16(gHt, ht, static_cast<uint32_t>(htSize) * 2u);
    }
}

// Parallel form of the same build.  Sequential first-come-first-served
// inserts leave every key in the first cell from its home that no earlier key
// took, so the table is the stable matching in which keys prefer cells nearer
// their home and every cell prefers the smaller slot (deferred acceptance,
// Gale and Shapley 1962).  It does not depend on the order of the proposals:
// every lane proposes its slots to their cells with an atomic min, and carries
// the slot that a cell gives up (its own or the one it displaced) to the next
// cell.  The proposals number the keys plus the sum of their distances from
// home, whatever the order.
//
// A later slot with a token already inserted meets the earlier entry on its
// probe path and is skipped (hisp_kernel_common.h:97-112).  With such slots
// inserted as keys of their own, each lies behind its token's first slot (same
// home, which that slot left no nearer cell free for), so a walk from the home
// finds every one of them; the table is then built again without them.
//
// A table of up to kInitLdsCells cells stands in LDS as 32-bit cells (the
// slot, all ones = empty): one returning atomic per proposal.  The bound is
// latency: a lane's chain of LDS round trips, four slots each at 4096 slots.
// The form it replaced (per-home counts, two scans of a contiguous run of
// cells per lane, a lane per cluster) read the table at strides that put half
// a wave on one bank: an admission of 61 such tables took 157 us, now 67.
constexpr int32_t kInitThreads = 1024;
constexpr int32_t kInitLdsCells = 32768;
constexpr int32_t kInitSmallThreads = 256;  // rows of up to kInitSmallSlots slots
constexpr int32_t kInitSmallSlots = 1024;
constexpr int kInitUnroll = 4;              // slots whose tokens a lane loads together

typedef __attribute__((address_space(1))) const int32_t GTok;
typedef __attribute__((address_space(1))) uint16_t GCell;
typedef uint32_t Chunk __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(1))) Chunk GChunk;

// The tokens of a row: read from the state, or, at admission, slot s holds
// token s for s < n0 (no token is held twice then).
template <bool kIdentity>
struct RowTokens {
    GTok *tok;
    int32_t n0;
    __device__ __forceinline__ int32_t operator()(int32_t s) const
    {
        if constexpr (kIdentity) return s < n0 ? s : -1;
        else return tok[s];
    }
};

template <bool kIdentity>
__device__ __forceinline__ void init_table_lds(uint8_t *smem, const RowTokens<kIdentity> token, GCell *gHt, int32_t dbs,
                                               int32_t H)
{
    constexpr uint32_t kEmpty = 0xFFFFFFFFu;
    const int32_t mask = H - 1, tid = threadIdx.x, nt = blockDim.x;
    uint32_t *cell = reinterpret_cast<uint32_t *>(smem);
    uint32_t *drop = cell + H;  // slots whose token an earlier slot holds
    const int32_t dropWords = (dbs + 31) / 32;
    if constexpr (!kIdentity) {
        for (int32_t i = tid; i < dropWords; i += nt) drop[i] = 0u;
    }
    for (int attempt = 0; attempt < 2; ++attempt) {
        for (int32_t i = tid; i < H / 4; i += nt) {
            reinterpret_cast<uint4 *>(cell)[i] = make_uint4(kEmpty, kEmpty, kEmpty, kEmpty);
        }
        __syncthreads();
        for (int32_t s0 = tid; s0 < dbs; s0 += kInitUnroll * nt) {
            int32_t t[kInitUnroll];
#pragma unroll
            for (int q = 0; q < kInitUnroll; ++q) t[q] = s0 + q * nt < dbs ? token(s0 + q * nt) : -1;
#pragma unroll
            for (int q = 0; q < kInitUnroll; ++q) {
                const int32_t s = s0 + q * nt;
                if (t[q] < 0) continue;
                if (!kIdentity && attempt != 0 && ((drop[s >> 5] >> (s & 31)) & 1u)) continue;
                uint32_t v = static_cast<uint32_t>(s);
                for (uint32_t c = ht_hash(t[q]) & static_cast<uint32_t>(mask);;) {
                    const uint32_t old = atomicMin(cell + c, v);
                    if (old == kEmpty) break;  // fewer keys than cells: every chain ends
                    v = old > v ? old : v;
                    c = (c + 1u) & static_cast<uint32_t>(mask);
                }
            }
        }
        __syncthreads();
        if constexpr (kIdentity) {
            break;
        } else {
            if (attempt != 0) break;
            int dup = 0;
            for (int32_t s0 = tid; s0 < dbs; s0 += kInitUnroll * nt) {
                int32_t t[kInitUnroll];
#pragma unroll
                for (int q = 0; q < kInitUnroll; ++q) t[q] = s0 + q * nt < dbs ? token(s0 + q * nt) : -1;
#pragma unroll
                for (int q = 0; q < kInitUnroll; ++q) {
                    const int32_t s = s0 + q * nt;
                    if (t[q] < 0) continue;
                    uint32_t c = ht_hash(t[q]) & static_cast<uint32_t>(mask);
                    for (uint32_t e = cell[c]; e != static_cast<uint32_t>(s) && e != kEmpty;) {
                        if (token(static_cast<int32_t>(e)) == t[q]) {
                            dup = 1;
                            atomicOr(drop + (s >> 5), 1u << (s & 31));
                            break;
                        }
                        c = (c + 1u) & static_cast<uint32_t>(mask);
                        e = cell[c];
                    }
                }
            }
            if (__syncthreads_or(dup) == 0) break;
        }
    }
    // an entry is slot + 1, 0 = empty: all ones plus one
    GChunk *out = reinterpret_cast<GChunk *>(gHt);
    for (int32_t i = tid; i < H / 8; i += nt) {
        const uint4 lo = reinterpret_cast<const uint4 *>(cell)[2 * i], hi = reinterpret_cast<const uint4 *>(cell)[2 * i + 1];
        auto two = [](uint32_t x, uint32_t y) { return ((x + 1u) & 0xFFFFu) | ((y + 1u) << 16); };
        out[i] = Chunk{two(lo.x, lo.y), two(lo.z, lo.w), two(hi.x, hi.y), two(hi.z, hi.w)};
    }
}

// The same build for tables beyond kInitLdsCells (65536 cells and more).  A
// hash has 16 bits, so every home lies in the first 65536 cells: those stand
// in LDS as the table's own 16-bit entries (compare and swap on the
// containing word), and the keys that run past them, in larger tables, take
// the cells from 65536 on in slot order (no key is homed there, so each cell
// takes the smallest slot waiting; they never wrap: a row holds fewer than
// 65536 keys).
//
// The slots go in increasing passes, each half of the cells left free, so
// that the proposals of a pass stay few however full the table gets; a cell
// taken in an earlier pass holds a smaller slot and is skipped by a bitmap
// (occ, with a bit per full word in `full`).  A pass is at least one slot per
// lane while the chains are short (homes spread evenly, as at admission), else
// at least kInitSmallPass: with the last 1006 of 65518 random tokens on 1024
// free cells in one pass, chains passed the limit below and the row was swept
// after all (four tables 6705 us, 1142 so).
//
// Homes packed into few cells make the proposals many (the square of the keys
// on one home): the row takes the one-wave sweep below, whose time does not
// depend on the distances.  A sample of the slots (every fourth, over 4096) is
// counted per 256 homes beforehand; more than twice the even share and 32 in
// one of them sends the row there (random tokens: ten and more standard
// deviations), and so does a chain of more than kInitMaxHops proposals.  (1024
// keys on the last 64 homes of a 65536-cell table: 577 us swept, 2799 when
// only the chains told.)
//
// A token held twice, or one beyond the bitmap that finds those, sends the
// row to the one-lane inserts.  Rows of more than 65535 slots are swept (two
// of 70000 random tokens 7 ms; minutes with one lane on the table in HBM).
//
// Against the sweep alone: four tables of 65518 slots, admission pattern, 4541
// -> 175 us with the calls around the build; 64 tables of 16000 random tokens
// 1379 -> 21 us; four of 60000 random tokens 4221 -> 368 us.
constexpr int32_t kWaveInitTokenBits = 1 << 20;
constexpr int32_t kFreeCap = 4;  // free cells counted between neighbouring first-free cells
constexpr int32_t kInitHomes = 65536;
constexpr int32_t kInitMaxHops = 512;
constexpr int32_t kInitLongChain = 16;                    // proposals past which later passes get smaller
constexpr int32_t kInitSmallPass = 64;                    // their least slots
constexpr int32_t kInitBuckets = 256;                     // sampled counts, of 256 homes each
constexpr int32_t kInitWords = kInitHomes / 64;           // words of the occ and spill bitmaps
constexpr int32_t kInitTailEnd = 2 * kInitHomes;          // no cell at or past it is ever taken
constexpr int32_t kInitHelpers = 3;                       // workgroups per row beside the one that builds

struct InitLargeLds {
    uint32_t cells[kInitHomes / 2];
    uint64_t occ[kInitWords], spill[kInitWords];
    uint64_t full[kInitWords / 64];
    uint32_t part[kInitThreads / 64 + 1];
    uint32_t bucket[kInitBuckets];
    int32_t longChain, stop;
};
static_assert(kWaveInitTokenBits / 8 <= sizeof(InitLargeLds::cells), "the token bitmap takes the cells' place");
static_assert(kInitWords == kInitThreads, "one bitmap word per lane");

__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Entry v proposes to cell c: 0 when the cell was empty, else the entry that
// goes on to the next cell.
__device__ __forceinline__ uint32_t propose16(uint32_t *cells, uint32_t c, uint32_t v)
{
    uint32_t *w = cells + (c >> 1);
    const uint32_t sh = (c & 1u) * 16u;
    uint32_t old = *w;
    for (;;) {
        const uint32_t cur = (old >> sh) & 0xFFFFu;
        if (cur != 0u && cur < v) return v;
        const uint32_t prev = atomicCAS(w, old, (old & ~(0xFFFFu << sh)) | (v << sh));
        if (prev == old) return cur;
        old = prev;
    }
}

// One wave inserts 64 slots at a time over a three-level bitmap of used
// cells: each key's first free cell at or after its home in the table before
// the batch, then the free cells in increasing order, each taken by the
// earliest key of the batch whose first free cell is at or before it -- linear
// probing's cells in slot order.  A batch whose probe wraps past the table's
// end, or that has fewer free cells than keys at or after its last first-free
// cell (its sweep could wrap), inserts its keys one by one.  The table is
// zeroed before.
template <bool kIdentity>
__device__ void init_table_sweep(uint8_t *smem, const RowTokens<kIdentity> token, GCell *gHt, int32_t dbs, int32_t H,
                                 uint64_t overflowSlot)
{
    const int32_t mask = H - 1;
    const int32_t lane = static_cast<int32_t>(__lane_id());
    // ---- used cells: word w bit i = cell 64w+i; full1 bit w = word w full;
    // full2 bit q = full1 word q full (bits past the last full1 word set)
    const int32_t nW = H >> 6, nS = nW >> 6, nT = (nS + 63) >> 6;
    uint64_t *used = reinterpret_cast<uint64_t *>(smem);
    uint64_t *full1 = used + nW;
    uint64_t *full2 = full1 + nS;
    for (int32_t i = lane; i < nW + nS; i += 64) used[i] = 0ull;
    for (int32_t i = lane; i < nT; i += 64) {
        const int32_t left = nS - i * 64;  // level-1 words covered by this word
        full2[i] = left >= 64 ? 0ull : ~((1ull << left) - 1ull);
    }
    wave_lds_sync();
    // first free cell in [x, H), -1 if none
    auto first_free = [&](int32_t x) -> int32_t {
        if (x >= H) return -1;
        int32_t w = x >> 6;
        const uint64_t u = used[w] | ((1ull << (x & 63)) - 1ull);
        if (u != ~0ull) return (w << 6) + __builtin_ctzll(~u);
        const int32_t w1 = w + 1;
        if (w1 >= nW) return -1;
        int32_t s1 = w1 >> 6;
        uint64_t f = full1[s1] | ((1ull << (w1 & 63)) - 1ull);
        if (f == ~0ull) {
            const int32_t s2 = s1 + 1;
            if (s2 >= nS) return -1;
            int32_t q = s2 >> 6;
            uint64_t g2 = full2[q] | ((1ull << (s2 & 63)) - 1ull);
            while (g2 == ~0ull) {
                if (++q >= nT) return -1;
                g2 = full2[q];
            }
            s1 = (q << 6) + __builtin_ctzll(~g2);
            f = full1[s1];
        }
        w = (s1 << 6) + __builtin_ctzll(~f);
        return (w << 6) + __builtin_ctzll(~used[w]);
    };
    // word w now holds bits u (written by lane 0); the levels above follow
    auto put_word = [&](int32_t w, uint64_t u) {
        if (lane == 0) {
            used[w] = u;
            if (u == ~0ull) {
                const int32_t s1 = w >> 6;
                const uint64_t f = full1[s1] | (1ull << (w & 63));
                full1[s1] = f;
                if (f == ~0ull) full2[s1 >> 6] |= 1ull << (s1 & 63);
            }
        }
        wave_lds_sync();
    };

    Guard g;
    const int32_t nb = (dbs + 63) >> 6;
    int32_t tNext = lane < dbs ? token(lane) : -1;
    for (int32_t bi = 0; bi < nb && g.code == 0; ++bi) {
        const int32_t s = (bi << 6) + lane;
        const int32_t t = tNext;
        tNext = s + 64 < dbs ? token(s + 64) : -1;  // the next batch's tokens, in flight meanwhile
        // (an entry is slot + 1 in 16 bits: slot 65535 writes an empty cell)
        const bool valid = s < dbs && t >= 0 && (s & 0xFFFF) != 0xFFFF;
        const uint64_t keys = __ballot(valid);
        if (keys == 0ull) continue;
        const int32_t h = valid ? static_cast<int32_t>(ht_hash(t)) & mask : 0;
        const int32_t tgt = valid ? first_free(h) : -1;
        const int32_t n = __popcll(keys);
        bool oneByOne = __ballot(valid && tgt < 0) != 0ull;
        // the keys in order of first-free cell (ties in slot order): rank by
        // comparing with every key, then each lane's cell and lane index move
        // to the lane of its rank (keys without a token rank last)
        int32_t rank = 0;
        if (!oneByOne) {
            for (uint64_t m = keys; m != 0ull; m &= m - 1ull) {
                const int32_t j = __builtin_ctzll(m);
                const int32_t tj = __builtin_amdgcn_readlane(tgt, j);
                rank += (tj < tgt || (tj == tgt && j < lane)) ? 1 : 0;
            }
            if (!valid) rank = n + __popcll(~keys & ((1ull << lane) - 1ull));
        }
        const int32_t sortedTgt = __builtin_amdgcn_ds_permute(rank << 2, tgt);
        const int32_t sortedLane = __builtin_amdgcn_ds_permute(rank << 2, lane);
        if (!oneByOne) {
            // free cells at or after the last first-free cell, counted up to the keys
            const int32_t tmax = __builtin_amdgcn_readlane(sortedTgt, n - 1);
            int32_t w = tmax >> 6;
            int32_t room = __popcll(~(used[w] | ((1ull << (tmax & 63)) - 1ull)));
            while (room < n) {
                const int32_t c = __builtin_amdgcn_readfirstlane(first_free((w + 1) << 6));
                if (c < 0) break;
                w = c >> 6;
                room += __popcll(~used[w]);
            }
            oneByOne = room < n;
        }
        if (oneByOne) {
            for (uint64_t m = keys; m != 0ull; m &= m - 1ull) {
                const int32_t j = __builtin_ctzll(m);
                const int32_t hj = __builtin_amdgcn_readlane(h, j);
                int32_t c = __builtin_amdgcn_readfirstlane(first_free(hj));
                if (c < 0) c = __builtin_amdgcn_readfirstlane(first_free(0));  // the probe wraps
                if (c < 0) {
                    g.code = kOverflowProbe;
                    break;
                }
                if (lane == j) gHt[c] = static_cast<uint16_t>(s + 1);
                put_word(c >> 6, used[c >> 6] | (1ull << (c & 63)));
            }
            continue;
        }
        // ---- keys that land on their own first-free cell, all at once.  In
        // rank order, key k's backlog b_k = max(0, b_{k-1} + 1 - D_k), D_k =
        // free cells in [t_{k-1}, t_k): the keys of earlier cells still
        // waiting when the sweep reaches t_k.  b_k = 0: key k takes t_k (the
        // earliest slot among keys of that cell).  D is counted up to
        // kFreeCap, which can only overstate b: such keys take the sweep.
        const bool rv = lane < n;
        const int32_t tk = sortedTgt;
        const int32_t tprev = __shfl_up(tk, 1);
        int32_t D = 0;
        if (rv && lane > 0 && tk > tprev) {
            D = 1;  // t_{k-1} itself
            for (int32_t x = tprev; D < kFreeCap;) {
                x = first_free(x + 1);
                if (x < 0 || x >= tk) break;
                ++D;
            }
        }
        // x -> max(P, x + Q) composed over ranks 0..k; rank 0 starts from b = 0
        int32_t P = 0, Q = lane == 0 ? -(1 << 24) : 1 - D;
        for (int32_t o = 1; o < 64; o <<= 1) {
            const int32_t Pp = __shfl_up(P, o), Qp = __shfl_up(Q, o);
            if (lane >= o) {
                P = max(P, Pp + Q);
                Q = Qp + Q;
            }
        }
        const bool direct = rv && P == 0;
        if (direct) {
            const int32_t slot = (bi << 6) + sortedLane;
            gHt[tk] = static_cast<uint16_t>(slot + 1);
            const int32_t w = tk >> 6;
            const uint64_t bit = 1ull << (tk & 63);
            if ((atomicOr(reinterpret_cast<unsigned long long *>(used) + w, bit) | bit) == ~0ull) {
                const int32_t s1 = w >> 6;
                const uint64_t bit1 = 1ull << (w & 63);
                if ((atomicOr(reinterpret_cast<unsigned long long *>(full1) + s1, bit1) | bit1) == ~0ull) {
                    atomicOr(reinterpret_cast<unsigned long long *>(full2) + (s1 >> 6), 1ull << (s1 & 63));
                }
            }
        }
        wave_lds_sync();
        const uint64_t congRank = __ballot(rv && !direct);
        if (congRank == 0ull) continue;
        // ---- the other keys: the sweep over the free cells, in rank order.
        // Their cells (ranked) move to lanes 0..m-1.
        const int32_t m = __popcll(congRank);
        const bool cg = (congRank >> lane) & 1ull;
        const int32_t below = __popcll(congRank & ((1ull << lane) - 1ull));
        const int32_t dest = cg ? below : m + (lane - below);
        const int32_t cTgt = __builtin_amdgcn_ds_permute(dest << 2, tk);
        const int32_t cLane = __builtin_amdgcn_ds_permute(dest << 2, sortedLane);
        uint64_t wait = 0ull;
        for (int32_t r = 0; r < m; ++r) wait |= 1ull << __builtin_amdgcn_readlane(cLane, r);
        // keys become ready in rank order as the cell passes their first-free
        // cell (which a key placed above may hold: the cell is the first free
        // one at or after it); the word holding the current cell stays in
        // registers
        uint64_t ready = 0ull;
        int32_t next = 0;  // keys of rank below it are ready or placed
        int32_t c = __builtin_amdgcn_readfirstlane(first_free(__builtin_amdgcn_readlane(cTgt, 0)));
        if (c < 0) {  // excluded by the room count; a corrupted launch only
            g.code = kOverflowProbe;
            break;
        }
        int32_t cw = c >> 6;
        uint64_t cbits = used[cw];
        while (wait != 0ull) {
            while (next < m && __builtin_amdgcn_readlane(cTgt, next) <= c) {
                ready |= 1ull << __builtin_amdgcn_readlane(cLane, next);
                ++next;
            }
            if (ready == 0ull) {  // no key waits at or before c: on to the next key's cell
                c = __builtin_amdgcn_readfirstlane(first_free(__builtin_amdgcn_readlane(cTgt, next)));
                if (c < 0) {
                    g.code = kOverflowProbe;
                    break;
                }
                if ((c >> 6) != cw) {
                    cw = c >> 6;
                    cbits = used[cw];
                }
                continue;
            }
            const int32_t j = __builtin_ctzll(ready);
            if (lane == j) gHt[c] = static_cast<uint16_t>(s + 1);
            cbits |= 1ull << (c & 63);
            put_word(cw, cbits);
            ready &= ~(1ull << j);
            wait &= ~(1ull << j);
            if (ready == 0ull) continue;  // the loop moves to the next key's cell
            // the next free cell: in the same word, else through the levels
            const uint64_t above = (c & 63) == 63 ? ~0ull : cbits | ((2ull << (c & 63)) - 1ull);
            if (above != ~0ull) {
                c = (cw << 6) + __builtin_ctzll(~above);
            } else {
                c = __builtin_amdgcn_readfirstlane(first_free((cw + 1) << 6));
                if (c < 0) {  // excluded by the room count; a corrupted launch only
                    g.code = kOverflowProbe;
                    break;
                }
                cw = c >> 6;
                cbits = used[cw];
            }
        }
    }
    if (lane == 0) report_overflow(overflowSlot, g.code);
}

template <bool kIdentity>
__device__ __forceinline__ void init_table_large(uint8_t *smem, const RowTokens<kIdentity> token, GCell *gHt,
                                                 int32_t padded, int32_t dbs, int32_t H, uint64_t overflowSlot)
{
    InitLargeLds &l = *reinterpret_cast<InitLargeLds *>(smem);
    const int32_t tid = threadIdx.x;
    constexpr int32_t NT = kInitThreads;
    // rows past 16-bit slots (no helpers; never at admission)
    const bool huge = !kIdentity && dbs >= kInitHomes;
    const int32_t zeroEnd = H < kInitTailEnd || huge ? H : kInitTailEnd;  // the helpers clear the rest
    auto clear_cells = [&]() {
        for (int32_t i = tid; i < kInitHomes / 8; i += NT) reinterpret_cast<uint4 *>(l.cells)[i] = make_uint4(0, 0, 0, 0);
    };
    auto clear_table = [&]() {
        for (int32_t i = tid; i < zeroEnd / 8; i += NT) reinterpret_cast<GChunk *>(gHt)[i] = Chunk{0u, 0u, 0u, 0u};
    };
    auto sweep = [&]() {
        clear_table();
        __threadfence_block();
        __syncthreads();
        if (tid < 64) init_table_sweep<kIdentity>(smem, token, gHt, dbs, H, overflowSlot);
    };
    clear_cells();
    l.spill[tid] = 0ull;
    if (!kIdentity && tid < kInitBuckets) l.bucket[tid] = 0u;
    if (tid == 0) l.longChain = l.stop = 0;
    __syncthreads();
    if constexpr (!kIdentity) {
        // repeated and out-of-range tokens; packed homes among the sampled slots
        const int32_t sampled = dbs <= kInitUnroll * NT ? (dbs < NT ? dbs : NT) : dbs / kInitUnroll;
        const uint32_t packed = 32u + 2u * static_cast<uint32_t>(sampled / kInitBuckets);
        bool inOrder = false;
        for (int32_t s0 = tid; s0 < dbs; s0 += kInitUnroll * NT) {
            int32_t t[kInitUnroll];
#pragma unroll
            for (int q = 0; q < kInitUnroll; ++q) t[q] = s0 + q * NT < dbs ? token(s0 + q * NT) : -1;
#pragma unroll
            for (int q = 0; q < kInitUnroll; ++q) {
                if (t[q] < 0) continue;
                // (the last homes' keys leave a larger table's homes at once)
                const uint32_t b = ht_hash(t[q]) / (kInitHomes / kInitBuckets);
                if (q == 0 && (b < kInitBuckets - 1 || H == kInitHomes) && atomicAdd(&l.bucket[b], 1u) >= packed) l.stop = 1;
                if (t[q] >= kWaveInitTokenBits) {
                    inOrder = true;
                    continue;
                }
                const uint32_t bit = 1u << (t[q] & 31);
                if (atomicOr(l.cells + (t[q] >> 5), bit) & bit) inOrder = true;
            }
        }
        if (__syncthreads_or(inOrder ? 1 : 0)) {
            clear_table();
            __threadfence_block();
            __syncthreads();
            if (tid == 0) {
                Guard g;
                const int32_t *tok = (const int32_t *)token.tok;
                for (int32_t s = 0; s < dbs && g.code == 0; ++s) {
                    const int32_t t = tok[s];
                    if (t >= 0) ht_insert((uint16_t *)gHt, tok, padded, t, s, H - 1, g);
                }
                report_overflow(overflowSlot, g.code);
            }
            return;
        }
        if (l.stop != 0 || huge) {
            sweep();
            return;
        }
        clear_cells();
        __syncthreads();
    }
    const bool wraps = H == kInitHomes;
    // the first cell at or after c that no earlier pass took, or kInitHomes
    auto next_free = [&](uint32_t c) -> uint32_t {
        uint32_t w = c >> 6;
        if (w >= static_cast<uint32_t>(kInitWords)) return kInitHomes;
        const uint64_t x = ~l.occ[w] & (~0ull << (c & 63u));
        if (x) return (w << 6) + static_cast<uint32_t>(__builtin_ctzll(x));
        for (++w; w < static_cast<uint32_t>(kInitWords); w = (w | 63u) + 1u) {
            const uint64_t f = ~l.full[w >> 6] & (~0ull << (w & 63u));
            if (f) {
                w = (w & ~63u) + static_cast<uint32_t>(__builtin_ctzll(f));
                return (w << 6) + static_cast<uint32_t>(__builtin_ctzll(~l.occ[w]));
            }
        }
        return kInitHomes;
    };
    int32_t least = NT;  // slots of a pass (at admission the chains are short)
    for (int32_t done = 0; done < dbs;) {
        const int32_t half = (kInitHomes - done) / 2;
        const int32_t end = min(dbs, done + (half > least ? half : least));
        const bool later = done > 0;
        bool longChain = false;
        for (int32_t s0 = done + tid; s0 < end; s0 += kInitUnroll * NT) {
            int32_t t[kInitUnroll];
#pragma unroll
            for (int q = 0; q < kInitUnroll; ++q) t[q] = s0 + q * NT < end ? token(s0 + q * NT) : -1;
#pragma unroll
            for (int q = 0; q < kInitUnroll; ++q) {
                if (t[q] < 0) continue;
                uint32_t v = static_cast<uint32_t>(s0 + q * NT) + 1u;
                uint32_t c = ht_hash(t[q]);  // 16 bits: the home
                int32_t hops = 0;
                for (;; ++hops) {
                    if (later) c = next_free(c);
                    if (c >= static_cast<uint32_t>(kInitHomes)) {
                        if (!wraps) {
                            atomicOr(reinterpret_cast<unsigned long long *>(l.spill) + ((v - 1u) >> 6), 1ull << ((v - 1u) & 63u));
                            break;
                        }
                        c = 0u;  // (fewer keys than cells: one is free)
                        continue;
                    }
                    v = propose16(l.cells, c, v);
                    if (v == 0u) break;
                    ++c;
                    if (hops >= kInitMaxHops) {
                        l.stop = 1;
                        break;
                    }
                }
                if constexpr (!kIdentity) longChain = longChain || hops > kInitLongChain;
            }
            if (*const_cast<volatile int32_t *>(&l.stop)) break;
        }
        if constexpr (!kIdentity) {
            if (longChain) l.longChain = 1;
        }
        __syncthreads();
        // (neither word is set again before the next barrier)
        if constexpr (!kIdentity) {
            if (l.longChain != 0) least = kInitSmallPass;
        }
        if (l.stop) {
            sweep();
            return;
        }
        done = end;
        if (done < dbs) {
            uint8_t *occ8 = reinterpret_cast<uint8_t *>(l.occ);
            for (int32_t i = tid; i < kInitHomes / 8; i += NT) {
                const uint4 v = reinterpret_cast<const uint4 *>(l.cells)[i];
                const uint32_t w[4] = {v.x, v.y, v.z, v.w};
                uint32_t m = 0u;
#pragma unroll
                for (int h = 0; h < 4; ++h) {
                    m |= ((w[h] & 0xFFFFu) != 0u ? 1u : 0u) << (2 * h);
                    m |= ((w[h] >> 16) != 0u ? 1u : 0u) << (2 * h + 1);
                }
                occ8[i] = static_cast<uint8_t>(m);
            }
            __syncthreads();
            const uint64_t fm = __ballot(l.occ[tid] == ~0ull);
            if ((tid & 63) == 0) l.full[tid >> 6] = fm;
            __syncthreads();
        }
    }
    for (int32_t i = tid; i < kInitHomes / 8; i += NT) {
        const uint4 v = reinterpret_cast<const uint4 *>(l.cells)[i];
        reinterpret_cast<GChunk *>(gHt)[i] = Chunk{v.x, v.y, v.z, v.w};
    }
    if (wraps) return;
    // the spilled slots in increasing order from cell 65536 on
    uint64_t sp = l.spill[tid];
    uint32_t inc = static_cast<uint32_t>(__builtin_popcountll(sp));
    const uint32_t mine = inc, lane = static_cast<uint32_t>(__lane_id());
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t o = static_cast<uint32_t>(__shfl_up(static_cast<int>(inc), d));
        if (lane >= static_cast<uint32_t>(d)) inc += o;
    }
    if (lane == 63u) l.part[tid >> 6] = inc;
    __syncthreads();
    uint32_t before = 0, total = 0;
    for (int w = 0; w < NT / 64; ++w) {
        if (w < (tid >> 6)) before += l.part[w];
        total += l.part[w];
    }
    uint32_t at = kInitHomes + before + inc - mine;
    for (; sp != 0ull; sp &= sp - 1ull) {
        gHt[at++] = static_cast<uint16_t>((static_cast<uint32_t>(tid) << 6) + static_cast<uint32_t>(__builtin_ctzll(sp)) + 1u);
    }
    // the empty cells after them: the cells up to the next chunk one by one
    const uint32_t end = kInitHomes + total, chunk0 = (end + 7u) / 8u;
    if (static_cast<uint32_t>(tid) < chunk0 * 8u - end) gHt[end + static_cast<uint32_t>(tid)] = 0;
    for (uint32_t i = chunk0 + static_cast<uint32_t>(tid); i < static_cast<uint32_t>(zeroEnd) / 8u; i += NT) {
        reinterpret_cast<GChunk *>(gHt)[i] = Chunk{0u, 0u, 0u, 0u};
    }
}

// kLarge: the form for tables beyond kInitLdsCells; workgroup y > 0 of a row
// clears its share of the cells that no key reaches.
template <bool kLarge>
__global__ __launch_bounds__(kInitThreads) void kvx_sieve_ht_init_par(KvxLaunch<HispSieveHtInitArgs> L)
{
    extern __shared__ __align__(16) uint8_t smem[];
    const HispSieveHtInitArgs &a = L.a;
    const int32_t numReqs = static_cast<int32_t>(a.numReqs);
    const int32_t poolSize = static_cast<int32_t>(a.poolSize);
    const int32_t padded = static_cast<int32_t>(a.paddedBufferSize);
    const int32_t H = static_cast<int32_t>(a.htSize);
    const int32_t b = blockIdx.x;  // the grid is exactly layerNum * numReqs
    const int32_t layer = b / numReqs;
    const int64_t reqIdx = static_cast<int64_t>(a.reqStart) + b % numReqs;
    if (reqIdx < 0 || reqIdx >= poolSize) return;
    const int64_t row = static_cast<int64_t>(layer) * poolSize + reqIdx;
    const RowTokens<false> token{reinterpret_cast<GTok *>(a.deviceBufferTokens) + row * padded, 0};
    GCell *gHt = reinterpret_cast<GCell *>(a.deviceBufferHt) + row * H;
    if constexpr (kLarge) {
        if (blockIdx.y != 0) {
            for (int32_t i = kInitTailEnd / 8 + (static_cast<int32_t>(blockIdx.y) - 1) * kInitThreads + threadIdx.x; i < H / 8;
                 i += kInitHelpers * kInitThreads) {
                reinterpret_cast<GChunk *>(gHt)[i] = Chunk{0u, 0u, 0u, 0u};
            }
            return;
        }
        init_table_large<false>(smem, token, gHt, padded, static_cast<int32_t>(a.deviceBufferSize), H, L.overflowSlot);
    } else {
        init_table_lds<false>(smem, token, gHt, static_cast<int32_t>(a.deviceBufferSize), H);
    }
}

// One request's state in every layer at admission, in one launch: slot s holds
// token s for s < n0 and none past it, the visited bits and the hand records
// cleared, the tables of those tokens, the request's lengths.  Workgroup x is
// layer x; in the large form workgroup y > 0 writes a share of everything but
// the cells below kInitTailEnd, which workgroup 0 builds meanwhile.  The
// tokens need not be read back: their slots are their numbers.  (As eight
// launches -- fills, a range, two copies of a scalar from the host, the table
// build -- an admission was bound by their submission, ~45 us of it.)
template <bool kLarge>
__global__ __launch_bounds__(kInitThreads) void kvx_admit(AdmitArgs a, uint64_t overflowSlot)
{
    extern __shared__ __align__(16) uint8_t smem[];
    const int32_t padded = static_cast<int32_t>(a.paddedBufferSize), H = static_cast<int32_t>(a.htSize);
    const int32_t tid = threadIdx.x, n0 = a.liveSlots;
    const int64_t row = static_cast<int64_t>(blockIdx.x) * a.poolSize + a.reqPoolIdx;
    GCell *gHt = reinterpret_cast<GCell *>(a.deviceBufferHt) + row * H;
    if (!kLarge || blockIdx.y != 0) {
        const int32_t parts = kLarge ? kInitHelpers : 1, part = kLarge ? static_cast<int32_t>(blockIdx.y) - 1 : 0;
        const int32_t step = parts * static_cast<int32_t>(blockDim.x), first = part * static_cast<int32_t>(blockDim.x) + tid;
        GChunk *tok4 = reinterpret_cast<GChunk *>(a.deviceBufferTokens + static_cast<uint64_t>(row) * padded * 4u);
        for (int32_t i = first; i < padded / 4; i += step) {
            auto at = [&](int32_t s) { return static_cast<uint32_t>(s < n0 ? s : -1); };
            tok4[i] = Chunk{at(4 * i), at(4 * i + 1), at(4 * i + 2), at(4 * i + 3)};
        }
        GChunk *vis4 = reinterpret_cast<GChunk *>(a.deviceBufferVisited + static_cast<uint64_t>(row) * a.visitedStrideB);
        for (int32_t i = first; i < static_cast<int32_t>(a.visitedStrideB) / 16; i += step) vis4[i] = Chunk{0u, 0u, 0u, 0u};
        if (part == 0 && tid < kHandStride / 4) {
            reinterpret_cast<GChunk *>(a.sieveHand + static_cast<uint64_t>(row) * kHandStride * 4u)[tid] = Chunk{0u, 0u, 0u, 0u};
        }
        if (blockIdx.x == 0 && part == 0 && tid == 0) {
            reinterpret_cast<__attribute__((address_space(1))) int32_t *>(a.prefillLens)[a.reqPoolIdx] = a.prefillLen;
            reinterpret_cast<__attribute__((address_space(1))) int64_t *>(a.reqHostBase)[a.reqBatchIdx] = a.hostBaseRow;
        }
        if constexpr (kLarge) {
            for (int32_t i = kInitTailEnd / 8 + first; i < H / 8; i += step) reinterpret_cast<GChunk *>(gHt)[i] = Chunk{0u, 0u, 0u, 0u};
            return;
        }
    }
    const RowTokens<true> token{nullptr, n0};
    if constexpr (kLarge) init_table_large<true>(smem, token, gHt, padded, n0, H, overflowSlot);
    else init_table_lds<true>(smem, token, gHt, n0, H);
}

}  // namespace

hipError_t sieve_set_lds_limit(size_t bytes)
{
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&kvx_sieve_update<true>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes));
    if (e != hipSuccess) return e;
    e = hipFuncSetAttribute(reinterpret_cast<const void *>(&kvx_sieve_ht_init<true>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes));
    if (e != hipSuccess) return e;
    e = hipFuncSetAttribute(reinterpret_cast<const void *>(&kvx_sieve_ht_init_par<false>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes));
    if (e != hipSuccess) return e;
    for (const void *f : {reinterpret_cast<const void *>(&kvx_sieve_ht_init_par<true>),
                          reinterpret_cast<const void *>(&kvx_admit<false>), reinterpret_cast<const void *>(&kvx_admit<true>)}) {
        e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes));
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t launch_sieve_update(const HispSieveUpdateArgs &a, uint64_t overflowSlot, int variant, size_t ldsBytes,
                               hipStream_t stream)
{
    KvxLaunch<HispSieveUpdateArgs> L{a, overflowSlot};
    const dim3 grid(a.maxNumReqs), block(256);
    if (variant == 0) {
        hipLaunchKernelGGL(kvx_sieve_update<true>, grid, block, ldsBytes, stream, L);
    } else {
        hipLaunchKernelGGL(kvx_sieve_update<false>, grid, block, 0, stream, L);
    }
    return hipGetLastError();
}

size_t sieve_ht_init_small_lds(uint32_t htSize, uint32_t dbs)
{
    // fewer keys than cells, or a chain of proposals would not end
    if (htSize < 1024u || htSize > static_cast<uint32_t>(kInitLdsCells) || dbs >= htSize) return 0;
    return static_cast<size_t>(htSize) * 4u + (dbs + 31u) / 32u * 4u;
}

size_t sieve_ht_init_large_lds(uint32_t htSize, uint32_t dbs)
{
    // fewer keys than cells
    if (htSize < static_cast<uint32_t>(kInitHomes) || htSize > (1u << 20) || dbs >= htSize) return 0;
    const size_t sweep = htSize / 8u + htSize / 512u + 8u * ((htSize + 262143u) / 262144u);
    return sweep > sizeof(InitLargeLds) ? sweep : sizeof(InitLargeLds);
}

hipError_t launch_admit(const AdmitArgs &a, uint32_t layers, uint64_t overflowSlot, size_t ldsBytes, bool large,
                        hipStream_t stream)
{
    if (large) {
        hipLaunchKernelGGL(kvx_admit<true>, dim3(layers, 1u + kInitHelpers), dim3(kInitThreads), ldsBytes, stream, a, overflowSlot);
    } else {
        const uint32_t threads = a.paddedBufferSize <= static_cast<uint32_t>(kInitSmallSlots) ? kInitSmallThreads : kInitThreads;
        hipLaunchKernelGGL(kvx_admit<false>, dim3(layers), dim3(threads), ldsBytes, stream, a, overflowSlot);
    }
    return hipGetLastError();
}

hipError_t launch_sieve_ht_init(const HispSieveHtInitArgs &a, uint64_t overflowSlot, size_t ldsBytes,
                                hipStream_t stream, InitForm form)
{
    KvxLaunch<HispSieveHtInitArgs> L{a, overflowSlot};
    const dim3 grid(a.layerNum * a.numReqs), block(256);
    if (form == InitForm::kSmall) {
        const uint32_t threads = a.deviceBufferSize <= static_cast<uint32_t>(kInitSmallSlots) ? kInitSmallThreads : kInitThreads;
        hipLaunchKernelGGL(kvx_sieve_ht_init_par<false>, grid, dim3(threads), ldsBytes, stream, L);
    } else if (form == InitForm::kLarge) {
        // (the rows of more than 65535 slots may take cells past kInitTailEnd)
        const bool tail = a.htSize > static_cast<uint32_t>(kInitTailEnd) && a.deviceBufferSize < static_cast<uint32_t>(kInitHomes);
        const uint32_t parts = tail ? 1u + kInitHelpers : 1u;
        hipLaunchKernelGGL(kvx_sieve_ht_init_par<true>, dim3(grid.x, parts), dim3(kInitThreads), ldsBytes, stream, L);
    } else if (ldsBytes != 0) {
        hipLaunchKernelGGL(kvx_sieve_ht_init<true>, grid, block, ldsBytes, stream, L);
    } else {
        hipLaunchKernelGGL(kvx_sieve_ht_init<false>, grid, block, 0, stream, L);
    }
    return hipGetLastError();
}

}  // namespace kvx

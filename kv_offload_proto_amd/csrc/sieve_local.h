// The table update of a SIEVE step that changes short clusters only, by the
// row's own workgroup at the end of the batch kernel (variant 5).
#pragma once

#include "kvx_internal.h"

#ifndef KVX_GM
#define KVX_GM __attribute__((address_space(1)))
#endif

namespace kvx {
namespace table_local {

typedef uint32_t Cells8 __attribute__((ext_vector_type(4)));  // eight table cells

// A row whose step changes short clusters only, by one workgroup with the
// cells that can be homes (the first 65536) in LDS as they are:
//  - a thread per cluster that lost a key walks it from its first deleted
//    cell on, each later entry moving into the leftmost hole at or after its
//    home (all of the step's deletions in the cluster at once, sieve_batch.hip);
//  - the new keys propose to the cells from their home on, all at once: a cell
//    that keeps an old entry refuses, one that holds a new key keeps the
//    earlier event's (the table of sequential inserts is the stable matching
//    of cells that prefer earlier events, found in any order of the
//    proposals).  An entry naming an evicted slot is a new key then, and the
//    hand evicts in ring order, so the ring offset of the slot is its event's
//    order: the cells need no second array.
// The cells that changed go back to HBM.  A row with a longer walk or chain, a
// cluster that runs past cell 65535, or a step whose hand turned past its
// start is left pending for the rebuild (sieve_table.hip), nothing written.
// The bound is latency: a staging round trip, about two token loads a walk,
// a few LDS round trips a key.  One row of 16384 slots, 470 misses: 19 us,
// where the rebuild took 98 (155 a call, 62 so; as a launch of its own, 59.6
// against 58.4 a call).
constexpr uint32_t kLocalCells = 65536;
constexpr uint32_t kLocalWalk = 64;    // cells of a walk (the holes are bits of a word)
constexpr uint32_t kLocalHops = 512;   // proposals of a chain
constexpr int kLocalLoads = kLocalCells / 8 / kBatchThreads;  // 16-byte chunks of cells a lane stages

constexpr uint32_t lds_bytes(uint32_t cells) { return cells * 2u + cells / 4u + kLocalCells / 8u; }

// tb: the row's rebuild scratch (evicted slots and new keys written, pending);
// N new keys, taken from `hand` on in ring order if ringOrder.  Every thread
// calls it, after a barrier behind those writes.
__device__ __forceinline__ void apply(const HispSieveUpdateArgs &a, KVX_GM uint32_t *tb, const TableLayout &t, int64_t reqIdx,
                                      uint32_t N, uint32_t hand, bool ringOrder, unsigned char *lds)
{
    __shared__ int32_t sStop;
    const uint32_t H = a.htSize, C = H < kLocalCells ? H : kLocalCells, padded = a.paddedBufferSize;
    const uint32_t dbs = a.deviceBufferSize;
    const uint32_t tid = threadIdx.x;
    KVX_GM Cells8 *ht8 = reinterpret_cast<KVX_GM Cells8 *>(reinterpret_cast<KVX_GM uint16_t *>(a.deviceBufferHt) + reqIdx * H);
    const KVX_GM int32_t *tok = reinterpret_cast<const KVX_GM int32_t *>(a.deviceBufferTokens) + reqIdx * padded;
    const KVX_GM uint32_t *newk = tb + t.newk;
    // the rebuild finds the per-home counts zeroed
    auto leave = [&]() {
        KVX_GM Cells8 *h4 = reinterpret_cast<KVX_GM Cells8 *>(tb + t.hist);
        for (uint32_t i = tid; i < C / 4u; i += kBatchThreads) h4[i] = Cells8{0u, 0u, 0u, 0u};
    };
    if (!ringOrder) {
        leave();
        return;
    }
    uint32_t *cells32 = reinterpret_cast<uint32_t *>(lds);
    uint16_t *cells = reinterpret_cast<uint16_t *>(lds);
    uint32_t *del = cells32 + C / 2u;        // deleted cells
    uint32_t *changed = del + C / 32u;       // cells to write back
    uint32_t *evict = changed + C / 32u;     // evicted slots, 65536 bits
    uint8_t *del8 = reinterpret_cast<uint8_t *>(del), *changed8 = reinterpret_cast<uint8_t *>(changed);
    // Whether the row is left to the rebuild is decided at a barrier, from
    // every thread's own flag; sStop only lets other waves' loops end early.
    // (Read behind a barrier, it could already hold the next phase's value in
    // a late wave, which would then leave alone.)
    bool stop = false;
    auto stop_now = [&]() {
        stop = true;
        *const_cast<volatile int32_t *>(&sStop) = 1;
    };
    auto stopped = [&]() { return *const_cast<volatile int32_t *>(&sStop) != 0; };
    auto refused = [&]() { return __syncthreads_or(stop ? 1 : 0) != 0; };
    auto evicted = [&](uint32_t s) { return (evict[s >> 5] >> (s & 31u)) & 1u; };
    Cells8 v[kLocalLoads];
#pragma unroll
    for (int q = 0; q < kLocalLoads; ++q) {
        const uint32_t i = tid + static_cast<uint32_t>(q) * kBatchThreads;
        if (i < C / 8u) v[q] = ht8[i];
    }
    for (uint32_t i = tid; i < kLocalCells / 32u; i += kBatchThreads) evict[i] = i < (dbs + 31u) / 32u ? tb[t.evict + i] : 0u;
    if (tid == 0) sStop = 0;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kLocalLoads; ++q) {
        const uint32_t i = tid + static_cast<uint32_t>(q) * kBatchThreads;
        if (i >= C / 8u) continue;
        reinterpret_cast<Cells8 *>(cells32)[i] = v[q];
        const uint32_t w[4] = {v[q].x, v[q].y, v[q].z, v[q].w};
        uint32_t m = 0u;
        bool taken = true;
#pragma unroll
        for (int h = 0; h < 8; ++h) {
            const uint32_t e = (w[h >> 1] >> (16 * (h & 1))) & 0xFFFFu;
            const uint32_t s = (e - 1u) & 0xFFFFu;
            taken = taken && e != 0u;
            m |= (e != 0u && evicted(s) ? 1u : 0u) << h;
        }
        del8[i] = static_cast<uint8_t>(m);
        changed8[i] = static_cast<uint8_t>(m);
        // a run of 64 taken cells (eight chunks of neighbouring lanes): walks
        // and chains would be too long
        uint64_t runs = __ballot(taken);
        runs &= runs >> 1;
        runs &= runs >> 2;
        runs &= runs >> 4;
        if (runs != 0ull) stop_now();
        // a key in a cell past 65535 has a home below it: cell 65535 is taken
        if (H > kLocalCells && i == kLocalCells / 8u - 1u && (v[q].w >> 16) != 0u) stop_now();
    }
    if (refused()) {
        leave();
        return;
    }
    const bool wraps = H <= kLocalCells;  // else cells past the staged ones are empty
    // clusters' first deleted cells: no deleted cell before them in the run
    uint32_t lead[kLocalCells / 32u / kBatchThreads];
#pragma unroll
    for (uint32_t q = 0; q < kLocalCells / 32u / kBatchThreads; ++q) {
        const uint32_t w = tid + q * kBatchThreads;
        lead[q] = 0u;
        if (w >= C / 32u) continue;
        for (uint32_t m = del[w]; m != 0u && !stopped(); m &= m - 1u) {
            const uint32_t c = (w << 5) + static_cast<uint32_t>(__builtin_ctz(m));
            bool first = true;
            uint32_t x = c;
            for (uint32_t n = 0;; ++n) {
                if (x == 0u && !wraps) break;
                x = (x - 1u) & (C - 1u);
                if (cells[x] == 0) break;
                if ((del[x >> 5] >> (x & 31u)) & 1u) {
                    first = false;
                    break;
                }
                if (n >= kLocalWalk) {
                    stop_now();
                    break;
                }
            }
            if (first) lead[q] |= 1u << (c & 31u);
        }
    }
    if (refused()) {
        leave();
        return;
    }
    // the clusters, four cells of a walk at a time (their tokens loaded together)
#pragma unroll
    for (uint32_t q = 0; q < kLocalCells / 32u / kBatchThreads; ++q) {
        for (uint32_t m = lead[q]; m != 0u && !stopped(); m &= m - 1u) {
            const uint32_t c = ((tid + q * kBatchThreads) << 5) + static_cast<uint32_t>(__builtin_ctz(m));
            uint64_t holes = 1ull;
            bool done = false;
            for (uint32_t o0 = 1; !done; o0 += 4u) {
                if (o0 + 4u > kLocalWalk) {
                    stop_now();
                    break;
                }
                uint32_t x[4], e[4];
                bool dl[4];
                int32_t tk[4];
                bool run = true;
#pragma unroll
                for (uint32_t h = 0; h < 4u; ++h) {
                    x[h] = c + o0 + h;
                    if (wraps) x[h] &= C - 1u;
                    e[h] = x[h] < C ? cells[x[h]] : 0u;  // (the cell after the staged ones is empty)
                    run = run && e[h] != 0u;
                    dl[h] = run && ((del[x[h] >> 5] >> (x[h] & 31u)) & 1u);
                    if (run && e[h] > padded) {  // only in a corrupted table: the rebuild takes the row
                        stop_now();
                        run = false;
                        e[h] = 0u;
                    }
                    tk[h] = run && !dl[h] ? tok[e[h] - 1u] : 0;
                }
#pragma unroll
                for (uint32_t h = 0; h < 4u; ++h) {
                    if (done) continue;
                    const uint32_t o = o0 + h;
                    if (e[h] == 0u) {
                        done = true;
                    } else if (dl[h]) {
                        holes |= 1ull << o;
                    } else {
                        // the home as an offset from c, 0 when it lies before
                        const uint32_t d = (x[h] - (ht_hash(tk[h]) & (H - 1u))) & (H - 1u);
                        const uint64_t at = d < o ? holes & (~0ull << (o - d)) : holes;
                        if (d == 0u || at == 0ull) continue;
                        const uint32_t t = static_cast<uint32_t>(__builtin_ctzll(at));
                        const uint32_t y = wraps ? (c + t) & (C - 1u) : c + t;
                        cells[y] = static_cast<uint16_t>(e[h]);
                        holes = (holes & ~(1ull << t)) | (1ull << o);
                        atomicOr(changed + (x[h] >> 5), 1u << (x[h] & 31u));
                    }
                }
            }
            for (; holes != 0ull; holes &= holes - 1ull) {
                const uint32_t y = c + static_cast<uint32_t>(__builtin_ctzll(holes));
                cells[wraps ? y & (C - 1u) : y] = 0;
            }
        }
    }
    if (refused()) {
        leave();
        return;
    }
    auto ring = [&](uint32_t s) { return s >= hand ? s - hand : s + dbs - hand; };
    for (uint32_t j = tid; j < N && !stopped(); j += kBatchThreads) {
        const uint32_t nk = newk[j];
        uint32_t c = nk >> 16, mine = nk & 0xFFFFu;
        for (uint32_t hops = 0;; ++hops) {
            if (c >= C && wraps) c = 0u;
            if (c >= C || hops >= kLocalHops) {
                stop_now();
                break;
            }
            uint32_t *w = cells32 + (c >> 1);
            const uint32_t sh = (c & 1u) * 16u;
            uint32_t old = *w, cur = 0u;
            bool placed = false;
            for (;;) {
                cur = (old >> sh) & 0xFFFFu;
                if (cur != 0u && (!evicted(cur - 1u) || ring(cur - 1u) < ring(mine - 1u))) break;
                const uint32_t prev = atomicCAS(w, old, (old & ~(0xFFFFu << sh)) | (mine << sh));
                if (prev == old) {
                    placed = true;
                    break;
                }
                old = prev;
            }
            if (placed) {
                atomicOr(changed + (c >> 5), 1u << (c & 31u));
                if (cur == 0u) break;
                mine = cur;
            }
            ++c;
        }
    }
    if (refused()) {
        leave();
        return;
    }
    for (uint32_t i = tid; i < C / 8u; i += kBatchThreads) {
        if (changed8[i] != 0) ht8[i] = reinterpret_cast<const Cells8 *>(cells32)[i];
    }
    if (tid == 0) tb[t.meta] = 0u;
}

}  // namespace table_local
}  // namespace kvx

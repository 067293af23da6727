"""CPU check of the winner rule of the one-launch import (kvx_gather_one,
csrc/rows.hip).

The rule (kvc_gather_rows.cpp:69-81 copies in position order, so the last
miss on a destination row wins): a position takes part when it is a miss with
a valid token, slot 0 <= s < 65536 and a pool row; its destination is
d = b * rows + s (b its request, rows = min(stride, 65536)); the winner of a
destination is its largest position.  The kernel takes the positions in use in
groups -- a request, or all of them at stride 0 -- and a group in spans of 16,
32 or 64.  A span's workgroup marks the slots of the group's positions after
the span in a bitmap; an own position wins when its slot is neither there nor
at a later own position, and, where the slot is at or past `rows`, at no
position of the later requests that reaches the same row.  Here that
decomposition is replayed and compared with the global rule by brute force,
over strides that keep requests apart, make neighbours share rows, or put every
request on the same rows, spans that end inside and past a request, every span
size, and fewer requests than the call was made for.
"""
import numpy as np
import pytest


def _spans(total, group):
    """gather_spans: (positions of a span, spans of a group, spans in all)."""
    if total == 0:
        return 16, 0, 0
    span = 16
    while span < 64 and total // span > 1024:
        span *= 2
    parts = -(-group // span)
    return span, parts, total // group * parts


def _inputs(rng, req, top_k, dbs):
    topk = rng.integers(-1, 50, size=req * top_k)
    slots = rng.integers(-1, dbs, size=req * top_k)
    slots[rng.random(req * top_k) < 0.01] = 70000  # outside the rule (>= 65536)
    miss = rng.random(req * top_k) < 0.6
    pool = np.where(rng.random(req) < 0.15, -1, np.arange(req))
    return topk, slots, miss, pool


def _part(p, topk, slots, miss, pool, top_k):
    """Slot of position p when it takes part in the winner rule, else -1."""
    s = int(slots[p])
    if not miss[p] or topk[p] < 0 or s < 0 or s >= 65536 or pool[p // top_k] < 0:
        return -1
    return s


def _global_winners(total, top_k, span, part):
    last = {}
    for p in range(total):
        s = part(p)
        if s >= 0:
            last[(p // top_k) * span + s] = p
    return {p for p in last.values()}


def _kernel_winners(total, top_k, rows, part):
    """The one-launch import's decisions, span by span."""
    group = total if rows == 0 else top_k
    span, parts, count = _spans(total, group)
    key = [part(p) for p in range(total)]
    won, seen = set(), []
    for blk in range(count):
        g, q = divmod(blk, parts)
        lo = g * group + q * span
        end = min((g + 1) * group, total)
        hi = min(lo + span, end)
        later = set(key[hi:end])
        for p in range(lo, hi):
            seen.append(p)
            k = key[p]
            if k < 0 or k in later or k in key[p + 1:hi]:
                continue
            if rows != 0 and k >= rows:  # also a row of the next k // rows requests
                b0 = p // top_k
                b1 = min(total // top_k - 1, b0 + k // rows)
                if any(key[x] == k - (x // top_k - b0) * rows for x in range((b0 + 1) * top_k, (b1 + 1) * top_k)):
                    continue
            won.add(p)
    assert seen == list(range(total))  # every position in use is in one span
    return won


@pytest.mark.parametrize("seed", range(6))
@pytest.mark.parametrize("req,top_k,dbs,stride", [
    (12, 20, 16, 16), (40, 7, 8, 8), (10, 48, 32, 16), (6, 100, 64, 0), (8, 64, 64, 64),
    (3, 33, 40, 70000), (5, 1, 4, 2), (1, 300, 50, 48),
    (12, 20, 17, 16), (20, 10, 9, 8),  # slots up to the rows themselves: only s == rows reaches the next request
])
def test_small_import_winners_equal_global_rule(seed, req, top_k, dbs, stride):
    _check(seed, req, top_k, dbs, stride, req)


@pytest.mark.parametrize("req,top_k,dbs,stride,num_real", [
    (40, 17, 16, 8, 3), (6, 100, 64, 0, 2), (6, 100, 64, 0, 0), (9, 64, 70, 16, 1),
    (40, 513, 96, 48, 40),   # spans of 32
    (40, 513, 96, 48, 30),   # 15390 positions: of 16
    (70, 513, 600, 512, 70),  # of 64, one position past eight of them
    (1, 8192, 4096, 0, 1),   # the longest group
])
def test_import_spans_equal_global_rule(req, top_k, dbs, stride, num_real):
    _check(req + top_k, req, top_k, dbs, stride, num_real)


def _check(seed, req, top_k, dbs, stride, num_real):
    rng = np.random.default_rng(seed * 7919 + req * 131 + top_k)
    topk, slots, miss, pool = _inputs(rng, req, top_k, dbs)
    total = num_real * top_k
    rows = min(stride, 65536)

    def part(p):
        return _part(p, topk, slots, miss, pool, top_k)

    assert _kernel_winners(total, top_k, rows, part) == _global_winners(total, top_k, rows, part)


def test_request_local_search_alone_misses_shared_rows():
    """The wider search is needed: with stride 0 (every request on the same
    rows) a search within each request keeps an earlier request's position that
    a later request overwrites."""
    top_k, span = 4, 0
    slots = np.array([3, 1, 2, 0, 3, 5, 6, 7])  # request 0's slot 3 is request 1's slot 3 too
    miss = np.ones(8, dtype=bool)
    topk = np.zeros(8, dtype=np.int64)
    pool = np.arange(2)

    def part(p):
        return _part(p, topk, slots, miss, pool, top_k)

    local = set()
    for p in range(8):
        end = (p // top_k + 1) * top_k
        if not any(part(q) == part(p) for q in range(p + 1, end)):
            local.add(p)
    glob = _global_winners(8, top_k, span, part)
    assert 0 in local and 0 not in glob
    assert _kernel_winners(8, top_k, span, part) == glob

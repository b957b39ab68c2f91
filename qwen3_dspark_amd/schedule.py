"""Split-K work lists.

Varlen / verification attention: balanced key segments.  The keys of all
requests, laid end to end in request order, are cut into `groups` runs of
(nearly) equal length, each cut moved to a 32-key tile boundary of the
request it falls in; the 8 workgroups of run w (one per KV head) run on
XCD w mod 8 (see XCDS).  A run may end
inside one request and start inside the next, so a request is held by one
or more segments (one per run it meets).  Every workgroup therefore reads
the same number of key rows, whatever the mix of context lengths, and a
request cut into several segments writes one set of FP32 partials per
segment for the split-K merge.  Segment partial slots are request-major, so
results do not depend on the cut points beyond the floating-point order of
the merge.

  list = [segment records, WORK_INTS each, grouped by run]
         [run ranges: groups + 1 record indices]
         [request records, REQ_INTS each]
  segment: request, first key, end key, partial slot (-1: the request has a
           single segment and writes its output), first query row, query
           length, key length, first key row (varlen) or resident slot (verify)
  request: first partial slot, segment count, first query row, query length

With measured per-XCD speeds (xcd_speed), run w's share of the cost is
proportional to the speed of its XCD, so that the XCDs finish together.
With two resident workgroups per CU, the runs dispatched second onto their
CUs get SECOND_SLOT_SHARE of that share (run_shares).

Draft attention: the same balanced segments over the context rows each
request streams (up to its largest anchor), one run per (workgroup, KV
head), cuts on 64-row ring-stage boundaries (draft_work).

Requests of more than DECODE_TOKENS query tokens (prompts) are attended by a
kernel with one workgroup per (segment, KV head, 32 query tokens); their
segments follow the runs' records and belong to no run (prompt_segments).
Balanced plans of batches that hold prompts have a list of their own
(mixed_plan): the runs are cut for the other requests alone, partial slots are
counted in tiles of 8 query tokens, and the prompts' workgroups are listed.

Without a list, both kernels walk fixed chunks of `chunk` rows in request
order over a grid sized from the row bound.
"""
import functools
from collections import namedtuple

import numpy as np

from ._device import upload

DEFAULT_CHUNK = 1024          # verification / varlen: fixed chunks when no list is given
TILE = 32                     # segment cuts fall on multiples of this many keys
MIN_SEGMENT = 256             # fewest keys a run is given (tiny calls use fewer runs)
RESIDENT_PER_CU = 2           # varlen/verify workgroups resident per CU (register budget)
XCDS = 8                      # MI355X: workgroup b runs on XCD b mod 8; varlen runs come in whole rounds of 8
SEGMENT_COST = 96             # keys' worth of fixed work per segment in balanced varlen plans (measured)
# Cost share of a balanced varlen run whose workgroups are dispatched after
# every CU already holds one: two resident workgroups share a CU, and the
# later one's waves lose issue arbitration to the older ones, so it streams
# ~15 % slower (measured; 0.6-0.9 all gain about the same).
SECOND_SLOT_SHARE = 0.75
DECODE_TOKENS = 8             # requests with more query tokens take the prefill kernel (attn.hip)
PROMPT_TOKENS = 32            # query tokens per prefill workgroup (two resident per CU)
# A prompt is cut while its segments keep this many keys on CUs of their own (in
# 1 / 2 / 4 / 8 / 16 segments, us a call: 200 tokens over 1,000 keys 26.7, 20.9, 17.5,
# 18.7, -; 128 over 4,096 61, 38, 26, 22, 23; 64 over 8,000 111, 63, 38, 27, 23) and this many
# where two workgroups share a CU (8 prompts of 100 tokens over 1,000 keys uncut 28,
# in halves 32; 256 over 8,000 in 4 / 8 43, 38).
MIN_PROMPT_SEGMENT = 256
SHARED_PROMPT_SEGMENT = 1024
MAX_PROMPT_SEGMENTS = 16      # more gain nothing: 16 / 24 / 32 of 64 tokens over 8,000 keys 22.8, 25.5, 25.9 us
# Prompts of up to TILED_TOKENS are attended as tiles of DECODE_TOKENS while their tiles'
# keys number at most TILED_KEYS per workgroup slot (two per CU): the prompt form
# waits for one 64-key stage after the other (~1 us each), which few tokens on an
# idle machine do not hide, while tiles read the keys once per 8 tokens.  Prompt
# form / tiles, us: 9 tokens over 700 keys 14.2 / 9.0, over 8,000 22.6 / 21.2; 64 over 300 14.0
# / 10.4, over 2,000 17.4 / 13.7, over 4,096 18.4 / 19; 96 over 700 16.4 / 11.9; 8 prompts of
# 64 tokens over 300 14.6 / 9.9, over 1,000 23.5 / 28.
TILED_TOKENS = 96
TILED_KEYS = 384
MAX_TILES = 64                # tiles that they add to a batch at most
DRAFT_TILE = 64               # draft cuts fall on multiples of the ring stage
DRAFT_SEGMENT_COST = 512      # balanced draft plans: fixed cost of a segment, in context rows (measured)
DRAFT_BLOCK_WEIGHT = 0.055    # balanced draft plans: extra cost of a row per block beyond the first (measured)
MIN_DRAFT_SEGMENT = 1024      # fewest context rows a draft run is given
# Fixed draft chunks when no list is given (a chunk carries up to 8 blocks
# of FP32 partials, so draft chunks are coarser).
DRAFT_CHUNK = 4096
MIN_DRAFT_CHUNK = 256         # the batch-sized draft chunk never falls below this many rows
WORK_INTS = 8
REQ_INTS = 4
PART_TILE_BYTES = 8 * 16 * (128 + 2) * 4      # split-K partials of one 8-token tile, every KV head

MixedCapacity = namedtuple('MixedCapacity', 'run_records prompt_records runs requests columns tiles')
MixedPlan = namedtuple('MixedPlan', 'records n_work runs requests columns tiles')


def check_chunk(chunk):
    """Refuses what the attention entry points refuse: the mixed one takes no chunk."""
    if chunk < TILE or chunk % TILE or chunk > 1 << 20:
        raise ValueError(f'chunk must be a multiple of {TILE} in [{TILE}, 2^20] (got {chunk})')


def n_chunks(n, chunk):
    return max(1, -(-int(n) // chunk))


def chunk_items(lengths, chunk):
    """[(request, chunk_index)] for all items, longest chunk first (stable)."""
    items = []
    for r, n in enumerate(lengths):
        n = int(n)
        for c in range(n_chunks(n, chunk)):
            items.append((min(chunk, n - c * chunk) if n > 0 else 0, r, c))
    items.sort(key=lambda x: -x[0])
    return [(r, c) for _, r, c in items]


def chunk_bound(n_req, rows_bound, chunk):
    """Upper bound on the number of items for n_req requests totalling at
    most rows_bound key rows (the C ABI's grid bound)."""
    return -(-int(rows_bound) // chunk) + int(n_req)


def _bases(lengths, chunk):
    first, acc = [], 0
    for n in lengths:
        first.append(acc)
        acc += n_chunks(n, chunk)
    return first


def run_count(total_keys, n_cu, row_tiles=1):
    """Runs for a balanced list: one workgroup per CU slot and KV head when
    there is enough work, about MIN_SEGMENT keys per run at least, in whole
    rounds of XCDS runs (run w executes on XCD w mod XCDS)."""
    slots = max(XCDS, (int(n_cu) * RESIDENT_PER_CU) // (8 * max(1, int(row_tiles))) // XCDS * XCDS)
    runs = max(1, min(slots, -(-int(total_keys) // MIN_SEGMENT)))
    return -(-runs // XCDS) * XCDS


def _flatten(n, per_run, record, request, loose=()):
    """Flatten per-run [(request, k0, k1)] segment lists into the int32 list
    format, giving split requests consecutive request-major partial slots in
    key order.  record(r, k0, k1, slot) and request(r, first, count) give the
    8 and 4 ints of a segment and a request.  loose: segments of no run, after
    the runs' records.  Returns (list, segment count, run count)."""
    loose = list(loose)
    keyed = [[] for _ in range(n)]               # first keys of each request's segments
    for run in [*per_run, loose]:
        for r, k0, _ in run:
            keyed[r].append(k0)
    first, slot, rank = [], 0, {}
    for r, keys in enumerate(keyed):
        if len(keys) <= 1:
            first.append(-1)
            continue
        # partial slot of a segment = first slot of its request + its key-order rank
        first.append(slot)
        rank[r] = {k0: slot + i for i, k0 in enumerate(sorted(keys))}
        slot += len(keys)
    out, ranges = [], [0]
    for run in per_run:
        for r, k0, k1 in run:
            out += record(r, k0, k1, rank[r][k0] if first[r] >= 0 else -1)
        ranges.append(ranges[-1] + len(run))
    for r, k0, k1 in loose:
        out += record(r, k0, k1, rank[r][k0] if first[r] >= 0 else -1)
    out += ranges
    for r in range(n):
        out += request(r, max(first[r], 0), len(keyed[r]))
    return out, ranges[-1] + len(loose), len(per_run)


def _segment_list(query_lengths, key_lengths, starts, per_run, loose=()):
    """Varlen/verify records: request, k0, k1, slot, first query row, query
    length, key length, start; request records: first slot, count, first
    query row, query length."""
    q0, acc = [], 0
    for q in query_lengths:
        q0.append(acc)
        acc += int(q)
    return _flatten(len(key_lengths), per_run,
                    lambda r, k0, k1, slot: (r, k0, k1, slot, q0[r], int(query_lengths[r]), int(key_lengths[r]),
                                             int(starts[r])),
                    lambda r, first, count: (first, count, q0[r], int(query_lengths[r])), loose)


def _balanced_runs(key_lengths, groups, tile, seg_cost=0, weights=None, shares=None):
    """Per-run [(request, k0, k1)] lists: the keys of all requests end to end,
    cut into `groups` runs of (nearly) equal cost, each cut moved down to a
    `tile` boundary of the request holding it.  A request costs seg_cost
    (the fixed work of starting a segment, in keys) plus its keys, each
    weighted by weights[r] (default 1), so runs that hold more request
    starts or heavier keys get fewer keys.  shares (one positive number per
    run) makes run w's cost proportional to shares[w] instead of equal."""
    n = len(key_lengths)
    groups = max(1, int(groups))
    if shares is None:
        bound = [w / groups for w in range(groups + 1)]
    else:
        if len(shares) != groups or min(shares) <= 0:
            raise ValueError('shares must give one positive number per run')
        bound, acc, tot = [0.0], 0.0, float(sum(shares))
        for x in shares:
            acc += float(x)
            bound.append(acc / tot)
    seg_cost = max(0.0, float(seg_cost))
    wt = [1.0] * n if weights is None else [max(1e-3, float(x)) for x in weights]
    begin, vbegin, total, vtotal = [], [], 0, 0.0
    for k, w in zip(key_lengths, wt):
        begin.append(total)
        vbegin.append(vtotal)
        total += int(k)
        vtotal += seg_cost + w * int(k)
    cuts, r, last = [0], 0, 0
    for w in range(1, groups):
        x = bound[w] * vtotal                         # cut in cost space
        while r + 1 < n and vbegin[r + 1] <= x:
            r += 1
        into = int((x - vbegin[r] - seg_cost) / wt[r])             # keys of request r before the cut
        at = begin[r] + (min(into, int(key_lengths[r])) // tile * tile if into > 0 else 0)
        if at > last:
            last = at
        cuts.append(last)
    cuts.append(total)
    per_run = [[] for _ in range(groups)]
    w = 0
    for r in range(n):
        a, kl = begin[r], int(key_lengths[r])
        while w + 1 < groups and cuts[w + 1] <= a:   # the run holding key position a
            w += 1
        if kl == 0:
            per_run[w].append((r, 0, 0))
            continue
        v, lo, end = w, a, a + kl
        while True:
            cut = cuts[v + 1]
            hi = cut if cut < end else end
            if hi > lo:
                per_run[v].append((r, lo - a, hi - a))
                lo = hi
            if cut >= end or v + 1 == groups:
                break
            v += 1
    return per_run


def xcd_shares(groups, xcd_speed):
    """Cost share of each of `groups` runs: the speed of the XCD it runs on
    (run w on XCD w mod XCDS), or None for equal runs."""
    if xcd_speed is None:
        return None
    speed = [float(x) for x in xcd_speed]
    if len(speed) != XCDS or min(speed) <= 0:
        raise ValueError(f'xcd_speed must give {XCDS} positive relative speeds')
    return [speed[w % XCDS] for w in range(int(groups))]


def second_slot_runs(groups, n_cu):
    """Runs whose workgroups are the second resident on their CUs, or an
    empty set.  Run w's workgroups are blockIdx.x = 8 (8 (w / 8) + g) + w mod
    8 (g = KV head); the dispatcher deals ids 0 .. n_cu - 1 one per CU first,
    so with exactly RESIDENT_PER_CU = 2 workgroups per CU (8 groups = 2 n_cu)
    and n_cu a multiple of 64 the runs w >= n_cu / 8 are the second ones.
    Any other launch shape gets no distinction."""
    groups = int(groups)
    if n_cu is None or int(n_cu) % 64 or 8 * groups != RESIDENT_PER_CU * int(n_cu):
        return frozenset()
    return frozenset(range(int(n_cu) // 8, groups))


def run_shares(groups, xcd_speed=None, n_cu=None):
    """Cost share of each of `groups` runs: its XCD's speed (xcd_shares;
    equal without xcd_speed), times SECOND_SLOT_SHARE for the runs of
    second_slot_runs(groups, n_cu); None when every share is equal."""
    shares = xcd_shares(groups, xcd_speed)
    second = second_slot_runs(groups, n_cu)
    if not second:
        return shares
    shares = shares or [1.0] * int(groups)
    return [x * (SECOND_SLOT_SHARE if w in second else 1.0) for w, x in enumerate(shares)]


def varlen_work(query_lengths, key_lengths, starts, groups, seg_cost=None, xcd_speed=None, n_cu=None):
    """Balanced plan: (flat int32 list, segment count, run count) for varlen (starts =
    first key row of each request) or verify (starts = resident slot of each
    request); groups = number of runs (workgroups per KV head); seg_cost
    (default SEGMENT_COST) the fixed cost of a segment in keys; xcd_speed
    (8 relative speeds) weights each run by the speed of its XCD; n_cu (the
    device's CU count) gives the second resident workgroups of each CU
    SECOND_SLOT_SHARE of a run's cost (run_shares).  The cut points depend
    on every request's length (and on xcd_speed), so a request's output can
    differ in the last bits between batches; request_work keeps them
    apart."""
    cost = SEGMENT_COST if seg_cost is None else seg_cost
    decode = [r for r, q in enumerate(query_lengths) if q <= DECODE_TOKENS]
    if len(decode) == len(key_lengths):
        runs, loose = _balanced_runs(key_lengths, groups, TILE, cost, shares=run_shares(groups, xcd_speed, n_cu)), ()
    else:
        # each cut of a prompt takes a run's cut from the others, so the segments
        # stay within varlen_list_bound; the others keep at least half of the runs
        loose = prompt_segments(query_lengths, key_lengths, (groups - 1) // 2 if decode else groups - 1, n_cu)
        n = groups - (len(loose) - (len(key_lengths) - len(decode)))
        runs = _decode_runs(decode, key_lengths, n, cost, xcd_speed, n_cu) + [[] for _ in range(groups - n)]
    return _segment_list(query_lengths, key_lengths, starts, runs, loose)


def _decode_runs(decode, key_lengths, groups, cost, xcd_speed, n_cu):
    """Balanced runs of the requests `decode` of a batch."""
    if not decode:
        return [[] for _ in range(groups)]
    return [[(decode[r], k0, k1) for r, k0, k1 in run]
            for run in _balanced_runs([key_lengths[r] for r in decode], groups, TILE, cost,
                                      shares=run_shares(groups, xcd_speed, n_cu))]


def prompt_segments(query_lengths, key_lengths, cuts, n_cu=None, pool=None):
    """[(request, k0, k1)] of the requests with more than DECODE_TOKENS query
    tokens, longest last: one segment each, so that nothing is merged, unless
    their (32-token tile, KV head) workgroups leave CUs idle over long keys (a
    later chunk of a prompt).  Then the request with the longest segments is cut
    once more, into equal parts of whole ring stages, while every part keeps
    MIN_PROMPT_SEGMENT keys, the workgroups fit two per CU, at most `cuts` cuts
    are made and the cut requests' segments fit `pool` partial tiles of 8 tokens."""
    prompts = [r for r, q in enumerate(query_lengths) if q > DECODE_TOKENS]
    tiles = {r: -(-int(query_lengths[r]) // PROMPT_TOKENS) for r in prompts}
    parts = dict.fromkeys(prompts, 1)
    per_head = int(n_cu or 256) // 8             # CUs per KV head
    used = sum(tiles.values())
    while prompts and cuts > 0:
        r = max(prompts, key=lambda x: key_lengths[x] / parts[x])
        need = -(-int(query_lengths[r]) // DECODE_TOKENS) * (2 if parts[r] == 1 else 1)
        used += tiles[r]
        least = MIN_PROMPT_SEGMENT if used <= per_head else SHARED_PROMPT_SEGMENT
        if (parts[r] == MAX_PROMPT_SEGMENTS or used > RESIDENT_PER_CU * per_head or pool is not None and need > pool
                or key_lengths[r] < least * (parts[r] + 1)):
            break
        parts[r], pool, cuts = parts[r] + 1, None if pool is None else pool - need, cuts - 1
    out = []
    for r in sorted(prompts, key=lambda x: key_lengths[x]):
        kl = int(key_lengths[r])
        at = [i * kl // parts[r] // DRAFT_TILE * DRAFT_TILE for i in range(parts[r])] + [kl]
        out += [(r, a, b) for a, b in zip(at, at[1:])]
    return out


def request_work(query_lengths, key_lengths, starts, chunk, groups):
    """Request-local plan: every request is cut at multiples of `chunk` of
    its own keys (at least one segment), so its output never depends on the
    other requests of the batch.  Segments go to the least-loaded of `groups`
    runs, longest first."""
    import heapq
    segs = []
    for r, kl in enumerate(key_lengths):
        kl = int(kl)
        for c in range(n_chunks(kl, chunk)):
            k0 = c * chunk
            segs.append((min(chunk, kl - k0) if kl > 0 else 0, r, k0, min(kl, k0 + chunk)))
    segs.sort(key=lambda x: (-x[0], x[1], x[2]))
    groups = -(-max(1, min(int(groups), len(segs))) // XCDS) * XCDS     # whole rounds over the XCDs
    heap = [(0, w) for w in range(groups)]
    per_run = [[] for _ in range(groups)]
    loose = [(r, k0, k1) for _, r, k0, k1 in reversed(segs) if query_lengths[r] > DECODE_TOKENS]
    for size, r, k0, k1 in segs:
        if query_lengths[r] > DECODE_TOKENS:
            continue
        load, w = heapq.heappop(heap)
        per_run[w].append((r, k0, k1))
        heapq.heappush(heap, (load + size + TILE, w))
    return _segment_list(query_lengths, key_lengths, starts, per_run, loose)


def varlen_list_bound(n_req, groups, rows_bound=0, chunk=None):
    """Most segment records a list over n_req requests holding at most
    rows_bound keys can have: n_req + groups - 1 for a balanced plan (each
    interior cut splits at most one request), ceil(rows_bound / chunk) +
    n_req for a request-local plan."""
    if chunk is None:
        return int(n_req) + int(groups) - 1
    return chunk_bound(n_req, rows_bound, chunk)


SPLITS = ('balanced', 'request')


def segment_plan(split, query_lengths, key_lengths, starts, groups, chunk, capacity=None, xcd_speed=None,
                 n_cu=None):
    """(flat int32 list, segment count, run count) of the named plan; the
    launch must pass the returned counts (n_work, n_groups).  xcd_speed,
    n_cu: see varlen_work (balanced plans only).

    capacity = (segments, runs) lays the list out in regions of fixed size:
    the records padded to `segments`, the run ranges to `runs` (trailing runs
    empty).  Every transaction of a bucket then launches with the same
    arguments and grid, which a captured graph replays."""
    if split == 'balanced':
        out, n_seg, runs = varlen_work(query_lengths, key_lengths, starts, groups, xcd_speed=xcd_speed, n_cu=n_cu)
    elif split == 'request':
        out, n_seg, runs = request_work(query_lengths, key_lengths, starts, chunk, groups)
    else:
        raise ValueError(f'split must be one of {SPLITS}')
    if capacity is None:
        return out, n_seg, runs
    seg_cap, run_cap = capacity
    if n_seg > seg_cap or runs > run_cap:
        raise ValueError('Segment plan exceeds its fixed capacity')
    base = WORK_INTS * n_seg
    ranges = out[base:base + runs + 1]
    padded = out[:base] + [0] * (WORK_INTS * (seg_cap - n_seg)) + ranges + [ranges[-1]] * (run_cap - runs)
    return padded + out[base + runs + 1:], seg_cap, run_cap


def _tile_count(n_req):
    """Most row tiles that mixed plans add to a batch's requests."""
    return min(n_req * (TILED_TOKENS // DECODE_TOKENS - 1), MAX_TILES)      # MAX_TILES from 6 requests on


def mixed_ints(c):
    """int32 length of a mixed list of capacity c."""
    return WORK_INTS * (c.run_records + c.prompt_records) + c.runs + 1 + REQ_INTS * c.requests + 2 * c.columns


@functools.lru_cache(maxsize=1024)
def mixed_capacity(n_req, query_tokens, key_capacity, max_q, n_cu, limit=None, short=True):
    """The regions of a fixed-capacity mixed list (MixedCapacity) for n_req
    requests of query_tokens query tokens in all, at most max_q > DECODE_TOKENS
    each (short: some may have up to TILED_TOKENS), and key_capacity keys in
    all; limit: the workspace's partial tiles.  List and partials take no more
    bytes than one balanced list of the whole batch would (a record per
    request and run, each of the longest request's tiles): a bucket's workspace
    then fits the memory budget it always did."""
    slots = max(XCDS, RESIDENT_PER_CU * n_cu // 8 // XCDS * XCDS)
    units = n_req + _tile_count(n_req) if short else 0
    runs = slots if short else XCDS
    longest = -(-max_q // DECODE_TOKENS)
    one_list = run_count(key_capacity, n_cu, longest)
    records = n_req + one_list - 1
    # what plans use at most: a tile per segment of the runs, and four per 32-token
    # workgroup of the prompts, which are cut only while all fit the CUs at once
    tiles = units + runs - 1 + PROMPT_TOKENS // DECODE_TOKENS * slots
    c = MixedCapacity(units + runs - 1, n_req + slots - 1, runs, max(units, n_req),
                      max(slots, query_tokens // PROMPT_TOKENS + n_req), 0)
    grown = 4 * (mixed_ints(c) - (WORK_INTS * records + one_list + 1 + REQ_INTS * n_req))
    tiles = min(tiles, records * longest - -(-grown // PART_TILE_BYTES))
    return c._replace(tiles=tiles if limit is None else min(tiles, limit))


def _tiled_requests(query_lengths, key_lengths, n_cu):
    """Prompts attended as tiles of DECODE_TOKENS in the runs: those of up to
    TILED_TOKENS, if all of their tiles' keys leave each workgroup slot few."""
    some = [r for r, q in enumerate(query_lengths) if DECODE_TOKENS < q <= TILED_TOKENS]
    tiles = [-(-query_lengths[r] // DECODE_TOKENS) for r in some]
    fits = (sum(tiles) - len(some) <= MAX_TILES
            and sum(t * key_lengths[r] for t, r in zip(tiles, some)) <= TILED_KEYS * RESIDENT_PER_CU * n_cu // 8)
    return some if fits else ()


def _tile_runs(units, columns):
    """Runs of row tiles alone (units as in _mixed_plan): a request's tiles are cut
    at the same keys into equal parts, 8 for every 8 MIN_SEGMENT keys while a part
    keeps two TILE, at most `columns` segments in all, a run each (a balanced cut would
    give most runs the end of one tile and the start of another, two segments'
    fixed work).  The tiles of a part are neighbours on one XCD, whose L2 they
    share."""
    share = max(1, columns // len(units))
    share = share // XCDS * XCDS or share
    tiles, segs = {}, []
    for u, unit in enumerate(units):
        tiles.setdefault(unit[0] & 0xffffff, []).append((u, unit[3]))
    for group in tiles.values():
        longest = max(k for _, k in group)
        parts = min(share, -(-longest // (XCDS * MIN_SEGMENT)) * XCDS, -(-longest // (2 * TILE)))
        at = [i * longest // parts // TILE * TILE for i in range(parts)] + [longest]
        for lo, hi in zip(at, at[1:]):
            segs += [(u, lo, min(hi, k)) for u, k in group if k > lo]
    depth = -(-len(segs) // XCDS)
    queues = [segs[x * depth:(x + 1) * depth] for x in range(XCDS)]
    rounds = min(columns // XCDS, depth)
    return [queues[x][j::rounds] for j in range(rounds) for x in range(XCDS)]


def mixed_plan(query_lengths, key_lengths, starts, n_cu, *, causal=True, capacity=None, xcd_speed=None,
               slot_balance=True):
    """Balanced plan of a batch that holds prompts (requests of more than
    DECODE_TOKENS query tokens), as dspark_mixed_attn_fwd takes it: MixedPlan(list,
    records, runs, request records, prompt columns, partial tiles).  The
    requests of up to DECODE_TOKENS are cut into runs by their own keys, as without
    prompts, with the tiles of _tiled_requests among them; other prompts are cut by
    prompt_segments.  capacity (mixed_capacity's) lays the list out in regions
    of fixed size, with counts that every transaction shares."""
    batch = (query_lengths, key_lengths, starts, n_cu, causal, capacity, xcd_speed, slot_balance)
    tiled = _tiled_requests(query_lengths, key_lengths, n_cu)
    plan = _mixed_plan(tiled, *batch)
    if plan is None and tiled:           # the capacity has too few partial tiles for row tiles
        plan = _mixed_plan((), *batch)
    if plan is None:
        raise ValueError('Segment plan exceeds its fixed capacity')
    return plan


def _mixed_plan(tiled, query_lengths, key_lengths, starts, n_cu, causal, capacity, xcd_speed, slot_balance):
    units, prompts, q0 = [], [], 0                # (first word, first query row, query length, key length, start)
    for r, (q, k) in enumerate(zip(query_lengths, key_lengths)):
        if q > DECODE_TOKENS and r not in tiled:
            prompts.append((r, q0, q, k, starts[r]))
        elif q <= DECODE_TOKENS:
            units.append((r, q0, q, k, starts[r]))
        else:
            for t in range(-(-q // DECODE_TOKENS)):
                row = DECODE_TOKENS * t
                n = min(DECODE_TOKENS, q - row)
                units.append((r | t << 24, q0 + row, n, k - q + row + n if causal else k, starts[r]))
        q0 += q
    per_head = max(XCDS, n_cu // 8 // XCDS * XCDS)                # CUs per KV head
    cuts, pool = RESIDENT_PER_CU * n_cu, None
    if capacity is not None:
        cuts, pool = capacity.prompt_records - len(prompts), capacity.tiles
        if prompts and units:                     # half each, and enough for 8 runs
            pool = max(pool // 2, min(len(units) + XCDS - 1, 2 * (XCDS - 1)))
    keys = [u[3] for u in units]
    if not units:
        per_run = [[] for _ in range(XCDS)]
    elif len(units) == sum(-(-query_lengths[r] // DECODE_TOKENS) for r in tiled):
        columns = per_head if prompts else RESIDENT_PER_CU * per_head
        per_run = _tile_runs(units, columns if pool is None else min(columns, max(XCDS, pool // XCDS * XCDS)))
    else:
        # At most one workgroup per CU: the other slot is the prompts'.  63 requests of
        # 7 tokens (157,000 keys) beside 64 tokens over 8,000 keys, 16 / 24 / 32 / 48
        # / 64 runs: 168, 138, 131, 139, 136 us; beside 4 prompts of 1,500
        # 184, 157, 169, 172, 181; alone 159, 123, 116, 127, 118.  And runs of twice
        # MIN_SEGMENT beside prompts: 6 requests with 4,700 keys beside 300 and 800
        # tokens, 8 / 16 / 24 / 32 runs: 24.9, 23.8, 24.3, 26.3.
        groups = min(run_count(sum(keys) // (2 if prompts else 1), n_cu), per_head)
        while pool is not None and groups > XCDS and min(len(units) + groups - 1, 2 * (groups - 1)) > pool:
            groups -= XCDS
        per_run = _balanced_runs(keys, groups, TILE, SEGMENT_COST,
                                 shares=run_shares(groups, xcd_speed, n_cu if slot_balance else None))
    spare = None
    if capacity is not None:
        held = {}
        for run in per_run:
            for u, _, _ in run:
                held[u] = held.get(u, 0) + 1
        spare = capacity.tiles - sum(c for c in held.values() if c > 1)
        if spare < 0:
            return None
    loose = prompt_segments([u[2] for u in prompts], [u[3] for u in prompts], cuts, n_cu, spare)
    n, every = len(units), units + prompts
    segs = [x for run in per_run for x in run] + [(n + p, k0, k1) for p, k0, k1 in loose]
    count = [0] * len(every)
    for u, _, _ in segs:
        count[u] += 1
    width, first_slot, tiles = [-(-u[2] // DECODE_TOKENS) for u in every], [], 0
    for c, w in zip(count, width):
        first_slot.append(tiles if c > 1 else -1)
        tiles += c * w if c > 1 else 0
    out, requests, ranges, nxt = [], [], [0], list(first_slot)
    if tiled:                            # a request's slots in key order, which balanced runs and prompts have
        slot = {}
        for seg in sorted(segs):
            slot[seg] = nxt[seg[0]]
            nxt[seg[0]] += width[seg[0]]
    for seg in segs:
        u, k0, k1 = seg
        word, row, q, k, start = every[u]
        if first_slot[u] < 0:
            out += (word, k0, k1, -1, row, q, k, start)
        elif tiled:
            out += (word, k0, k1, slot[seg], row, q, k, start)
        else:
            out += (word, k0, k1, nxt[u], row, q, k, start)
            nxt[u] += width[u]
    for (_, row, q, _, _), f, c in zip(every, first_slot, count):
        requests += (f if c > 1 else 0, c, row, q)
    for run in per_run:
        ranges.append(ranges[-1] + len(run))
    groups, first = len(per_run), ranges[-1]
    columns = _prompt_columns(prompts, loose, first if capacity is None else capacity.run_records, causal)
    if capacity is None:
        return MixedPlan(out + ranges + requests + columns, len(segs), groups, len(every), len(columns) // 2, tiles)
    c = capacity
    if (first > c.run_records or len(loose) > c.prompt_records or groups > c.runs or len(every) > c.requests
            or len(columns) > 2 * c.columns):
        return None
    cut, n_work = WORK_INTS * first, c.run_records + c.prompt_records
    padded = np.zeros(mixed_ints(c), dtype=np.int32)
    after = WORK_INTS * n_work + c.runs + 1
    for at, part in ((0, out[:cut]), (WORK_INTS * c.run_records, out[cut:]),
                     (WORK_INTS * n_work, ranges + [first] * (c.runs - groups)), (after, requests),
                     (after + REQ_INTS * c.requests, columns)):
        padded[at:at + len(part)] = part
    return MixedPlan(padded, n_work, c.runs, c.requests, c.columns, c.tiles)


def _prompt_columns(prompts, loose, first, causal):
    """(1 + record, tile) of every 32-token tile of the prompts' segments, the
    records counted from `first`, most keys first."""
    out = []
    for i, (p, k0, k1) in enumerate(loose, 1 + first):
        _, _, q, k, _ = prompts[p]
        seen = k - q + PROMPT_TOKENS if causal else k            # keys up to the first tile's last token
        out += [(k0 - min(k1, seen + PROMPT_TOKENS * t), i, t) for t in range(-(-q // PROMPT_TOKENS))]
    out.sort()
    return [x for column in out for x in column[1:]]


def draft_work(context_lengths, cu_blocks, anchors, groups=None, *, chunk=None, offsets=None):
    """Draft plan: (flat int32 list, segment count, run count).  Request r
    streams its context up to its largest anchor (the rows any of its blocks
    sees), and the segment ending a request also attends its blocks' own rows.
      * chunk given (the default plan): every request is cut at multiples of
        `chunk` of its own rows, one segment per run (workgroup), longest
        first, so the hardware dispatcher balances the ragged tail (each
        workgroup's 128 KiB ring fills a CU's LDS, one resident per CU);
      * else: the rows of all requests, end to end, are cut into `groups` runs
        of equal cost at DRAFT_TILE boundaries: a request costs
        DRAFT_SEGMENT_COST plus its rows weighted by 1 + DRAFT_BLOCK_WEIGHT
        per block beyond the first (more blocks, more MFMA and LDS work per
        row).

      segment: request, k0, k1, partial slot (-1: one segment), first block,
               block count, largest anchor, 1 + offsets[r] (0 without
               offsets, or when it does not fit in 31 bits: the kernel then
               reads ctx_off[r] itself)
      request: first partial slot, segment count, first block, block count
    """
    amax = [max(anchors[cu_blocks[r]:cu_blocks[r + 1]]) for r in range(len(context_lengths))]
    off1 = [0] * len(amax) if offsets is None else [int(o) + 1 if 0 <= int(o) < 2 ** 31 - 1 else 0 for o in offsets]
    if any(not 0 <= a <= int(c) for a, c in zip(amax, context_lengths)):
        raise ValueError('Anchors must lie in [0, context length]')
    if chunk is not None:
        # One segment per run: the partial slots follow from the chunk numbers,
        # so the list is written out directly (64 requests in 290 us of host time
        # against _flatten's 470, before every round's first draft launch).
        segs, requests, slots = [], [], 0
        for r, n in enumerate(amax):
            count = n_chunks(n, chunk)
            tail = (cu_blocks[r], cu_blocks[r + 1] - cu_blocks[r])
            first = slots if count > 1 else -1
            for c in range(count):
                k0 = c * chunk
                k1 = min(n, k0 + chunk)
                segs.append((k0 - k1, r, k0, k1, first + c if count > 1 else -1, *tail, n, off1[r]))
            slots += count if count > 1 else 0
            requests += (max(first, 0), count, *tail)
        segs.sort()                                  # longest first; then request and k0, which are distinct
        out = [x for s in segs for x in s[1:]]
        return out + list(range(len(segs) + 1)) + requests, len(segs), len(segs)
    nb = [cu_blocks[r + 1] - cu_blocks[r] for r in range(len(amax))]
    per_run = _balanced_runs(amax, groups, DRAFT_TILE, DRAFT_SEGMENT_COST,
                             [1.0 + DRAFT_BLOCK_WEIGHT * (b - 1) for b in nb])
    return _flatten(len(amax), per_run,
                    lambda r, k0, k1, slot: (r, k0, k1, slot, cu_blocks[r], cu_blocks[r + 1] - cu_blocks[r], amax[r],
                                             off1[r]),
                    lambda r, first, count: (first, count, cu_blocks[r], cu_blocks[r + 1] - cu_blocks[r]))


def draft_chunk_for(visible_rows, n_cu):
    """Fixed draft chunk sized to a batch: its visible context rows (each
    request's largest anchor, summed) cut into about one (chunk, KV head)
    item per CU, in multiples of DRAFT_TILE rows, between MIN_DRAFT_CHUNK
    and DRAFT_CHUNK.  A batch that fills the CUs at DRAFT_CHUNK keeps it; a
    small one is cut finer, so that its few requests still spread over every
    CU (at the price of split-K partials and their merge)."""
    per_head = max(1, int(n_cu) // 8)
    rows = -(-max(1, int(visible_rows)) // per_head)
    rows = -(-rows // DRAFT_TILE) * DRAFT_TILE
    return max(MIN_DRAFT_CHUNK, min(DRAFT_CHUNK, rows))


def draft_run_count(total_rows, n_cu):
    """Draft runs per KV head: one workgroup per CU (its 128 KiB ring fills
    the CU's LDS), never fewer than MIN_DRAFT_SEGMENT rows per run."""
    return max(1, min(max(1, int(n_cu) // 8), -(-int(total_rows) // MIN_DRAFT_SEGMENT)))


def upload_work(records, device):
    """int32 device copy of a work list via the pinned staging ring."""
    return upload(device, records)

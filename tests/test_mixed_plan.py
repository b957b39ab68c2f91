"""Plans of batches that hold prompts (schedule.mixed_plan): the kernels trust
these lists, so every row tile's keys are covered exactly once, the merge
records name the slots that the segments write, and the fixed-capacity form
always fits its regions, which take no more memory than one balanced list of
the batch.  And what such a plan must not lose: a prompt leaves the decoding
requests their workgroups, and a few query tokens over a long context are
spread over the CUs."""
import numpy as np
import pytest

from qwen3_dspark_amd.schedule import (DECODE_TOKENS, PART_TILE_BYTES, REQ_INTS, WORK_INTS, mixed_capacity,
                                       mixed_ints, mixed_plan, run_count)

N_CU = 256


def read(plan):
    n, ints = plan.n_work, [int(x) for x in plan.records]
    rec = [ints[WORK_INTS * i:WORK_INTS * (i + 1)] for i in range(n)]
    ranges = ints[WORK_INTS * n:WORK_INTS * n + plan.runs + 1]
    rest = ints[WORK_INTS * n + plan.runs + 1:]
    reqs = [rest[REQ_INTS * i:REQ_INTS * (i + 1)] for i in range(plan.requests)]
    columns = rest[REQ_INTS * plan.requests:]
    assert len(columns) == 2 * plan.columns and plan.runs % 8 == 0
    return rec, ranges, reqs, [(a - 1, t) for a, t in zip(columns[::2], columns[1::2]) if a]


def check(ql, kl, starts, plan, causal=True):
    """The list against the batch; returns the columns (workgroups per KV head)
    of the decoding requests and of each prompt."""
    rec, ranges, reqs, columns = read(plan)
    assert ranges[0] == 0 and sorted(ranges) == ranges
    q0 = np.concatenate([[0], np.cumsum(ql)])
    assert sorted(columns) == [(i, t) for i in range(ranges[-1], len(rec)) for t in range(-(-rec[i][5] // 32))]
    rows = {}                                  # (first row, rows) -> segments
    for i, (w0, k0, k1, slot, first_row, n, keys, start) in enumerate(rec):
        if n == 0:
            continue
        r, t = w0 & 0xffffff, w0 >> 24
        assert start == starts[r] and first_row == q0[r] + DECODE_TOKENS * t
        if i >= ranges[-1]:
            assert t == 0 and n == ql[r] > DECODE_TOKENS and keys == kl[r]
        else:
            assert n == min(DECODE_TOKENS, ql[r] - DECODE_TOKENS * t)
            assert keys == (kl[r] - ql[r] + DECODE_TOKENS * t + n if causal else kl[r])
        rows.setdefault((first_row, n), []).append((k0, k1, slot, keys, i))
    assert sorted(x for a, n in rows for x in range(a, a + n)) == list(range(q0[-1]))
    merged = {(m[2], m[3]): m for m in reqs if m[3]}
    assert sorted(merged) == sorted(rows)
    used = []
    for key, segs in rows.items():
        segs.sort()
        assert segs[0][0] == 0 and segs[-1][1] == segs[0][3]
        assert all(a[1] == b[0] and a[1] % 32 == 0 for a, b in zip(segs, segs[1:]))
        first, count = merged[key][:2]
        assert count == len(segs)
        slots, tiles = [s[2] for s in segs], -(-key[1] // 8)
        assert slots == ([-1] if count == 1 else [first + tiles * i for i in range(count)])
        if count > 1:
            used += range(first, first + tiles * count)
    assert len(set(used)) == len(used) and all(0 <= x < plan.tiles for x in used)
    busy = sum(b > a for a, b in zip(ranges, ranges[1:]))
    prompts = {a: len(s) * -(-n // 32) for (a, n), s in rows.items() if n > DECODE_TOKENS}
    return busy, prompts


def one_list_bytes(n, keys, max_q):
    """What one balanced list over the whole batch reserves."""
    tiles = -(-max_q // 8)
    runs = run_count(keys, N_CU, tiles)
    records = n + runs - 1
    return 4 * (WORK_INTS * records + runs + 1 + REQ_INTS * n) + PART_TILE_BYTES * records * tiles


def capacity_bytes(c):
    return 4 * mixed_ints(c) + PART_TILE_BYTES * c.tiles


BATCHES = [([9], [9]), ([9], [709]), ([64], [2064]), ([96], [396]), ([97], [1000]), ([16, 9, 33], [16, 4000, 40]),
           ([7] * 4 + [9], [2000, 300, 7, 5000, 8009]), ([7, 1, 8, 64], [100, 9, 8, 900]), ([20] * 40, [200] * 40),
           ([300], [4000]), ([7] * 63 + [1000], [8000] * 63 + [1000]), ([9, 1000, 7], [8009, 1000, 700]),
           ([1024] * 16, [1024] * 16), ([9] * 4096, [9] * 4096), ([16] * 8, [4096] * 8), ([7] * 3, [900, 20, 7])]


@pytest.mark.parametrize('ql,kl', BATCHES)
@pytest.mark.parametrize('causal', [True, False])
def test_every_key_once(ql, kl, causal):
    starts = [3 * i for i in range(len(ql))]
    check(ql, kl, starts, mixed_plan(ql, kl, starts, N_CU, causal=causal), causal)


@pytest.mark.parametrize('ql,kl', BATCHES)
def test_fixed_capacity(ql, kl):
    """Every batch of a bucket fits its regions, whose sizes depend on the bucket
    alone and take no more bytes than one list did."""
    rng = np.random.default_rng(len(ql) + sum(kl))
    n, keys, max_q = len(ql), sum(kl), max(max(ql), DECODE_TOKENS + 1)
    cap = mixed_capacity(n, sum(ql), keys, max_q, N_CU)
    assert capacity_bytes(cap) <= one_list_bytes(n, keys, max_q)
    starts = list(range(n))
    counts = None
    for _ in range(6 if n < 100 else 1):
        plan = mixed_plan(ql, kl, starts, N_CU, capacity=cap)
        check(ql, kl, starts, plan)
        assert counts in (None, plan[1:])
        counts = plan[1:]
        assert counts == (cap.run_records + cap.prompt_records, cap.runs, cap.requests, cap.columns, cap.tiles)
        ql = [int(rng.integers(1, q + 1)) for q in ql]
        kl = [q + int(rng.integers(0, k - q + 1)) for q, k in zip(ql, kl)]


def test_random_buckets_fit():
    rng = np.random.default_rng(3)
    for _ in range(400):
        n = int(rng.choice([1, 1, 2, 3, 8, 20, 64]))
        max_q = int(np.exp(rng.uniform(np.log(9), np.log(2000))))
        ql = [int(np.exp(rng.uniform(0, np.log(max_q + .99)))) for _ in range(n)]
        kl = [q + int(np.exp(rng.uniform(0, np.log(9000)))) - 1 for q in ql]
        bound = sum(kl) + int(rng.integers(0, 5000))
        cap = mixed_capacity(n, sum(ql), bound, max_q, N_CU)
        if min(ql) > 96:
            exact = mixed_capacity(n, sum(ql), bound, max_q, N_CU, None, False)
            check(ql, kl, list(range(n)), mixed_plan(ql, kl, list(range(n)), N_CU, capacity=exact))
        assert capacity_bytes(cap) <= one_list_bytes(n, bound, max_q)
        check(ql, kl, list(range(n)), mixed_plan(ql, kl, list(range(n)), N_CU, capacity=cap))
        # a family of an arena whose partials are as many as its own shape would have
        again = mixed_capacity(n, sum(ql), bound, max_q, N_CU, cap.tiles)
        assert again == cap


@pytest.mark.parametrize('tokens', [9, 64, 300, 1000])
@pytest.mark.parametrize('fixed', [False, True])
def test_a_chunk_leaves_the_decoding_requests_their_workgroups(tokens, fixed):
    """63 requests of 7 tokens over 8,000 keys keep a workgroup per CU beside a
    chunk of a prompt, whatever its length."""
    ql, kl = [7] * 63 + [tokens], [8000] * 63 + [8000 + tokens]
    cap = mixed_capacity(64, sum(ql), sum(kl), tokens, N_CU) if fixed else None
    busy, _ = check(ql, kl, list(range(64)), mixed_plan(ql, kl, list(range(64)), N_CU, capacity=cap))
    assert busy * 8 >= N_CU


@pytest.mark.parametrize('tokens', [9, 16, 32, 64])
@pytest.mark.parametrize('keys', [2000, 4096, 8000])
def test_a_short_chunk_over_a_long_context_is_spread(tokens, keys):
    """At least 14 workgroups per KV head: as 8-token requests over the same keys
    have (8 to 32), where one list gave a chunk 1 to 7."""
    ql, kl = [tokens], [keys + tokens]
    for cap in (None, mixed_capacity(1, tokens, kl[0], tokens, N_CU)):
        busy, prompts = check(ql, kl, [0], mixed_plan(ql, kl, [0], N_CU, capacity=cap))
        assert (busy if not prompts else sum(prompts.values())) >= min(14, -(-keys // 256))


@pytest.mark.parametrize('split', ['balanced', 'request'])
def test_lists_of_the_families_of_one_arena(split, monkeypatch):
    """An arena takes the elementwise maximum of its families' shapes, whose lists
    have fewer runs where a request is long: every family's lists and partials
    still fit, with as many runs as a list of its own wherever those do."""
    from types import SimpleNamespace
    from qwen3_dspark_amd import kv_device as kd
    monkeypatch.setattr(kd, 'cu_count', lambda device: N_CU)
    rng = np.random.default_rng(3)
    fields = ('request_count', 'query_tokens', 'key_capacity', 'maximum_query_length')
    first = [[(4, 19, 22958, 8), (4, 78, 22958, 40)], [(3, 19, 11732, 8), (3, 40, 11732, 40)],
             [(1, 7, 16000, 7), (1, 9, 16000, 9)], [(128, 128, 1 << 20, 1), (1, 17, 17, 17)]]
    for i in range(3000):
        if i < len(first):
            arena = first[i]
        else:
            arena = []
            for _ in range(int(rng.integers(1, 4))):
                n, longest = int(rng.choice([1, 2, 3, 8, 33, 128])), int(rng.choice([1, 7, 8, 9, 17, 40, 97, 1000]))
                q = int(rng.integers(max(n, longest), n * longest + 1)) if n * longest > n + longest else n * longest
                arena.append((n, q, q + int(rng.integers(0, n * 8000)), longest))
        arena = [SimpleNamespace(**dict(zip(fields, f))) for f in arena]
        top = SimpleNamespace(**{name: max(getattr(f, name) for f in arena) for name in fields})
        mixed = kd._mixed_shape(top, None, split)
        tiles = (mixed.tiles if mixed is not None else
                 kd._list_shape(top, None, 512, split)[0] * -(-top.maximum_query_length // 8))
        ints = kd._list_ints(top, None, 512, split)
        for f in arena:
            c = kd._mixed_shape(f, None, split, tiles)
            if c is not None:
                assert mixed_ints(c) <= ints and c.tiles <= tiles
                continue
            records, runs = kd._fitting_shape(f, None, 512, split, ints, tiles)
            assert runs >= 8 and runs % 8 == 0
            size = 8 * records + runs + 1 + 4 * f.request_count
            width = -(-f.maximum_query_length // 8)
            assert size <= ints and records * width <= tiles
            own = kd._list_shape(f, None, 512, split)
            own_size = 8 * own[0] + own[1] + 1 + 4 * f.request_count
            assert (records, runs) == own or own_size > ints or own[0] * width > tiles

"""The work whose speed is measured, each case one pass through the package's
public entry points as a serving program drives them: verification rounds and
prompt prefill over the persistent KV store, packed forwards over the
append-order cache with their rollback, multi-block draft attention, draft
context appends, and the sampling law on both sides of a round.

A case is a dict of plain values.  Request lengths are drawn from its
`lengths` number, tensor values from the seed given to prepare, so one case
has the same sizes under every seed.  The attention geometry is the
package's: 16 query heads, 8 KV heads, head dim 128; hidden 1024, five draft
layers, vocabulary 151,936.
"""
import math
import random

import torch

DEV = 'cuda'
HQ, HKV, D, HIDDEN, VOCAB, BLOCK = 16, 8, 128, 1024, 151936, 7
SCALE = D ** -0.5
EPS, THETA = 1e-6, 1e6
ROW = HKV * D * 2                      # bytes of one K or V row, bf16


def listed():
    return [
        # Four users, short cached contexts: each request is admitted with its
        # prefix, verified once through all 28 layers, committed, retired.
        # Small launches: host and launch latency count.
        dict(name='verify_4_retire', kind='verify', requests=4, q_min=7, q_max=7, ctx_min=64, ctx_max=512, layers=28,
             projected=False, retire=True, lengths=1),
        # A mid-sized batch, every layer from its hidden states: q/k/v
        # projection, norm and RoPE into the scratch, then attention.
        dict(name='verify_32_projected', kind='verify', requests=32, q_min=7, q_max=7, ctx_min=256, ctx_max=2048,
             layers=28, projected=True, retire=False, lengths=2),
        # A full batch of long ragged contexts, ragged proposals, staged by the
        # attention launch (8 of the 28 layers, for memory).
        dict(name='verify_64_long', kind='verify', requests=64, q_min=1, q_max=8, ctx_min=256, ctx_max=8192, layers=8,
             projected=False, retire=False, lengths=3),
        # New prompts enter the store: one ragged prefill transaction, every
        # row committed.
        dict(name='prefill_4_prompts', kind='verify', requests=4, q_min=200, q_max=1500, ctx_min=0, ctx_max=0,
             layers=8, projected=True, retire=True, lengths=4),
        # Append-order cache: a packed forward with two new prompts among
        # requests that verify a few tokens, over four layers, then the
        # rollback of what was not accepted.
        dict(name='packed_mixed', kind='packed', decode=6, prompts=2, q_min=1, q_max=8, prompt_min=300,
             prompt_max=1000, ctx_min=100, ctx_max=1500, layers=4, lengths=5),
        # Two requests, one block each, in the autocast form (FP32 Q and K).
        dict(name='draft_2_amp', kind='draft', requests=2, blocks_min=1, blocks_max=1, ctx_min=90, ctx_max=130,
             layers=5, amp=True, indexed=False, lengths=6),
        # Sixteen requests, four blocks each.
        dict(name='draft_16', kind='draft', requests=16, blocks_min=4, blocks_max=4, ctx_min=128, ctx_max=1024,
             layers=5, amp=False, indexed=False, lengths=7),
        # A full batch, 1 to 8 blocks each, long ragged contexts.
        dict(name='draft_64_long', kind='draft', requests=64, blocks_min=1, blocks_max=8, ctx_min=256, ctx_max=8192,
             layers=5, amp=False, indexed=False, lengths=8),
        # The rows a round committed enter the draft's context.
        dict(name='append_round', kind='append', requests=64, rows_min=1, rows_max=8, ctx_min=0, ctx_max=1000,
             lengths=9),
        # Sixteen prompts enter the draft's context.
        dict(name='append_prompts', kind='append', requests=16, rows_min=128, rows_max=1024, ctx_min=0, ctx_max=0,
             lengths=10),
        # LM head and the float64 verification law of a full round.
        dict(name='speculate_64', kind='speculate', requests=64, proposed_min=7, proposed_max=7, temperature=0.8,
             lengths=11),
        # The draft's side: its laws from FP32 logits, and a draw from each.
        dict(name='laws_64', kind='laws', rows=64, dtype='float32', temperature=0.8, lengths=12),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(math.exp(rng.uniform(math.log(max(lo, 1)), math.log(hi + 1))))))


def _cost(case):
    w = work(case)
    return max(w['bytes'], w['flops'] / 50)


def draw(rng):
    limit = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(('verify', 'verify', 'prefill', 'packed', 'draft', 'draft', 'append', 'speculate', 'laws'))
        seed = rng.randrange(1 << 20)
        if kind == 'verify':
            hi = _log_int(rng, 64, 8192)
            case = dict(kind='verify', requests=_log_int(rng, 1, 64), q_min=rng.randint(1, 7),
                        q_max=rng.randint(7, 8), ctx_min=hi // rng.choice((2, 4, 32)), ctx_max=hi,
                        layers=rng.choice((4, 8, 28)), projected=rng.random() < .5, retire=False, lengths=seed)
        elif kind == 'prefill':
            hi = _log_int(rng, 9, 4096)
            cached = rng.random() < .4          # a later chunk of a prompt
            top = _log_int(rng, 64, 4096) if cached else 0
            case = dict(kind='verify', requests=_log_int(rng, 1, 16), q_min=max(1, hi // rng.choice((1, 2, 8))),
                        q_max=hi, ctx_min=top // 2, ctx_max=top, layers=rng.choice((4, 8)),
                        projected=rng.random() < .5, retire=not cached, lengths=seed)
        elif kind == 'packed':
            hi, top = _log_int(rng, 16, 2048), _log_int(rng, 64, 2048)
            case = dict(kind='packed', decode=rng.randint(1, 16), prompts=rng.randint(0, 3), q_min=1,
                        q_max=rng.randint(1, 8), prompt_min=hi // 2, prompt_max=hi, ctx_min=top // 8, ctx_max=top,
                        layers=rng.choice((2, 4)), lengths=seed)
        elif kind == 'draft':
            hi = _log_int(rng, 32, 8192)
            case = dict(kind='draft', requests=_log_int(rng, 1, 64), blocks_min=1, blocks_max=rng.randint(1, 8),
                        ctx_min=hi // rng.choice((2, 4, 32)), ctx_max=hi, layers=5, amp=rng.random() < .25,
                        indexed=rng.random() < .3, lengths=seed)
        elif kind == 'append':
            hi = _log_int(rng, 1, 1024)
            top = rng.choice((0, 1000))
            case = dict(kind='append', requests=_log_int(rng, 1, 64), rows_min=max(1, hi // 8), rows_max=hi,
                        ctx_min=0, ctx_max=top, lengths=seed)
        elif kind == 'speculate':
            hi = rng.randint(1, 8)
            case = dict(kind='speculate', requests=_log_int(rng, 1, 64), proposed_min=rng.randint(1, hi),
                        proposed_max=hi, temperature=rng.choice((0.6, 0.8, 1.0)), lengths=seed)
        else:
            case = dict(kind='laws', rows=_log_int(rng, 1, 64), dtype=rng.choice(('float32', 'bfloat16')),
                        temperature=rng.choice((0.6, 0.8, 1.0)), lengths=seed)
        if _cost(case) <= limit and _fits(case):
            return case


def _fits(case):
    """Bounds the state of a drawn case (three fit one card with room to spare)."""
    if case['kind'] == 'verify':
        rows = case['requests'] * (case['ctx_max'] + case['q_max'])
        return rows * case['layers'] <= 64 * 8200 * 8 and case['requests'] * case['q_max'] <= 16384
    if case['kind'] == 'draft':
        return case['requests'] * case['ctx_max'] <= 64 * 8192
    return True


# -- sizes of a case ----------------------------------------------------------

def _ints(rng, lo, hi, n):
    """n sizes in [lo, hi], even over their logarithm where the range spans more than a factor of ten."""
    if lo > 0 and hi > 10 * lo:
        return [_log_int(rng, lo, hi) for _ in range(n)]
    return [rng.randint(lo, hi) for _ in range(n)]


def _sizes(case):
    rng = random.Random(case['lengths'])
    kind = case['kind']
    if kind == 'verify':
        n = case['requests']
        return dict(c=_ints(rng, case['ctx_min'], case['ctx_max'], n), q=_ints(rng, case['q_min'], case['q_max'], n),
                    kept=[rng.random() for _ in range(n)])
    if kind == 'packed':
        n, p = case['decode'], case['prompts']
        decode = [min(a, 8) for a in _ints(rng, case['q_min'], case['q_max'], n)]
        return dict(c=_ints(rng, case['ctx_min'], case['ctx_max'], n) + [0] * p,
                    q=decode + _ints(rng, case['prompt_min'], case['prompt_max'], p))
    if kind == 'draft':
        c = _ints(rng, case['ctx_min'], case['ctx_max'], case['requests'])
        most = [1] * len(c) if case['indexed'] else [rng.randint(case['blocks_min'], case['blocks_max']) for _ in c]
        return dict(c=c, anchors=[[x] + [rng.randint(0, x) for _ in range(b - 1)] for x, b in zip(c, most)])
    if kind == 'append':
        n = case['requests']
        return dict(rows=_ints(rng, case['rows_min'], case['rows_max'], n),
                    c=[rng.randint(case['ctx_min'], case['ctx_max']) for _ in range(n)])
    if kind == 'speculate':
        return dict(n=[rng.randint(case['proposed_min'], case['proposed_max']) for _ in range(case['requests'])])
    return {}


def _accepted(s):
    """Rows each request of a retiring round keeps: of a prompt all, of a proposal a prefix."""
    return [q if c == 0 else int(k * (q + 1)) for c, q, k in zip(s['c'], s['q'], s['kept'])]


# -- inputs, from the seed alone ---------------------------------------------

def _rand(g, *shape, scale=1.0, dtype=torch.bfloat16):
    x = torch.empty(shape, dtype=torch.float32, device=DEV).normal_(0.0, scale, generator=g)
    return x if dtype == torch.float32 else x.to(dtype)


def _layer_weights(g):
    """One layer's q/k/v projections and q/k norms."""
    proj = [_rand(g, n * D, HIDDEN, scale=HIDDEN ** -0.5) for n in (HQ, HKV, HKV)]
    norms = [torch.empty(D, device=DEV).uniform_(0.7, 1.5, generator=g).bfloat16() for _ in range(2)]
    return (*proj, *norms)


def _inputs(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    kind, s = case['kind'], _sizes(case)
    if kind in ('verify', 'packed'):
        L, rows, cached = case['layers'], sum(s['q']), sum(s['c'])
        x = dict(ctx_k=[_rand(g, cached, HKV, D) for _ in range(L)], ctx_v=[_rand(g, cached, HKV, D) for _ in range(L)])
        if case.get('projected'):
            x.update(weights=[_layer_weights(g) for _ in range(L)], hidden=[_rand(g, rows, HIDDEN) for _ in range(L)])
        else:
            x.update(q=[_rand(g, rows, HQ, D, scale=1.5) for _ in range(L)],
                     k=[_rand(g, rows, HKV, D) for _ in range(L)], v=[_rand(g, rows, HKV, D) for _ in range(L)])
        return s, x
    if kind == 'draft':
        L, rows, cached = case['layers'], BLOCK * sum(map(len, s['anchors'])), sum(s['c'])
        qk = torch.float32 if case['amp'] else torch.bfloat16
        return s, dict(ctx_k=[_rand(g, cached, HKV, D, dtype=qk) for _ in range(L)],
                       ctx_v=[_rand(g, cached, HKV, D) for _ in range(L)],
                       q=[_rand(g, rows, HQ, D, scale=1.5, dtype=qk) for _ in range(L)],
                       k=[_rand(g, rows, HKV, D, dtype=qk) for _ in range(L)],
                       v=[_rand(g, rows, HKV, D) for _ in range(L)])
    if kind == 'append':
        features = 5 * HIDDEN
        weights = [_layer_weights(g) for _ in range(5)]
        return s, dict(fc=_rand(g, HIDDEN, features, scale=features ** -0.5),
                       norm=torch.empty(HIDDEN, device=DEV).uniform_(0.5, 1.5, generator=g).bfloat16(),
                       layers=[(w[1], w[4], w[2]) for w in weights],
                       features=[_rand(g, 1, n, features) for n in s['rows']])
    if kind == 'speculate':
        rows = sum(s['n']) + len(s['n'])
        head = _rand(g, VOCAB, HIDDEN, scale=0.06)
        hidden = _rand(g, rows, HIDDEN)
        # the draft's laws: near the target's, as a trained draft's are
        take, at = [], 0
        for n in s['n']:
            take += range(at, at + n)
            at += n + 1
        logits = hidden[take].float() @ head.float().t() + _rand(g, len(take), VOCAB, scale=0.5, dtype=torch.float32)
        laws = torch.softmax(logits.double() / case['temperature'], -1)
        del logits
        tokens = torch.empty(len(take), dtype=torch.long, device=DEV)
        for i in range(0, len(take), 64):
            tokens[i:i + 64] = torch.multinomial(laws[i:i + 64], 1, generator=g)[:, 0]
        return s, dict(head=head, hidden=hidden, laws=laws, tokens=tokens,
                       uniforms=torch.rand(rows, generator=g, device=DEV, dtype=torch.float64))
    return s, dict(logits=_rand(g, case['rows'], VOCAB, scale=2.0, dtype=getattr(torch, case['dtype'])),
                   uniforms=torch.rand(case['rows'], generator=g, device=DEV, dtype=torch.float64))



# -- prepare ------------------------------------------------------------------

def _prepare_verify(case, s, x):
    from qwen3_dspark_amd.persistent_kv import Bucket, PersistentTargetKV
    from qwen3_dspark_amd.prologue import QKVPrologue
    n = len(s['c'])
    ceiling, most = case['ctx_max'], case['q_max']
    store = PersistentTargetKV(layers=case['layers'], slots=n, context_capacity=ceiling + most,
                               max_query_tokens=sum(s['q']), heads=HKV, dim=D, device=DEV)
    bucket = Bucket(tuple(s['q']), (ceiling,) * n, 'perf case')
    store.register_bucket(bucket)
    keys = list(torch.stack(x['ctx_k']).split(s['c'], dim=1))
    values = list(torch.stack(x['ctx_v']).split(s['c'], dim=1))
    st = dict(kind='verify', store=store, bucket=bucket, layers=range(case['layers']), retire=case['retire'],
              names=[f'r{i}' for i in range(n)], accepted=_accepted(s))
    if case['projected']:
        st.update(prologues=[QKVPrologue(*w, eps=EPS, theta=THETA) for w in x['weights']], hidden=x['hidden'])
    else:
        st.update(q=x['q'], k=x['k'], v=x['v'])
    if case['retire']:
        st['prefix'] = [(k.contiguous(), v.contiguous()) if c else None for k, v, c in zip(keys, values, s['c'])]
    else:
        st['handles'] = [store.add_request(r) for r in st['names']]
        for h, k, v in zip(st['handles'], keys, values):
            if k.shape[1]:
                store.load_prefix(h, k, v)
    return st


def _prepare_packed(case, s, x):
    from qwen3_dspark_amd.kernels import HipVarlenKernel
    from qwen3_dspark_amd.packed_kv import AppendOrderKV
    kv = AppendOrderKV(layers=case['layers'], device=DEV)
    names = [f'r{i}' for i in range(len(s['c']))]
    for r in names:
        kv.add_request(r)
    rows = lambda t: t.transpose(0, 1)[None].contiguous()
    old = {r: c for r, c in zip(names, s['c']) if c}
    kv.append(old, [(rows(k), rows(v)) for k, v in zip(x['ctx_k'], x['ctx_v'])])
    return dict(kind='packed', kv=kv, kernel=HipVarlenKernel(DEV), lengths=dict(zip(names, s['c'])),
                chunks=dict(zip(names, s['q'])), q=x['q'], new=[(rows(k), rows(v)) for k, v in zip(x['k'], x['v'])])


def _prepare_draft(case, s, x):
    from qwen3_dspark_amd.draft import DraftKVPool, HipDraftAttention
    names = [f'r{i}' for i in range(len(s['c']))]
    st = dict(kind='draft', q=x['q'], k=x['k'], v=x['v'], layers=range(case['layers']))
    if case['indexed']:
        # the append-order pool [1, 8, N, 128] read through a layout's gather
        # indices: 16-row appends of the requests in turn
        order, taken = [], [0] * len(s['c'])
        while any(t < c for t, c in zip(taken, s['c'])):
            for r, c in enumerate(s['c']):
                n = min(16, c - taken[r])
                order += [(r, taken[r] + i) for i in range(n)]
                taken[r] += n
        first = [sum(s['c'][:r]) for r in range(len(s['c']))]
        at = torch.tensor([first[r] + p for r, p in order], device=DEV)
        own = [(r, c + i) for r, c in enumerate(s['c']) for i in range(BLOCK)]
        to = lambda pairs: [torch.tensor(col, dtype=torch.long, device=DEV) for col in zip(*pairs)]
        head_major = lambda t: t.transpose(0, 1)[None].contiguous()
        qr, qp = to(own)
        kr, kp = to(order + own)
        st.update(metadata=(qr, qp, kr, kp), kernel=HipDraftAttention(DEV),
                  pool=[(head_major(k[at]), head_major(v[at])) for k, v in zip(x['ctx_k'], x['ctx_v'])])
        return st
    pool = DraftKVPool(layers=case['layers'], slots=len(names), capacity=case['ctx_max'] + BLOCK, device=DEV,
                       key_dtype=torch.float32 if case['amp'] else torch.bfloat16, value_dtype=torch.bfloat16)
    for r in names:
        pool.add_request(r)
    pool.append_projected({r: c for r, c in zip(names, s['c']) if c}, list(zip(x['ctx_k'], x['ctx_v'])))
    st.update(pool=pool, anchors=dict(zip(names, s['anchors'])))
    return st


def _prepare_append(case, s, x):
    from qwen3_dspark_amd.draft import DraftKVPool
    from qwen3_dspark_amd.draft_projection import DraftContextProjector
    names = [f'r{i}' for i in range(len(s['c']))]
    projector = DraftContextProjector(x['fc'], x['norm'], x['layers'], eps=EPS, theta=THETA)
    pool = DraftKVPool(layers=5, slots=len(names), capacity=case['ctx_max'] + case['rows_max'], device=DEV,
                       projector=projector)
    for r in names:
        pool.add_request(r)
    old = {r: c for r, c in zip(names, s['c']) if c}
    if old:
        # an append never reads the rows before it: zeros, so that the
        # returned pool shows the appended rows alone
        zero = torch.zeros(sum(old.values()), HKV, D, dtype=torch.bfloat16, device=DEV)
        pool.append_projected(old, [(zero, zero)] * 5)
    return dict(kind='append', pool=pool, lengths=dict(zip(names, s['c'])), chunks=dict(zip(names, x['features'])))


def prepare(case, seed):
    s, x = _inputs(case, seed)
    kind = case['kind']
    if kind == 'verify':
        return _prepare_verify(case, s, x)
    if kind == 'packed':
        return _prepare_packed(case, s, x)
    if kind == 'draft':
        return _prepare_draft(case, s, x)
    if kind == 'append':
        return _prepare_append(case, s, x)
    if kind == 'speculate':
        from qwen3_dspark_amd.sampling import TargetHead
        return dict(kind=kind, head=TargetHead(x['head']), hidden=x['hidden'], laws=x['laws'], tokens=x['tokens'],
                    uniforms=x['uniforms'], counts=s['n'], budgets=[64] * len(s['n']), temperature=case['temperature'])
    return dict(kind=kind, logits=x['logits'], uniforms=x['uniforms'], temperature=case['temperature'])


# -- run ------------------------------------------------------------------------

def _run_verify(st):
    store = st['store']
    if st['retire']:
        handles = [store.add_request(r) for r in st['names']]
        for h, p in zip(handles, st['prefix']):
            if p:
                store.load_prefix(h, *p)
    else:
        handles = st['handles']
    tx = store.begin(handles, st['bucket'])
    outs = []
    for layer in st['layers']:
        if 'prologues' in st:
            query = store.stage_projected(tx, layer, st['hidden'][layer], st['prologues'][layer])
            outs.append(store.attend(tx, layer, query))
        else:
            outs.append(store.attend(tx, layer, st['q'][layer], keys=st['k'][layer], values=st['v'][layer]))
    if not st['retire']:
        store.abort(tx)
        return dict(out=outs, scratch_keys=store.scratch_keys, scratch_values=store.scratch_values)
    store.commit(tx, dict(zip(handles, st['accepted'])))
    for h in handles:
        store.remove_request(h)
    return dict(out=outs, keys=store.keys, values=store.values)


def _run_packed(st):
    from qwen3_dspark_amd.layout import PackedLayout
    kv, chunks, lengths = st['kv'], st['chunks'], st['lengths']
    markers, positions = [], []
    for r, n in chunks.items():
        markers += [kv.marker(r)] * n
        positions += range(lengths[r], lengths[r] + n)
    meta = torch.tensor([markers, positions], dtype=torch.long).to(DEV)
    layout = PackedLayout.from_metadata(meta[0], meta[1], torch.cat((kv.key_requests, meta[0])),
                                        torch.cat((kv.key_positions, meta[1])))
    outs, packed = [], None
    for layer, (q, new) in enumerate(zip(st['q'], st['new'])):
        packed = layout.gather_kv(*kv.append_layer(layer, *new))
        outs.append(st['kernel'](q, *packed, layout, scale=SCALE))
    kv.commit_rows(chunks)
    for r in chunks:
        kv.crop(r, lengths[r])
    return dict(out=outs, keys=packed[0], values=packed[1])


def _run_draft(st):
    if 'metadata' in st:
        from qwen3_dspark_amd.layout import PackedLayout
        layout = PackedLayout.from_metadata(*st['metadata'])
        return [st['kernel'].over_append_order_pool(st['q'][l], st['k'][l], st['v'][l], *st['pool'][l], layout,
                                                    scale=SCALE) for l in st['layers']]
    pool = st['pool']
    batch = pool.batch(st['anchors'])
    return [pool.attention(l, st['q'][l], st['k'][l], st['v'][l], batch) for l in st['layers']]


def run(st):
    kind = st['kind']
    if kind == 'verify':
        return _run_verify(st)
    if kind == 'packed':
        return _run_packed(st)
    if kind == 'draft':
        return _run_draft(st)
    if kind == 'append':
        pool = st['pool']
        pool.append_committed(st['chunks'])
        for r, n in st['lengths'].items():
            pool.crop(r, n)
        return dict(keys=pool.keys, values=pool.values)
    from qwen3_dspark_amd.sampling import logits_to_probabilities, sample_categorical, verify_proposals
    if kind == 'speculate':
        logits = st['head'](st['hidden'])
        rounds = verify_proposals(logits, st['tokens'], st['laws'], st['uniforms'], counts=st['counts'],
                                  temperature=st['temperature'], max_new_tokens=st['budgets'])
        # the emitted tokens end to end, padded: how many there are depends on the draws
        tokens = torch.cat([r.tokens for r in rounds])
        tokens = torch.nn.functional.pad(tokens, (0, len(logits) - len(tokens)), value=-1)
        return dict(logits=logits, tokens=tokens,
                    accepted=torch.tensor([r.accepted_draft_tokens for r in rounds]),
                    draws=torch.tensor([r.draws for r in rounds]))
    laws = logits_to_probabilities(st['logits'], st['temperature'])
    return dict(laws=laws, tokens=sample_categorical(laws, st['uniforms']))


# -- work -----------------------------------------------------------------------

def work(case):
    kind, s = case['kind'], _sizes(case)
    if kind in ('verify', 'packed'):
        L, rows, cached = case['layers'], sum(s['q']), sum(s['c'])
        pairs = sum(q * c + q * (q + 1) // 2 for q, c in zip(s['q'], s['c']))
        out = 2 * rows * HQ * D                                   # attention output, bf16
        if case.get('projected'):
            weights = (HQ + 2 * HKV) * D * HIDDEN
            nbytes = 2 * weights + 2 * rows * HIDDEN + 2 * ROW * rows + 2 * ROW * cached + out
            flops = 2 * rows * weights + 4 * HQ * D * pairs
        else:
            # queries, new and cached rows in, output and staged rows out
            nbytes = 2 * out + 4 * ROW * rows + 2 * ROW * cached
            flops = 4 * HQ * D * pairs
        nbytes, flops = L * nbytes, L * flops
        if kind == 'verify' and case['retire']:
            # prefixes in and into the store (whose rows the layers then
            # read, counted above), accepted rows into it
            nbytes += L * 4 * ROW * cached + L * 2 * ROW * sum(_accepted(s))
        if kind == 'packed':
            nbytes += L * 2 * ROW * cached                        # the gathered rows are outputs
        return dict(bytes=nbytes, flops=flops)
    if kind == 'draft':
        L, rows = case['layers'], BLOCK * sum(map(len, s['anchors']))
        seen = sum(max(a) for a in s['anchors'])
        pairs = sum(BLOCK * (x + BLOCK) for a in s['anchors'] for x in a)
        k = 2 if case['amp'] else 1                               # FP32 K and Q
        return dict(bytes=L * ((seen + rows) * (k + 1) * ROW + rows * HQ * D * 2 * (k + 1)),
                    flops=L * 4 * HQ * D * pairs)
    if kind == 'append':
        rows, features = sum(s['rows']), 5 * HIDDEN
        weights = HIDDEN * features + 5 * 2 * HKV * D * HIDDEN
        return dict(bytes=2 * weights + 2 * rows * features + 5 * 2 * ROW * rows, flops=2 * rows * weights)
    if kind == 'speculate':
        rows = sum(s['n']) + len(s['n'])
        # the head's weights and hidden rows in, the logits out and read by
        # the law; a draft law row is read where a proposal is rejected, about
        # one per request
        return dict(bytes=2 * VOCAB * HIDDEN + 2 * rows * HIDDEN + 4 * rows * VOCAB + 8 * VOCAB * len(s['n']),
                    flops=2 * rows * VOCAB * HIDDEN)
    each = 4 if case['dtype'] == 'float32' else 2
    return dict(bytes=case['rows'] * VOCAB * (each + 16), flops=case['rows'] * VOCAB * 24)


# -- tolerance ------------------------------------------------------------------

def tolerance(case):
    # bf16 results are 2e-3 to 3.6e-3 (2-norm) from the 64-bit ones, whatever
    # the order of the sums, so two correct implementations stay within
    # 5e-3 of each other; the float64 laws are 2e-16 away.
    if case['kind'] == 'laws':
        return dict(rel=1e-14, max=1e-13, differ=0.0)
    return dict(rel=1e-2, max=0.1, differ=0.0)


# -- the same in 64 bits, plain torch --------------------------------------------

def _softmax(x):
    # written out: torch's float64 softmax on the GPU is off by 1e-7
    e = torch.exp(x - x.amax(-1, keepdim=True))
    return e / e.sum(-1, keepdim=True)


def _attend(q, k, v, visible=None):
    """q [n, 16, d], k/v [m, 8, d] in float64 -> [n, 16, d]; visible: [n, m] mask or None.  Head by head: small
    enough for long prompts."""
    out = torch.empty_like(q)
    for h in range(HQ):
        x = (q[:, h] @ k[:, h // 2].t()) * SCALE
        if visible is not None:
            x = x.masked_fill(~visible, -math.inf)
        out[:, h] = _softmax(x) @ v[:, h // 2]
    return out


def _norm(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _rope(x, positions):
    inv = 1.0 / (THETA ** (torch.arange(0, D, 2, dtype=torch.float) / D))
    angle = (positions.float()[:, None] * inv.to(DEV)).double()       # the model's float32 table
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]
    lo, hi = x[..., :D // 2], x[..., D // 2:]
    return torch.cat((lo * cos - hi * sin, hi * cos + lo * sin), -1)


def _exact_rows(case, s, x):
    """Per layer: new q, k, v rows in float64, and the attention over the cached and new rows."""
    positions = torch.cat([torch.arange(c, c + q, device=DEV) for c, q in zip(s['c'], s['q'])])
    news, outs = [], []
    for layer in range(case['layers']):
        if case.get('projected'):
            wq, wk, wv, nq, nk = x['weights'][layer]
            h = x['hidden'][layer].double()
            heads = lambda w: (h @ w.double().t()).view(len(h), -1, D)
            q = _rope(_norm(heads(wq), nq), positions)
            k, v = _rope(_norm(heads(wk), nk), positions), heads(wv)
        else:
            q, k, v = (x[n][layer].double() for n in 'qkv')
        out, at, row = [], 0, 0
        for c, n in zip(s['c'], s['q']):
            keys = torch.cat((x['ctx_k'][layer][at:at + c].double(), k[row:row + n]))
            vals = torch.cat((x['ctx_v'][layer][at:at + c].double(), v[row:row + n]))
            seen = torch.arange(c + n, device=DEV)[None] <= torch.arange(c, c + n, device=DEV)[:, None]
            out.append(_attend(q[row:row + n], keys, vals, seen))
            at, row = at + c, row + n
        news.append((k, v))
        outs.append(torch.cat(out))
    return news, outs


def exact(case, seed):
    s, x = _inputs(case, seed)
    kind = case['kind']
    if kind == 'verify':
        news, outs = _exact_rows(case, s, x)
        if not case['retire']:
            return dict(out=outs, scratch_keys=torch.stack([k for k, _ in news]),
                        scratch_values=torch.stack([v for _, v in news]))
        n, cap = len(s['c']), case['ctx_max'] + case['q_max']
        stores = []
        for which, ctx in enumerate((x['ctx_k'], x['ctx_v'])):
            store = torch.zeros(case['layers'], n, cap, HKV, D, dtype=torch.float64, device=DEV)
            for layer in range(case['layers']):
                at = row = 0
                for r, (c, q, keep) in enumerate(zip(s['c'], s['q'], _accepted(s))):
                    store[layer, r, :c] = ctx[layer][at:at + c].double()
                    store[layer, r, c:c + keep] = news[layer][which][row:row + keep]
                    at, row = at + c, row + q
            stores.append(store)
        return dict(out=outs, keys=stores[0], values=stores[1])
    if kind == 'packed':
        news, outs = _exact_rows(case, s, x)
        last = []
        for which, ctx in enumerate((x['ctx_k'], x['ctx_v'])):
            pieces, at, row = [], 0, 0
            for c, q in zip(s['c'], s['q']):
                pieces += [ctx[-1][at:at + c].double(), news[-1][which][row:row + q]]
                at, row = at + c, row + q
            last.append(torch.cat(pieces))
        return dict(out=outs, keys=last[0], values=last[1])
    if kind == 'draft':
        outs = []
        for layer in range(case['layers']):
            out, at, row = [], 0, 0
            for c, anchors in zip(s['c'], s['anchors']):
                for a in anchors:
                    own = slice(row, row + BLOCK)
                    keys = torch.cat((x['ctx_k'][layer][at:at + a], x['k'][layer][own])).bfloat16().double()
                    vals = torch.cat((x['ctx_v'][layer][at:at + a], x['v'][layer][own])).double()
                    out.append(_attend(x['q'][layer][own].bfloat16().double(), keys, vals))
                    row += BLOCK
                at += c
            outs.append(torch.cat(out))
        return outs
    if kind == 'append':
        n, cap = len(s['c']), case['ctx_max'] + case['rows_max']
        keys = torch.zeros(5, n, HKV, cap, D, dtype=torch.float64, device=DEV)
        values = torch.zeros_like(keys)
        for r, (f, c) in enumerate(zip(x['features'], s['c'])):
            h = _norm(f[0].double() @ x['fc'].double().t(), x['norm'])
            positions = torch.arange(c, c + len(h), device=DEV)
            for layer, (wk, nk, wv) in enumerate(x['layers']):
                k = _rope(_norm((h @ wk.double().t()).view(-1, HKV, D), nk), positions)
                keys[layer, r, :, c:c + len(h)] = k.transpose(0, 1)
                values[layer, r, :, c:c + len(h)] = (h @ wv.double().t()).view(-1, HKV, D).transpose(0, 1)
        return dict(keys=keys, values=values)
    if kind == 'speculate':
        return dict(logits=x['hidden'].double() @ x['head'].double().t(), tokens=None, accepted=None, draws=None)
    return dict(laws=_softmax(x['logits'].double() / case['temperature']), tokens=None)

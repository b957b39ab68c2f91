"""dspark_mixed_attn_fwd: batches of prompts, chunks of prompts and decoding
requests at the sizes where a plan changes form (row tiles in the runs, alone
and among decoding requests; prompts cut and uncut; partials of tiles and of
prompts; nothing to merge), packed and from the store, staged by the launch or
before it, against the CPU oracle at the attention tolerance."""
import pytest
import torch

from helpers import SCALE, SEED, attention_gate, bits, f64, randn_bf16, segments
from oracle import cref
from test_gpu_prefill import layout_of

pytestmark = pytest.mark.gpu
DEV = torch.device('cuda:0')

BATCHES = [([9], [0]), ([9], [700]), ([16, 64], [0, 300]), ([96], [300]), ([97], [300]), ([12, 33, 9], [1500, 0, 40]),
           ([7, 7, 9], [600, 30, 1900]), ([8, 1, 64, 200], [500, 0, 1200, 0]), ([17], [3000]), ([40, 7], [2500, 900]),
           ([64, 7, 7, 300], [1800, 700, 9, 1900]), ([20] * 20, [30] * 20)]


@pytest.mark.parametrize('ql,ctx', BATCHES)
def test_packed(ql, ctx):
    from qwen3_dspark_amd.kernels import HipDraftVarlenKernel, HipVarlenKernel
    print(f'[mixed] packed q={ql} ctx={ctx}', flush=True)
    layout, q, k, v = layout_of(ql, [c + n for c, n in zip(ctx, ql)])
    cu_q = layout.cu_query.tolist()
    for cls in (HipVarlenKernel, HipDraftVarlenKernel):
        out = cls(DEV)(q.to(DEV), k.to(DEV), v.to(DEV), layout, scale=SCALE)
        ref = cref.varlen_attention(bits(q), bits(k), bits(v), cu_q, layout.cu_key.tolist(), causal=cls.causal,
                                    scale=SCALE)
        attention_gate(f64(out), ref, segments(cu_q))


@pytest.mark.parametrize('ql,ctx', BATCHES)
def test_store(ql, ctx):
    """Through a bucket and through a family that also takes other lengths;
    rows past a context and other slots hold NaN."""
    from qwen3_dspark_amd.persistent_kv import Bucket, PersistentTargetKV, QueryFamily
    print(f'[mixed] store q={ql} ctx={ctx}', flush=True)
    gen = torch.Generator().manual_seed(SEED + sum(ql) + sum(ctx))
    n, rows = len(ql), sum(ql)
    store = PersistentTargetKV(layers=1, slots=n + 1, context_capacity=3400, max_query_tokens=rows, heads=8, dim=128,
                               device=DEV)
    store.keys.fill_(float('nan'))
    store.values.fill_(float('nan'))
    handles = [store.add_request(f'r{i}') for i in range(n)][::-1]
    for h, c in zip(handles, ctx):
        if c:
            kv = randn_bf16(gen, 2, 1, c, 8, 128).to(DEV)
            store.load_prefix(h, kv[0], kv[1])
    bucket = Bucket(tuple(ql), tuple(c + 100 for c in ctx), 'mixed')
    family = QueryFamily(n, rows, max(ql) + 20, rows + sum(ctx) + 500, 3400, 'mixed family')
    store.register_bucket(bucket)
    store.register_families((family,))
    q, nk, nv = (randn_bf16(gen, rows, h, 128).to(DEV) for h in (16, 8, 8))
    cu_q = [sum(ql[:i]) for i in range(n + 1)]
    ref = cref.verify_attention(bits(q), bits(store.keys[0]), bits(store.values[0]), bits(nk), bits(nv),
                                [h.index for h in handles], ctx, cu_q, scale=SCALE)
    for shape in (bucket, family):
        tx = store.begin(handles, shape, query_lengths=tuple(ql))
        store.scratch_keys.zero_()
        out = store.attend(tx, 0, q, keys=nk, values=nv)
        assert torch.equal(store.scratch_keys[0], nk) and torch.equal(store.scratch_values[0], nv)
        attention_gate(f64(out), ref, segments(cu_q))
        store.abort(tx)
        tx = store.begin(handles, shape, query_lengths=tuple(ql))
        store.stage_layer(tx, 0, nk, nv)
        assert torch.equal(store.attend(tx, 0, q), out)
        store.abort(tx)


def test_families_of_one_arena():
    """A decoding family and one with prompts share a workspace: the lists and
    partials of both fit, whatever the transaction holds."""
    from qwen3_dspark_amd.persistent_kv import PersistentTargetKV, QueryFamily
    gen = torch.Generator().manual_seed(SEED)
    store = PersistentTargetKV(layers=1, slots=4, context_capacity=3000, max_query_tokens=400, heads=8, dim=128,
                               device=DEV)
    handles = [store.add_request(f'r{i}') for i in range(4)]
    ctx = [2500, 40, 1800, 700]
    for h, c in zip(handles, ctx):
        kv = randn_bf16(gen, 2, 1, c, 8, 128).to(DEV)
        store.load_prefix(h, kv[0], kv[1])
    small = QueryFamily(4, 20, 8, 6000, 3000, 'decoding')
    large = QueryFamily(4, 220, 200, 6000, 3000, 'with prompts')
    store.register_families((small, large))
    for family, ql in ((small, (7, 1, 8, 4)), (large, (7, 200, 9, 4)), (large, (55, 55, 55, 55)), (small, (5,) * 4),
                       (large, (1, 1, 18, 200))):
        rows = sum(ql)
        q, nk, nv = (randn_bf16(gen, rows, h, 128).to(DEV) for h in (16, 8, 8))
        tx = store.begin(handles, family, query_lengths=ql)
        out = store.attend(tx, 0, q, keys=nk, values=nv)
        cu_q = [sum(ql[:i]) for i in range(5)]
        ref = cref.verify_attention(bits(q), bits(store.keys[0]), bits(store.values[0]), bits(nk), bits(nv),
                                    [h.index for h in handles], ctx, cu_q, scale=SCALE)
        attention_gate(f64(out), ref, segments(cu_q))
        store.abort(tx)


@pytest.mark.parametrize('split', ['balanced', 'request'])
def test_a_decoding_family_in_an_arena_of_fewer_partials(split):
    """Four decoding requests beside a family of 40 tokens at most: a list of
    their own would have more runs than the arena's partials hold."""
    from qwen3_dspark_amd.persistent_kv import PersistentTargetKV, QueryFamily
    gen = torch.Generator().manual_seed(SEED)
    store = PersistentTargetKV(layers=1, slots=4, context_capacity=6000, max_query_tokens=78, heads=8, dim=128,
                               device=DEV, split=split)
    handles = [store.add_request(f'r{i}') for i in range(4)]
    ctx = [5900, 5800, 5700, 5500]
    for h, c in zip(handles, ctx):
        kv = randn_bf16(gen, 2, 1, c, 8, 128).to(DEV)
        store.load_prefix(h, kv[0], kv[1])
    small = QueryFamily(4, 19, 8, 22958, 6000, 'decoding')
    large = QueryFamily(4, 78, 40, 22978, 6000, 'with prompts')
    store.register_families((small, large))
    for family, ql in ((small, (7, 1, 8, 3)), (large, (7, 40, 9, 22)), (small, (4, 5, 5, 5))):
        rows = sum(ql)
        q, nk, nv = (randn_bf16(gen, rows, h, 128).to(DEV) for h in (16, 8, 8))
        tx = store.begin(handles, family, query_lengths=ql)
        out = store.attend(tx, 0, q, keys=nk, values=nv)
        cu_q = [sum(ql[:i]) for i in range(5)]
        ref = cref.verify_attention(bits(q), bits(store.keys[0]), bits(store.values[0]), bits(nk), bits(nv),
                                    [h.index for h in handles], ctx, cu_q, scale=SCALE)
        attention_gate(f64(out), ref, segments(cu_q))
        store.abort(tx)


@pytest.mark.parametrize('chunk', [0, 33, 1 << 21])
@pytest.mark.parametrize('tokens', [5, 40])
def test_a_chunk_that_the_other_calls_refuse(chunk, tokens):
    """Refused on the host whatever the plan, packed and from the store."""
    from qwen3_dspark_amd.kernels import HipVarlenKernel
    from qwen3_dspark_amd.persistent_kv import Bucket, PersistentTargetKV
    layout, q, k, v = layout_of([tokens], [tokens])
    with pytest.raises((ValueError, RuntimeError)):
        HipVarlenKernel(DEV, chunk=chunk)(q.to(DEV), k.to(DEV), v.to(DEV), layout, scale=SCALE)
    store = PersistentTargetKV(layers=1, slots=1, context_capacity=128, max_query_tokens=64, heads=8, dim=128,
                               device=DEV, chunk=chunk)
    bucket = Bucket((tokens,), (64,), 'chunk')
    store.register_bucket(bucket)
    tx = store.begin([store.add_request('r')], bucket, query_lengths=(tokens,))
    with pytest.raises((ValueError, RuntimeError)):
        store.attend(tx, 0, q.to(DEV), keys=k.to(DEV), values=v.to(DEV))


@pytest.mark.parametrize('split', ['balanced', 'request'])
def test_captured_rounds_with_prompts(split):
    """One captured program for a bucket of prompts and short requests, replayed
    over contexts that change which of them are cut or attended by row tiles: every
    replay equals the eager call."""
    from qwen3_dspark_amd.graph import VerificationGraph
    from qwen3_dspark_amd.persistent_kv import Bucket, PersistentTargetKV
    gen = torch.Generator().manual_seed(SEED)
    ql, ceiling = (7, 64, 9, 200), 6000
    rows = sum(ql)
    store = PersistentTargetKV(layers=2, slots=8, context_capacity=6400, max_query_tokens=rows, heads=8, dim=128,
                               device=DEV, split=split)
    contexts = (0, 300, 20, 5900, 700, 2500, 64, 4000)
    handles = [store.add_request(f'r{i}') for i in range(8)]
    for h, c in zip(handles, contexts):
        if c:
            kv = randn_bf16(gen, 2, 2, c, 8, 128).to(DEV)
            store.load_prefix(h, kv[0], kv[1])
    bucket = Bucket(ql, (ceiling,) * 4, 'captured prompts')
    store.register_bucket(bucket)
    graph = VerificationGraph(store, bucket).capture()
    cu_q = [sum(ql[:i]) for i in range(5)]
    for chosen in ((0, 1, 2, 6), (3, 5, 7, 4), (1, 0, 3, 6), (7, 2, 5, 3), (0, 1, 2, 6)):
        some = [handles[i] for i in chosen]
        ctx = [store.length(h) for h in some]
        print(f'[mixed] captured split={split} ctx={ctx}', flush=True)
        q, nk, nv = (randn_bf16(gen, 2, rows, h, 128).to(DEV) for h in (16, 8, 8))
        tx = store.begin(some, bucket)
        eager = [store.attend(tx, l, q[l], keys=nk[l], values=nv[l]) for l in range(2)]
        store.abort(tx)
        torch.cuda.synchronize()
        tx = store.begin(some, bucket)
        graph.query.copy_(q)
        graph.keys.copy_(nk)
        graph.values.copy_(nv)
        out = graph.wait(graph.submit(tx))
        assert all(torch.equal(out[l], eager[l]) for l in range(2))
        ref = cref.verify_attention(bits(q[1]), bits(store.keys[1]), bits(store.values[1]), bits(nk[1]), bits(nv[1]),
                                    [h.index for h in some], ctx, cu_q, scale=SCALE)
        attention_gate(f64(out[1]), ref, segments(cu_q))
        store.commit(tx, {h: min(n, 5) for h, n in zip(some, ql)})

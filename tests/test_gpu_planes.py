"""Short prompts attended by row tiles in launches whose plan is not a balanced
one: fixed chunks without a work list (on both sides of the key bound that decides),
request-local lists, packed and from the store, and lists whose prompts stand
in the runs or after them, against the CPU oracle at the attention tolerance."""
import pytest
import torch

from helpers import SCALE, SEED, attention_gate, bits, f64, randn_bf16, segments
from oracle import cref
from test_gpu_prefill import layout_of

pytestmark = pytest.mark.gpu
DEV = torch.device('cuda:0')


@pytest.mark.parametrize('ql,kl,cap', [((9,), (9,), 9), ((9, 5, 64), (300, 1100, 400), 2000),
                                       ((9, 5, 64), (300, 1100, 400), 3072), ((9, 5, 64), (300, 1100, 400), 3073),
                                       ((17, 33, 1), (17, 2100, 5), 2400), ((65, 9), (65, 1500), 1565)])
def test_fixed_chunks(ql, kl, cap):
    from qwen3_dspark_amd.kernels import HipCapacityKernel
    from qwen3_dspark_amd.layout import PersistentAttentionLayout
    exact, q, k, v = layout_of(list(ql), list(kl))
    tail = torch.full((cap - sum(kl), 8, 128), float('nan'), dtype=torch.bfloat16)
    layout = PersistentAttentionLayout(ql, kl, exact.cu_query, exact.cu_key, cap, max(kl), max(ql))
    out = HipCapacityKernel(DEV)(q.to(DEV), torch.cat((k, tail)).to(DEV), torch.cat((v, tail)).to(DEV), layout,
                                 scale=SCALE)
    cu_q = exact.cu_query.tolist()
    ref = cref.varlen_attention(bits(q), bits(k), bits(v), cu_q, exact.cu_key.tolist(), causal=True, scale=SCALE)
    attention_gate(f64(out), ref, segments(cu_q))


@pytest.mark.parametrize('ql,ctx', [([9, 16, 40, 7], [0, 2000, 600, 30]), ([64, 65, 8], [704, 0, 900]),
                                    ([33, 9, 200], [1500, 2100, 40])])
def test_request_local_store(ql, ctx):
    """Staged by the launch: outputs, scratch, and the bits of each request alone."""
    from qwen3_dspark_amd.persistent_kv import Bucket, PersistentTargetKV
    gen = torch.Generator().manual_seed(SEED + sum(ql))
    n, rows = len(ql), sum(ql)
    store = PersistentTargetKV(layers=1, slots=n, context_capacity=2400, max_query_tokens=rows, heads=8, dim=128,
                               device=DEV, split='request', chunk=512)
    handles = [store.add_request(f'r{i}') for i in range(n)]
    for h, c in zip(handles, ctx):
        if c:
            kv = randn_bf16(gen, 2, 1, c, 8, 128).to(DEV)
            store.load_prefix(h, kv[0], kv[1])
        store.keys[:, h.index, c:] = float('nan')
        store.values[:, h.index, c:] = float('nan')
    q, nk, nv = (randn_bf16(gen, rows, h, 128).to(DEV) for h in (16, 8, 8))
    cu_q = [sum(ql[:i]) for i in range(n + 1)]

    def attend(which):
        bucket = Bucket(tuple(ql[i] for i in which), tuple(ctx[i] + 9 for i in which), f'planes {which}')
        store.register_bucket(bucket)
        at = torch.cat([torch.arange(cu_q[i], cu_q[i + 1]) for i in which]).to(DEV)
        tx = store.begin([handles[i] for i in which], bucket)
        out = store.attend(tx, 0, q[at], keys=nk[at], values=nv[at])
        assert torch.equal(store.scratch_keys[0, :len(at)], nk[at])
        assert torch.equal(store.scratch_values[0, :len(at)], nv[at])
        store.abort(tx)
        return out
    out = attend(range(n))
    ref = cref.verify_attention(bits(q), bits(store.keys[0]), bits(store.values[0]), bits(nk), bits(nv),
                                [h.index for h in handles], ctx, cu_q, scale=SCALE)
    attention_gate(f64(out), ref, segments(cu_q))
    for i in range(n):
        assert torch.equal(attend([i]), out[cu_q[i]:cu_q[i + 1]])


@pytest.mark.parametrize('ql,kl', [([9, 7, 64], [700, 40, 300]), ([20, 100, 33, 8], [900, 1100, 33, 2000])])
def test_records_in_runs_or_in_none(ql, kl):
    """A list may hold a prompt's records in any run or after the last: the same bits."""
    from qwen3_dspark_amd import _native
    from qwen3_dspark_amd.schedule import WORK_INTS, request_work
    layout, q, k, v = layout_of(ql, kl)
    q, k, v = (t.to(DEV) for t in (q, k, v))
    starts = layout.cu_key.tolist()[:-1]
    out, n, runs = request_work(ql, kl, starts, 512, 16)
    base = WORK_INTS * n
    ranges = out[base:base + runs + 1]
    assert ranges[-1] < n                                   # prompts after the runs
    inside = out[:base] + ranges[:-1] + [n] + out[base + runs + 1:]     # the last run takes them
    tiles = -(-max(ql) // 8)
    ws = torch.zeros(_native.load().dspark_attn_workspace_bytes(n, 0, tiles, 512), dtype=torch.uint8, device=DEV)
    got = []
    for records in (out, inside):
        work = torch.tensor(records, dtype=torch.int32, device=DEV)
        o = torch.full_like(q, float('nan'))
        _native.call('dspark_varlen_attn_fwd', q.data_ptr(), k.data_ptr(), v.data_ptr(), layout.cu_query.data_ptr(),
                     layout.cu_key.data_ptr(), len(ql), len(q), len(k), max(ql), 1, SCALE, 512, work.data_ptr(), n,
                     runs, o.data_ptr(), ws.data_ptr(), ws.numel(), _native.stream_handle(DEV))
        got.append(o)
    assert torch.equal(*got)
    cu_q = layout.cu_query.tolist()
    ref = cref.varlen_attention(bits(q), bits(k), bits(v), cu_q, layout.cu_key.tolist(), causal=True, scale=SCALE)
    attention_gate(f64(got[0]), ref, segments(cu_q))

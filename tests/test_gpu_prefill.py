"""Attention of requests with more than 8 query tokens (prefill_attn_kernel)
at the sizes where it can go wrong: the edges of its 16-token row groups,
32-token workgroups and 64-key stages, prompts beside verifying requests,
later chunks of a prompt with their keys cut, all three kernels' forms
(exact, noncausal, capacity) and the store's staged form, against the CPU
oracle at the attention tolerance."""
import pytest
import torch

from helpers import SCALE, SEED, attention_gate, bits, f64, randn_bf16, segments
from oracle import cref
from test_gpu_varlen import make_packed

pytestmark = pytest.mark.gpu
DEV = torch.device('cuda:0')

SHAPES = [([9], [9]), ([16, 17], [16, 60]), ([32, 33, 48], [95, 33, 64]), ([63, 64, 65], [63, 128, 129]),
          ([128, 7, 1, 200], [128, 300, 1, 333]), ([12, 8, 9], [2500, 1100, 9]), ([300], [4000]), ([129, 257], [1300, 257])]


def layout_of(q_lens, k_lens):
    from qwen3_dspark_amd.layout import PackedLayout
    meta, q, k, v = make_packed(torch.Generator().manual_seed(SEED + sum(k_lens)), q_lens, k_lens)
    return PackedLayout.from_metadata(*(m.to(DEV) for m in meta)), q, k, v


@pytest.mark.parametrize('q_lens,k_lens', SHAPES)
@pytest.mark.parametrize('split', ['balanced', 'request'])
def test_packed_prompts_against_oracle(q_lens, k_lens, split):
    from qwen3_dspark_amd.kernels import HipDraftVarlenKernel, HipVarlenKernel
    print(f'[prefill] q={q_lens} k={k_lens} {split}', flush=True)
    layout, q, k, v = layout_of(q_lens, k_lens)
    cu_q, cu_k = layout.cu_query.tolist(), layout.cu_key.tolist()
    for cls in (HipVarlenKernel, HipDraftVarlenKernel):
        kernel = cls(DEV, split=split, chunk=512)
        out = kernel(q.to(DEV), k.to(DEV), v.to(DEV), layout, scale=SCALE)
        ref = cref.varlen_attention(bits(q), bits(k), bits(v), cu_q, cu_k, causal=cls.causal, scale=SCALE)
        attention_gate(f64(out), ref, segments(cu_q))
        if split == 'request':      # a request alone: the bits it has in the batch
            for r, (n, m) in enumerate(zip(q_lens, k_lens)):
                lone, _, _, _ = layout_of([n], [m])
                one = kernel(q[cu_q[r]:cu_q[r + 1]].to(DEV), k[cu_k[r]:cu_k[r + 1]].to(DEV),
                             v[cu_k[r]:cu_k[r + 1]].to(DEV), lone, scale=SCALE)
                assert torch.equal(one, out[cu_q[r]:cu_q[r + 1]])


def test_capacity_tail_prompts():
    """Fixed chunks without a work list; the capacity tail is never read."""
    from qwen3_dspark_amd.kernels import HipCapacityKernel
    from qwen3_dspark_amd.layout import PersistentAttentionLayout
    q_lens, k_lens, cap = (70, 5, 16), (1500, 1030, 16), 4000
    exact, q, k, v = layout_of(list(q_lens), list(k_lens))
    layout = PersistentAttentionLayout(q_lens, k_lens, exact.cu_query, exact.cu_key, cap, 2000, 80)
    tail = torch.full((cap - sum(k_lens), 8, 128), float('nan'), dtype=torch.bfloat16)
    out = HipCapacityKernel(DEV)(q.to(DEV), torch.cat((k, tail)).to(DEV), torch.cat((v, tail)).to(DEV), layout,
                                 scale=SCALE)
    cu_q = exact.cu_query.tolist()
    ref = cref.varlen_attention(bits(q), bits(k), bits(v), cu_q, exact.cu_key.tolist(), causal=True, scale=SCALE)
    attention_gate(f64(out), ref, segments(cu_q))


@pytest.mark.parametrize('qls,ctx', [([100, 7, 33], [0, 900, 50]), ([9, 64, 1, 130], [31, 0, 700, 1900])])
def test_store_prefill_and_chunks(qls, ctx):
    """A store transaction mixing prompts, later chunks and verification,
    staged by the attention launch: outputs, scratch and untouched rows."""
    from qwen3_dspark_amd.persistent_kv import Bucket, PersistentTargetKV
    print(f'[prefill store] q={qls} ctx={ctx}', flush=True)
    gen = torch.Generator().manual_seed(SEED + sum(qls))
    n, cap = len(qls), 2100
    pool = PersistentTargetKV(layers=1, slots=n, context_capacity=cap, max_query_tokens=sum(qls), heads=8, dim=128,
                              device=DEV)
    handles = [pool.add_request(f'r{i}') for i in range(n)]
    for h, c in zip(handles, ctx):
        if c:
            kv = randn_bf16(gen, 2, 1, c, 8, 128).to(DEV)
            pool.load_prefix(h, kv[0], kv[1])
        pool.keys[:, h.index, c:] = float('nan')
        pool.values[:, h.index, c:] = float('nan')
    bucket = Bucket(tuple(qls), (1950,) * n, 'prompts')
    pool.register_bucket(bucket)
    q, nk, nv = (randn_bf16(gen, sum(qls), h, 128).to(DEV) for h in (16, 8, 8))
    tx = pool.begin(handles, bucket)
    out = pool.attend(tx, 0, q, keys=nk, values=nv)
    assert torch.equal(pool.scratch_keys[0], nk) and torch.equal(pool.scratch_values[0], nv)
    cu_q = [sum(qls[:i]) for i in range(n + 1)]
    ref = cref.verify_attention(bits(q), bits(pool.keys[0]), bits(pool.values[0]), bits(nk), bits(nv),
                                [h.index for h in handles], ctx, cu_q, scale=SCALE)
    attention_gate(f64(out), ref, segments(cu_q))


def test_values_past_a_rows_limit_never_reach_it():
    """An infinite value row at token j leaves every 8-token group before
    j's untouched, in the same workgroup and 32-key tile."""
    from qwen3_dspark_amd.kernels import HipVarlenKernel
    layout, q, k, v = layout_of([80], [80])
    kernel = HipVarlenKernel(DEV)
    clean = kernel(q.to(DEV), k.to(DEV), v.to(DEV), layout, scale=SCALE)
    for j in (8, 20, 31, 63, 64):
        bad = v.clone()
        bad[j] = float('inf')
        out = kernel(q.to(DEV), k.to(DEV), bad.to(DEV), layout, scale=SCALE)
        assert torch.equal(out[:j // 8 * 8], clean[:j // 8 * 8])
        assert not torch.isfinite(out[j:]).any()


@pytest.mark.parametrize('q_lens,k_lens', [([300], [300]), ([1024], [1024]), ([200], [1200]), ([97, 128, 200], [700, 2000, 1064])])
def test_error_is_that_of_the_output_rounding(q_lens, k_lens):
    """The probabilities reach V to 15 bits and everything else is FP32, so the
    2-norm error is the one rounding of the outputs to bf16, however few key
    groups a request has (one bf16 probability operand is 10 to 40 % above it).
    Requests of the prompt form: a balanced plan attends up to 96 tokens as
    decoding requests are."""
    from qwen3_dspark_amd.kernels import HipVarlenKernel
    layout, q, k, v = layout_of(q_lens, k_lens)
    q = (q.float() * 1.5).bfloat16()
    out = HipVarlenKernel(DEV)(q.to(DEV), k.to(DEV), v.to(DEV), layout, scale=SCALE).double().cpu()
    wrong = rounding = 0.0
    for a, b, n, m in zip(layout.cu_query.tolist(), layout.cu_key.tolist(), q_lens, k_lens):
        seen = torch.arange(m)[None] <= torch.arange(m - n, m)[:, None]
        for h in range(16):
            x = (q[a:a + n, h].double() @ k[b:b + m, h // 2].double().t() * SCALE).masked_fill(~seen, -torch.inf)
            ref = torch.softmax(x, -1) @ v[b:b + m, h // 2].double()
            wrong += (out[a:a + n, h] - ref).square().sum()
            rounding += (ref.bfloat16().double() - ref).square().sum()
    # what is left off: probabilities at 1.5 x 2^-15 and FP32 sums, each under 1 % of
    # the rounding's 2^-8 / sqrt(12) to the outputs' own scale
    assert wrong.sqrt() <= 1.02 * rounding.sqrt()


@pytest.mark.parametrize('value', [float('inf'), -float('inf')])
def test_an_infinite_value_row_gives_its_infinity(value):
    """Not NaN: every part of a visible key's weight has its sign.  One infinite
    row per request; equal keys, so that its weight is far from underflow."""
    from qwen3_dspark_amd.kernels import HipVarlenKernel
    for n, j in ((20, 3), (64, 40), (200, 100), (300, 299)):
        layout, q, k, v = layout_of([n], [n])
        v[j] = value
        k[:] = k[:1]
        out = HipVarlenKernel(DEV)(q.to(DEV), k.to(DEV), v.to(DEV), layout, scale=SCALE)
        assert bool((out[j:] == value).all()) and bool(torch.isfinite(out[:j // 8 * 8]).all())

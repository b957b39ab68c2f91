"""The 128-token projection tiles (wide_gemm.h) at the edges of a tile: the
draft context projection forced onto them against the fused 64-token tiles and
the float64 oracle, and the verify-layer prologue from 513 tokens on against
the oracle."""
import numpy as np
import pytest
import torch

from helpers import SEED, f64, randn_bf16
from oracle import draft_proj, qkv
from test_gpu_draft_projection import HIDDEN, gate, make_weights, projector
from test_gpu_prologue import gate as prologue_gate, weights as prologue_weights

pytestmark = pytest.mark.gpu
DEV = torch.device('cuda:0')


@pytest.mark.parametrize('counts', [[1], [127], [100, 28], [1, 128], [255, 2, 3], [300]])
def test_wide_projection_tiles(counts):
    """Rows against the oracle on the same fc output, and against the fused
    tiles: FP32 sums in another order, so nearly all outputs are equal and the
    rest within two bf16 ulps (2^-6 relative, plus 2^-12 near zero)."""
    gen = torch.Generator().manual_seed(SEED + sum(counts))
    fc, cn, per = make_weights(gen, layers=2)
    proj = projector(fc, cn, per)
    total = sum(counts)
    x = randn_bf16(gen, total, HIDDEN)
    records = torch.tensor([[len(counts) - 1 - i, 3 * i, sum(counts[:i]), n] for i, n in enumerate(counts)],
                           dtype=torch.int32, device=DEV)
    out = {}
    for path in ('fused', 'wide'):
        keys = torch.zeros(2, len(counts), 8, 320, 128, dtype=torch.bfloat16, device=DEV)
        values = torch.zeros_like(keys)
        flag = torch.zeros(1, dtype=torch.int32, device=DEV)
        proj.project_into(x.to(DEV), records, len(counts), keys, values, flag=flag, path=path)
        assert int(flag.item()) == 0
        out[path] = (f64(keys), f64(values))
    pos = np.concatenate([np.arange(3 * i, 3 * i + n) for i, n in enumerate(counts)])
    ref = draft_proj.project_context_kv(None, None, f64(cn), [(f64(a), f64(b), f64(c)) for a, b, c in per], pos,
                                        fc_out=f64(x))
    for layer in range(2):
        for which in range(2):
            got = np.concatenate([out['wide'][which][layer, len(counts) - 1 - i, :, 3 * i:3 * i + n].transpose(1, 0, 2)
                                  for i, n in enumerate(counts)])
            gate(got, ref[layer][which])
    for a, b in zip(out['fused'], out['wide']):
        d = np.abs(a - b)
        assert (d <= 2.0 ** -6 * np.maximum(np.abs(a), np.abs(b)) + 2.0 ** -12).all()
        assert (d > 0).mean() <= 1e-3
    bad = x.clone()
    bad[total - 1] = float('inf')
    proj.project_into(bad.to(DEV), records, len(counts), keys, values, flag=flag, path='wide')
    assert int(flag.item()) == 1


@pytest.mark.parametrize('tokens', [513, 640, 769])
def test_wide_prologue_against_oracle(tokens):
    from qwen3_dspark_amd.prologue import QKVPrologue
    gen = torch.Generator().manual_seed(SEED + tokens)
    w = prologue_weights(gen)
    x, pos = randn_bf16(gen, tokens, HIDDEN), torch.randint(0, 9000, (tokens,), generator=gen)
    pro = QKVPrologue(*(t.to(DEV) for t in w), eps=1e-6, theta=1e6)
    formed = pro(x.to(DEV), pos.to(DEV))
    read = pro(x.to(DEV), pos.to(DEV), rope=pro.rope_table(pos.to(DEV)))
    ref = qkv.qkv_prologue(f64(x), *(f64(t) for t in w), pos.numpy())
    for a, b, r in zip(formed, read, ref):
        assert torch.equal(a, b)
        prologue_gate(a, r)

"""The launch count that append_committed reports is the number of launches that
its projection made, on every path of the dispatch."""
import pytest
import torch

from helpers import SEED, randn_bf16
from test_gpu_draft_projection import FEATS, LAYERS, make_weights, projector

pytestmark = pytest.mark.gpu
DEV = torch.device('cuda:0')


@pytest.mark.parametrize('rows,gemm', [(1, False), (64, False), (400, False), (130, True)])
def test_reported_launches_are_those_made(rows, gemm, monkeypatch):
    from qwen3_dspark_amd import _native, draft_projection
    from qwen3_dspark_amd.draft import DraftKVPool
    if gemm:
        monkeypatch.setattr(draft_projection, 'GEMM_MIN_TOKENS', 1)
        monkeypatch.setattr(draft_projection, 'GEMM_CHUNK', 64)
    gen = torch.Generator().manual_seed(SEED + rows)
    proj = projector(*make_weights(gen))
    pool = DraftKVPool(layers=LAYERS, slots=1, capacity=512, device=DEV, projector=proj)
    pool.add_request('r')
    # each entry point's kernels, and the library GEMM that goes with an epilogue
    kernels = {'dspark_draft_kv_project': 1, 'dspark_draft_kv_project_rows': 2, 'dspark_draft_kv_epilogue': 2}
    made, real = [1], _native.call                                  # fc
    monkeypatch.setattr(_native, 'call', lambda name, *args: (made.append(kernels.get(name, 0)), real(name, *args))[1])
    work = pool.append_committed({'r': randn_bf16(gen, 1, rows, FEATS).to(DEV)})
    assert work['projection_launches'] == sum(made)

"""append_committed's feature packing (dspark_rows_pack): the one-launch pack of
aligned bf16 chunks against the same append with the chunks in forms that are
concatenated first, bit for bit, and the refusal of a non-finite feature
wherever it stands."""
import pytest
import torch

from helpers import SEED, randn_bf16
from test_gpu_draft_projection import FEATS, LAYERS, make_weights, projector

pytestmark = pytest.mark.gpu
DEV = torch.device('cuda:0')


def append(proj, chunks):
    from qwen3_dspark_amd.draft import DraftKVPool
    pool = DraftKVPool(layers=LAYERS, slots=len(chunks), capacity=300, device=DEV, projector=proj)
    for r in chunks:
        pool.add_request(r)
    pool.append_committed(chunks)
    return pool


@pytest.mark.parametrize('counts', [[1], [3], [1, 1, 1], [5, 200, 2], [7] * 33])
def test_pack_equals_concatenation(counts):
    gen = torch.Generator().manual_seed(SEED + sum(counts))
    proj = projector(*make_weights(gen))
    chunks = {f'r{i}': randn_bf16(gen, 1, n, FEATS).to(DEV) for i, n in enumerate(counts)}
    want = append(proj, chunks)
    # bf16 chunks off the 16-byte grid, FP32 chunks, and chunks with strided rows
    shifted, strided = {}, {}
    for r, x in chunks.items():
        flat = torch.empty(x.numel() + 1, dtype=torch.bfloat16, device=DEV)
        shifted[r] = flat[1:].view(x.shape).copy_(x)
        strided[r] = torch.stack((x, x), dim=2).flatten(2)[..., :FEATS]
    for other in (shifted, {r: x.float() for r, x in chunks.items()}, strided):
        got = append(proj, other)
        assert torch.equal(got.keys, want.keys) and torch.equal(got.values, want.values)
    for where in ((0, 0), (len(counts) - 1, -1)):
        for bad in (float('nan'), float('-inf')):
            wrong = dict(chunks)
            name = f'r{where[0]}'
            wrong[name] = chunks[name].clone()
            wrong[name].view(-1)[where[1]] = bad
            with pytest.raises(ValueError, match='finite'):
                append(proj, wrong)

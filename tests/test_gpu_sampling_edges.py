"""Laws, draws and verification at the edges of the kernels' tiles: a
probability workgroup's 4,096 values, a draw batch's 320 values of a segment
(256 segments per law), a wave's 64 chunks of a row's statistics, and
proposals of none to 255 tokens, against the oracle."""
import numpy as np
import pytest
import torch

from helpers import SEED
from oracle import sampling as oracle

pytestmark = pytest.mark.gpu
DEV = torch.device('cuda:0')


def as_tuple(r):
    return (tuple(int(t) for t in r.tokens.tolist()), r.accepted_draft_tokens, r.rejected_index, r.extra_token_kind,
            r.stop_reason)


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float32])
@pytest.mark.parametrize('vocab', [1, 255, 4095, 4096, 4097, 256 * 320, 256 * 320 + 1, 64 * 8192 + 1])
def test_laws_and_draws(vocab, dtype):
    from qwen3_dspark_amd.sampling import logits_to_probabilities, sample_categorical
    gen = torch.Generator(device=DEV).manual_seed(SEED + vocab)
    logits = (torch.randn(3, vocab + 3, generator=gen, device=DEV) * 3).to(dtype)[:, 1:vocab + 1]   # rows off 16 bytes
    logits[0, vocab // 2] = 120.0             # a peaked row: most of its law underflows in the ratio
    if vocab > 1:
        logits[0, 0] = -600.0
    probs = logits_to_probabilities(logits, 0.8)
    ref = oracle.logits_to_probabilities(logits.float().cpu().numpy(), 0.8)
    np.testing.assert_allclose(probs.cpu().numpy(), ref, rtol=1e-12, atol=1e-300)
    u = torch.tensor([0.3, 0.77, 0.999], dtype=torch.float64, device=DEV)
    assert sample_categorical(probs, u).tolist() == [oracle.sample_categorical(row, x)
                                                     for row, x in zip(ref, u.tolist())]


@pytest.mark.parametrize('counts,vocab', [((0, 255, 1, 8), 300), ((7, 0, 9), 256 * 320 + 77), ((2, 1), 64 * 8192 + 5)])
def test_verification(counts, vocab):
    from qwen3_dspark_amd.sampling import logits_to_probabilities, sample_categorical, verify_proposals
    gen = torch.Generator(device=DEV).manual_seed(SEED + vocab)
    rows, n = sum(counts) + len(counts), sum(counts)
    target = (torch.randn(rows, vocab, generator=gen, device=DEV) * 2).to(torch.bfloat16)
    first = np.cumsum([0] + [c + 1 for c in counts])
    own = [int(first[r]) + j for r, c in enumerate(counts) for j in range(c)]
    q = logits_to_probabilities(target[own].float() + 0.1 * torch.randn(n, vocab, generator=gen, device=DEV), 0.8)
    tokens = sample_categorical(q, torch.rand(n, generator=gen, device=DEV, dtype=torch.float64))
    uniforms = torch.rand(rows, generator=gen, device=DEV, dtype=torch.float64) * 0.9
    got = verify_proposals(target, tokens, q, uniforms, counts=counts, temperature=0.8,
                           max_new_tokens=[300] * len(counts))
    p_h = oracle.logits_to_probabilities(target.float().cpu().numpy(), 0.8)
    q_h, t_h, u_h = q.cpu().numpy(), tokens.cpu().numpy(), uniforms.cpu().numpy()
    for r, c in enumerate(counts):
        a = int(first[r])
        ref = oracle.verify_proposal(t_h[a - r:a - r + c], q_h[a - r:a - r + c], p_h[a:a + c + 1], u_h[a:a + c + 1],
                                     max_new_tokens=300)
        assert as_tuple(got[r]) == (ref.tokens, ref.accepted_draft_tokens, ref.rejected_index, ref.extra_token_kind,
                                    ref.stop_reason), r
        assert got[r].draws == ref.draws


@pytest.mark.parametrize('value', [float('nan'), float('inf'), -float('inf'), 3.0e38, -3.0e38, -600.0])
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float32])
def test_a_value_of_a_full_chunk(dtype, value):
    """A full aligned chunk whose terms are all normal takes the short exp; one
    NaN or infinity in it is refused, and one finite value whose term underflows
    takes the general exp."""
    from qwen3_dspark_amd.sampling import logits_to_probabilities
    gen = torch.Generator(device=DEV).manual_seed(SEED)
    logits = torch.randn(4, 3 * 8192, generator=gen, device=DEV).to(dtype)
    logits[2, 8192 + 4321] = value
    if not np.isfinite(value):
        with pytest.raises(ValueError, match='finite'):
            logits_to_probabilities(logits, 0.8)
        return
    ref = oracle.logits_to_probabilities(logits.float().cpu().numpy(), 0.8)
    np.testing.assert_allclose(logits_to_probabilities(logits, 0.8).cpu().numpy(), ref, rtol=1e-12, atol=1e-300)

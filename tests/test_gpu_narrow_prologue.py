"""The prologue's 32-token tiles (at most 256 tokens): the sums of the 64-token
tiles in the same order, so every row has the bits it has in a longer call."""
import pytest
import torch

from helpers import SEED

pytestmark = pytest.mark.gpu
DEV = torch.device('cuda:0')


@pytest.mark.parametrize('table', [True, False])
@pytest.mark.parametrize('hidden', [128, 256, 384, 512, 1024])          # 1 to 8 ring stages
@pytest.mark.parametrize('tokens', [1, 31, 32, 33, 64, 225, 256])
def test_rows_have_the_bits_of_a_longer_call(tokens, hidden, table):
    from qwen3_dspark_amd.prologue import QKVPrologue
    gen = torch.Generator(device=DEV).manual_seed(SEED + tokens + hidden)
    w = [(torch.randn(n, hidden, generator=gen, device=DEV) * 0.05).bfloat16() for n in (2048, 1024, 1024)]
    norms = [torch.rand(128, generator=gen, device=DEV).add(0.5).bfloat16() for _ in range(2)]
    pro = QKVPrologue(*w, *norms)
    x = torch.randn(300, hidden, generator=gen, device=DEV).bfloat16()
    pos = torch.randint(0, 8192, (300,), generator=gen, device=DEV)
    rope = pro.rope_table(pos) if table else None
    want = pro(x, pos, rope=rope)
    k, v = (torch.full((tokens + 2, 8, 128), 7.0, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    got = pro(x[:tokens], pos[:tokens], k_out=k, v_out=v, rope=rope[:tokens] if table else None)
    for a, b in zip(got, want):
        assert torch.equal(a[:tokens], b[:tokens])
    assert bool((k[tokens:] == 7.0).all()) and bool((v[tokens:] == 7.0).all())

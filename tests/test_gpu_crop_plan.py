"""The crop plan at the edges of its tiles and on both sides of the line
between its one-launch and three-launch forms, against a mask on the CPU."""
import pytest
import torch

from qwen3_dspark_amd import _native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n', [1, 63, 64, 1023, 1024, 1025, 5000, 32767, 32768, 32769, 36864, 36865, 100003])
@pytest.mark.parametrize('keep', ['some', 'none of it', 'nothing at all', 'everything'])
def test_crop_plan_is_the_stable_compaction(n, keep):
    gen = torch.Generator().manual_seed(n)
    kr = torch.randint(0, 3, (n,), generator=gen)
    if keep == 'nothing at all':
        kr.fill_(1)
    kp = torch.randint(0, 100, (n,), generator=gen)
    length = {'some': 40, 'none of it': 0, 'nothing at all': 0, 'everything': 100}[keep]
    want = torch.nonzero((kr != 1) | (kp < length)).flatten()
    m = want.numel()
    dkr, dkp = kr.cuda(), kp.cuda()
    plan, okr, okp = (torch.full((m + 8,), -7, device='cuda') for _ in range(3))
    ws = torch.empty(_native.load().dspark_crop_plan_workspace_bytes(n), dtype=torch.uint8, device='cuda')
    _native.call('dspark_crop_plan', dkr.data_ptr(), dkp.data_ptr(), n, 1, length, plan.data_ptr(), okr.data_ptr(),
                 okp.data_ptr(), ws.data_ptr(), ws.numel(), _native.stream_handle(dkr.device))
    for got, exact in ((plan, want), (okr, kr[want]), (okp, kp[want])):
        assert torch.equal(got[:m].cpu(), exact)
        assert bool((got[m:] == -7).all())

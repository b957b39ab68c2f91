"""The launch stream that entry points receive is torch's current stream of
the device, inside and outside a stream context and in another thread."""
import threading

import pytest
import torch

from qwen3_dspark_amd import _native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('device', ['cuda', 'cuda:0'])
def test_stream_handle_is_the_current_stream(device):
    device = torch.device(device)
    side = torch.cuda.Stream(device)
    main = torch.cuda.current_stream(device).cuda_stream
    seen = []
    assert _native.stream_handle(device) == main
    with torch.cuda.stream(side):
        assert _native.stream_handle(device) == side.cuda_stream != main
        worker = threading.Thread(target=lambda: seen.append(_native.stream_handle(device)))
        worker.start()
        worker.join()
    assert _native.stream_handle(device) == main and seen == [main]

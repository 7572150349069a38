"""Calls without a stream run on PyTorch's current one."""
import pytest

import shtamd

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def test_default_stream_is_torchs_current_one():
    assert shtamd._stream_handle(None) == torch.cuda.current_stream().cuda_stream
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert shtamd._stream_handle(None) == side.cuda_stream
    assert shtamd._stream_handle(None) == torch.cuda.current_stream().cuda_stream
    assert shtamd._stream_handle(side) == side.cuda_stream and shtamd._stream_handle(7) == 7

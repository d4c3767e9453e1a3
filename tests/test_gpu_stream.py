"""capi.stream_ptr is the current stream's handle: the default stream as None,
a side stream inside its context, and the default one again after it."""
import pytest
import torch

from taraference_amd import capi

pytestmark = pytest.mark.gpu


def test_stream_ptr_follows_the_current_stream(gpu):
    assert capi.stream_ptr() == (torch.cuda.current_stream().cuda_stream or None)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert capi.stream_ptr() == side.cuda_stream
    assert capi.stream_ptr() == (torch.cuda.current_stream().cuda_stream or None)
    assert capi.stream_ptr(side) == side.cuda_stream

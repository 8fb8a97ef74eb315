"""_lib.current_stream: the handle of torch's current stream, on every stream and in every form of the device."""
import pytest
import torch

from semi_pd_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("device", [None, 0, "cuda", "cuda:0", torch.device("cuda"), torch.device("cuda", 0)])
def test_handle_of_the_current_stream(device):
    for stream in (torch.cuda.default_stream(), torch.cuda.Stream(), torch.cuda.Stream()):
        with torch.cuda.stream(stream):
            assert _lib.current_stream(device) == torch.cuda.current_stream().cuda_stream == stream.cuda_stream
    assert _lib.current_stream(device) == torch.cuda.default_stream().cuda_stream

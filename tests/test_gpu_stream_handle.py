"""The stream handle that the bindings pass down is the current stream's, for
every way to name the device."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def test_stream_handle_is_the_current_streams(cuda):
    from circulant_attention._functions import stream_ptr
    for s in (torch.cuda.default_stream(cuda), torch.cuda.Stream(cuda)):
        with torch.cuda.stream(s):
            for d in (None, cuda, torch.device("cuda"), "cuda:0"):
                assert (stream_ptr(d).value or 0) == s.cuda_stream

"""Calls without a stream go to the current one: the handle taken without a Stream
object is the one the object has, outside and inside a stream context."""
import pytest

from astc_encoder_amd import encoder

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def test_current_stream_handle():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    torch.zeros(1, device="cuda")
    assert encoder._stream_handle(None) == torch.cuda.current_stream().cuda_stream
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert encoder._stream_handle(None) == side.cuda_stream
    assert encoder._stream_handle(side) == side.cuda_stream
    assert encoder._stream_handle(None) == torch.cuda.current_stream().cuda_stream

"""The stream handle the Python mirror passes on: the current stream of the current device."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def test_stream_handle_is_the_current_streams():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from slime_amd.ca import _stream
    assert (_stream().value or 0) == torch.cuda.current_stream().cuda_stream
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        assert _stream().value == s.cuda_stream
    assert _stream(s).value == s.cuda_stream
    assert (_stream().value or 0) == torch.cuda.current_stream().cuda_stream

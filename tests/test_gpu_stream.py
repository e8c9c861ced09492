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


@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
def test_new_parameters_reach_a_step_on_a_side_stream(dtype):
    """set_params uploads the weights (and, in bf16, lays them out on the device); a projection
    that follows at once on a stream of its own reads the new ones. It holds the result, not
    the wait that ends set_params: the blocking copies after the layout kernel, on the same
    stream, would be likely to cover for it."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import numpy as np
    from slime_amd import Pseudopod
    G, D = 32, 64
    C = 8 * D
    rng = np.random.default_rng(5)
    z = np.zeros
    ca = Pseudopod(1, G, 8, D, dtype, 0.1)
    x = torch.from_numpy(rng.random((1, G, G, C), dtype=np.float32)).to("cuda", ca.torch_dtype)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    for s in (1.0, 2.0, 0.5, 4.0):  # W = s I: V = s X exactly, for powers of two
        w = (s * np.eye(C, dtype=np.float32))[None]
        ca.set_params(dict(WP=w, WI=w, WV=w, K=z((1, 8, 9), np.float32), mu=z((1, 8), np.float32),
                           sigma=np.ones((1, 8), np.float32), M=np.eye(8, dtype=np.float32)[None]))
        with torch.cuda.stream(side):
            P, I, V = ca.project(x)
        side.synchronize()
        assert torch.equal(V, s * x)
        assert torch.equal(P, s * x)

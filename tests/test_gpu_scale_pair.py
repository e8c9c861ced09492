"""The mass factor's pair (hi, lo) is applied with one rounding: fp32 outputs of a step are the
unscaled outputs times the fp64 factor to half a unit of the last place (2^-24 relative,
and 2^-40 more for the rounding of x * lo). Adding x * lo to a rounded x * hi would lose
lo almost always, and the rounding of the ratio would bias every element alike."""
import numpy as np
import pytest

from slime_amd import Pseudopod, make_params, make_state
from slime_amd.synthetic import CAConfig

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("G,D", [(16, 64), (24, 16)])
def test_step_output_is_the_unscaled_output_times_the_factor(G, D):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    cfg = CAConfig("pair", B=3, G=G, H=8, D=D, dtype="fp32", steps=1, w_std=0.05)
    x = torch.from_numpy(make_state(cfg, seed=5)).cuda()
    with Pseudopod(cfg.B, G, 8, D, "fp32") as e:
        e.set_params(make_params(cfg, seed=4))
        hist = torch.empty((2,) + e.state_shape, device="cuda")
        hist[0] = x
        scales = e.rollout(hist)  # hist[1]: before the factor
        y = e.forward(x)
        torch.cuda.synchronize()
    s = scales[1].repeat_interleave(D, -1)[:, None, None, :]
    ref = hist[1].double() * s
    lo = (scales[1] - scales[1].float().double()).abs() / scales[1].abs()
    assert float(lo.max()) > 2.0 ** -27  # the low part matters here
    over = (y.double() - ref).abs() - ref.abs() * (2.0 ** -24 + 2.0 ** -40)
    assert float(over.max()) <= 0.0, float((over / ref.abs().clamp_min(1e-30)).max() * 2 ** 24)
    assert np.isfinite(float(y.sum()))

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


def test_matrix_core_stencil_reads_the_state_in_the_recorded_order():
    """bf16, D = 64: the stencil reads a stored state x as fma(x, lo, x * hi), the order in
    which histories of this type were made; the other order changes their bits. With dt = 0
    and one non-zero element per (batch, head, tile), a step's input sum is the sum of those
    products, two of them here, added in fp64."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    cfg = CAConfig("pair", B=32, G=8, H=8, D=64, dtype="bf16", steps=1, w_std=0.05)
    rng = np.random.default_rng(3)
    p = make_params(cfg, seed=4)
    p["M"] = np.diag(rng.uniform(0.4, 1.6, 8)).astype(np.float32)[None]
    x = np.zeros((32, 2, 32, 8, 64), np.float32)  # [B][tile][cell][head][channel]
    for b, t, h in np.ndindex(32, 2, 8):
        x[b, t, rng.integers(32), h, rng.integers(64)] = rng.uniform(0.5, 2.0)
    with Pseudopod(32, 8, 8, 64, "bf16", dt=0.0) as e:
        e.set_params(p)
        hist = torch.zeros((3,) + e.state_shape, device="cuda", dtype=torch.bfloat16)
        hist[0] = torch.from_numpy(x).view(e.state_shape).to("cuda", torch.bfloat16)
        scales = e.rollout(hist).cpu().numpy()
        mass_in = e.mass()[0]
    stored = hist[1].float().cpu().numpy().astype(np.float64).reshape(x.shape).sum((2, 4))  # [B][tile][head]
    hi = scales[1].astype(np.float32)[:, None]
    lo = (scales[1][:, None] - hi).astype(np.float32).astype(np.float64)
    # x is 8 bits, so both products are exact in fp64
    ref = ((stored * hi).astype(np.float32) + stored * lo).astype(np.float32).astype(np.float64).sum(1)
    other = (stored * hi + (stored * lo).astype(np.float32)).astype(np.float32).astype(np.float64).sum(1)
    assert (ref != other).sum() > 10  # the orders are told apart
    assert np.array_equal(mass_in, ref)

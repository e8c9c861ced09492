"""The two kinds of partial sums of the fitness at their edges: grids of one Gram unit (64
cells) and of unit counts the chunks do not divide, every head width and storage type, and
histories around the states per pass (2, 4, 8), against fp64 numpy: moments and Gram to
fp64 sums, so coherence and rank agree to their fp32 rounding (2^-24 relative) plus the
solver's own 1e-6 threshold, 1e-6 in all."""
import numpy as np
import pytest

from slime_amd import Pseudopod, round_bf16

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(autouse=True)
def _needs_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


@pytest.mark.parametrize("dtype,B,G,D,T", [
    ("bf16", 1, 8, 8, 2), ("fp32", 2, 8, 16, 3), ("fp32", 1, 8, 32, 2), ("bf16", 3, 24, 64, 2),
    ("fp32", 3, 24, 64, 5), ("bf16", 2, 40, 32, 4), ("fp32", 5, 40, 8, 9), ("bf16", 1, 56, 16, 8),
    ("fp32", 1, 136, 64, 2),
])
def test_fitness_matches_numpy(oracle, dtype, B, G, D, T):
    print(f"[case] {dtype} B={B} G={G} D={D} T={T}", flush=True)
    rng = np.random.default_rng(G + D + T)
    hist = rng.random((T, B, G, G, 8 * D), dtype=np.float32)
    for t in range(1, T):
        hist[t] = 0.6 * hist[t - 1] + 0.4 * hist[t]
    if dtype == "bf16":
        hist = round_bf16(hist)
    dev = torch.from_numpy(hist).cuda().to(torch.bfloat16 if dtype == "bf16" else torch.float32)
    with Pseudopod(B, G, 8, D, dtype) as e:
        er, coh, fit = (v.cpu().numpy() for v in e.fitness(dev))
        sweeps = e.jacobi_sweeps()
    rer, rcoh, rfit = oracle.fitness(oracle.OracleConfig(B=B, G=G, H=8, D=D), hist)
    # coherence again, independently of the oracle
    x = hist.astype(np.float64).reshape(T, B, G * G, 8, D).transpose(0, 1, 3, 2, 4).reshape(T, B * 8, -1)
    x -= x.mean(-1, keepdims=True)
    rho = [(x[t] * x[t - 1]).sum(-1) / np.sqrt((x[t] ** 2).sum(-1) * (x[t - 1] ** 2).sum(-1)) for t in range(1, T)]
    np.testing.assert_allclose(coh.ravel(), (np.mean(rho, 0) + 1) / 2, atol=1e-6)
    np.testing.assert_allclose(coh, rcoh, atol=1e-6)
    np.testing.assert_allclose(er, rer, rtol=1e-6, atol=1e-6)
    np.testing.assert_allclose(fit, rfit, rtol=1e-6, atol=1e-6)
    gram = oracle.gram(oracle.OracleConfig(B=B, G=G, H=8, D=D), hist[-1])
    want = [[oracle.jacobi_eigs(gram[b, h])[1] for h in range(8)] for b in range(B)]
    np.testing.assert_array_equal(sweeps, np.array(want))

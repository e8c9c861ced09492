"""The generic stencil's forms at the sizes where the choice between them changes: the same
cells computed with heads in parallel (one small grid) and one head after the other (a batch
of copies of that grid, past the rule's tile counts) give the same bits, output and conserved
sums, since both mix the heads in the same order; the small grid is checked against the
oracle elsewhere (test_gpu_parity)."""
import numpy as np
import pytest

from slime_amd import Pseudopod, make_params, make_state
from slime_amd.synthetic import CAConfig

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("cons", [0, 1])
@pytest.mark.parametrize("dtype,D,G,copies,per_cell", [
    ("fp32", 8, 8, 600, False), ("bf16", 8, 16, 160, True),    # 2 and 8 tiles; 1200 and 1280
    ("fp32", 16, 16, 40, True), ("bf16", 16, 24, 40, False),   # 8 and 18 tiles; 320 and 720
    ("fp32", 32, 40, 6, False), ("bf16", 32, 16, 40, True),    # 50 and 8 tiles; 300 and 320
])
def test_parallel_heads_match_serial_heads(dtype, D, G, copies, per_cell, cons):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    print(f"[case] {dtype} D={D} G={G} x{copies} per_cell={per_cell} cons={cons}", flush=True)
    cfg = CAConfig("var", B=1, G=G, H=8, D=D, dtype=dtype, steps=1, w_std=0.1, growth_per_cell=per_cell)
    p = make_params(cfg, seed=3)
    dt = torch.bfloat16 if dtype == "bf16" else torch.float32
    x = torch.from_numpy(make_state(cfg, seed=4)).cuda().to(dt)
    g = torch.Generator(device="cuda").manual_seed(5)
    P, I, V = (torch.randn(x.shape, generator=g, device="cuda").to(dt) for _ in range(3))
    outs, masses = [], []
    for B in (1, copies):
        with Pseudopod(B, G, 8, D, dtype, growth_per_cell=per_cell, conservation=cons) as e:
            e.set_params(p)
            y = e.flow_lenia(*(t.expand(B, -1, -1, -1).contiguous() for t in (x, P, I, V)))
            mi, mo = e.mass()
            outs.append(y)
            masses.append((mi, mo))
    assert torch.isfinite(outs[0].float()).all()
    assert torch.equal(outs[1], outs[0].expand_as(outs[1]))
    for one, many in zip(masses[0], masses[1]):
        # the same lanes' sums added in fp64 in another order: about ten roundings of 2^-53 of
        # the sum of magnitudes, which is below 2^9 of the sum itself
        np.testing.assert_allclose(many, np.broadcast_to(one, many.shape), rtol=2.0 ** -40)


@pytest.mark.parametrize("D,G", [(64, 16), (64, 96), (16, 16), (32, 64)])
def test_per_cell_conservation_in_the_stencil(D, G):
    """fp32: every (cell, head) of the output keeps its input's sum; cells whose output sums
    to zero (an all-zero patch) stay zero. Tolerance: the sums of D values in fp32, the
    factor and the stored products, 8 u sum|y| each way, plus the per-head factor's distance
    from 1, which the rescale applies to both sides alike."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    cfg = CAConfig("cc", B=1, G=G, H=8, D=D, dtype="fp32", steps=1, w_std=0.1)
    x = torch.from_numpy(make_state(cfg, seed=6)).cuda() + 0.1
    g = torch.Generator(device="cuda").manual_seed(7)
    P, I, V = (torch.randn(x.shape, generator=g, device="cuda") for _ in range(3))
    x[:, :6, :6] = 0  # and, one cell further in, no value flows in either
    V[:, :6, :6] = 0
    with Pseudopod(1, G, 8, D, "fp32", conservation=1) as e:
        e.set_params(make_params(cfg, seed=3))
        y = e.flow_lenia(x, P, I, V)
        torch.cuda.synchronize()
    s = lambda t: t.double().reshape(G, G, 8, D).sum(-1)  # noqa: E731
    assert torch.isfinite(y).all() and float(y[:, 1:5, 1:5].abs().max()) == 0.0
    bound = 16 * 2.0 ** -24 * (s(y.abs()) + s(x.abs())) + 1e-6
    assert float(((s(y) - s(x)).abs() - bound).max()) <= 0.0

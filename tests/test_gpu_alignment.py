"""States that start one element into their buffers, inputs and outputs of every entry point
that takes one: bit for bit what aligned tensors give, with the elements around an output
left alone. Shapes: the matrix-core stencil and the generic one, products in tiles of 256
and 64, each storage type."""
import ctypes

import numpy as np
import pytest

from slime_amd import Pseudopod, make_params, make_state
from slime_amd._lib import Grads, check
from slime_amd.synthetic import CAConfig

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

SHAPES = [("bf16", 32, 64), ("bf16", 24, 16), ("fp32", 16, 64), ("fp32", 24, 8)]


@pytest.fixture(autouse=True)
def _needs_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


class Off:
    """A tensor one element into its buffer, with a known element on either side."""

    def __init__(self, t):
        self.buf = torch.full((t.numel() + 2,), 7.0, dtype=t.dtype, device="cuda")
        self.t = self.buf[1:-1].view(t.shape)
        self.t.copy_(t)
        assert self.t.is_contiguous() and self.t.data_ptr() % 16

    def same(self, ref):
        return torch.equal(self.t, ref) and float(self.buf[0]) == 7.0 and float(self.buf[-1]) == 7.0


def _engine(dtype, G, D, B=2, **kw):
    cfg = CAConfig("a", B=B, G=G, H=8, D=D, dtype=dtype, steps=1, w_std=0.05)
    e = Pseudopod(B, G, 8, D, dtype, **kw)
    e.set_params(make_params(cfg, seed=4))
    return e, [torch.from_numpy(make_state(cfg, seed=s)).to("cuda", e.torch_dtype) for s in (5, 6)]


def _ptrs(*ts):
    return [ctypes.c_void_p(t.data_ptr()) for t in ts]


@pytest.mark.parametrize("chain", [0, 1, 2])
@pytest.mark.parametrize("dtype,G,D", SHAPES)
def test_project_and_flow(dtype, G, D, chain):
    print(f"[case] project, flow {dtype} G={G} D={D} chain={chain}", flush=True)
    e, (x, _) = _engine(dtype, G, D, pvi_chain=chain)
    with e:
        ref = e.project(x)
        y = e.flow_lenia(x, *ref)
        ox, outs = Off(x), [Off(torch.zeros_like(x)) for _ in range(3)]
        check(e.lib.slime_ca_project(e._h, *_ptrs(ox.t, *(o.t for o in outs)), None))
        oy = Off(torch.zeros_like(x))
        e.flow_lenia(ox.t, *(o.t for o in outs), out=oy.t)
        torch.cuda.synchronize()
        assert all(o.same(r) for o, r in zip(outs, ref))
        assert oy.same(y) and ox.same(x)


@pytest.mark.parametrize("dtype,G,D", SHAPES)
def test_step_and_rollout(dtype, G, D):
    print(f"[case] step, rollout {dtype} G={G} D={D}", flush=True)
    e, (x, _) = _engine(dtype, G, D)
    with e:
        for n in (0, 1, 2, 3):
            ref = e.forward(x, n_steps=n)
            ox, oy = Off(x), Off(torch.zeros_like(x))
            e.forward(ox.t, out=oy.t, n_steps=n)
            torch.cuda.synchronize()
            assert oy.same(ref) and ox.same(x), n
            e.forward(ox.t, out=ox.t, n_steps=n)  # in place
            torch.cuda.synchronize()
            assert ox.same(ref), n
        hist = torch.zeros((4,) + e.state_shape, dtype=x.dtype, device="cuda")
        hist[0] = x
        oh = Off(hist)
        scales = e.rollout(hist)
        oscales = e.rollout(oh.t)
        torch.cuda.synchronize()
        assert oh.same(hist) and torch.equal(scales, oscales)


@pytest.mark.parametrize("dtype,G,D", SHAPES)
def test_backward(dtype, G, D):
    print(f"[case] backward {dtype} G={G} D={D}", flush=True)
    e, (x, target) = _engine(dtype, G, D)
    with e:
        loss, gx, grads = e.backward(x, target)
        ox, ot, og = Off(x), Off(target), Off(torch.zeros_like(gx))
        got = {k: torch.empty_like(v) for k, v in grads.items()}
        gs = Grads(*[got[k].data_ptr() for k in ("WP", "WI", "WV", "K", "mu", "sigma", "M")])
        oloss = ctypes.c_double()
        check(e.lib.slime_ca_backward(e._h, *_ptrs(ox.t, ot.t, og.t), ctypes.byref(gs), ctypes.byref(oloss), None))
        torch.cuda.synchronize()
        assert oloss.value == loss and og.same(gx)
        for k, v in grads.items():
            assert torch.equal(got[k], v), k


@pytest.mark.parametrize("dtype,G,D", SHAPES)
def test_organism(dtype, G, D):
    print(f"[case] organism {dtype} G={G} D={D}", flush=True)
    e, _ = _engine(dtype, G, D, B=1)
    conc = torch.from_numpy(np.random.default_rng(2).random((G, G), np.float32)).cuda()
    zero = torch.zeros((G, G, 8 * D), dtype=e.torch_dtype, device="cuda")
    with e:
        res = []
        for a, b in ((zero.clone(), zero.clone()), (Off(zero), Off(zero))):
            field, erank, mass = conc.clone(), torch.zeros(2, device="cuda"), torch.zeros(8, device="cuda")
            e.neural_ca_update(field, *(t.t if isinstance(t, Off) else t for t in (a, b)), erank, 1, mass_buffer=mass)
            torch.cuda.synchronize()
            res.append((field, erank, mass, a, b))
        (f0, r0, m0, a0, b0), (f1, r1, m1, a1, b1) = res
        assert a1.same(a0) and b1.same(b0)
        assert torch.equal(f0, f1) and torch.equal(r0, r1) and torch.equal(m0, m1)
